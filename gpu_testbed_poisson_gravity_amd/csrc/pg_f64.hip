// FP64 entry of the solver (the reference's FLOAT8 build, Makefile:22, Header/Macro.h:35) and the standalone FP64
// gravity update (CPU_GravitySolver.cpp:34-79).  The SOR kernel is in pg_sor_blocks.hip, the MG kernel in pg_mg.hip.

#include <hip/hip_runtime.h>

#include "pg_geometry.h"
#include "pg_kernels.h"

#pragma clang fp contract(off)

namespace pgamd {
namespace {

constexpr int kT64 = 256;

// Standalone FP64 gravity update from an output window in HBM (the Poisson = false path).
__global__ void __launch_bounds__(kT64) gravity64_kernel(const double* __restrict__ pot, double* __restrict__ flu,
                                                         int npatch, int gg, double gra_const, int p5) {
  const int P = blockIdx.x;
  if (P >= npatch) return;
  const int G = gra_nxt(gg);
  const double* pp = pot + (size_t)P * G * G * G;
  double* f = flu + (size_t)P * kNComp * kPatchCells;
  for (int t = threadIdx.x; t < kPatchCells; t += kT64) {
    const int i = t % kPatchSize, j = (t / kPatchSize) % kPatchSize, k = t / (kPatchSize * kPatchSize);
    const int x = i + gg, y = j + gg, z = k + gg;
    auto Q = [&](int dz, int dy, int dx) { return pp[((z + dz) * G + (y + dy)) * G + (x + dx)]; };
    double ax, ay, az;
    if (p5) {
      ax = gra_const * (-Q(0, 0, 2) + Q(0, 0, -2) + 8.0 * Q(0, 0, 1) - 8.0 * Q(0, 0, -1));
      ay = gra_const * (-Q(0, 2, 0) + Q(0, -2, 0) + 8.0 * Q(0, 1, 0) - 8.0 * Q(0, -1, 0));
      az = gra_const * (-Q(2, 0, 0) + Q(-2, 0, 0) + 8.0 * Q(1, 0, 0) - 8.0 * Q(-1, 0, 0));
    } else {
      ax = gra_const * (Q(0, 0, 1) - Q(0, 0, -1));
      ay = gra_const * (Q(0, 1, 0) - Q(0, -1, 0));
      az = gra_const * (Q(1, 0, 0) - Q(-1, 0, 0));
    }
    const double rho = f[t];
    double px = f[kPatchCells + t], py = f[2 * kPatchCells + t], pz = f[3 * kPatchCells + t];
    const double temp = 0.5 / rho;
    const double eint = f[4 * kPatchCells + t] - temp * (px * px + py * py + pz * pz);
    px = px - rho * ax;
    py = py - rho * ay;
    pz = pz - rho * az;
    f[kPatchCells + t] = px;
    f[2 * kPatchCells + t] = py;
    f[3 * kPatchCells + t] = pz;
    f[4 * kPatchCells + t] = eint + temp * (px * px + py * py + pz * pz);
  }
}

}  // namespace

hipError_t launch_uniform64(const UniformBatch64& b, const SolveParams64& p, hipStream_t s) {
  if (b.npatch <= 0) return hipSuccess;
  if (b.scheme == kSchemeMG) return launch_mg_uniform64(b, p, s);
  return launch_sor_blocks64(b, p, s);
}

hipError_t launch_gravity64(const double* pot, double* flu, int npatch, int gra_ghost, double gra_const, int p5,
                            hipStream_t stream) {
  if (npatch <= 0) return hipSuccess;
  hipLaunchKernelGGL(gravity64_kernel, dim3(npatch), dim3(kT64), 0, stream, pot, flu, npatch, gra_ghost, gra_const,
                     p5);
  return hipGetLastError();
}

}  // namespace pgamd
