// Coarse-to-fine potential interpolation of one coarse cell, and the enumeration of a solve cube's Dirichlet
// layer (device code shared by the SOR, MG and network kernels).  Restates CPU_PoissonSolver_SOR.cpp:110-203 with the reference's operation order, for the FP32
// kernels and the FP64 ones (the reference's FLOAT8 build).
#pragma once

#include <hip/hip_runtime.h>

#include "pg_geometry.h"

#pragma clang fp contract(off)

namespace pgamd {

// One coarse cell's 8 children: CQUAD (13 signed slopes summed in slope order, then + parent) or QUAD
// (27-point tensor product of the weights {5,30,-3}/32 and {-3,30,5}/32).  Same operation order as the
// reference so that results are identical in either precision (every constant is exact in both).
template <typename T>
__device__ __forceinline__ void interp_children(const T (&v)[3][3][3], int int_scheme, T (&ch)[2][2][2]) {
  if (int_scheme == kIntCQuad) {
    const T c8 = T(0.125), c64 = T(0.015625), c512 = T(0.001953125);
    T S[13];
    S[0] = c8 * (v[1][1][2] - v[1][1][0]);
    S[1] = c8 * (v[1][2][1] - v[1][0][1]);
    S[2] = c8 * (v[2][1][1] - v[0][1][1]);
    S[3] = c64 * (v[0][1][2] - v[0][1][0]);
    S[4] = c64 * (v[0][2][1] - v[0][0][1]);
    S[5] = c64 * (v[1][0][2] - v[1][0][0]);
    S[6] = c64 * (v[1][2][2] - v[1][2][0]);
    S[7] = c64 * (v[2][1][2] - v[2][1][0]);
    S[8] = c64 * (v[2][2][1] - v[2][0][1]);
    S[9] = c512 * (v[0][0][2] - v[0][0][0]);
    S[10] = c512 * (v[0][2][2] - v[0][2][0]);
    S[11] = c512 * (v[2][0][2] - v[2][0][0]);
    S[12] = c512 * (v[2][2][2] - v[2][2][0]);
#pragma unroll
    for (int cz = 0; cz < 2; cz++)
#pragma unroll
      for (int cy = 0; cy < 2; cy++)
#pragma unroll
        for (int cx = 0; cx < 2; cx++) {
          const int sx = cx ? 1 : -1, sy = cy ? 1 : -1, sz = cz ? 1 : -1;
          const int sg[13] = {sx,      sy,      sz,           -sx * sz,      -sy * sz,      -sx * sy,    sx * sy,
                              sx * sz, sy * sz, sx * sy * sz, -sx * sy * sz, -sx * sy * sz, sx * sy * sz};
          T a = sg[0] > 0 ? S[0] : -S[0];
#pragma unroll
          for (int q = 1; q < 13; q++) a = sg[q] > 0 ? a + S[q] : a - S[q];
          ch[cz][cy][cx] = a + v[1][1][1];
        }
  } else {
    const T Mp[3] = {T(-0.09375), T(0.9375), T(0.15625)};
    const T Mm[3] = {T(0.15625), T(0.9375), T(-0.09375)};
#pragma unroll
    for (int cz = 0; cz < 2; cz++)
#pragma unroll
      for (int cy = 0; cy < 2; cy++)
#pragma unroll
        for (int cx = 0; cx < 2; cx++) {
          T a = T(0);
#pragma unroll
          for (int dk = 0; dk < 3; dk++)
#pragma unroll
            for (int dj = 0; dj < 3; dj++)
#pragma unroll
              for (int di = 0; di < 3; di++) {
                const T wz = cz ? Mp[dk] : Mm[dk];
                const T wy = cy ? Mp[dj] : Mm[dj];
                const T wx = cx ? Mp[di] : Mm[di];
                a = a + v[dk][dj][di] * wz * wy * wx;
              }
          ch[cz][cy][cx] = a;
        }
  }
}

// The same operations child by child, arranged for few registers: at(dk, dj, di) is the value at that offset (0..2) of the
// 3^3 neighbourhood, and the eight sums advance together, a slope (or neighbour) at a time, so that little besides them is
// live.  FENCE: keeps the compiler from loading the whole neighbourhood first.  The kernels that keep their cells in
// registers during the interpolation use this form (FP64 block SOR, ghost size 5: 300 bytes of spills per lane with the
// form above, none with this one); the compact one-wavefront SOR kernel allocates its 256 registers better with the form
// above (1.00 against 1.22 ms for 16384 patches).
template <bool FENCE, typename T, class At>
__device__ __forceinline__ void interp_children_at(At at, int int_scheme, T (&ch)[2][2][2]) {
  auto fence = [](int q) {
    if (FENCE && q % 4 == 3) __builtin_amdgcn_sched_barrier(0);
  };
  if (int_scheme == kIntCQuad) {
    // slope q: scale, and the offsets of its two values; its sign in child (cz, cy, cx) is the product of the signs of the
    // axes in `ax` (bit 0 x, 1 y, 2 z), negated where `neg`
    constexpr struct {
      float scale;
      int p[3], m[3], ax;
      bool neg;
    } S[13] = {{0.125f, {1, 1, 2}, {1, 1, 0}, 1, false},       {0.125f, {1, 2, 1}, {1, 0, 1}, 2, false},
               {0.125f, {2, 1, 1}, {0, 1, 1}, 4, false},       {0.015625f, {0, 1, 2}, {0, 1, 0}, 5, true},
               {0.015625f, {0, 2, 1}, {0, 0, 1}, 6, true},     {0.015625f, {1, 0, 2}, {1, 0, 0}, 3, true},
               {0.015625f, {1, 2, 2}, {1, 2, 0}, 3, false},    {0.015625f, {2, 1, 2}, {2, 1, 0}, 5, false},
               {0.015625f, {2, 2, 1}, {2, 0, 1}, 6, false},    {0.001953125f, {0, 0, 2}, {0, 0, 0}, 7, false},
               {0.001953125f, {0, 2, 2}, {0, 2, 0}, 7, true},  {0.001953125f, {2, 0, 2}, {2, 0, 0}, 7, true},
               {0.001953125f, {2, 2, 2}, {2, 2, 0}, 7, false}};
#pragma unroll
    for (int q = 0; q < 13; q++) {
      const T s = T(S[q].scale) * (at(S[q].p[0], S[q].p[1], S[q].p[2]) - at(S[q].m[0], S[q].m[1], S[q].m[2]));
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const int minus = ((S[q].ax & 1) && !(e & 1)) + ((S[q].ax & 2) && !(e & 2)) + ((S[q].ax & 4) && !(e & 4)) + S[q].neg;
        T& a = ch[e >> 2][(e >> 1) & 1][e & 1];
        if (q == 0)
          a = minus & 1 ? -s : s;
        else
          a = minus & 1 ? a - s : a + s;
      }
      fence(q);
    }
    const T parent = at(1, 1, 1);
#pragma unroll
    for (int e = 0; e < 8; e++) ch[e >> 2][(e >> 1) & 1][e & 1] = ch[e >> 2][(e >> 1) & 1][e & 1] + parent;
  } else {
    const T Mp[3] = {T(-0.09375), T(0.9375), T(0.15625)};
    const T Mm[3] = {T(0.15625), T(0.9375), T(-0.09375)};
#pragma unroll
    for (int e = 0; e < 8; e++) ch[e >> 2][(e >> 1) & 1][e & 1] = T(0);
#pragma unroll
    for (int q = 0; q < 27; q++) {
      const int dk = q / 9, dj = q / 3 % 3, di = q % 3;
      const T v = at(dk, dj, di);
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const T wz = e & 4 ? Mp[dk] : Mm[dk];
        const T wy = e & 2 ? Mp[dj] : Mm[dj];
        const T wx = e & 1 ? Mp[di] : Mm[di];
        T& a = ch[e >> 2][(e >> 1) & 1][e & 1];
        a = a + v * wz * wy * wx;
      }
      fence(q);
    }
  }
}

// Coarse cell q (1-based i, j, k of the NC^3 block that has children in the cube) of the interpolation
// loop: every cell, or (SHELL) only the 2 NC^2 + 4 (NC-1)(NC-2) cells on the outer layer of the block, whose
// children include every cell of the cube's Dirichlet layer (the only cells a zero start or a caller's guess
// leaves to the interpolation).
template <int NC, bool SHELL>
__device__ __forceinline__ void coarse_cell(int q, int& i, int& j, int& k) {
  if (!SHELL) {
    i = q % NC + 1;
    j = (q / NC) % NC + 1;
    k = q / (NC * NC) + 1;
    return;
  }
  constexpr int F = NC * NC, RING = 4 * (NC - 1);
  if (q < 2 * F) {   // the bottom and top faces
    const int t = q % F;
    k = q < F ? 1 : NC;
    i = t % NC + 1;
    j = t / NC + 1;
    return;
  }
  const int r = q - 2 * F, t = r % RING;   // the ring of each layer in between
  k = r / RING + 2;
  if (t < 2 * NC) {
    j = t < NC ? 1 : NC;
    i = t % NC + 1;
  } else {
    const int u = t - 2 * NC;
    i = u < NC - 2 ? 1 : NC;
    j = u % (NC - 2) + 2;
  }
}

// Cell q of the outer layer of an N^3 cube (faces z = 0 and N-1, then the ring of each layer in between).
template <int N>
__device__ __forceinline__ void shell_cell(int q, int& x, int& y, int& z) {
  constexpr int F = N * N, RING = 4 * (N - 1);
  if (q < 2 * F) {
    z = q < F ? 0 : N - 1;
    const int t = q % F;
    x = t % N;
    y = t / N;
    return;
  }
  const int r = q - 2 * F, t = r % RING;
  z = r / RING + 1;
  if (t < 2 * N) {
    y = t < N ? 0 : N - 1;
    x = t % N;
  } else {
    const int u = t - 2 * N;
    x = u < N - 2 ? 0 : N - 1;
    y = u % (N - 2) + 1;
  }
}

}  // namespace pgamd
