// Red-black SOR with several wavefronts per patch on gfx950: every FP64 solve (the reference's FLOAT8 build, Makefile:22,
// Header/Macro.h:35), and the FP32 batches for which it is faster than one wavefront per patch (pg_sor.hip): all at ghost
// sizes 1 to 3, where that kernel leaves lanes idle, and those too small to fill the GPU with it (sor_blocks_limit).
//
// Reference behaviour reproduced (bit for bit at equal iteration counts):
//   interpolation  CPU_PoissonSolver_SOR.cpp:110-203
//   SOR sweep      CPU_PoissonSolver_SOR.cpp:215-270
//   stall rule     CPU_PoissonSolver_SOR.cpp:273-283
//   window         CPU_PoissonSolver_SOR.cpp:303-311
//   gravity        CPU_GravitySolver.cpp:34-79
//
// Work split.  A thread owns a 2x2 block of z-columns (x in {2m+1, 2m+2}, y in {2yb+1, 2yb+2}) over H planes and keeps
// its cells' phi and Const*rho in registers: 16 cells and 64 registers in FP64 at ghost size 5, which leaves room for
// three waves per SIMD.  H is even, so that which of a block's cells has which colour does not depend on the thread.
//
// Layout.  The cube in LDS, split by colour c = (x+y+z)&1: word c*CS + z*PL + y*HP + (x>>1).  Every neighbour of an
// owned cell sits at a compile-time offset from one lane register (the cell across the x pair even at the cell's own word,
// in the other colour), the Dirichlet layer included.  A cell update costs two LDS reads (across the x pair and the y
// pair), one more at the ends of a chunk of planes, and one write.  HP and PL were chosen for the fewest bank conflicts of
// 32 lanes per cycle (FP32) or 16 (FP64): none at ghost sizes 1 and 5.  (Tried: HP from N/2 to N/2 + 3, PL from N HP to N HP +
// 16, both lane orders; counted: over the groups of lanes that share a cycle, the most different words on one bank among the
// lanes' own words, which every other access is a constant away from.)
// FP64 at ghost size 5 keeps a column's cells of one colour together instead, so that the two cells of a thread's column
// are one 16-byte read or write (BlockGeo::PAIRS): 64 lanes in 4 cycles, as an 8-byte read.  It was bound by the LDS (70%
// busy, VALU 64%); now the LDS is busy for half of the time and the VALU for 62%, and what is left is their latency with
// three patches (12 waves) per CU.  MI355X, 4096 patches to a relative residual of 1e-10: 1148 -> 1055 us (1004 with wave
// sums for the stopping test); with 10 words per column and rows shifted in turn (writes with two-way conflicts) 1113 us.
//
// The one-wavefront kernel decides where to stop on FP32 sums in its own order.  The FP32 form here must stop at the same
// iteration: it compares sums reduced as a tree over the workgroup, and where the two sides are within 2e-5 of each other
// (five times the rounding either order can leave) it forms the sums again in the other kernel's order, unless no order can
// change the answer: a NaN (sums of absolute values have one in every order or in none; the comparison is then false), or
// residuals that repeat those of the last iteration.  A patch of zeros or with a NaN in it runs to the last iteration under
// the stall rule and would otherwise form them every time: 256 GS-5 patches, 1000 iterations, one patch of zeros 5.14 -> 1.09 ms
// (one-wavefront kernel 2.14), one with a NaN 5.14 -> 0.88 ms (2.14).

#include <hip/hip_runtime.h>

#include <cfloat>
#include <climits>

#include "pg_geometry.h"
#include "pg_interp.h"
#include "pg_kernels.h"
#include "pg_reduce.h"

#pragma clang fp contract(off)

namespace pgamd {
namespace {

// HELP: workgroup of HELP times the waves that own cells; the others only share the work before and after the iterations.
template <int GS, typename T, int PLANES, int HELP = 1>
struct BlockGeo {
  static constexpr Geo g = geo_of(GS);
  static constexpr int N = g.N, R = g.R, C = g.C, U = g.U;
  static constexpr int MX = R / 2, LP = MX * MX;          // blocks per row / per plane
  static constexpr int H = PLANES;                        // planes per thread
  static constexpr int CHUNKS = R / H;
  static constexpr int OWNERS = LP * CHUNKS;
  static constexpr int THREADS = (OWNERS + 63) / 64 * 64 * HELP;
  static constexpr int FACES = HELP > 1 ? OWNERS : 0;     // first thread with a face's coarse cell (interpolation)
  static constexpr int EDGES = HELP > 1 ? FACES + 6 * LP : 0;
  static_assert(HELP == 1 || (OWNERS == 64 && EDGES + 12 * MX + 8 <= THREADS), "one wave of owners, one item per helper");
  static constexpr bool F64 = sizeof(T) == 8;
  static constexpr int HP = N / 2 + (GS == 1 || GS == 4 || (GS == 5 && !F64) ? 1 : 0);
  static constexpr int PL = N * HP + (GS == 1 && !F64 ? 12 : GS == 2 ? (F64 ? 3 : 1) : GS == 4 && F64 ? 2 : 0);
  // One order of the stopping sums for both plane counts of FP64 ghost size 3, which the batch size chooses between: with two
  // planes per thread, consecutive threads have the two halves of a four-plane chunk; with four, a thread adds its halves
  // apart.  The sums over the threads are binary trees, so the rest of the order is the same.
  static constexpr bool ONE_ORDER = F64 && GS == 3;
  static constexpr int PARTS = ONE_ORDER && PLANES == 4 ? 2 : 1;   // sums per thread
  __device__ static constexpr int part(int zi) { return PARTS == 2 ? zi >> 1 : 0; }
  // Pairs: a column's interior cells of one colour lie together, so that a thread's two are one 16-byte word; x pairs of
  // columns are XP words apart (their two Dirichlet cells last), rows RP.  A 16-byte read serves lanes 0-3, 12-15 and 20-27 of
  // 32 in a cycle, then the others; a write 8 lanes of 32 banks: XP is 2 modulo 16 and RP 8 modulo 16, without conflicts.
  static constexpr bool PAIRS = F64 && GS == 5 && PLANES == 4;
  static constexpr int XP = R + 2, RP = (N / 2 * XP + 7) / 16 * 16 + 8;
  static_assert(!PAIRS || (XP % 16 == 2 && RP >= N / 2 * XP), "bank-free");
  static constexpr bool XMAJOR = GS >= 3 && !PAIRS;       // lane order within a plane: x blocks slow
  static constexpr int CS = PAIRS ? N * RP : N * PL;      // words per colour
  static constexpr int NC = C - 2;                        // coarse cells with children in the cube, per axis
  static constexpr int WAVES = THREADS / 64 / HELP;       // with cells
  static constexpr int RED = 2 * CS;                      // two pairs of wave sums
  static constexpr int SCRATCH = RED + 4 * WAVES;         // FP32: 2H values per column (ordered sums), one result
  static constexpr int WORDS = SCRATCH + (F64 ? 0 : 2 * H * 64 + 1);
  static_assert(C * C * C <= 2 * CS, "the coarse potential fits where the cube goes");
  // cube cell on two or three faces
  __device__ static bool edge(int x, int y, int z) {
    return (x == 0 || x == N - 1) + (y == 0 || y == N - 1) + (z == 0 || z == N - 1) > 1;
  }
  __device__ static int column(int x, int y) { return y * RP + (x >> 1) * XP + (x & 1) * (R / 2); }
  __device__ static int word(int x, int y, int z) {
    const int c = ((x + y + z) & 1) * CS;
    if (PAIRS) return z == 0 || z == N - 1 ? c + y * RP + (x >> 1) * XP + R + (x & 1) : c + column(x, y) + ((z - 1) >> 1);
    return c + z * PL + y * HP + (x >> 1);
  }
};

// A thread's cells.
template <int GS, typename T, int PLANES, int HELP = 1>
struct Block {
  using G = BlockGeo<GS, T, PLANES, HELP>;
  static constexpr int H = G::H;
  T phi[2][2][H], cr[2][2][H];   // [yy][xx][zi]; cr = Const*rho
  int x0, y0, z0;                // cube coordinates of the first cell, all odd
  static constexpr int kX1 = G::XP - G::R / 2;   // pairs: words from the first column of a block to the second
  int own;                       // word of (x0, y0, z0) without its colour
  int below[2], above[2];        // pairs: offsets of the words below and above the chunk in a column
  int chunk, column;             // chunk of planes; lane of the column in the one-wavefront kernel
  bool active;

  __device__ __forceinline__ void init(int t) {
    active = t < G::OWNERS;
    if (!active) t = 0;   // reads stay in range; nothing is written
    const bool halves = G::ONE_ORDER && H == 2;
    const int u = halves ? t >> 1 : t;
    chunk = u / G::LP;
    const int cb = u - chunk * G::LP, a = cb / G::MX, b = cb - a * G::MX;
    if (halves) chunk = 2 * chunk + (t & 1);
    const int m = G::XMAJOR ? a : b, yb = G::XMAJOR ? b : a;
    x0 = 2 * m + 1;
    y0 = 2 * yb + 1;
    z0 = chunk * H + 1;
    if (G::PAIRS) {
      static_assert(!G::PAIRS || (H == 4 && G::OWNERS == G::THREADS), "two cells of each colour per column");
      own = G::column(x0, y0) + 2 * chunk;
#pragma unroll
      for (int xx = 0; xx < 2; xx++) {
        const int end = xx ? G::R : G::R / 2 + 1;   // the column's Dirichlet cell
        below[xx] = chunk ? -1 : end;
        above[xx] = chunk < G::CHUNKS - 1 ? 2 : end - 2 * chunk;
      }
    } else {
      own = z0 * G::PL + y0 * G::HP + m;
    }
    column = GS >= 4 ? m * G::MX + yb : yb * G::MX + m;
  }
  static constexpr int xx_of(int c, int yy, int zi) { return (c + yy + zi + 1) & 1; }
  __device__ __forceinline__ int word(int c, int yy, int xx, int zi) const {
    if (G::PAIRS) return own + c * G::CS + yy * G::RP + xx * kX1 + (zi >> 1);
    return own + c * G::CS + zi * G::PL + yy * G::HP + xx;
  }
  // Residual of the cell of colour c at (yy, zi), reference operand order (CPU_PoissonSolver_SOR.cpp:247-250).
  template <int c, int yy, int zi>
  __device__ __forceinline__ T residual(const T* __restrict__ lds) const {
    constexpr int xx = xx_of(c, yy, zi);
    const int o = word(1 - c, yy, xx, zi);
    const T kp = zi + 1 < H ? phi[yy][xx][zi + 1 < H ? zi + 1 : 0] : lds[o + G::PL];
    const T km = zi > 0 ? phi[yy][xx][zi > 0 ? zi - 1 : 0] : lds[o - G::PL];
    const T jo = lds[yy == 0 ? o - G::HP : o + G::HP], io = lds[o];
    const T jp = yy == 0 ? phi[1][xx][zi] : jo, jm = yy == 1 ? phi[0][xx][zi] : jo;
    const T ip = xx == 0 ? phi[yy][1][zi] : io, im = xx == 1 ? phi[yy][0][zi] : io;
    return kp + km + jp + jm + ip + im - T(6) * phi[yy][xx][zi] - cr[yy][xx][zi];
  }
  // Pairs: residuals of colour c in column (yy, xx), r[2 zi + yy].
  template <int c, int yy, int xx>
  __device__ __forceinline__ void column_residuals(const T* __restrict__ lds, T (&r)[2 * H]) const {
    constexpr int zs = (c + 1 + yy + xx) & 1, b = (1 - c) * G::CS;
    const int o = own + b + yy * G::RP + xx * kX1;
    struct alignas(16) Two { T v[2]; };
    const Two io = *reinterpret_cast<const Two*>(lds + o + (xx ? G::R / 2 : -G::R / 2));
    const Two jo = *reinterpret_cast<const Two*>(lds + o + (yy ? G::RP : -G::RP));
    const T end = lds[o + (zs ? above[xx] : below[xx])];
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int zi = zs + 2 * u;
      const T kp = zi + 1 < H ? phi[yy][xx][zi + 1 < H ? zi + 1 : 0] : end;
      const T km = zi > 0 ? phi[yy][xx][zi > 0 ? zi - 1 : 0] : end;
      const T jp = yy == 0 ? phi[1][xx][zi] : jo.v[u], jm = yy == 1 ? phi[0][xx][zi] : jo.v[u];
      const T ip = xx == 0 ? phi[yy][1][zi] : io.v[u], im = xx == 1 ? phi[yy][0][zi] : io.v[u];
      r[2 * zi + yy] = kp + km + jp + jm + ip + im - T(6) * phi[yy][xx][zi] - cr[yy][xx][zi];
    }
  }
  // f(q, yy, xx, zi, residual) for every cell of colour c, q = 2 zi + yy
  template <int c, int q = 0, class F>
  __device__ __forceinline__ void each(const T* __restrict__ lds, F f) const {
    if constexpr (G::PAIRS) {
      T r[2 * H];
      column_residuals<c, 0, 0>(lds, r);
      column_residuals<c, 0, 1>(lds, r);
      column_residuals<c, 1, 0>(lds, r);
      column_residuals<c, 1, 1>(lds, r);
#pragma unroll
      for (int i = 0; i < 2 * H; i++) f(i, i & 1, xx_of(c, i & 1, i >> 1), i >> 1, r[i]);
    } else if constexpr (q < 2 * H) {
      const T r = residual<c, (q & 1), (q >> 1)>(lds);
      f(q, q & 1, xx_of(c, q & 1, q >> 1), q >> 1, r);
      each<c, q + 1>(lds, f);
    }
  }
  template <int c>
  __device__ __forceinline__ void publish(T* __restrict__ lds) const {
    if (G::PAIRS) {   // every thread owns a block
      struct alignas(16) Two { T v[2]; };
#pragma unroll
      for (int yy = 0; yy < 2; yy++)
#pragma unroll
        for (int xx = 0; xx < 2; xx++) {
          const int zs = (c + 1 + yy + xx) & 1;
          *reinterpret_cast<Two*>(lds + word(c, yy, xx, 0)) = Two{{phi[yy][xx][zs], phi[yy][xx][zs + 2 < H ? zs + 2 : 0]}};
        }
    } else if (active) {
#pragma unroll
      for (int zi = 0; zi < H; zi++)
#pragma unroll
        for (int yy = 0; yy < 2; yy++) lds[word(c, yy, xx_of(c, yy, zi), zi)] = phi[yy][xx_of(c, yy, zi)][zi];
    }
  }
  template <class F>
  __device__ __forceinline__ void cells(F f) {
#pragma unroll
    for (int yy = 0; yy < 2; yy++)
#pragma unroll
      for (int xx = 0; xx < 2; xx++)
#pragma unroll
        for (int zi = 0; zi < H; zi++) f(yy, xx, zi);
  }
};

// Coarse potential into LDS, where the cube will go.
template <class G, typename T>
__device__ __forceinline__ void blocks_stage(T* __restrict__ lds, const T* __restrict__ cpot, int t) {
  constexpr int C3 = G::C * G::C * G::C, SI = (C3 + G::THREADS - 1) / G::THREADS;
  T v[SI];
#pragma unroll
  for (int u = 0; u < SI; u++) v[u] = t + u * G::THREADS < C3 ? cpot[t + u * G::THREADS] : T(0);
#pragma unroll
  for (int u = 0; u < SI; u++)
    if (t + u * G::THREADS < C3) lds[t + u * G::THREADS] = v[u];
}

// Children of staged coarse cell (i, j, k).
template <int C, typename T>
__device__ __forceinline__ void blocks_children(const T* __restrict__ stage, int i, int j, int k, int int_scheme, T (&ch)[2][2][2]) {
  const T* c = stage + ((k - 1) * C + j - 1) * C + i - 1;
  interp_children_at<sizeof(T) == 8>([&](int dk, int dj, int di) { return c[(dk * C + dj) * C + di]; }, int_scheme, ch);
}

// Interpolated cube into LDS, even ghost sizes: children of every coarse cell (SHELL: of those that reach the Dirichlet
// layer) in registers until the staged coarse potential has been read.
template <class G, bool SHELL, typename T>
__device__ __forceinline__ void blocks_interpolate_even(T* __restrict__ lds, int int_scheme, int t) {
  constexpr int NC = G::NC, N = G::N;
  constexpr int CELLS = SHELL ? 2 * NC * NC + 4 * (NC - 1) * (NC - 2) : NC * NC * NC;
  constexpr int ITEMS = (CELLS + G::THREADS - 1) / G::THREADS;
  static_assert(G::U == 0 && ITEMS <= 2, "aligned with the coarse cells");
  T ch[ITEMS][2][2][2];
#pragma unroll
  for (int u = 0; u < ITEMS; u++) {
    const int q = t + u * G::THREADS;
    if (q < CELLS) {
      int i, j, k;
      coarse_cell<NC, SHELL>(q, i, j, k);
      blocks_children<G::C>(lds, i, j, k, int_scheme, ch[u]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < ITEMS; u++) {
    const int q = t + u * G::THREADS;
    if (q < CELLS) {
      int i, j, k;
      coarse_cell<NC, SHELL>(q, i, j, k);
#pragma unroll
      for (int e = 0; e < 8; e++)
        lds[G::word(2 * (i - 1) + (e & 1), 2 * (j - 1) + ((e >> 1) & 1), 2 * (k - 1) + (e >> 2))] = ch[u][e >> 2][(e >> 1) & 1][e & 1];
    }
  }
}

// Odd ghost sizes: a thread's block is whole coarse cells, whose children go straight to its registers (interior: with
// the interpolated start); the faces' coarse cells are shared out and their children written once the staged coarse
// potential has been read.  The cube's edges and corners, which no stencil reads, go straight to a window that has them.
template <int GS, typename T, int PLANES, int HELP>
__device__ __forceinline__ void blocks_interpolate_odd(Block<GS, T, PLANES, HELP>& o, T* __restrict__ lds, T* __restrict__ out, bool interior,
                                                       bool whole, int int_scheme, int t) {
  using G = BlockGeo<GS, T, PLANES, HELP>;
  constexpr int NC = G::NC, N = G::N, C = G::C, MX = G::MX, LP = G::LP, FI = (6 * LP + G::THREADS - 1) / G::THREADS;
  // helpers take the faces and the edges while the owners are at their blocks
  auto face_item = [&](int u) { return (unsigned)(t - G::FACES + u * G::THREADS); };
  static_assert(G::U == 1 && NC == MX + 2, "blocks are coarse cells");
  if (interior && (HELP == 1 || o.active)) {
#pragma unroll
    for (int kk = 0; kk < G::H / 2; kk++) {
      T ch[2][2][2];
      blocks_children<C>(lds, (o.x0 + 3) >> 1, (o.y0 + 3) >> 1, ((o.z0 + 3) >> 1) + kk, int_scheme, ch);
#pragma unroll
      for (int e = 0; e < 8; e++) o.phi[(e >> 1) & 1][e & 1][2 * kk + (e >> 2)] = ch[e >> 2][(e >> 1) & 1][e & 1];
    }
  }
  T face[FI][4];
#pragma unroll
  for (int u = 0; u < FI; u++) {
    const int q = face_item(u), f = q / LP, r = q - f * LP, b = r / MX, a = r - b * MX, ax = f >> 1, end = f & 1 ? NC : 1;
    if ((unsigned)q < 6 * LP) {
      T ch[2][2][2];
      blocks_children<C>(lds, ax == 0 ? end : a + 2, ax == 0 ? a + 2 : ax == 1 ? end : b + 2, ax == 2 ? end : b + 2, int_scheme, ch);
      const int s = 1 - (f & 1);   // the child on the Dirichlet layer
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int c1 = e & 1, c2 = e >> 1;
        const T vx = s ? ch[c2][c1][1] : ch[c2][c1][0], vy = s ? ch[c2][1][c1] : ch[c2][0][c1],
                vz = s ? ch[1][c2][c1] : ch[0][c2][c1];
        face[u][e] = ax == 0 ? vx : ax == 1 ? vy : vz;
      }
    }
  }
  if (whole) {
    for (int q = t >= G::EDGES ? t - G::EDGES : t + G::THREADS; q < 12 * MX + 8; q += G::THREADS) {
      const int ed = q / MX, ax = q < 12 * MX ? ed >> 2 : 3, bits = q < 12 * MX ? ed & 3 : q - 12 * MX, a = q - ed * MX + 2;
      const int e0 = bits & 1 ? NC : 1, e1 = bits & 2 ? NC : 1, e2 = bits & 4 ? NC : 1;
      const int i = ax == 0 ? a : e0, j = ax == 1 ? a : ax == 0 ? e0 : e1, k = ax == 2 ? a : ax == 3 ? e2 : e1;
      T ch[2][2][2];
      blocks_children<C>(lds, i, j, k, int_scheme, ch);
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const int x = 2 * i - 3 + (e & 1), y = 2 * j - 3 + ((e >> 1) & 1), z = 2 * k - 3 + (e >> 2);
        const bool in = x >= 0 && x < N && y >= 0 && y < N && z >= 0 && z < N;
        if (in && G::edge(x, y, z)) out[(z * N + y) * N + x] = ch[e >> 2][(e >> 1) & 1][e & 1];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < FI; u++) {
    const int q = face_item(u), f = q / LP, r = q - f * LP, b = r / MX, a = r - b * MX, d = f & 1 ? N - 1 : 0;
    if ((unsigned)q < 6 * LP) {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int p = 2 * a + 1 + (e & 1), w = 2 * b + 1 + (e >> 1);
        lds[f < 2 ? G::word(d, p, w) : f < 4 ? G::word(p, d, w) : G::word(p, w, d)] = face[u][e];
      }
    }
  }
}

// Sum of the waves' values (one wave: each lane has it).
template <int WAVES, typename T>
__device__ __forceinline__ void blocks_put(T wave, T* red) {
  if (WAVES > 1 && (threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = wave;
}
template <int WAVES, typename T>
__device__ __forceinline__ T blocks_get(T wave, const T* red) {
  if constexpr (WAVES == 1)
    return wave;
  else
    return tree_sum<WAVES>(red);
}

// Orders the LDS accesses of the threads with cells: a workgroup barrier, or beside helpers, where one wave has them all, only a
// compiler fence (a wave's LDS operations execute in order).
template <class G>
__device__ __forceinline__ void blocks_sync() {
  if (G::THREADS > 64 * G::WAVES) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
    __syncthreads();
  }
}

// Sums of a and b over the workgroup, the same bits in every thread.  No barrier afterwards: the next use of the same
// `red` comes after at least one other barrier.
template <class G, typename T>
__device__ __forceinline__ void blocks_sum2(T& a, T& b, T* red) {
  a = wave_sum_dpp(a);
  b = wave_sum_dpp(b);
  blocks_put<G::WAVES>(a, red);
  blocks_put<G::WAVES>(b, red + G::WAVES);
  blocks_sync<G>();
  a = blocks_get<G::WAVES>(a, red);
  b = blocks_get<G::WAVES>(b, red + G::WAVES);
}

// The sums of the one-wavefront kernel (FP32): per column, the cells of a colour from the bottom up, lane `column` of the
// first wave; then the wave's lanes as that kernel adds them.  Every thread calls these and gets the result.
template <int GS, int PLANES>
struct OrderedSums {
  using B = Block<GS, float, PLANES>;
  using G = BlockGeo<GS, float, PLANES>;
  // sum of |r| over a column (r[q] of one colour), in the threads of the first wave
  __device__ static float column(const B& o, const float (&r)[2 * G::H], float* lds) {
    float* s = lds + G::SCRATCH;
    float acc = 0.0f;
#pragma unroll 1
    for (int k = 0; k < G::CHUNKS; k++) {
      if (o.active && o.chunk == k) {
#pragma unroll
        for (int q = 0; q < 2 * G::H; q++) s[q * 64 + o.column] = fabsf(r[q]);
      }
      __syncthreads();
      if (threadIdx.x < G::LP) {
#pragma unroll
        for (int q = 0; q < 2 * G::H; q++) acc += s[q * 64 + threadIdx.x];
      }
      __syncthreads();
    }
    return acc;
  }
  // sum of |phi| over a column from the published cube: y, x, then z upwards
  __device__ static float column_phi(const float* lds) {
    float acc = 0.0f;
    const int t = threadIdx.x;
    if (t < G::LP) {
      const int a = t / G::MX, b = t % G::MX, m = GS >= 4 ? a : b, yb = GS >= 4 ? b : a;
#pragma unroll 1
      for (int e = 0; e < 4; e++)
#pragma unroll 1
        for (int z = 1; z <= G::R; z++) acc += fabsf(lds[G::word(2 * m + 1 + (e & 1), 2 * yb + 1 + (e >> 1), z)]);
    }
    return acc;
  }
  // v of the first wave's lanes, added as that kernel does; dpp: its order for the relative-residual test at one patch per
  // wavefront
  __device__ static float wave(float v, bool dpp, float* lds) {
    float* s = lds + G::SCRATCH + 2 * G::H * 64;
    v = threadIdx.x < G::LP ? v : 0.0f;
    if (threadIdx.x < 64) {
      v = dpp ? wave_sum_dpp(v) : wave_sum_butterfly(v);
      if (threadIdx.x == 0) *s = v;
    }
    __syncthreads();
    v = *s;
    __syncthreads();
    return v;
  }
};

// Whether the order of summation could decide between a and b: true where either is infinite (it may have overflowed in one
// order only), false for NaN, which sums of absolute values have in every order or in none.  FLT_MIN: products below it are
// subnormal and round by more than the relative bound.
__device__ __forceinline__ bool too_close(float a, float b) { return fabsf(a - b) <= 2e-5f * a + 2e-5f * b + FLT_MIN || a == b; }

// Whether any thread's residuals differ from those of the last iteration.
template <int WAVES, class B, int NQ>
__device__ __forceinline__ bool blocks_moved(const B& o, const float (&r1)[NQ], const float (&p1)[NQ], const float (&r0)[NQ],
                                             const float (&p0)[NQ], float* red) {
  bool moved = false;
#pragma unroll
  for (int q = 0; q < NQ; q++) moved |= r1[q] != p1[q] || r0[q] != p0[q];
  float any = __ballot(o.active && moved) ? 1.0f : 0.0f;
  blocks_put<WAVES>(any, red);
  __syncthreads();
  return blocks_get<WAVES>(any, red) > 0.0f;
}

// Gravity update of one patch from the potential in LDS; idx gives the word of cell (x, y, z) of the cube.
template <int GS, int THREADS, typename PT, typename T, class Idx>
__device__ __forceinline__ void blocks_gravity(const T* __restrict__ lds, Idx idx, T* __restrict__ flu, int t, const PT& P) {
  constexpr int CELLS = (kPatchCells + THREADS - 1) / THREADS, FC = CELLS < 4 ? CELLS : 4;   // four cells' fluid at a time
#pragma unroll 1
  for (int q0 = t; q0 < kPatchCells; q0 += FC * THREADS) {
  T f[FC][kNComp];
#pragma unroll
  for (int u = 0; u < FC; u++)
#pragma unroll
    for (int v = 0; v < kNComp; v++) f[u][v] = q0 + u * THREADS < kPatchCells ? flu[v * kPatchCells + q0 + u * THREADS] : T(1);
#pragma unroll
  for (int u = 0; u < FC; u++) {
    const int q = q0 + u * THREADS;
    if (q >= kPatchCells) break;
    const int x = q % kPatchSize + GS, y = q / kPatchSize % kPatchSize + GS, z = q / (kPatchSize * kPatchSize) + GS;
    T acc[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
      auto c = [&](int d) { return lds[idx(x + (a == 0 ? d : 0), y + (a == 1 ? d : 0), z + (a == 2 ? d : 0))]; };
      acc[a] = P.p5 ? P.gra_const * (-c(2) + c(-2) + T(8) * c(1) - T(8) * c(-1)) : P.gra_const * (c(1) - c(-1));
    }
    T px = f[u][1], py = f[u][2], pz = f[u][3];
    const T temp = T(0.5) / f[u][0];
    const T eint = f[u][4] - temp * (px * px + py * py + pz * pz);
    px = px - f[u][0] * acc[0];
    py = py - f[u][0] * acc[1];
    pz = pz - f[u][0] * acc[2];
    flu[kPatchCells + q] = px;
    flu[2 * kPatchCells + q] = py;
    flu[3 * kPatchCells + q] = pz;
    flu[4 * kPatchCells + q] = eint + temp * (px * px + py * py + pz * pz);
  }
  }
}

// One patch.  wave_dpp (FP32): the one-wavefront kernel's order of the relative-residual sums.
template <int GS, int PLANES, int HELP, typename PT, typename T = typename PT::real>
__device__ __forceinline__ void blocks_patch(T* __restrict__ lds, const T* __restrict__ rho, const T* __restrict__ cpot,
                                             const T* __restrict__ guess, T* __restrict__ out, T* __restrict__ flu,
                                             int* iters, int* status, const PT& P, bool wave_dpp) {
  using G = BlockGeo<GS, T, PLANES, HELP>;
  using Ordered = OrderedSums<GS, PLANES>;
  constexpr int N = G::N, R = G::R, H = G::H, THREADS = G::THREADS;
  constexpr bool ORDERED = !G::F64;
  const int t = threadIdx.x;
  T* red = lds + G::RED;
  Block<GS, T, PLANES, HELP> o;
  o.init(t);

  // Const*rho first where that pays: its loads run beside those of the coarse potential; after the interpolation they are a
  // second memory round trip (4096 FP64 GS-5 patches 1007 -> 979 us, 4096 FP32 GS-3 165 -> 159).  At FP64 GS 1 to 4 the
  // registers held over the interpolation cost 1 to 2%.
  constexpr bool EARLY = !G::F64 || GS == 5;
  auto cell_of = [&](int yy, int xx, int zi) { return ((o.z0 - 1 + zi) * R + o.y0 - 1 + yy) * R + o.x0 - 1 + xx; };
  if (EARLY) o.cells([&](int yy, int xx, int zi) { o.cr[yy][xx][zi] = P.cst * rho[cell_of(yy, xx, zi)]; });

  const int W = gra_nxt(P.gra_ghost), og = GS - P.gra_ghost;
  // A. the solve cube: the interpolated coarse potential (a zero start or an interior guess needs only its Dirichlet
  // layer) or the caller's whole cube
  if (P.init_mode == 3) {
    for (int q = t; q < N * N * N; q += THREADS) lds[G::word(q % N, q / N % N, q / (N * N))] = guess[q];
  } else {
    blocks_stage<G>(lds, cpot, t);
    __syncthreads();
    if constexpr (G::U == 1)
      blocks_interpolate_odd(o, lds, out, P.init_mode == 0, og == 0, P.int_scheme, t);
    else if (P.init_mode != 0)
      blocks_interpolate_even<G, true>(lds, P.int_scheme, t);
    else
      blocks_interpolate_even<G, false>(lds, P.int_scheme, t);
  }
  __syncthreads();

  // B. owned cells
  o.cells([&](int yy, int xx, int zi) {
    const int gi = cell_of(yy, xx, zi);
    if (!EARLY) o.cr[yy][xx][zi] = P.cst * rho[gi];
    T& ph = o.phi[yy][xx][zi];
    if (P.init_mode == 1) ph = T(0);
    if (P.init_mode == 2) ph = guess[gi];
    if (P.init_mode == 3 || (P.init_mode == 0 && G::U == 0)) ph = lds[o.word((xx + yy + zi + 1) & 1, yy, xx, zi)];
  });
  if (P.init_mode == 1 || P.init_mode == 2 || (P.init_mode == 0 && G::U == 1)) {
    o.template publish<0>(lds);
    o.template publish<1>(lds);
  }
  __syncthreads();

  bool fell_back = false;
  int it_done = P.max_iter, st = kStatusMaxIter;
  if (HELP == 1 || o.active) {   // helpers wait for the owners after the iterations
    // B'. a caller guess whose relative residual exceeds guess_tol is replaced by the zero guess
    T res[2 * H], black[2 * H];   // residuals of one colour: the pass being tested, and the last second pass
    if (P.init_mode >= 2 && P.guess_tol > T(0)) {
      T nums[G::PARTS] = {}, dens[G::PARTS] = {};
      o.template each<1>(lds, [&](int q, int, int, int zi, T r) { nums[G::part(zi)] += fabs(res[q] = r); });
      o.template each<0>(lds, [&](int q, int, int, int zi, T r) { nums[G::part(zi)] += fabs(black[q] = r); });
      o.cells([&](int yy, int xx, int zi) { dens[G::part(zi)] += fabs(o.phi[yy][xx][zi]); });
      T num = o.active ? tree_sum<G::PARTS>(nums) : T(0), den = o.active ? tree_sum<G::PARTS>(dens) : T(0);
      blocks_sum2<G>(num, den, red);
      bool keep = num <= P.guess_tol * den;
      if constexpr (ORDERED) {
        if (too_close(num, P.guess_tol * den)) {
          float n1 = Ordered::column(o, res, lds);
          n1 += Ordered::column(o, black, lds);
          n1 = Ordered::wave(n1, false, lds);
          keep = n1 <= P.guess_tol * Ordered::wave(Ordered::column_phi(lds), false, lds);
        }
      }
      fell_back = !keep;
      blocks_sync<G>();
      if (fell_back) {
        o.cells([&](int yy, int xx, int zi) { o.phi[yy][xx][zi] = T(0); });
        o.template publish<0>(lds);
        o.template publish<1>(lds);
      }
      blocks_sync<G>();
    }

    // C. red-black iterations: pass 0 updates the cells with x + y + z odd (colour 1), pass 1 the others
    const bool stall = P.term_mode == 0, relres = P.term_mode == 1;
    const int first_check = P.min_iter > 1 ? P.min_iter : 1;
    T old = T(FLT_MAX), black_sum[G::PARTS] = {};   // Residual_Total_Old = __FLT_MAX__ (CPU_PoissonSolver_SOR.cpp:215)
    T prev1[2 * H], prev0[2 * H];           // residuals of the last iteration (stall rule, FP32)
#pragma unroll
    for (int q = 0; q < 2 * H; q++) black[q] = prev1[q] = prev0[q] = T(0);
    for (int it = 0; it < P.max_iter; it++) {
      T sum[G::PARTS] = {};
      if (relres && it >= first_check && (it - first_check) % P.check_every == 0) {
        // first-colour residuals before the pass, second-colour ones |1 - omega| times those of the last pass
        T dens[G::PARTS] = {};
        o.template each<1>(lds, [&](int q, int, int, int zi, T r) { sum[G::part(zi)] += fabs(res[q] = r); });
        o.cells([&](int yy, int xx, int zi) { dens[G::part(zi)] += fabs(o.phi[yy][xx][zi]); });
#pragma unroll
        for (int h = 0; h < G::PARTS; h++) sum[h] = sum[h] + P.damp * black_sum[h];
        T num = o.active ? tree_sum<G::PARTS>(sum) : T(0), den = o.active ? tree_sum<G::PARTS>(dens) : T(0);
        blocks_sum2<G>(num, den, red);
        bool stop = num <= P.rel_tol * den;
        if constexpr (ORDERED) {
          if (too_close(num, P.rel_tol * den)) {
            float n1 = Ordered::column(o, res, lds);
            n1 = n1 + P.damp * Ordered::column(o, black, lds);
            n1 = Ordered::wave(n1, wave_dpp, lds);
            stop = n1 <= P.rel_tol * Ordered::wave(Ordered::column_phi(lds), wave_dpp, lds);
          }
        }
        if (stop) {
          it_done = it;
          st = kStatusConverged;
          break;
        }
#pragma unroll
        for (int q = 0; q < 2 * H; q++) {
          T& ph = o.phi[q & 1][o.xx_of(1, q & 1, q >> 1)][q >> 1];
          ph = ph + P.w6 * res[q];
        }
      } else if (stall) {
        o.template each<1>(lds, [&](int q, int yy, int xx, int zi, T r) {
          if (ORDERED) res[q] = r;
          sum[G::part(zi)] += fabs(r);
          o.phi[yy][xx][zi] = o.phi[yy][xx][zi] + P.w6 * r;
        });
      } else {
        o.template each<1>(lds, [&](int, int yy, int xx, int zi, T r) { o.phi[yy][xx][zi] = o.phi[yy][xx][zi] + P.w6 * r; });
      }
      o.template publish<1>(lds);
      blocks_sync<G>();
      if (stall || (it + 1 >= first_check && (it + 1 - first_check) % P.check_every == 0)) {
#pragma unroll
        for (int h = 0; h < G::PARTS; h++) black_sum[h] = T(0);
        o.template each<0>(lds, [&](int q, int yy, int xx, int zi, T r) {
          if (ORDERED) black[q] = r;
          black_sum[G::part(zi)] += fabs(r);
          o.phi[yy][xx][zi] = o.phi[yy][xx][zi] + P.w6 * r;
        });
      } else {
        o.template each<0>(lds, [&](int, int yy, int xx, int zi, T r) { o.phi[yy][xx][zi] = o.phi[yy][xx][zi] + P.w6 * r; });
      }
      o.template publish<0>(lds);
      if (stall) {
#pragma unroll
        for (int h = 0; h < G::PARTS; h++) sum[h] = sum[h] + black_sum[h];
        T tot = o.active ? tree_sum<G::PARTS>(sum) : T(0);
        T* r2 = red + 2 * G::WAVES;
        tot = wave_sum_dpp(tot);
        blocks_put<G::WAVES>(tot, r2);
        blocks_sync<G>();
        tot = blocks_get<G::WAVES>(tot, r2);
        if (it + 1 >= P.min_iter) {
          bool grew = tot > old;
          if constexpr (ORDERED) {
            // as too_close, but for two infinities, which any order has except within rounding of FLT_MAX; written out because
            // with the call 8 GS-5 patches under this rule take 43.9 us, so 42.9
            if (__builtin_expect(fabsf(tot - old) <= 2e-5f * tot + 2e-5f * old + FLT_MIN &&
                                     (tot != old || blocks_moved<G::WAVES>(o, res, prev1, black, prev0, red)),
                                 0)) {
              float a = Ordered::column(o, res, lds);
              a += Ordered::column(o, black, lds);
              a = Ordered::wave(a, false, lds);
              float b = FLT_MAX;
              if (it > 0) {
                b = Ordered::column(o, prev1, lds);
                b += Ordered::column(o, prev0, lds);
                b = Ordered::wave(b, false, lds);
              }
              grew = a > b;
            }
          }
          if (grew) {
            it_done = it + 1;
            st = kStatusConverged;
            break;
          }
        }
        old = tot;
        if (ORDERED) {
#pragma unroll
          for (int q = 0; q < 2 * H; q++) {
            prev1[q] = res[q];
            prev0[q] = black[q];
          }
        }
      } else {
        blocks_sync<G>();
      }
    }
  }

  // non-finite check over the interior, count and status
  bool bad = false;
  o.cells([&](int yy, int xx, int zi) { bad |= !isfinite(o.phi[yy][xx][zi]); });
  if (__syncthreads_or(o.active && bad)) st |= kStatusNonFinite;
  if (fell_back) st |= kStatusFallback;
  if (t == 0) {
    if (iters) *iters = it_done;
    if (status) *status = st;
  }

  // D. output window and the fused gravity update: from a dense copy of the window, or from the cube itself where the
  // window is all of it
  if (og == 0) {
    for (int q = t; q < N * N * N; q += THREADS) {
      const int x = q % N, y = q / N % N, z = q / (N * N);
      if (G::U == 0 || P.init_mode == 3 || !G::edge(x, y, z)) out[q] = lds[G::word(x, y, z)];
    }
    if (P.fuse_gravity && flu) blocks_gravity<GS, THREADS>(lds, [](int x, int y, int z) { return G::word(x, y, z); }, flu, t, P);
  } else {
    if (o.active)
      o.cells([&](int yy, int xx, int zi) {
        const int x = o.x0 + xx - og, y = o.y0 + yy - og, z = o.z0 + zi - og;
        if ((unsigned)x < (unsigned)W && (unsigned)y < (unsigned)W && (unsigned)z < (unsigned)W)
          lds[(z * W + y) * W + x] = o.phi[yy][xx][zi];
      });
    __syncthreads();
    for (int q = t; q < W * W * W; q += THREADS) out[q] = lds[q];
    if (P.fuse_gravity && flu)
      blocks_gravity<GS, THREADS>(lds, [=](int x, int y, int z) { return ((z - og) * W + y - og) * W + x - og; }, flu, t, P);
  }
}

// Waves per SIMD the kernel is asked to be compiled for.  FP64, with what the registers then allow beside the LDS: GS 1, 4 (16
// single waves of 17); GS 2, 5 (comes out at 76 registers, 6: more than the eleven workgroups of two waves); GS 3, 3 (two
// planes 76 registers, six workgroups of four waves beside seven; four planes 130, six of two beside seven); GS 4, 5 (80, 6:
// the four workgroups of six waves); GS 5, 3 (138, the three of four).  FP32 4 in 128 registers (16 cells per thread) or 6 in
// 80 (8 cells), 5 at GS 1.
constexpr int blocks_waves(int gs, bool f64, int planes) {
  return f64 ? (gs == 1 ? 4 : gs == 2 || gs == 4 ? 5 : 3) : planes == 4 ? 4 : gs == 1 ? 5 : 6;
}

template <int GS, int PLANES, typename PT, int HELP, typename G = BlockGeo<GS, typename PT::real, PLANES, HELP>>
__global__ void __launch_bounds__(G::THREADS, blocks_waves(GS, G::F64, PLANES))
    sor_blocks_kernel(UniformBatchT<typename PT::real> b, PT P, int wave_dpp) {
  using T = typename PT::real;
  extern __shared__ __align__(16) unsigned char blocks_smem[];
  constexpr int N3 = G::N * G::N * G::N, R3 = G::R * G::R * G::R, C3 = G::C * G::C * G::C;
  const int p = blockIdx.x;
  if (p >= b.npatch) return;
  const int W = gra_nxt(P.gra_ghost);
  blocks_patch<GS, PLANES, HELP>(reinterpret_cast<T*>(blocks_smem), b.rho + (size_t)p * R3, b.cpot + (size_t)p * C3,
                           b.guess ? b.guess + (size_t)p * (P.init_mode == 3 ? N3 : R3) : nullptr,
                           b.pot_out + (size_t)p * W * W * W, b.flu ? b.flu + (size_t)p * kNComp * kPatchCells : nullptr,
                           b.iters ? b.iters + p : nullptr, b.status ? b.status + p : nullptr, P, wave_dpp != 0);
}

// The patches of SOR tasks [first, first + gridDim.x / ppw) of a mixed batch, ppw to a task.
template <int GS, int PLANES, typename G = BlockGeo<GS, float, PLANES>>
__global__ void __launch_bounds__(G::THREADS, blocks_waves(GS, false, PLANES))
    sor_blocks_tasks_kernel(MixedBatch b, int first, int ppw, SolveParams P, int wave_dpp) {
  extern __shared__ __align__(16) unsigned char blocks_smem[];
  const Task tk = b.tasks[first + blockIdx.x / ppw];
  const int slot = blockIdx.x % ppw;
  if (tk.gs != GS || slot >= tk.count) return;   // a malformed plan never runs with another ghost size's layout
  const int patch = b.perm[tk.first + slot];
  if (patch < 0 || patch >= b.npatch) return;
  const PatchDesc d = b.desc[patch];
  const int W = gra_nxt(P.gra_ghost);
  blocks_patch<GS, PLANES, 1>(reinterpret_cast<float*>(blocks_smem), b.rho + d.rho_off, b.cpot + d.cpot_off,
                           b.guess ? b.guess + d.rho_off : nullptr, b.pot_out + (size_t)patch * W * W * W,
                           b.flu ? b.flu + (size_t)patch * kNComp * kPatchCells : nullptr, b.iters ? b.iters + patch : nullptr,
                           b.status ? b.status + patch : nullptr, P, wave_dpp != 0);
}

template <int GS, int PLANES, int HELP = 1, typename PT>
hipError_t launch_as(const UniformBatchT<typename PT::real>& b, const PT& p, bool wave_dpp, hipStream_t s) {
  using T = typename PT::real;
  using G = BlockGeo<GS, T, PLANES, HELP>;
  static_assert(sizeof(T) * G::WORDS <= 64 * 1024, "fits the default dynamic LDS limit");
  hipLaunchKernelGGL((sor_blocks_kernel<GS, PLANES, PT, HELP>), dim3(b.npatch), dim3(G::THREADS), sizeof(T) * G::WORDS, s, b, p,
                     wave_dpp ? 1 : 0);
  return hipGetLastError();
}

template <int GS, int PLANES>
hipError_t launch_tasks_as(const MixedBatch& b, const SolveParams& p, int ppw, int first, int count, hipStream_t s) {
  using G = BlockGeo<GS, float, PLANES>;
  hipLaunchKernelGGL((sor_blocks_tasks_kernel<GS, PLANES>), dim3(count * ppw), dim3(G::THREADS), sizeof(float) * G::WORDS, s,
                     b, first, ppw, p, ppw == 1 ? 1 : 0);
  return hipGetLastError();
}

// Two planes per thread instead of four at ghost sizes 3 and 5 (FP32 only at 5: FP64 has the paired layout for four): twice
// the waves per patch, for batches that leave the GPU short of them.  MI355X, us per call with 4 / 2 planes (interpolated
// start, FP32 stall rule; FP64 to 1e-10): GS 3, 8 patches 50 / 36, 1024: 62 / 54, 1536: 75 / 70, 2048: 82 / 96; GS 5, 8:
// 59 / 42, 512: 76 / 63, 768: 84 / 74, 1024: 95 / 103.  FP64 GS 3, 8: 124 / 94, 512: 159 / 132, 1024: 190 / 205; GS 5, 8:
// 122 / 124, 256: 140 / 144, 512: 185 / 214, 4096: 1004 / 1250.
bool two_planes(int gs, bool f64, int npatch) { return npatch <= (gs == 3 ? (f64 ? 512 : 1536) : (f64 ? 0 : 768)); }

// Helpers at FP64 ghost size 1, where one wave owns a patch and would do its interpolation (four coarse cells per lane, one
// after the other), window and gravity update by itself: 8 us beside the launch, where the iterations take 0.6 us each.  Three
// more waves share those, and the owner needs no barriers.  MI355X, us per call without / with helpers, 8 patches: 10
// iterations 19.9 / 13.4, 40: 37.7 / 29.7; 512: 22.4 / 16.3, 41.2 / 33.4; 1536 (six workgroups to a CU, one round): 32.5 /
// 27.3, 52.9 / 47.5; 2048: 36.6 / 40.6, 58.4 / 75.4.  The 256-thread kernel before the block form: 8 patches 13.2, 33.8; 512:
// 18.1, 44.5.
constexpr int kHelpersTo = 1536;

template <typename PT>
hipError_t launch_blocks(const UniformBatchT<typename PT::real>& b, const PT& p, bool wave_dpp, hipStream_t s) {
  constexpr bool F64 = sizeof(typename PT::real) == 8;
  const bool two = two_planes(b.gs, F64, b.npatch);
  switch (b.gs) {
    case 1:
      if constexpr (F64) {
        if (b.npatch <= kHelpersTo) return launch_as<1, 2, 4>(b, p, wave_dpp, s);
      }
      return launch_as<1, 2>(b, p, wave_dpp, s);
    case 2: return launch_as<2, 2>(b, p, wave_dpp, s);
    case 3: return two ? launch_as<3, 2>(b, p, wave_dpp, s) : launch_as<3, 4>(b, p, wave_dpp, s);
    case 4: return launch_as<4, 2>(b, p, wave_dpp, s);
    case 5:
      if constexpr (!F64) {
        if (two) return launch_as<5, 2>(b, p, wave_dpp, s);
      }
      return launch_as<5, 4>(b, p, wave_dpp, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace

// Largest batch for which the block form is the faster one.  MI355X, us per call, one wavefront per patch (or group) / blocks,
// FP32, 10, 40 and 150 iterations with a test every 2:
//   GS 1   256 patches 42/19 80/39 215/110   4096: 53/36 93/62 232/162   8192: 69/63 111/110 266/293   16384: 139/122 224/215 510/524
//   GS 2   256: 32/14 76/37 239/120   4096: 52/42 114/112 331/357   5120: 79/48 184/131 554/409   16384: 188/127 405/357 1268/1155
//   GS 3   1024: 37/23 91/60 280/190   2048: 45/35 110/90 332/276   16384: 313/230 761/575 2475/1944
//   GS 4   1024: 40/27 100/80 320/260   1152: 43/35 106/107 333/359   1536: 45/43 111/132 340/453
//   GS 5   1024: 47/32 113/84 358/258   1152: 51/43 122/119 377/389   1536: 54/46 128/126 379/410
// GS 1 to 3: the one-wavefront kernel uses 25 of 32 lanes at GS 2 and 36 of 64 at GS 3.  It is ahead only where its waves just
// fill a round and the solve is long (above some 60 iterations, 3700 to 4096 patches at GS 2, 7300 to 8192 and 16384 at GS 1).
// GS 4 and 5: 1024 patches are four workgroups to a CU; beyond, long solves lose (the one-wavefront kernel needs fewer
// reductions and reads once a launch fills the GPU).
int sor_blocks_limit(int gs) { return gs <= 3 ? INT_MAX : 1024; }

hipError_t launch_sor_blocks(const UniformBatch& b, const SolveParams& p, bool wave_dpp, hipStream_t s) {
  return launch_blocks(b, p, wave_dpp, s);
}

hipError_t launch_sor_blocks64(const UniformBatch64& b, const SolveParams64& p, hipStream_t s) {
  return launch_blocks(b, p, false, s);
}

hipError_t launch_sor_blocks_tasks(const MixedBatch& b, const SolveParams& p, int gs, int ppw, int first, int count,
                                   hipStream_t s) {
  if (count <= 0) return hipSuccess;
  const bool two = two_planes(gs, false, count * ppw);
  switch (gs) {
    case 1: return launch_tasks_as<1, 2>(b, p, ppw, first, count, s);
    case 2: return launch_tasks_as<2, 2>(b, p, ppw, first, count, s);
    case 3: return two ? launch_tasks_as<3, 2>(b, p, ppw, first, count, s) : launch_tasks_as<3, 4>(b, p, ppw, first, count, s);
    case 4: return launch_tasks_as<4, 2>(b, p, ppw, first, count, s);
    case 5: return two ? launch_tasks_as<5, 2>(b, p, ppw, first, count, s) : launch_tasks_as<5, 4>(b, p, ppw, first, count, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace pgamd
