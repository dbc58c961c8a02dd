// Per-patch multigrid V-cycle on gfx950: one workgroup per patch, level 0 in registers with its neighbours exchanged
// through LDS, the coarser levels in LDS.
//
// Reference behaviour reproduced (bit for bit in FP32 for the same number of V-cycles):
//   level schedule        CPU_PoissonSolver_MG.cpp:62-87      (GPU: CUPOT_PoissonSolver_MG.cu:16-53)
//   V-cycle driver        CPU_PoissonSolver_MG.cpp:213-258    (GPU: CUPOT_PoissonSolver_MG.cu:414-463)
//   smoother              CPU_PoissonSolver_MG.cpp:392-441
//   defect / error        CPU_PoissonSolver_MG.cpp:460-514
//   restriction           CPU_PoissonSolver_MG.cpp:533-616
//   prolongation          CPU_PoissonSolver_MG.cpp:635-684
//   window                CPU_PoissonSolver_MG.cpp:348-358
//
// Bound: VALU issue and LDS reads, about evenly (GS 5, per patch and V-cycle of 3+3 sweeps: 9.4k wave VALU
// instructions over 4 SIMDs and 8.9k LDS cycles).  The first form kept every cell and its right-hand side's index
// arithmetic in 256 threads and read all seven operands from LDS.  MI355X, 4096 GS-5 patches: 551 -> 222 us.

#include <hip/hip_runtime.h>

#include <cfloat>

#include "pg_geometry.h"
#include "pg_kernels.h"
#include "pg_interp.h"
#include "pg_reduce.h"

#pragma clang fp contract(off)

namespace pgamd {

// Level schedule: N_{l+1} = (N_l + 1)/2 while that is >= 3 (at most 4 levels for N <= 18).
struct MgLevels {
  int n[4];
  int nlv;
  int nbottom;
};

constexpr MgLevels mg_levels_of(int n0) {
  MgLevels L{{n0, 0, 0, 0}, 1, 0};
  while ((L.n[L.nlv - 1] + 1) / 2 >= 3 && L.nlv < 4) {
    L.n[L.nlv] = (L.n[L.nlv - 1] + 1) / 2;
    L.nlv++;
  }
  L.nbottom = L.n[L.nlv - 1] == 3 ? 1 : 7;
  return L;
}

// Work split.  A thread owns a 2x2 block of z-columns (x in {2m+1, 2m+2}, y in {2yb+1, 2yb+2}) over H planes of level
// 0 and keeps those cells' solution and right-hand side in registers; LDS serves the neighbours outside the block.
// H is even, so that which of a block's cells has which colour does not depend on the thread, and divides R:
// H = 4 where that fills the waves (GS 3: 108 of 128 threads, GS 5: 256), else 2 (GS 1: 64, GS 2: 125 of 128,
// GS 4: 343 of 384).  A cell of a coarser level belongs to one thread, two neighbours along x where the level has more
// cells than the workgroup threads (mg_coarse_cells).
//
// Level-0 layout in LDS: colour c = (x+y+z)&1, plane z, then the plane's cells of that colour as
// [y parity][y/2][x/2] (interior coordinates), so consecutive threads touch consecutive words; then the plane's
// Dirichlet cells of that colour (y = 0, y = N-1, x = 0, x = N-1; MX each).  Where those and the planes start decides
// the bank conflicts of the edge threads' reads and of waves that span two chunks of planes: the constants below were
// found by search over the 32 lanes and 32 banks of an LDS cycle (GS 5: none left; with everything packed, half of
// the LDS cycles of a V-cycle were conflicts, and LDS was the bound).  Searched: P, the faces' first words within P, and xs 1 or
// MX, from random starts by single moves; counted: over all half waves and the seven addresses of a colour pass (own, ylo, yhi,
// both xlo and both xhi), the most different words on one bank.
// The cube's edges and corners, which no stencil reads, are not stored.  While the coarse levels run, the solution
// is in registers only and the interior of this array holds the defect, rows of R in the same places.
constexpr int kMgRows = 32;   // rows of 16 lanes in the largest workgroup
struct MgBlock {
  int lpp;              // thread indices per chunk of planes (LP, or one more: an even pitch for 7x7 blocks)
  int P;                // words per colour and plane
  int x0, x1, xs;       // x = 0 and x = N-1 cells: first word and stride per y block
  int y0, y1;           // y = 0 and y = N-1 cells, stride 1
};
constexpr MgBlock mg_block(int gs) {
  switch (gs) {
    case 1: return {16, 72, 59, 52, 4, 44, 48};
    case 2: return {25, 94, 52, 74, 1, 84, 89};
    case 3: return {36, 137, 83, 74, 6, 126, 120};
    case 4: return {50, 185, 127, 135, 7, 106, 113};
    default: return {64, 224, 135, 128, 8, 216, 192};
  }
}

// cells of a coarse level per thread: one where the workgroup covers the level, else two neighbours along x
constexpr int mg_coarse_cells(int n) { return n <= 8 ? 1 : 2; }

template <int GS>
struct MgGeo {
  static constexpr Geo g = geo_of(GS);
  static constexpr int N = g.N, R = g.R, C = g.C, U = g.U;
  static constexpr MgLevels L = mg_levels_of(N);
  static constexpr int NLV = L.nlv;
  static constexpr int n(int l) { return L.n[l]; }
  static constexpr int MX = R / 2, LP = MX * MX;          // blocks per row / per plane
  static constexpr int H = GS == 3 || GS == 5 ? 4 : 2;    // planes per thread
  static constexpr MgBlock B = mg_block(GS);
  static constexpr int OWNERS = B.lpp * (R / H);          // threads up to the last that owns level-0 cells
  static constexpr int THREADS = (OWNERS + 63) / 64 * 64;
  static constexpr int P = B.P;
  static constexpr int CS = N * P;                        // words per colour
  // Coarse levels 1..NLV-1: solution and (but for the last) defect.  Row pitch n-1: the zero border cell x = n-1 of a
  // row is the x = 0 cell of the next, and likewise for planes (at n = 9 the pitch of 8 also makes the prolongation's
  // reads conflict-free).
  static constexpr int cn(int l) { return ((n(l) - 1) * (n(l) - 1) + n(l)) * (n(l) - 1) + 1; }
  static constexpr int off_sol(int l) {
    int s = 2 * CS;
    for (int k = 1; k < l; k++) s += 2 * cn(k);
    return s;
  }
  static constexpr int off_def(int l) { return off_sol(l) + cn(l); }
  static constexpr int COARSE = off_sol(NLV - 1) + cn(NLV - 1) - 2 * CS;
  static constexpr int STAGE = C * C * C;                 // the coarse potential, before the levels are used
  static constexpr int off_red() { return 2 * CS + (COARSE > STAGE ? COARSE : STAGE); }
  static constexpr int FLOATS = off_red() + 2 * kMgRows;  // two sums, a row of 16 lanes each
  static_assert(off_red() >= N * N * N, "the dense window fits below the sums");
  // threads that own cells of coarse level l
  static constexpr int coarse_owners(int l) {
    const int m = n(l) - 2;
    return mg_coarse_cells(n(l)) == 1 ? m * m * m : m * m * ((m + 1) / 2);
  }
  // Word of interior cell (x, y) of a plane's colour block, and of the Dirichlet cell of a face: face f = 2 * axis +
  // side, tangential coordinates u, v (y, z on the x faces; x, z on the y faces; x, y on the z faces), 1..R.
  __device__ static int in_plane(int x, int y) { return ((y - 1) & 1) * LP + ((y - 1) >> 1) * MX + ((x - 1) >> 1); }
  __device__ static int face_slot(int f, int u, int v) {
    const int side = f & 1, col = ((side + u + v) & 1) * CS;   // N - 1 is odd
    if (f < 2) return col + v * P + (side ? B.x1 : B.x0) + B.xs * ((u - 1) >> 1);
    if (f < 4) return col + v * P + (side ? B.y1 : B.y0) + ((u - 1) >> 1);
    return col + (side ? N - 1 : 0) * P + in_plane(u, v);
  }
  // word of cube cell (x, y, z) with at most one coordinate on the Dirichlet layer; -1 for edges and corners
  __device__ static int slot(int x, int y, int z) {
    const bool bx = x == 0 || x == N - 1, by = y == 0 || y == N - 1, bz = z == 0 || z == N - 1;
    if (bx + by + bz > 1) return -1;
    return bx ? face_slot(x > 0, y, z) : by ? face_slot(2 + (y > 0), x, z) : ((x + y + z) & 1) * CS + z * P + in_plane(x, y);
  }
};
// Waves per SIMD mg_patch is compiled for: FP32 fits 4 in 128 registers and FP64 2 in 256; with two planes per thread one
// more (not at ghost size 1, whose single wave does all the rest of a patch and would spill), and at ghost size 4 another
// one: its workgroups of six waves then fit four to a CU instead of three (FP32 8192 patches 493 -> 452 us, FP64 2776 ->
// 2051 us, for 28 bytes of spills that cost a lone patch 8%).
constexpr int mg_waves(int gs, size_t word) { return (word == 8 ? 2 : 4) + (gs == 2 || gs == 4) + (gs == 4); }
// workgroup of mg_patch_cells: one thread per cell of a colour
constexpr int mg_cell_threads(int gs) { return gs == 1 ? 256 : 512; }
constexpr int kMgMaxThreads = MgGeo<4>::THREADS;   // workgroup of the persistent kernel, enough for any ghost size

__device__ __forceinline__ constexpr int nat(int n, int x, int y, int z) { return (z * n + y) * n + x; }
// word of a coarse level's cell
__device__ __forceinline__ constexpr int cnat(int n, int x, int y, int z) { return nat(n - 1, x, y, z); }

// A value the compiler cannot see through: what is derived from it is computed again each time (a V-cycle, a task)
// instead of being kept in registers across the loop.
template <bool ON = true>
__device__ __forceinline__ int opaque(int v) {
  if (ON) asm volatile("" : "+v"(v));
  return v;
}

// Orders the LDS accesses of the calling threads: a workgroup barrier, or for levels owned by one wave only a
// compiler fence (a wave's LDS operations execute in order).
template <bool ONE_WAVE>
__device__ __forceinline__ void level_sync() {
  if (ONE_WAVE) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
    __syncthreads();
  }
}

// Block-wide sums of two values over the first ROWS rows of 16 threads (the others have zeros), in an order that does not
// depend on the workgroup's size: rows by DPP, then the row sums through LDS as a tree (shuffles over the wave would cross
// the LDS crossbar twelve times in a row).
template <int ROWS, typename T>
__device__ __forceinline__ void block_sum2(T& a, T& b, T* red) {
  static_assert(ROWS <= kMgRows, "room for the row sums");
  a = row_sum(a);
  b = row_sum(b);
  const int w = threadIdx.x >> 4;
  if ((threadIdx.x & 15) == 0) {
    red[w] = a;
    red[kMgRows + w] = b;
  }
  __syncthreads();
  a = tree_sum<ROWS>(red);
  b = tree_sum<ROWS>(red + kMgRows);
  __syncthreads();
}

// A thread's level-0 cells: solution, right-hand side and LDS addresses (words; the compile-time part of an address
// is the colour, the plane within the thread's H planes and the y parity).
template <int GS, typename T>
struct MgOwned {
  using M = MgGeo<GS>;
  static constexpr int H = M::H;
  T phi[2][2][H], rhs[2][2][H];   // [yy][xx][zi]
  int x0, y0, z0;                 // cube coordinates of the first cell
  int own, ylo, yhi, xlo[2], xhi[2];
  bool active;

  __device__ __forceinline__ void init(int t) {
    constexpr int LPP = M::B.lpp;
    int zc = t / LPP, cb = t - zc * LPP;
    active = t < M::OWNERS && cb < M::LP;
    if (!active) zc = cb = 0;   // reads stay in range; nothing is written
    const int yb = cb / M::MX, m = cb - yb * M::MX;
    x0 = 2 * m + 1;
    y0 = 2 * yb + 1;
    z0 = zc * H + 1;
    const int pz = z0 * M::P;
    own = pz + cb;
    ylo = pz + (yb > 0 ? M::LP + cb - M::MX : M::B.y0 + m);
    yhi = pz + (yb < M::MX - 1 ? cb + M::MX : M::B.y1 + m);
#pragma unroll
    for (int yy = 0; yy < 2; yy++) {
      xlo[yy] = pz + (m > 0 ? yy * M::LP + cb - 1 : M::B.x0 + M::B.xs * yb);
      xhi[yy] = pz + (m < M::MX - 1 ? yy * M::LP + cb + 1 : M::B.x1 + M::B.xs * yb);
    }
  }
  // which cell of a row pair has colour c (z0 is odd)
  static constexpr int xx_of(int c, int yy, int zi) { return (c + yy + zi + 1) & 1; }
  // sum of the six neighbours of cell (yy, xx, zi) of colour c, reference order k+ k- j+ j- i+ i-
  template <int c, int yy, int zi>
  __device__ __forceinline__ T neighbours(const T* __restrict__ lds) const {
    constexpr int xx = xx_of(c, yy, zi), oc = (1 - c) * M::CS + zi * M::P;
    const T kp = zi + 1 < H ? phi[yy][xx][zi + 1 < H ? zi + 1 : 0] : lds[own + oc + M::P + yy * M::LP];
    const T km = zi > 0 ? phi[yy][xx][zi > 0 ? zi - 1 : 0] : lds[own + oc - M::P + yy * M::LP];
    const T jo = lds[(yy == 0 ? ylo : yhi) + oc], io = lds[(xx == 0 ? xlo[yy] : xhi[yy]) + oc];
    const T jp = yy == 0 ? phi[1][xx][zi] : jo, jm = yy == 1 ? phi[0][xx][zi] : jo;
    const T ip = xx == 0 ? phi[yy][1][zi] : io, im = xx == 1 ? phi[yy][0][zi] : io;
    return kp + km + jp + jm + ip + im;
  }
  template <int c>
  __device__ __forceinline__ void publish(T* __restrict__ lds) const {
    if (active) {
#pragma unroll
      for (int zi = 0; zi < H; zi++)
#pragma unroll
        for (int yy = 0; yy < 2; yy++) lds[own + c * M::CS + zi * M::P + yy * M::LP] = phi[yy][xx_of(c, yy, zi)][zi];
    }
  }
  // calls f(yy, xx, zi, neighbour sum) for every cell of colour c, with the loads ahead of the arithmetic
  template <int c, class F>
  __device__ __forceinline__ void each(const T* __restrict__ lds, F f) const {
    each_at<c, 0>(lds, f);
  }
  template <int c, int q, class F>
  __device__ __forceinline__ void each_at(const T* __restrict__ lds, F f) const {
    if constexpr (q < 2 * H) {
      const T nb = neighbours<c, (q & 1), (q >> 1)>(lds);
      f(q & 1, xx_of(c, q & 1, q >> 1), q >> 1, nb);
      each_at<c, q + 1>(lds, f);
    }
  }
};

// Sums of two values per cell over the patch, for the error estimate and the guess check.  At ghost sizes 1 and 2 the batch
// size decides between mg_patch and mg_patch_cells (mg_small), and what a patch returns must not: both add in the order of
// mg_patch_cells, whose threads hold an x pair each, four consecutive ones to a block of mg_patch.  The cells of a pair come
// first (colour 0, then 1), then the pairs of a block by y and z, then the blocks as a tree over the threads.
template <int GS, typename T>
struct MgSums {
  static constexpr bool PAIRS = GS <= 2;
  static constexpr int NP = PAIRS ? 2 * MgGeo<GS>::H : 1;
  T a[NP] = {}, b[NP] = {};
  __device__ __forceinline__ void add(int yy, int zi, T va, T vb) {
    const int q = PAIRS ? 2 * zi + yy : 0;
    a[q] += va;
    b[q] += vb;
  }
  __device__ __forceinline__ void total(bool active, T& sa, T& sb, T* red) const {
    sa = active ? tree_sum<NP>(a) : T(0);
    sb = active ? tree_sum<NP>(b) : T(0);
    block_sum2<MgGeo<GS>::THREADS / 16>(sa, sb, red);
  }
};

// One red-black Gauss-Seidel sweep of level 0 (CPU_PoissonSolver_MG.cpp:392-441); both colours are published.
template <int GS, typename T>
__device__ __forceinline__ void smooth_level0(MgOwned<GS, T>& o, T* __restrict__ lds, T dh2) {
  const T one_six = T(1) / T(6);
  o.template each<1>(lds, [&](int yy, int xx, int zi, T nb) { o.phi[yy][xx][zi] = one_six * (nb - dh2 * o.rhs[yy][xx][zi]); });
  o.template publish<1>(lds);
  __syncthreads();
  o.template each<0>(lds, [&](int yy, int xx, int zi, T nb) { o.phi[yy][xx][zi] = one_six * (nb - dh2 * o.rhs[yy][xx][zi]); });
  o.template publish<0>(lds);
  __syncthreads();
}

// A thread's cells of a coarse level: (x, y, z), and with K = 2 also (x+1, y, z), x odd.
template <int n>
struct MgCoarse {
  static constexpr int m = n - 2, K = mg_coarse_cells(n), HW = (m + K - 1) / K;
  int x, y, z, id;
  bool active, two;
  __device__ __forceinline__ void init(int t) {
    active = t < m * m * HW;
    const int h = t % HW;
    y = (t / HW) % m + 1;
    z = active ? t / (HW * m) + 1 : 1;
    x = K * h + 1;
    two = K == 2 && active && x < m;
    id = cnat(n, x, y, z);
  }
  __device__ __forceinline__ bool has(int xx) const { return xx ? two : active; }
};

// sum of the six neighbours of a coarse level's cell
template <int n, typename T>
__device__ __forceinline__ T coarse_neighbours(const T* __restrict__ p) {
  constexpr int ys = n - 1, zs = ys * ys;
  return p[zs] + p[-zs] + p[ys] + p[-ys] + p[1] + p[-1];
}

// FROM_ZERO: the solution is zero before the first sweep, whatever its interior holds: the first pass reads nothing.
template <int n, bool ONE_WAVE, bool FROM_ZERO, typename T, int K>
__device__ __forceinline__ void smooth_coarse(const MgCoarse<n>& k, T* __restrict__ sol, const T (&rhs)[K], T dh2, int times) {
  const T one_six = T(1) / T(6);
  const int odd = (k.x + k.y + k.z) & 1;                    // colour of the first cell
  const int x1 = K == 2 ? 1 - odd : 0, x0 = K == 2 ? odd : 0;   // the cell of either colour
  const bool h1 = K == 2 ? k.has(x1) : k.active && odd, h0 = K == 2 ? k.has(x0) : k.active && !odd;
  T *p1 = sol + k.id + x1, *p0 = sol + k.id + x0;
  const T q1 = dh2 * (x1 ? rhs[K - 1] : rhs[0]), q0 = dh2 * (x0 ? rhs[K - 1] : rhs[0]);
  for (int s = 0; s < times; s++) {
    if (FROM_ZERO && s == 0) {
      if (h1) *p1 = one_six * (T(0) - q1);
    } else {
      if (h1) *p1 = one_six * (coarse_neighbours<n>(p1) - q1);
    }
    level_sync<ONE_WAVE>();
    if (h0) *p0 = one_six * (coarse_neighbours<n>(p0) - q0);
    level_sync<ONE_WAVE>();
  }
}

// 27-point restriction with ratio (nf-1)/(nc-1) at the thread's coarse cells (CPU_PoissonSolver_MG.cpp:533-616); row(y,
// z) is the word of the fine defect's (0, y, z).
template <int nc, int nf, typename T, class Row, int K>
__device__ __forceinline__ void restrict_to(const MgCoarse<nc>& k, const T* __restrict__ f, Row row, T (&rhs)[K]) {
  const T ratio = T(nf - 1) / T(nc - 1);
#pragma unroll
  for (int xx = 0; xx < K; xx++) rhs[xx] = T(0);
  if (!k.active) return;
  T w[2 + K][3];   // z, y, and the cells' x
  int ctr[2 + K];
#pragma unroll
  for (int a = 0; a < 2 + K; a++) {
    const T x = T(a == 0 ? k.z : a == 1 ? k.y : a == 2 || !k.two ? k.x : k.x + 1) * ratio;
    ctr[a] = int(x + T(0.5));
    w[a][0] = T(0.5) * (T(ctr[a]) + T(0.5) - x);
    w[a][2] = T(0.5) - w[a][0];
    w[a][1] = T(0.5);
  }
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) {
      const T* r = f + row(ctr[1] - 1 + b, ctr[0] - 1 + a) - 1;
      const T wzy = w[0][a] * w[1][b];
#pragma unroll
      for (int d = 0; d < 3; d++)
#pragma unroll
        for (int xx = 0; xx < K; xx++) rhs[xx] = rhs[xx] + wzy * w[2 + xx][d] * r[ctr[2 + xx] + d];
    }
}

// Trilinear prolongation weights of fine coordinate i: lower coarse coordinate and the two weights.
template <int nc, int nf, typename T>
__device__ __forceinline__ int prolong_axis(int i, T (&w)[2]) {
  const T x = T(i) * (T(nc - 1) / T(nf - 1));
  const int lo = int(x);
  w[0] = T(lo + 1) - x;
  w[1] = T(1) - w[0];
  return lo;
}

// The prolongation at one fine cell from the coarse corner c0; wzy[a][b] the z and y weights' products.  Terms in the
// order 000,001,010,100,011,110,101,111 of (z,y,x) (CPU_PoissonSolver_MG.cpp:635-684).
template <int nc, typename T>
__device__ __forceinline__ T prolong_cell(const T* __restrict__ c0, const T (&wzy)[2][2], const T (&wx)[2]) {
  constexpr int order[8][3] = {{0, 0, 0}, {0, 0, 1}, {0, 1, 0}, {1, 0, 0}, {0, 1, 1}, {1, 1, 0}, {1, 0, 1}, {1, 1, 1}};
  T s = T(0);
#pragma unroll
  for (int t = 0; t < 8; t++) {
    const int a = order[t][0], b = order[t][1], d = order[t][2];
    s = s + wzy[a][b] * wx[d] * c0[cnat(nc, d, b, a)];
  }
  return s;
}

// Correction of the thread's level-0 cells of one colour (ODD: colour 1) from level 1, published.
template <bool ODD, int GS, typename T>
__device__ __forceinline__ void prolongate_level0(MgOwned<GS, T>& o, T* __restrict__ lds) {
  using M = MgGeo<GS>;
  constexpr int n1 = M::n(1), N = M::N;
  const T* cs = lds + M::off_sol(1);
  T wx[2][2], wy[2][2];
  int lx[2], ly[2];
  const int x0 = opaque(o.x0), y0 = opaque(o.y0), z0 = opaque(o.z0);
#pragma unroll
  for (int u = 0; u < 2; u++) {
    lx[u] = prolong_axis<n1, N>(x0 + u, wx[u]);
    ly[u] = prolong_axis<n1, N>(y0 + u, wy[u]);
  }
#pragma unroll
  for (int zi = 0; zi < M::H; zi++) {
    T wz[2];
    const int lz = prolong_axis<n1, N>(z0 + zi, wz);
#pragma unroll
    for (int yy = 0; yy < 2; yy++) {
      const int xx = o.xx_of(ODD, yy, zi);
      const T wzy[2][2] = {{wz[0] * wy[yy][0], wz[0] * wy[yy][1]}, {wz[1] * wy[yy][0], wz[1] * wy[yy][1]}};
      o.phi[yy][xx][zi] = o.phi[yy][xx][zi] + prolong_cell<n1>(cs + cnat(n1, lx[xx], ly[yy], lz), wzy, wx[xx]);
    }
  }
  o.template publish<ODD>(lds);
}

// Coarse level l and below: the correction for the right-hand side in rhs (the thread's cells), left in the level's
// solution array.  Called by all threads, or by the first wave alone once a level fits it.
template <int GS, int l, bool ONE_WAVE, typename PT, typename T = typename PT::real>
__device__ __forceinline__ void coarse_cycle(T* __restrict__ lds, const MgCoarse<MgGeo<GS>::n(l)>& k, const T (&rhs)[MgCoarse<MgGeo<GS>::n(l)>::K], const PT& P) {
  using M = MgGeo<GS>;
  constexpr int n = M::n(l);
  const T dh = P.dh * T(M::N - 1) / T(n - 1), dh2 = dh * dh;
  T* sol = lds + M::off_sol(l);
  if constexpr (l == M::NLV - 1) {
    smooth_coarse<n, ONE_WAVE, true>(k, sol, rhs, dh2, M::L.nbottom);
  } else {
    if (P.mg_npre == 0) {
      if (k.active) sol[k.id] = T(0);
      if (k.two) sol[k.id + 1] = T(0);
      level_sync<ONE_WAVE>();
    }
    smooth_coarse<n, ONE_WAVE, true>(k, sol, rhs, dh2, P.mg_npre);
    T* def = lds + M::off_def(l);
    const T m_dh2 = T(-1) / dh2;
#pragma unroll
    for (int xx = 0; xx < k.K; xx++)
      if (k.has(xx)) {
        const T* p = sol + k.id + xx;
        def[k.id + xx] = m_dh2 * (coarse_neighbours<n>(p) - T(6) * p[0]) + rhs[xx];
      }
    level_sync<ONE_WAVE>();
    constexpr int nn = M::n(l + 1);
    constexpr bool NEXT_ONE = M::coarse_owners(l + 1) <= 64;
    if (!NEXT_ONE || threadIdx.x < 64) {
      MgCoarse<nn> kn;
      kn.init(opaque(threadIdx.x));
      T rn[MgCoarse<nn>::K];
      restrict_to<nn, n>(kn, def, [](int y, int z) { return cnat(n, 0, y, z); }, rn);
      coarse_cycle<GS, l + 1, NEXT_ONE>(lds, kn, rn, P);
    }
    if (NEXT_ONE && !ONE_WAVE) __syncthreads();
    const T* cs = lds + M::off_sol(l + 1);
    T wz[2], wy[2];
    const int lz = prolong_axis<nn, n>(k.z, wz), ly = prolong_axis<nn, n>(k.y, wy);
    const T wzy[2][2] = {{wz[0] * wy[0], wz[0] * wy[1]}, {wz[1] * wy[0], wz[1] * wy[1]}};
    // the next sweep overwrites colour 1 from colour 0: only colour 0 is corrected, unless there is no sweep
    auto correct = [&](int xx) {
      T wx[2];
      const int lx = prolong_axis<nn, n>(k.x + xx, wx);
      sol[k.id + xx] = sol[k.id + xx] + prolong_cell<nn>(cs + cnat(nn, lx, ly, lz), wzy, wx);
    };
    const int odd = (k.x + k.y + k.z) & 1, x0 = k.K == 2 ? odd : 0;
    const bool all = P.mg_npost == 0;
    if (k.K == 2 ? k.has(x0) : k.active && (!odd || all)) correct(x0);
    if (k.K == 2 && all && k.has(1 - x0)) correct(1 - x0);
    level_sync<ONE_WAVE>();
    smooth_coarse<n, ONE_WAVE, false>(k, sol, rhs, dh2, P.mg_npost);
  }
}

// Gravity update of cell q of the patch proper from the potential at c (strides 1, sy, sz) and the cell's fluid f
// (CPU_GravitySolver.cpp:34-79).
template <typename PT, typename T>
__device__ __forceinline__ void gravity_cell(const T* __restrict__ c, int sy, int sz, const T (&f)[kNComp], T* __restrict__ flu,
                                             int q, const PT& P) {
  T acc[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const int d = a == 0 ? 1 : a == 1 ? sy : sz;
    acc[a] = P.p5 ? P.gra_const * (-c[2 * d] + c[-2 * d] + T(8) * c[d] - T(8) * c[-d]) : P.gra_const * (c[d] - c[-d]);
  }
  T px = f[1], py = f[2], pz = f[3];
  const T temp = T(0.5) / f[0];
  const T eint = f[4] - temp * (px * px + py * py + pz * pz);
  px = px - f[0] * acc[0];
  py = py - f[0] * acc[1];
  pz = pz - f[0] * acc[2];
  flu[kPatchCells + q] = px;
  flu[2 * kPatchCells + q] = py;
  flu[3 * kPatchCells + q] = pz;
  flu[4 * kPatchCells + q] = eint + temp * (px * px + py * py + pz * pz);
}

template <typename PT, typename T>
__device__ __forceinline__ void mg_report(int iter, T error, bool fell_back, int* iters, int* status, const PT& P) {
  int st = error <= P.mg_tol ? kStatusConverged : kStatusMaxIter;
  if (!(error == error) || error == T(INFINITY)) st |= kStatusNonFinite;
  if (fell_back) st |= kStatusFallback;
  if (iters) *iters = iter;
  if (status) *status = st;
}

// One patch: interpolation, V-cycles until Error <= tol or max_iter, window and optional gravity.  PT is the
// parameter type, SolveParams (FP32) or SolveParams64 (FP64); T its element type; THREADS the workgroup's size.
template <int GS, int THREADS, typename PT, typename T = typename PT::real>
__device__ void mg_patch(T* __restrict__ lds, const T* __restrict__ rho, const T* __restrict__ cpot,
                         const T* __restrict__ guess, T* __restrict__ out, T* __restrict__ flu, int* iters,
                         int* status, const PT& P) {
  using M = MgGeo<GS>;
  constexpr int N = M::N, R = M::R, C = M::C, U = M::U, H = M::H;
  static_assert(THREADS >= M::THREADS, "one thread per level-0 block of columns");
  static_assert(M::NLV >= 2, "at least one coarse level");
  T* red = lds + M::off_red();
  const int G = gra_nxt(P.gra_ghost), og = GS - P.gra_ghost;
  const int t = opaque(threadIdx.x);

  // Interpolation, from the coarse potential staged where the coarse levels go.  The cube's edges and corners are
  // final and go straight to a window that has them (og = 0).
  MgOwned<GS, T> o;
  o.init(t);
  T* stage = lds + 2 * M::CS;
  {
    constexpr int SI = (M::STAGE + THREADS - 1) / THREADS;
    T v[SI];
#pragma unroll
    for (int u = 0; u < SI; u++) v[u] = t + u * THREADS < M::STAGE ? cpot[t + u * THREADS] : T(0);
#pragma unroll
    for (int u = 0; u < SI; u++)
      if (t + u * THREADS < M::STAGE) stage[t + u * THREADS] = v[u];
  }
  __syncthreads();
  constexpr int NC = C - 2, MX = M::MX;
  auto children = [&](int i, int j, int k, T (&ch)[2][2][2]) {
    const T* c = stage + ((k - 1) * C + j - 1) * C + i - 1;
    interp_children_at<false>([&](int dk, int dj, int di) { return c[(dk * C + dj) * C + di]; }, P.int_scheme, ch);
  };
  if constexpr (U == 1) {
    // A thread's block is whole coarse cells: straight into registers.  The faces' coarse cells and, for a window that
    // has them, the edges' and corners' are shared out.
    if (P.init_mode == 0) {
#pragma unroll
      for (int kk = 0; kk < H / 2; kk++) {
        T ch[2][2][2];
        children((o.x0 + 3) >> 1, (o.y0 + 3) >> 1, ((o.z0 + 3) >> 1) + kk, ch);
#pragma unroll
        for (int e = 0; e < 8; e++) o.phi[(e >> 1) & 1][e & 1][2 * kk + (e >> 2)] = ch[e >> 2][(e >> 1) & 1][e & 1];
      }
    }
    for (int q = t; q < 6 * M::LP; q += THREADS) {
      const int f = q / M::LP, r = q - f * M::LP, b = r / MX, a = r - b * MX, ax = f >> 1, end = f & 1 ? NC : 1;
      T ch[2][2][2];
      children(ax == 0 ? end : a + 2, ax == 0 ? a + 2 : ax == 1 ? end : b + 2, ax == 2 ? end : b + 2, ch);
      const int s = 1 - (f & 1);   // the child on the Dirichlet layer
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int c1 = e & 1, c2 = e >> 1;
        const T vx = s ? ch[c2][c1][1] : ch[c2][c1][0], vy = s ? ch[c2][1][c1] : ch[c2][0][c1],
                vz = s ? ch[1][c2][c1] : ch[0][c2][c1];
        lds[M::face_slot(f, 2 * a + 1 + c1, 2 * b + 1 + c2)] = ax == 0 ? vx : ax == 1 ? vy : vz;
      }
    }
    if (og == 0) {
      for (int q = t; q < 12 * MX + 8; q += THREADS) {
        const int ed = q / MX, ax = q < 12 * MX ? ed >> 2 : 3, bits = q < 12 * MX ? ed & 3 : q - 12 * MX, a = q - ed * MX + 2;
        const int e0 = bits & 1 ? NC : 1, e1 = bits & 2 ? NC : 1, e2 = bits & 4 ? NC : 1;
        const int i = ax == 0 ? a : e0, j = ax == 1 ? a : ax == 0 ? e0 : e1, k = ax == 2 ? a : ax == 3 ? e2 : e1;
        T ch[2][2][2];
        children(i, j, k, ch);
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const int x = 2 * i - 3 + (e & 1), y = 2 * j - 3 + ((e >> 1) & 1), z = 2 * k - 3 + (e >> 2);
          const int nb = (x == 0 || x == N - 1) + (y == 0 || y == N - 1) + (z == 0 || z == N - 1);
          const bool in = x >= 0 && x < N && y >= 0 && y < N && z >= 0 && z < N;
          if (in && nb > 1) out[nat(N, x, y, z)] = ch[e >> 2][(e >> 1) & 1][e & 1];
        }
      }
    }
  } else {
    for (int q = t; q < NC * NC * NC; q += THREADS) {
      const int i = q % NC + 1, j = (q / NC) % NC + 1, k = q / (NC * NC) + 1;
      T ch[2][2][2];
      children(i, j, k, ch);
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const int x = 2 * (i - 1) + (e & 1), y = 2 * (j - 1) + ((e >> 1) & 1), z = 2 * (k - 1) + (e >> 2);
        const int sl = M::slot(x, y, z);
        if (sl >= 0)
          lds[sl] = ch[e >> 2][(e >> 1) & 1][e & 1];
        else if (og == 0)
          out[nat(N, x, y, z)] = ch[e >> 2][(e >> 1) & 1][e & 1];
      }
    }
  }
  __syncthreads();
  for (int q = t; q < M::COARSE; q += THREADS) stage[q] = T(0);   // the coarse levels' borders stay zero

  // level-0 cells into registers; initial-guess modes
#pragma unroll
  for (int yy = 0; yy < 2; yy++)
#pragma unroll
    for (int xx = 0; xx < 2; xx++)
#pragma unroll
      for (int zi = 0; zi < H; zi++) {
        const int c = (xx + yy + zi + 1) & 1;
        const int gi = ((o.z0 - 1 + zi) * R + (o.y0 - 1 + yy)) * R + (o.x0 - 1 + xx);
        o.rhs[yy][xx][zi] = P.poi_coeff * rho[gi];  // CPU_PoissonSolver_MG.cpp:200-207
        T& ph = o.phi[yy][xx][zi];
        if (U == 0 && P.init_mode == 0) ph = lds[o.own + c * M::CS + zi * M::P + yy * M::LP];
        if (P.init_mode == 1) ph = T(0);
        if (P.init_mode == 2) ph = guess[gi];
        if (P.init_mode == 3) ph = guess[nat(N, o.x0 + xx, o.y0 + yy, o.z0 + zi)];   // whole-cube guess: its interior
      }
  if (U == 1 || P.init_mode != 0) {
    o.template publish<0>(lds);
    o.template publish<1>(lds);
  }
  __syncthreads();

  // Reject a caller guess whose relative residual sum|R| / sum|phi| (the SOR residual in the reference
  // operand order, Const = Poi_Coeff dh^2, over the interior) exceeds guess_tol: start from the zero guess,
  // as the SOR kernel does, and report it in the status.
  bool fell_back = false;
  if (P.init_mode >= 2 && P.guess_tol > T(0)) {
    MgSums<GS, T> a;
    auto add = [&](int yy, int xx, int zi, T nb) {
      const int gi = ((o.z0 - 1 + zi) * R + (o.y0 - 1 + yy)) * R + (o.x0 - 1 + xx);
      a.add(yy, zi, fabs(nb - T(6) * o.phi[yy][xx][zi] - P.cst * rho[gi]), fabs(o.phi[yy][xx][zi]));
    };
    o.template each<0>(lds, add);
    o.template each<1>(lds, add);
    T num, den;
    a.total(o.active, num, den, red);
    fell_back = !(num <= P.guess_tol * den);
    if (fell_back) {
#pragma unroll
      for (int yy = 0; yy < 2; yy++)
#pragma unroll
        for (int xx = 0; xx < 2; xx++)
#pragma unroll
          for (int zi = 0; zi < H; zi++) o.phi[yy][xx][zi] = T(0);
      o.template publish<0>(lds);
      o.template publish<1>(lds);
    }
    __syncthreads();
  }

  constexpr int n1 = M::n(1);
  constexpr bool ONE1 = M::coarse_owners(1) <= 64;
  const T dh2 = P.dh * P.dh, m_dh2 = T(-1) / dh2;
  int iter = 0;
  T error = T(FLT_MAX);
  while (iter < P.mg_max_iter && error > P.mg_tol) {
    for (int s = 0; s < P.mg_npre; s++) smooth_level0<GS>(o, lds, dh2);
    // defect -(lap(sol) - rhs) (CPU_PoissonSolver_MG.cpp:460-514), over the published solution
    {
      T d[2][2][H];
      auto defect = [&](int yy, int xx, int zi, T nb) {
        d[yy][xx][zi] = m_dh2 * (nb - T(6) * o.phi[yy][xx][zi]) + o.rhs[yy][xx][zi];
      };
      o.template each<0>(lds, defect);
      o.template each<1>(lds, defect);
      __syncthreads();
      if (o.active) {
        T* r = lds + o.z0 * M::P + (o.y0 >> 1) * R + o.x0 - 1;
#pragma unroll
        for (int zi = 0; zi < H; zi++)
#pragma unroll
          for (int yy = 0; yy < 2; yy++)
#pragma unroll
            for (int xx = 0; xx < 2; xx++) r[yy * M::CS + zi * M::P + xx] = d[yy][xx][zi];
      }
    }
    __syncthreads();
    if (!ONE1 || t < 64) {
      MgCoarse<n1> k1;
      k1.init(opaque(t));
      T r1[MgCoarse<n1>::K];
      restrict_to<n1, N>(k1, lds, [](int y, int z) { return ((y - 1) & 1) * M::CS + z * M::P + ((y - 1) >> 1) * R - 1; }, r1);
      coarse_cycle<GS, 1, ONE1>(lds, k1, r1, P);
    }
    __syncthreads();
    // Prolongate, correct and publish again.  The next sweep overwrites colour 1 from colour 0: only colour 0 is corrected,
    // unless there is no sweep.
    prolongate_level0<false>(o, lds);
    if (P.mg_npost == 0) prolongate_level0<true>(o, lds);
    __syncthreads();
    for (int s = 0; s < P.mg_npost; s++) smooth_level0<GS>(o, lds, dh2);
    MgSums<GS, T> a;
    auto sums = [&](int yy, int xx, int zi, T nb) {
      a.add(yy, zi, fabs(m_dh2 * (nb - T(6) * o.phi[yy][xx][zi]) + o.rhs[yy][xx][zi]), fabs(o.phi[yy][xx][zi]));
    };
    o.template each<0>(lds, sums);
    o.template each<1>(lds, sums);
    T sd, ss;
    a.total(o.active, sd, ss, red);
    error = P.dh * P.dh * sd / ss;
    iter++;
  }

  // status: converged / max_iter / non-finite
  if (t == 0) mg_report(iter, error, fell_back, iters, status, P);

  // the fluid is requested before the window is laid out: one memory round trip
  constexpr int FC = (kPatchCells + THREADS - 1) / THREADS;
  const bool gravity = P.fuse_gravity && flu;
  T fl[FC][kNComp];
  if (gravity) {
#pragma unroll
    for (int u = 0; u < FC; u++)
#pragma unroll
      for (int v = 0; v < kNComp; v++) fl[u][v] = t + u * THREADS < kPatchCells ? flu[v * kPatchCells + t + u * THREADS] : T(1);
  }
  // Window (CPU_PoissonSolver_MG.cpp:348-358) and fused gravity, from a dense copy of the window.  A window of the
  // whole cube also has the faces (its edges and corners were written at the start).
  constexpr int FI = (6 * M::LP + THREADS - 1) / THREADS;
  T face[FI][4];
  auto faces = [&](auto f) {
#pragma unroll
    for (int u = 0; u < FI; u++) {
      const int q = t + u * THREADS;
      if (q < 6 * M::LP) {
        const int fc = q / M::LP, r = q - fc * M::LP, b = r / MX, a = r - b * MX;
#pragma unroll
        for (int e = 0; e < 4; e++) f(face[u][e], fc, 2 * a + 1 + (e & 1), 2 * b + 1 + (e >> 1));
      }
    }
  };
  if (og == 0) {
    faces([&](T& v, int f, int u, int w) { v = lds[M::face_slot(f, u, w)]; });
    __syncthreads();
  }
  if (o.active) {
#pragma unroll
    for (int zi = 0; zi < H; zi++)
#pragma unroll
      for (int yy = 0; yy < 2; yy++)
#pragma unroll
        for (int xx = 0; xx < 2; xx++) {
          const int x = o.x0 + xx - og, y = o.y0 + yy - og, z = o.z0 + zi - og;
          if ((unsigned)x < (unsigned)G && (unsigned)y < (unsigned)G && (unsigned)z < (unsigned)G)
            lds[nat(G, x, y, z)] = o.phi[yy][xx][zi];
        }
  }
  if (og == 0)
    faces([&](T& v, int f, int u, int w) {
      const int d = f & 1 ? N - 1 : 0;
      lds[f < 2 ? nat(N, d, u, w) : f < 4 ? nat(N, u, d, w) : nat(N, u, w, d)] = v;
    });
  __syncthreads();
  for (int q = t; q < G * G * G; q += THREADS) {
    if (og == 0) {
      const int i = q % N, j = (q / N) % N, k = q / (N * N);
      if ((i == 0 || i == N - 1) + (j == 0 || j == N - 1) + (k == 0 || k == N - 1) > 1) continue;
    }
    out[q] = lds[q];
  }
  if (gravity) {
#pragma unroll
    for (int u = 0; u < FC; u++) {
      const int q = t + u * THREADS;
      if (q >= kPatchCells) break;
      const int i = q % kPatchSize, j = (q / kPatchSize) % kPatchSize, k = q / (kPatchSize * kPatchSize);
      gravity_cell(lds + nat(G, i + P.gra_ghost, j + P.gra_ghost, k + P.gra_ghost), G, G * G, fl[u], flu, q, P);
    }
  }
  __syncthreads();
}

// One patch of ghost size 1 or 2 in the shortest time: a thread has one cell of each colour, every neighbour comes from
// LDS (natural layout).  The blocks of mg_patch leave one or two waves to do everything, which is the better use of a
// full GPU and the slower of the two for a patch by itself.
template <int GS, typename PT, typename T = typename PT::real>
__device__ void mg_patch_cells(T* __restrict__ lds, const T* __restrict__ rho, const T* __restrict__ cpot,
                               const T* __restrict__ guess, T* __restrict__ out, T* __restrict__ flu, int* iters,
                               int* status, const PT& P) {
  using M = MgGeo<GS>;
  constexpr int N = M::N, R = M::R, C = M::C, U = M::U, NC = C - 2, THREADS = mg_cell_threads(GS), LAST = R * R * R / 2 - 1;
  static_assert(LAST < THREADS && N * N * N <= 2 * M::CS && M::NLV >= 2, "one cell of each colour per thread");
  static_assert(M::H == 2 && M::B.lpp == M::LP && THREADS == 4 * M::THREADS, "four threads to a block of mg_patch");
  T *sol = lds, *def = lds + M::FLOATS, *red = lds + M::off_red(), *stage = lds + 2 * M::CS;
  constexpr bool FRESH = sizeof(T) == 4;   // FP64 is compiled for fewer waves and keeps its weights in registers
  const int t = threadIdx.x;
  for (int q = t; q < M::STAGE; q += THREADS) stage[q] = cpot[q];
  const bool active = t <= LAST;
  // an x pair, four threads to the 2x2x2 cells that a thread of mg_patch has (see MgSums)
  const int tc = active ? t : LAST, tb = tc >> 2, cb = tb % M::LP;
  const int x = 2 * (cb % M::MX) + 1, y = 2 * (cb / M::MX) + 1 + (tc & 1), z = 2 * (tb / M::LP) + 1 + (tc >> 1 & 1);
  const int x1 = (y + z) & 1;   // which of x, x + 1 has colour 1
  const int id[2] = {nat(N, x + 1 - x1, y, z), nat(N, x + x1, y, z)};   // by colour
  T rh[2], gu[2] = {T(0), T(0)};
  auto owned_rho = [&](int c) { return rho[nat(R, x - 1 + (c ? x1 : 1 - x1), y - 1, z - 1)]; };
#pragma unroll
  for (int c = 0; c < 2; c++) {
    rh[c] = owned_rho(c);
    if (P.init_mode == 2) gu[c] = guess[nat(R, x - 1 + (c ? x1 : 1 - x1), y - 1, z - 1)];
    if (P.init_mode == 3) gu[c] = guess[id[c]];
  }
  __syncthreads();
  if (t < NC * NC * NC) {
    const int i = t % NC + 1, j = (t / NC) % NC + 1, k = t / (NC * NC) + 1;
    T ch[2][2][2];
    const T* c = stage + nat(C, i - 1, j - 1, k - 1);
    interp_children_at<false>([&](int dk, int dj, int di) { return c[nat(C, di, dj, dk)]; }, P.int_scheme, ch);
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const int fx = 2 * (i - 1) + (e & 1) - U, fy = 2 * (j - 1) + ((e >> 1) & 1) - U, fz = 2 * (k - 1) + (e >> 2) - U;
      if (fx >= 0 && fx < N && fy >= 0 && fy < N && fz >= 0 && fz < N) sol[nat(N, fx, fy, fz)] = ch[e >> 2][(e >> 1) & 1][e & 1];
    }
  }
  static_assert(NC * NC * NC <= THREADS, "one coarse cell per thread");
  __syncthreads();
  for (int q = t; q < M::COARSE; q += THREADS) stage[q] = T(0);
  if (P.init_mode != 0 && active) {
    sol[id[0]] = gu[0];
    sol[id[1]] = gu[1];
  }
  __syncthreads();
  auto nb = [&](int i) { return sol[i + N * N] + sol[i - N * N] + sol[i + N] + sol[i - N] + sol[i + 1] + sol[i - 1]; };
  bool fell_back = false;
  if (P.init_mode >= 2 && P.guess_tol > T(0)) {
    T num = T(0), den = T(0);
#pragma unroll
    for (int c = 0; c < 2; c++) {
      num += fabs(nb(id[c]) - T(6) * sol[id[c]] - P.cst * rh[c]);
      den += fabs(sol[id[c]]);
    }
    if (!active) num = den = T(0);
    block_sum2<THREADS / 16>(num, den, red);
    fell_back = !(num <= P.guess_tol * den);
    if (fell_back && active) sol[id[0]] = sol[id[1]] = T(0);
    __syncthreads();
  }
  rh[0] = P.poi_coeff * rh[0];
  rh[1] = P.poi_coeff * rh[1];
  const T one_six = T(1) / T(6), dh2 = P.dh * P.dh, m_dh2 = T(-1) / dh2, q0 = dh2 * rh[0], q1 = dh2 * rh[1];
  auto smooth = [&](int times) {
    for (int s = 0; s < times; s++) {
      if (active) sol[id[1]] = one_six * (nb(id[1]) - q1);
      __syncthreads();
      if (active) sol[id[0]] = one_six * (nb(id[0]) - q0);
      __syncthreads();
    }
  };
  constexpr int n1 = M::n(1);
  static_assert(M::coarse_owners(1) <= 64, "the coarse levels fit a wave");
  int iter = 0;
  T error = T(FLT_MAX);
  while (iter < P.mg_max_iter && error > P.mg_tol) {
    smooth(P.mg_npre);
    if (active)
#pragma unroll
      for (int c = 0; c < 2; c++) def[id[c]] = m_dh2 * (nb(id[c]) - T(6) * sol[id[c]]) + rh[c];
    __syncthreads();
    if (t < 64) {
      MgCoarse<n1> k1;
      k1.init(opaque<FRESH>(t));
      T r1[MgCoarse<n1>::K];
      restrict_to<n1, N>(k1, def, [](int yf, int zf) { return nat(N, 0, yf, zf); }, r1);
      coarse_cycle<GS, 1, true>(lds, k1, r1, P);
    }
    __syncthreads();
    {
      T wy[2], wz[2];
      const int px = opaque<FRESH>(x), py = opaque<FRESH>(y), pz = opaque<FRESH>(z);
      const int ly = prolong_axis<n1, N>(py, wy), lz = prolong_axis<n1, N>(pz, wz);
      const T wzy[2][2] = {{wz[0] * wy[0], wz[0] * wy[1]}, {wz[1] * wy[0], wz[1] * wy[1]}};
#pragma unroll
      for (int u = 0; u < 2; u++) {
        T wx[2];
        const int lx = prolong_axis<n1, N>(px + u, wx);
        T* p = sol + nat(N, px + u, py, pz);
        if (active) *p = *p + prolong_cell<n1>(lds + M::off_sol(1) + cnat(n1, lx, ly, lz), wzy, wx);
      }
    }
    __syncthreads();
    smooth(P.mg_npost);
    T sd = T(0), ss = T(0);
#pragma unroll
    for (int c = 0; c < 2; c++) {
      sd += fabs(m_dh2 * (nb(id[c]) - T(6) * sol[id[c]]) + rh[c]);
      ss += fabs(sol[id[c]]);
    }
    if (!active) sd = ss = T(0);
    block_sum2<THREADS / 16>(sd, ss, red);
    error = P.dh * P.dh * sd / ss;
    iter++;
  }
  if (t == 0) mg_report(iter, error, fell_back, iters, status, P);
  const int G = gra_nxt(P.gra_ghost), og = GS - P.gra_ghost;
  for (int q = t; q < G * G * G; q += THREADS) out[q] = sol[nat(N, q % G + og, q / G % G + og, q / (G * G) + og)];
  if (P.fuse_gravity && flu) {
    for (int q = t; q < kPatchCells; q += THREADS) {
      T f[kNComp];
#pragma unroll
      for (int v = 0; v < kNComp; v++) f[v] = flu[v * kPatchCells + q];
      gravity_cell(sol + nat(N, q % 8 + GS, q / 8 % 8 + GS, q / 64 + GS), N, N * N, f, flu, q, P);
    }
  }
}

// How a batch is run: mg_patch, or for a small batch at ghost sizes 1 and 2 mg_patch_cells (see mg_small), at ghost size 3
// mg_patch with twice the threads (see mg_wide).
enum MgForm { kMgBlocks, kMgCells, kMgWide };

template <int GS, MgForm F, typename T>
struct MgLaunch {
  static constexpr int THREADS = F == kMgCells ? mg_cell_threads(GS) : MgGeo<GS>::THREADS * (F == kMgWide ? 2 : 1);
  static constexpr int WAVES = F == kMgCells ? (sizeof(T) == 8 ? 2 : 6) : mg_waves(GS, sizeof(T));
  static constexpr size_t LDS = sizeof(T) * (MgGeo<GS>::FLOATS + (F == kMgCells ? MgGeo<GS>::N * MgGeo<GS>::N * MgGeo<GS>::N : 0));
};

template <int GS, MgForm F, typename PT, typename T>
__device__ __forceinline__ void mg_run(T* lds, const T* rho, const T* cpot, const T* guess, T* out, T* flu, int* iters, int* status,
                                       const PT& P) {
  if constexpr (F == kMgCells)
    mg_patch_cells<GS>(lds, rho, cpot, guess, out, flu, iters, status, P);
  else
    mg_patch<GS, MgLaunch<GS, F, T>::THREADS>(lds, rho, cpot, guess, out, flu, iters, status, P);
}

template <int GS, MgForm F, typename PT, typename L = MgLaunch<GS, F, typename PT::real>>
__global__ void __launch_bounds__(L::THREADS, L::WAVES) mg_uniform_kernel(UniformBatchT<typename PT::real> b, PT P) {
  using T = typename PT::real;
  extern __shared__ __align__(16) unsigned char mg_smem[];
  T* lds = reinterpret_cast<T*>(mg_smem);
  using M = MgGeo<GS>;
  constexpr int R3 = M::R * M::R * M::R, C3 = M::C * M::C * M::C;
  const int p = blockIdx.x;
  if (p >= b.npatch) return;
  const int G = gra_nxt(P.gra_ghost);
  constexpr int N3 = M::N * M::N * M::N;
  mg_run<GS, F>(lds, b.rho + (size_t)p * R3, b.cpot + (size_t)p * C3,
                b.guess ? b.guess + (size_t)p * (P.init_mode == 3 ? N3 : R3) : nullptr,
                b.pot_out + (size_t)p * G * G * G, b.flu ? b.flu + (size_t)p * kNComp * kPatchCells : nullptr,
                b.iters ? b.iters + p : nullptr, b.status ? b.status + p : nullptr, P);
}

size_t lds_bytes_mg(int gs) {
  switch (gs) {
    case 1: return sizeof(float) * MgGeo<1>::FLOATS;
    case 2: return sizeof(float) * MgGeo<2>::FLOATS;
    case 3: return sizeof(float) * MgGeo<3>::FLOATS;
    case 4: return sizeof(float) * MgGeo<4>::FLOATS;
    case 5: return sizeof(float) * MgGeo<5>::FLOATS;
  }
  return 0;
}

// Largest batch for mg_patch_cells.  Measured on MI355X, us per call (interpolated start, 3+3 smoothing), mg_patch /
// mg_patch_cells after 1, 2 and 3 V-cycles (mg_patch's set-up is the longer, its V-cycle the shorter in a full GPU): FP32 GS 1,
// 1025 patches 21.9/14.4 27.1/21.6 32.3/28.7, 1536: 24.4/17.8 29.7/26.5 35.4/34.6, 2048: 25.9/21.8 31.7/32.7 37.2/43.0; GS 2,
// 513: 16.8/14.7 22.6/24.3 28.6/33.5 (two workgroups per CU to 512).  FP64, which goes on to six V-cycles for 1e-10: GS 1, 513:
// 23.0/15.6 29.3/22.7 35.3/30.4, 768: 24.7/17.9 31.4/25.2 38.0/32.8, 1024: 26.6/25.9 33.0/36.9 39.2/47.9; GS 2, 257: 18.7/22.6
// 26.3/35.4 33.9/48.1 (one per CU to 256).
static bool mg_small(int gs, size_t word, int n) {
  if (gs == 1) return n <= (word == 8 ? 768 : 1536);
  return gs == 2 && n <= (word == 8 ? 256 : 512);
}

// Twice the threads for mg_patch at ghost size 3, one patch to a CU: the second half shares the interpolation, the window and
// the gravity update.  us per call with 128 / 256 threads, 1, 3 and 6 V-cycles: FP32, 8 patches 20.0/17.5 38.9/36.9 67.5/65.8,
// 256: 20.7/18.4 39.6/37.5 67.0/65.4, 320: 21.7/19.8 41.2/40.4 69.8/70.7; FP64, 8: 21.6/19.7 44.3/42.7 78.0/76.9, 256:
// 22.9/21.3 44.9/44.4 76.9/76.5, 320: 27.1/25.3 53.6/53.9 92.2/94.4.
static bool mg_wide(int gs, int n) { return gs == 3 && n <= 256; }

template <int GS, MgForm F, typename PT>
static hipError_t launch_mg_as(const UniformBatchT<typename PT::real>& b, const PT& p, hipStream_t s) {
  using L = MgLaunch<GS, F, typename PT::real>;
  if (L::LDS > 64 * 1024)   // the FP64 levels of the larger cubes exceed the default dynamic LDS limit
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&mg_uniform_kernel<GS, F, PT>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)L::LDS);
  hipLaunchKernelGGL((mg_uniform_kernel<GS, F, PT>), dim3(b.npatch), dim3(L::THREADS), L::LDS, s, b, p);
  return hipGetLastError();
}

template <int GS, typename PT>
static hipError_t launch_mg(const UniformBatchT<typename PT::real>& b, const PT& p, hipStream_t s) {
  if constexpr (GS <= 2) {
    if (mg_small(GS, sizeof(typename PT::real), b.npatch)) return launch_mg_as<GS, kMgCells>(b, p, s);
  }
  if constexpr (GS == 3) {
    if (mg_wide(GS, b.npatch)) return launch_mg_as<GS, kMgWide>(b, p, s);
  }
  return launch_mg_as<GS, kMgBlocks>(b, p, s);
}

// Persistent MG kernel of a mixed batch: each workgroup pulls one patch at a time from the queue.
__global__ void __launch_bounds__(kMgMaxThreads) mg_persistent_kernel(MixedBatch b, ParamsByGs P) {
  extern __shared__ float lds[];
  __shared__ int s_task;
  for (;;) {
    if (threadIdx.x == 0) s_task = (int)atomicAdd(b.counter, 1u);
    __syncthreads();
    const int t = s_task;
    __syncthreads();
    if (t >= b.ntasks) break;
    const Task tk = b.tasks[t];
    const int patch = b.perm[tk.first];
    if (patch < 0 || patch >= b.npatch || tk.gs < 1 || tk.gs > kMaxGhost) continue;  // malformed plan: skip
    const PatchDesc d = b.desc[patch];
    const SolveParams& Q = P.p[tk.gs];
    const int G = gra_nxt(Q.gra_ghost);
    const float* rho = b.rho + d.rho_off;
    const float* cpot = b.cpot + d.cpot_off;
    const float* guess = b.guess ? b.guess + d.rho_off : nullptr;
    float* out = b.pot_out + (size_t)patch * G * G * G;
    float* flu = b.flu ? b.flu + (size_t)patch * kNComp * kPatchCells : nullptr;
    int* it = b.iters ? b.iters + patch : nullptr;
    int* st = b.status ? b.status + patch : nullptr;
    switch (tk.gs) {
      case 1: mg_patch<1, kMgMaxThreads>(lds, rho, cpot, guess, out, flu, it, st, Q); break;
      case 2: mg_patch<2, kMgMaxThreads>(lds, rho, cpot, guess, out, flu, it, st, Q); break;
      case 3: mg_patch<3, kMgMaxThreads>(lds, rho, cpot, guess, out, flu, it, st, Q); break;
      case 4: mg_patch<4, kMgMaxThreads>(lds, rho, cpot, guess, out, flu, it, st, Q); break;
      default: mg_patch<5, kMgMaxThreads>(lds, rho, cpot, guess, out, flu, it, st, Q); break;
    }
  }
}

// The MG tasks [first, first + gridDim.x) of one ghost size, one patch per workgroup (no task loop: the
// patch solve compiles as in the uniform kernel, without the persistent kernel's spills).
template <int GS, MgForm F, typename L = MgLaunch<GS, F, float>>
__global__ void __launch_bounds__(L::THREADS, L::WAVES) mg_tasks_kernel(MixedBatch b, int first, SolveParams Q) {
  extern __shared__ float lds[];
  const Task tk = b.tasks[first + blockIdx.x];
  const int patch = b.perm[tk.first];
  if (patch < 0 || patch >= b.npatch || tk.gs != GS) return;   // malformed plan: skip (uniform per workgroup)
  const PatchDesc d = b.desc[patch];
  const int G = gra_nxt(Q.gra_ghost);
  mg_run<GS, F>(lds, b.rho + d.rho_off, b.cpot + d.cpot_off, b.guess ? b.guess + d.rho_off : nullptr,
                b.pot_out + (size_t)patch * G * G * G, b.flu ? b.flu + (size_t)patch * kNComp * kPatchCells : nullptr,
                b.iters ? b.iters + patch : nullptr, b.status ? b.status + patch : nullptr, Q);
}

template <int GS, MgForm F>
static void launch_mg_tasks_form(const MixedBatch& b, const SolveParams& p, int first, int count, hipStream_t s) {
  using L = MgLaunch<GS, F, float>;
  hipLaunchKernelGGL((mg_tasks_kernel<GS, F>), dim3(count), dim3(L::THREADS), L::LDS, s, b, first, p);
}

template <int GS>
static void launch_mg_tasks_as(const MixedBatch& b, const SolveParams& p, int first, int count, hipStream_t s) {
  if constexpr (GS <= 2) {
    if (mg_small(GS, sizeof(float), count)) return launch_mg_tasks_form<GS, kMgCells>(b, p, first, count, s);
  }
  if constexpr (GS == 3) {
    if (mg_wide(GS, count)) return launch_mg_tasks_form<GS, kMgWide>(b, p, first, count, s);
  }
  launch_mg_tasks_form<GS, kMgBlocks>(b, p, first, count, s);
}

hipError_t launch_mg_tasks(const MixedBatch& b, const SolveParams& p, int gs, int first, int count, hipStream_t s) {
  if (count <= 0) return hipSuccess;
  switch (gs) {
    case 1: launch_mg_tasks_as<1>(b, p, first, count, s); break;
    case 2: launch_mg_tasks_as<2>(b, p, first, count, s); break;
    case 3: launch_mg_tasks_as<3>(b, p, first, count, s); break;
    case 4: launch_mg_tasks_as<4>(b, p, first, count, s); break;
    case 5: launch_mg_tasks_as<5>(b, p, first, count, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

int mg_persistent_blocks_per_cu(size_t lds) {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void*>(&mg_persistent_kernel),
                                                   kMgMaxThreads, lds) != hipSuccess)
    return 0;
  return n;
}

hipError_t launch_mg_persistent(const MixedBatch& b, const ParamsByGs& p, int grid, size_t lds, hipStream_t s) {
  if (b.ntasks <= 0) return hipSuccess;
  hipLaunchKernelGGL(mg_persistent_kernel, dim3(grid), dim3(kMgMaxThreads), lds, s, b, p);
  return hipGetLastError();
}

hipError_t launch_mg_uniform(const UniformBatch& b, const SolveParams& p, hipStream_t s) {
  switch (b.gs) {
    case 1: return launch_mg<1>(b, p, s);
    case 2: return launch_mg<2>(b, p, s);
    case 3: return launch_mg<3>(b, p, s);
    case 4: return launch_mg<4>(b, p, s);
    case 5: return launch_mg<5>(b, p, s);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_mg_uniform64(const UniformBatch64& b, const SolveParams64& p, hipStream_t s) {
  switch (b.gs) {
    case 1: return launch_mg<1>(b, p, s);
    case 2: return launch_mg<2>(b, p, s);
    case 3: return launch_mg<3>(b, p, s);
    case 4: return launch_mg<4>(b, p, s);
    case 5: return launch_mg<5>(b, p, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace pgamd
