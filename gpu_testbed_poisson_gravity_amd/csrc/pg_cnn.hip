// Learned warm start: a small 3D CNN that predicts the correction from the interpolated coarse potential
// to the converged potential on the whole solve interior, trained on solutions of the solver itself.
// No reference counterpart (the reference always starts from the interpolated cube).
//
// Network (activations BF16 channel-last, weights BF16, accumulation and master weights FP32):
//   frame   the 18^3 solve cube of ghost size 5 (smaller cubes centred, zeros around), with the fields
//           q0 = interp/s and q1 = 64 r/s on the solve interior and zero elsewhere, s = max|interp| over the
//           solve cube, r the SOR residual of the interpolated cube (reference operand order), i.e. the
//           right-hand side of A e = r that the correction e to the interpolated start satisfies (e has zero
//           Dirichlet values, so the boundary enters through r alone)
//   x0      [n][10^3][16]: space-to-depth of the zero-extended 20^3 frame (fine index f = 2c - 1 + d per
//           axis, channel ((dz*2+dy)*2+dx)*2 + q), so that coarse voxels 1..8 hold the 2^3 blocks of the
//           16^3 interior and the voxels with a coordinate 0 or 9 are zero (the first layer's padding)
//   y1      relu(conv3(x0) + b1)                        10^3 -> 8^3, 16 channels
//   yl      y_{l-1} + relu(conv3(pad(y_{l-1})) + bl)    l = 2..5, 8^3 (residual blocks, zero padding)
//   D       conv3(pad(y5)) + b6                         8^3, 8 channels = the 2^3 sub-cells (linear)
//   guess   interp + s * D[o][p] at interior frame index 2o + p (depth-to-space)
// Activations are stored padded (10^3 with a zero border) so that every layer is the same valid 3^3
// convolution: 10^3 x 16 channels in, 8^3 x 16 channels out, K = 27 taps x 16 channels = 432.
//
// Convolutions are implicit GEMMs on the gfx950 matrix cores (v_mfma_f32_16x16x32_bf16): the weights are
// the A operand (rows = 16 output channels), the activations the B operand (columns = 16 output voxels of a
// tile), K made of (tap, channel) pairs so that each lane's 8 consecutive K values are 8 channels of one input
// voxel (one 16-byte LDS read).  MFMA lane layout (16x16x32): A[i][k] with i = lane%16, k = 8*(lane/16)+0..7;
// B[k][j] with j = lane%16, k = 8*(lane/16)+0..7; D[i][j] with j = lane%16, i = 4*(lane/16)+0..3.  So a lane
// loads the channels of voxel lane%16 and receives output channels 4*(lane/16)..+3 of that same voxel: the
// epilogue reads and writes 4 consecutive channels (8 bytes) at once.
// Forward K order: 15 steps c = dz*5 + s; step c covers the in-plane positions 2s and 2s+1 (position
// dy*3 + dx, 16 channels each) of tap plane dz; position 9 is a pad with zero weights whose A operand
// repeats position 8.  Grouping the steps by dz lets the fused kernel read an input plane once and feed it
// to the three output planes that use it.  The input gradient is the same convolution with the taps reversed.

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "pg_cnn.h"
#include "pg_geometry.h"
#include "pg_interp.h"
#include "pg_kernels.h"

#pragma clang fp contract(off)

namespace pgamd {
namespace cnn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef uint16_t u16;

__device__ __forceinline__ float bf2f(u16 v) { return __uint_as_float(((uint32_t)v) << 16); }
// round to nearest even (one v_cvt_pk_bf16_f32 on gfx950); every kernel here uses this one conversion
__device__ __forceinline__ u16 f2bf(float f) { return __builtin_bit_cast(u16, (__bf16)f); }

// Two floats as two BF16 values in one word (the first one low): one two-source v_cvt_pk_bf16_f32, the same
// rounding as f2bf.
__device__ __forceinline__ uint32_t pack2_bf16(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2){a, b}, bf16x2));
}
// Four floats as four BF16 values (8 bytes, the first one lowest).
__device__ __forceinline__ uint2 pack4_bf16(float a, float b, float c, float d) {
  return make_uint2(pack2_bf16(a, b), pack2_bf16(c, d));
}
__device__ __forceinline__ float bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

union Pack8 {
  bf16x8 v;
  uint4 u;
  u16 h[8];
};

constexpr int kThreads = 256;
constexpr int S = kCnnPadded;   // 10: padded input edge
constexpr int So = kCnnEdge;    // 8: output edge
constexpr int CH = 16;          // channels
constexpr int K = 27 * CH;      // 432
constexpr int KZ = 15;          // forward K steps: 3 dz x 5 position pairs
constexpr int KF = KZ * 32;     // 480 = kCnnKF
static_assert(KF == kCnnKF, "forward weight layout");
constexpr int kTZ = 2;          // output z-planes per workgroup
constexpr int kSlabs = So / kTZ;
constexpr int kPlane = S * S * CH;  // bf16 values per padded plane

// Step c of this lane's A operand from the lane-major copy WL of one layer ([15][64][8]).
__device__ __forceinline__ bf16x8 load_weight_step(const u16* __restrict__ WL, int c) {
  Pack8 p;
  p.u = *reinterpret_cast<const uint4*>(WL + ((size_t)c * 64 + (threadIdx.x & 63)) * 8);
  return p.v;
}

// B operand of the forward layout (row j = lane%16 of [16][480]) for the 15 steps.
__device__ __forceinline__ void load_weights_fwd(const u16* __restrict__ W, bf16x8 (&wreg)[KZ]) {
  const int j = threadIdx.x & 15, kq = 8 * ((threadIdx.x & 63) >> 4);
#pragma unroll
  for (int c = 0; c < KZ; c++) {
    Pack8 p;
    p.u = *reinterpret_cast<const uint4*>(W + j * KF + c * 32 + kq);
    wreg[c] = p.v;
  }
}

// Activation buffers in LDS (the fused kernels): planes of [half][10 x 10 voxels][8 channels] BF16, the halves kHalfV
// values apart.  A 16-byte read serves 16 lanes per cycle from 64 banks: lanes 0-3, 12-15 and 20-27 of each half wave, then
// the others (measured; 16 consecutive lanes do not share a cycle).  So a tile of 16 voxels is rows r and r + 4 (640 bytes
// apart) with lane j at x = tile_x(j), and the halves lie 1664 bytes apart: half a wave's lanes 0-3, 12-15 (half 0) and
// 20-27 (half 1) then read 16 different bank quads.  With halves of 1600 bytes and x = j % 8 each read took 8 cycles or
// more in place of 4.
constexpr int kHalfV = S * S * 8 + 32;
constexpr int kPlaneV = 2 * kHalfV;   // per plane
__device__ __forceinline__ int tile_x(int j) { return (j & 7) ^ ((j & 8) >> 1); }
__device__ __forceinline__ int tile_dy(int j) { return (j & 8) >> 1; }   // 0 or 4

// In-plane position (dy*3 + dx) and channel half read by lane group g = lane/16 at position pair s.
__device__ __forceinline__ int fwd_pos(int s, int g) { return min(2 * s + (g >> 1), 8); }

// ---- forward convolution ------------------------------------------------------------------------------
// MODE 0: y = relu(h) (layer 1);  MODE 1: y = x_centre + relu(h) (layers 2-5), both written into the
// interior of a padded [n][10^3][16] BF16 buffer whose border stays zero;  MODE 2: D = h for the first 8 channels,
// FP32 [n][8^3][8] (output layer).  One workgroup: kTZ output planes of one sample.
template <int MODE>
__global__ void __launch_bounds__(kThreads) conv_fwd_kernel(const u16* __restrict__ X, const u16* __restrict__ W,
                                                            const float* __restrict__ bias, u16* __restrict__ Y,
                                                            float* __restrict__ D) {
  __shared__ uint4 smem[(kTZ + 2) * kPlane / 8];
  const u16* xs = reinterpret_cast<const u16*>(smem);
  const int n = blockIdx.x / kSlabs, z0 = (blockIdx.x % kSlabs) * kTZ;
  const uint4* src = reinterpret_cast<const uint4*>(X + ((size_t)n * S + z0) * kPlane);
  for (int i = threadIdx.x; i < (kTZ + 2) * kPlane / 8; i += kThreads) smem[i] = src[i];
  bf16x8 wreg[KZ];
  load_weights_fwd(W, wreg);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, co0 = 4 * g;   // this lane's output channels co0..co0+3
  const float4 b4 = *reinterpret_cast<const float4*>(bias + co0);
  __syncthreads();
  constexpr int M = kTZ * So * So;   // 128 output voxels: 8 tiles, 2 per wave
  for (int t = wave; t < M / 16; t += kThreads / 64) {
    const int v = t * 16 + (lane & 15);   // this lane's voxel: its B-operand column and its D column
    const int lz = v / (So * So), oy = (v / So) % So, ox = v % So;
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < KZ; c++) {
      const int dz = c / 5, pos = fwd_pos(c % 5, g), dy = pos / 3, dx = pos % 3;
      Pack8 a;
      a.u = *reinterpret_cast<const uint4*>(xs + (((lz + dz) * S + oy + dy) * S + ox + dx) * CH + 8 * (g & 1));
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wreg[c], a.v, acc, 0, 0, 0);
    }
    const float h0 = acc[0] + b4.x, h1 = acc[1] + b4.y, h2 = acc[2] + b4.z, h3 = acc[3] + b4.w;
    const size_t o = (((size_t)n * So + z0 + lz) * So + oy) * So + ox;  // voxel in the 8^3 output
    if (MODE == 2) {
      if (co0 < kCnnOut) *reinterpret_cast<float4*>(D + o * kCnnOut + co0) = make_float4(h0, h1, h2, h3);
    } else {
      float o0 = fmaxf(h0, 0.0f), o1 = fmaxf(h1, 0.0f), o2 = fmaxf(h2, 0.0f), o3 = fmaxf(h3, 0.0f);
      if (MODE == 1) {
        const uint2 rx = *reinterpret_cast<const uint2*>(xs + (((lz + 1) * S + oy + 1) * S + ox + 1) * CH + co0);
        o0 += bf_lo(rx.x);
        o1 += bf_hi(rx.x);
        o2 += bf_lo(rx.y);
        o3 += bf_hi(rx.y);
      }
      *reinterpret_cast<uint2*>(Y + ((((size_t)n * S + z0 + lz + 1) * S + oy + 1) * S + ox + 1) * CH + co0) =
          pack4_bf16(o0, o1, o2, o3);
    }
  }
}

// ---- training pass -----------------------------------------------------------------------------------------

// Forward, loss and the gradients of every layer's output, one workgroup (16 waves) per sample: activations and output
// gradients pass from layer to layer through two LDS buffers, each lane's own gradients and ReLU masks stay in its
// registers, and memory only sees what weight_grad_kernel reads (y1..y5 and dH of every layer).
//
// The input gradient of a layer is the same padded convolution of dH with the weights transposed and its taps reversed,
// so one routine serves both directions: weights are the A operand, and a lane has channels 4*(lane/16)..+3 of voxel
// lane%16 of its wave's tiles.  A wave owns kTiles tiles one above the other in z (y rows r and r + 4) and walks the
// kTiles + 2 input planes they need: 20 operand reads for 30 products, in the K order of conv_fwd_kernel.
//
// Buffers: ten planes with a zero border but for the packed input, whose border is the caller's.
//
// Loss: e = D - T, mean(e^2), and with res_weight the residual r = stencil(e) that the error leaves in the guess on the
// 16^3 frame (fine cell 2o + p of output voxel o, sub-cell p): dY = 2 e / count + res_weight * 2 / count * stencil(r) (the
// stencil is symmetric with the zero exterior).  One partial sum per workgroup.
//
// Bound by the chain of twelve short phases: with one sample per CU the LDS unit, the matrix cores and the VALU are each
// busy for about a quarter of it; a third of the time is the launch and the 57 MB to and from memory.  MI355X, 256
// samples: 35 us (512 threads 35.5 us; each wave loading its own weights 37 us with 512 threads and 43 us with 1024; with
// the two-way conflicts of unpadded halves 44 us); 247 us as 19 launches (a layer each, the ReLU masks, the two terms of
// the loss) that passed gradients and pre-activations through memory.
constexpr int kTrainThreads = 1024;
constexpr int kTiles = kCnnVox / 16 / (kTrainThreads / 64);   // per wave
constexpr int kTBuf = S * kPlaneV;                   // u16 per buffer
// FP32 frame of the loss with a zero halo.  Eight rows are 16 modulo 32 and the plane pitch is odd: the cells that half a
// wave reads for its sub-cells (two y rows, two z planes, every other x) fall on 32 banks.
constexpr int kFY = 18, kFZ = 18 * kFY + 1, kFrame = 18 * kFZ;
struct TrainLds {
  u16 a[kTBuf], b[kTBuf];              // packed input, activations, dH
  u16 w[2][16 * KF];                   // weights of this layer and of the next, lane-major
  float e[kFrame + 2], r[kFrame + 2];
  float red[kTrainThreads / 64];
};
static_assert(sizeof(TrainLds) <= 160 * 1024 && sizeof(TrainLds) % 16 == 0, "one workgroup per CU");

struct TrainOut {
  u16* y[kCnnLayers];   // y[1..5]: layer outputs, padded [n][10^3][16]
  u16* dh;              // [6][n][8^3][16]
  float* loss;          // one partial per workgroup, host memory
};

// A value the compiler cannot see through: addresses derived from it are computed in each phase, not kept across them.
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// This lane's voxel of tile k is (z + k, y, x); its channels are co0..co0+3.
struct TrainLane {
  int z, y, x, co0;
  __device__ __forceinline__ TrainLane() {
    const int tid = opaque(threadIdx.x), wave = tid >> 6, lane = tid & 63;
    z = kTiles * (wave >> 2);
    y = (wave & 3) + tile_dy(lane);
    x = tile_x(lane);
    co0 = 4 * (lane >> 4);
  }
  // the four channels of tile k in a buffer (8 bytes)
  __device__ __forceinline__ u16* at(u16* buf, int k) const {
    return buf + (z + k + 1) * kPlaneV + (co0 >> 3) * kHalfV + ((y + 1) * S + x + 1) * 8 + (co0 & 7);
  }
  __device__ __forceinline__ int voxel(int k) const { return ((z + k) * So + y) * So + x; }
  __device__ __forceinline__ int padded(int k) const { return ((z + k + 1) * S + y + 1) * S + x + 1; }
};

// Barrier for what the buffers hand over: the stores to memory, which only the next kernel reads, stay in flight.
__device__ __forceinline__ void train_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A layer's weights: requested into registers one layer ahead, written to LDS when that layer ends, read by every wave.
// (Each wave loading its 15 KB from L2 through the L1 was a quarter of the kernel.)
constexpr int kWVec = 16 * KF / 8, kWFetch = (kWVec + kTrainThreads - 1) / kTrainThreads;
__device__ __forceinline__ void train_fetch(const u16* __restrict__ W, int l, uint4 (&f)[kWFetch]) {
#pragma unroll
  for (int j = 0; j < kWFetch; j++) {
    const int i = threadIdx.x + j * kTrainThreads;
    f[j] = i < kWVec ? reinterpret_cast<const uint4*>(W + (size_t)(l - 1) * 16 * KF)[i] : make_uint4(0, 0, 0, 0);
  }
}
__device__ __forceinline__ void train_put(u16* w, const uint4 (&f)[kWFetch]) {
#pragma unroll
  for (int j = 0; j < kWFetch; j++) {
    const int i = threadIdx.x + j * kTrainThreads;
    if (i < kWVec) reinterpret_cast<uint4*>(w)[i] = f[j];
  }
}

// Zero the border of the buffer that held the packed input.
__device__ __forceinline__ void train_zero_border(u16* buf) {
#pragma unroll 1
  for (int i = opaque(threadIdx.x); i < kCnnPadVox * 2; i += kTrainThreads) {
    const int vox = i >> 1, x = vox % S, y = vox / S % S, z = vox / (S * S);
    if (x == 0 || x == S - 1 || y == 0 || y == S - 1 || z == 0 || z == S - 1)
      *reinterpret_cast<uint4*>(buf + z * kPlaneV + (i & 1) * kHalfV + (y * S + x) * 8) = make_uint4(0, 0, 0, 0);
  }
}

__device__ __forceinline__ float4 train_bias(const float* __restrict__ P, int l) {
  return *reinterpret_cast<const float4*>(P + (size_t)(l - 1) * kCnnLayerParams + 16 * K + 4 * ((threadIdx.x & 63) >> 4));
}

__device__ __forceinline__ void train_conv(const u16* in, const u16* wl, floatx4 (&acc)[kTiles]) {
  bf16x8 w[KZ];
#pragma unroll
  for (int c = 0; c < KZ; c++) w[c] = load_weight_step(wl, c);
  const TrainLane t;
  const int g = t.co0 >> 2;
  const u16* base = in + t.z * kPlaneV + (g & 1) * kHalfV + (t.y * S + t.x) * 8;
#pragma unroll
  for (int k = 0; k < kTiles; k++) acc[k] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int p = 0; p < kTiles + 2; p++)
#pragma unroll
    for (int s = 0; s < 5; s++) {
      const int pos = fwd_pos(s, g);
      Pack8 a;
      a.u = *reinterpret_cast<const uint4*>(base + p * kPlaneV + ((pos / 3) * S + pos % 3) * 8);
#pragma unroll
      for (int k = 0; k < kTiles; k++)
        if (p >= k && p <= k + 2) acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[(p - k) * 5 + s], a.v, acc[k], 0, 0, 0);
    }
}

// Forward epilogue of layers 1..5: relu(h) (+ the layer's input) to the other buffer and to memory; returns the mask bits.
__device__ __forceinline__ uint32_t train_relu(u16* in, u16* out, bool res, const floatx4 (&acc)[kTiles],
                                               const float4& b, u16* __restrict__ Y) {
  const TrainLane t;
  uint32_t mask = 0;
#pragma unroll
  for (int k = 0; k < kTiles; k++) {
    const float h0 = acc[k][0] + b.x, h1 = acc[k][1] + b.y, h2 = acc[k][2] + b.z, h3 = acc[k][3] + b.w;
    const uint2 hb = pack4_bf16(h0, h1, h2, h3);   // the mask is that of the stored precision
    mask |= ((uint32_t)(bf_lo(hb.x) > 0.0f) | (uint32_t)(bf_hi(hb.x) > 0.0f) << 1 | (uint32_t)(bf_lo(hb.y) > 0.0f) << 2 |
             (uint32_t)(bf_hi(hb.y) > 0.0f) << 3)
            << (4 * k);
    float o0 = fmaxf(h0, 0.0f), o1 = fmaxf(h1, 0.0f), o2 = fmaxf(h2, 0.0f), o3 = fmaxf(h3, 0.0f);
    uint2 rx = *reinterpret_cast<const uint2*>(t.at(in, k));
    rx = res ? rx : make_uint2(0, 0);
    o0 += bf_lo(rx.x);
    o1 += bf_hi(rx.x);
    o2 += bf_lo(rx.y);
    o3 += bf_hi(rx.y);
    const uint2 ob = pack4_bf16(o0, o1, o2, o3);
    *reinterpret_cast<uint2*>(t.at(out, k)) = ob;
    *reinterpret_cast<uint2*>(Y + t.padded(k) * CH + t.co0) = ob;
  }
  return opaque(mask);   // kept as bits, not as the 16 values they come from
}

// 7-point stencil (six neighbours - 6 a) at a cell of a frame.
__device__ __forceinline__ float train_stencil(const float* a) {
  return (((((a[kFZ] + a[-kFZ]) + a[kFY]) + a[-kFY]) + a[1]) + a[-1]) - 6.0f * a[0];
}

// Loss of the sample's output h6 = acc + b; dY of the lane's four channels (zero for the dead ones).
__device__ __forceinline__ void train_loss(TrainLds& s, const floatx4 (&acc)[kTiles], const float4& b,
                                           const float* __restrict__ T, float inv, float kr, bool res, float& se, float& sr,
                                           float (&dy)[kTiles][4]) {
  const TrainLane t;
  const bool live = t.co0 < kCnnOut;   // sub-cells of z parity co0 / 4
  const int f0 = (2 * t.z + (t.co0 >> 2 & 1) + 1) * kFZ + (2 * t.y + 1) * kFY + 2 * t.x + 1;
#pragma unroll
  for (int k = 0; k < kTiles; k++)
#pragma unroll
    for (int c = 0; c < 4; c++) dy[k][c] = 0.0f;
  if (live) {
#pragma unroll
    for (int k = 0; k < kTiles; k++) {
      const float* tv = T + t.voxel(k) * kCnnOut + t.co0;   // any alignment
      const float d[4] = {(acc[k][0] + b.x) - tv[0], (acc[k][1] + b.y) - tv[1], (acc[k][2] + b.z) - tv[2], (acc[k][3] + b.w) - tv[3]};
      float* ef = s.e + f0 + 2 * k * kFZ;
#pragma unroll
      for (int c = 0; c < 4; c++) {
        se += d[c] * d[c];
        dy[k][c] = d[c] * inv;
        ef[(c >> 1) * kFY + (c & 1)] = d[c];
      }
    }
  }
  train_barrier();
  if (!res) return;
  constexpr int kPlanes = kTrainThreads / 256;   // per pass
  const int q = opaque(threadIdx.x), fr = ((q >> 8) + 1) * kFZ + ((q >> 4 & 15) + 1) * kFY + (q & 15) + 1;
#pragma unroll
  for (int j = 0; j < 16 / kPlanes; j++) {
    const int f = fr + kPlanes * j * kFZ;
    const float v = train_stencil(s.e + f);
    s.r[f] = v;
    sr += v * v;
  }
  train_barrier();
  if (live) {
#pragma unroll
    for (int k = 0; k < kTiles; k++)
#pragma unroll
      for (int c = 0; c < 4; c++) dy[k][c] += kr * train_stencil(s.r + f0 + 2 * k * kFZ + (c >> 1) * kFY + (c & 1));
  }
}

// dH of a layer from dY and its mask bits, to a buffer and to memory.
__device__ __forceinline__ void train_mask(const float (&dy)[kTiles][4], uint32_t mask, u16* out,
                                           u16* __restrict__ dH) {
  const TrainLane t;
#pragma unroll
  for (int k = 0; k < kTiles; k++) {
    const uint32_t m = mask >> (4 * k);
    const uint2 v = pack4_bf16(m & 1 ? dy[k][0] : 0.0f, m & 2 ? dy[k][1] : 0.0f, m & 4 ? dy[k][2] : 0.0f, m & 8 ? dy[k][3] : 0.0f);
    *reinterpret_cast<uint2*>(t.at(out, k)) = v;
    *reinterpret_cast<uint2*>(dH + t.voxel(k) * CH + t.co0) = v;
  }
}

__global__ void __launch_bounds__(kTrainThreads, kTrainThreads / 256) train_pass_kernel(const u16* __restrict__ X0, const u16* __restrict__ WL,
                                                                      const u16* __restrict__ WT, const float* __restrict__ P,
                                                                      const float* __restrict__ T, int n, float res_weight,
                                                                      TrainOut out) {
  __shared__ __align__(16) TrainLds lds;
  const float inv = 2.0f / ((float)(n * kCnnVox) * kCnnOut), kr = res_weight * (2.0f / ((float)n * kCnnOutputs));
  float se = 0.0f, sr = 0.0f;
  for (int i = threadIdx.x; i < (int)(sizeof(TrainLds) / 16); i += kTrainThreads)
    reinterpret_cast<uint4*>(&lds)[i] = make_uint4(0, 0, 0, 0);
  train_barrier();
  for (int smp = blockIdx.x; smp < n; smp += gridDim.x) {
    floatx4 acc[kTiles];
    uint32_t mask1 = 0;   // ReLU masks: layer 1, and 16 bits each of layers 2..5 (5 lowest)
    uint64_t masks = 0;
    float dy[kTiles][4];
    uint4 f[kWFetch];
    train_fetch(WL, 1, f);
    const uint4* src = reinterpret_cast<const uint4*>(X0 + (size_t)smp * kCnnInput);
    for (int i = opaque(threadIdx.x); i < kCnnPadVox * 2; i += kTrainThreads) {
      const int vox = i >> 1;
      *reinterpret_cast<uint4*>(lds.a + vox / (S * S) * kPlaneV + (i & 1) * kHalfV + vox % (S * S) * 8) = src[i];
    }
    train_put(lds.w[1], f);
    train_barrier();
    // A layer reads one buffer and one weight buffer and writes the others; what is rewritten was last read before the
    // barrier that ended the layer before.  Forward layer l has weights l & 1, backward layer l those of the other parity.
    // The loops over layers stay rolled: a workgroup has one sample or few, and runs from a cold instruction cache.
#pragma unroll 1
    for (int l = 1; l < kCnnLayers; l++) {
      u16 *in = l & 1 ? lds.a : lds.b, *o = l & 1 ? lds.b : lds.a;
      const float4 b = train_bias(P, l);
      train_fetch(WL, l + 1, f);
      train_conv(in, lds.w[l & 1], acc);
      if (l == 2) train_zero_border(lds.a);   // of the packed input
      const uint32_t m = train_relu(in, o, l > 1, acc, b, out.y[l] + (size_t)smp * kCnnInput);
      if (l == 1)
        mask1 = m;
      else
        masks = masks << 16 | m;
      train_put(lds.w[l + 1 & 1], f);
      train_barrier();
    }
    const float4 b6 = train_bias(P, kCnnLayers);
    train_fetch(WT, kCnnLayers, f);
    train_conv(lds.b, lds.w[0], acc);
    train_put(lds.w[1], f);
    train_loss(lds, acc, b6, T + (size_t)smp * kCnnOutputs, inv, kr, res_weight > 0.0f, se, sr, dy);
    const size_t layer = (size_t)n * kCnnVox * CH;
    u16* dh = out.dh + (size_t)smp * kCnnVox * CH + (kCnnLayers - 1) * layer;
    train_mask(dy, 0xffffu, lds.b, dh);
    train_barrier();
#pragma unroll
    for (int k = 0; k < kTiles; k++)
#pragma unroll
      for (int c = 0; c < 4; c++) dy[k][c] = 0.0f;   // layer 6 has no residual path
#pragma unroll 1
    for (int l = kCnnLayers; l > 1; l--) {
      u16 *in = l & 1 ? lds.a : lds.b, *o = l & 1 ? lds.b : lds.a;
      if (l > 2) train_fetch(WT, l - 1, f);
      train_conv(in, lds.w[l + 1 & 1], acc);
#pragma unroll
      for (int k = 0; k < kTiles; k++)
#pragma unroll
        for (int c = 0; c < 4; c++) dy[k][c] += acc[k][c];
      dh -= layer;
      train_mask(dy, l > 2 ? (uint32_t)masks : mask1, o, dh);
      masks >>= 16;
      if (l > 2) train_put(lds.w[l & 1], f);
      train_barrier();
    }
  }
  float s = se + res_weight * sr;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if ((threadIdx.x & 63) == 0) lds.red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    float sum = lds.red[0];
    for (int i = 1; i < kTrainThreads / 64; i++) sum += lds.red[i];
    __hip_atomic_store(out.loss + blockIdx.x, sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Weight and bias gradients of all six layers, one launch: dW[co][tap*16+ci] = sum_{n,v} dH[n][v][co] X[n][v+tap][ci]
// and db[co] = sum_{n,v} dH[n][v][co].  Block (b, l) sums the samples b, b + gridDim.x, ... of layer l + 1 in its
// accumulators and writes one partial in the parameter layout of a layer (W [16][432], b [16]).
//
// GEMM with rows co, columns ci and K = voxels, one 16x16 tile per tap.  Both operands need 8 consecutive voxels of
// one channel per lane, so a sample is staged transposed, [z][y][channel][8 x] (row pitch 272 B: the transposing
// writes of 8 rows then fall on different banks, and a wave's operand read is four contiguous 256 B pieces).  A tap's
// x shift is applied to the dH row in registers (voxels shifted out of the row meet the zero x border of X), so one
// X operand serves three taps: per 32 voxels a wave reads 4 operands for its 9 tiles (wave = dz).  A tenth tile with
// a column of ones is the bias gradient.
// Layer 1's input may hold any values in its border (the caller's array): its y and z border rows are staged like the
// others and the two x border columns are added by two extra K steps gathered from memory.
// Bound by staging (LDS writes, L2 reads).  MI355X, 256 samples: 12.2 us per layer and, with one partial per half
// sample summed by a serial loop, 1.06 ms per layer for the sums; now see grad_reduce_kernel.
constexpr int kWThreads = 192;     // three waves, one per dz
constexpr int kTRow = 136;         // u16 per staged row: 16 channels x 8 voxels and 8 of padding
constexpr int kXRows = S * S, kHRows = So * So;

// Two voxels' 8 channels (h: channel half) into a staged row, as (voxel, voxel + 1) pairs per channel.
__device__ __forceinline__ void stage_pair(u16* row, int xp, int h, const uint4& v0, const uint4& v1) {
  const uint32_t a[4] = {v0.x, v0.y, v0.z, v0.w}, b[4] = {v1.x, v1.y, v1.z, v1.w};
  uint32_t* d = reinterpret_cast<uint32_t*>(row + 64 * h) + xp;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    d[8 * j] = (a[j] & 0xffffu) | (b[j] << 16);
    d[8 * j + 4] = (a[j] >> 16) | (b[j] & 0xffff0000u);
  }
}

struct GradInputs {
  const u16* x[kCnnLayers];   // input of each layer, padded [n][10^3][16]
};

template <bool BORDER>
__device__ __forceinline__ void weight_grad_block(const u16* __restrict__ X, const u16* __restrict__ dH, int n,
                                                  float* __restrict__ out, u16* xs, u16* hs) {
  const int lane = threadIdx.x & 63, dz = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
  if (!BORDER)   // the zero y and z border of the activations
    for (int i = threadIdx.x; i < kXRows * kTRow / 8; i += kWThreads) {
      const int r = i / (kTRow / 8), y = r % S, z = r / S;
      if (y == 0 || y == S - 1 || z == 0 || z == S - 1) reinterpret_cast<uint4*>(xs)[i] = make_uint4(0, 0, 0, 0);
    }
  floatx4 acc[9], accb = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < 9; t++) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  Pack8 one;
  one.u = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);
  for (int smp = blockIdx.x; smp < n; smp += gridDim.x) {
    const uint4* xg = reinterpret_cast<const uint4*>(X + (size_t)smp * kCnnInput);
    const uint4* hg = reinterpret_cast<const uint4*>(dH + (size_t)smp * kCnnVox * CH);
    constexpr int XR = BORDER ? kXRows : kHRows;
    for (int i = threadIdx.x; i < XR * 8; i += kWThreads) {
      const int r = i >> 3, xp = i & 3, h = (i >> 2) & 1;
      const int z = BORDER ? r / S : r / So + 1, y = BORDER ? r % S : r % So + 1;
      const uint4* s = xg + ((z * S + y) * S + 2 * xp + 1) * 2 + h;
      stage_pair(xs + (z * S + y) * kTRow, xp, h, s[0], s[2]);
    }
    for (int i = threadIdx.x; i < kHRows * 8; i += kWThreads) {
      const int r = i >> 3, xp = i & 3, h = (i >> 2) & 1;
      const uint4* s = hg + (r * So + 2 * xp) * 2 + h;
      stage_pair(hs + r * kTRow, xp, h, s[0], s[2]);
    }
    __syncthreads();
#pragma unroll 2
    for (int ks = 0; ks < kHRows / 4; ks++) {
      const int z = ks >> 1, y = 4 * (ks & 1) + g;
      Pack8 a[3], b;
      a[1].u = *reinterpret_cast<const uint4*>(hs + (z * So + y) * kTRow + 8 * c);
      const uint4 d = a[1].u;
      const uint32_t s01 = __builtin_amdgcn_alignbit(d.y, d.x, 16), s12 = __builtin_amdgcn_alignbit(d.z, d.y, 16),
                     s23 = __builtin_amdgcn_alignbit(d.w, d.z, 16);
      a[0].u = make_uint4(s01, s12, s23, d.w >> 16);   // dx = 0: input voxel x meets output voxel x + 1
      a[2].u = make_uint4(d.x << 16, s01, s12, s23);   // dx = 2: output voxel x - 1
#pragma unroll
      for (int dy = 0; dy < 3; dy++) {
        b.u = *reinterpret_cast<const uint4*>(xs + ((z + dz) * S + y + dy) * kTRow + 8 * c);
#pragma unroll
        for (int dx = 0; dx < 3; dx++)
          acc[3 * dy + dx] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[dx].v, b.v, acc[3 * dy + dx], 0, 0, 0);
      }
      if (dz == 0) accb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1].v, one.v, accb, 0, 0, 0);
    }
    if (BORDER) {   // x = 0 meets output voxel 0 at dx = 0, x = 9 output voxel 7 at dx = 2; K = 32 (z, y) rows
      const u16* xb = X + (size_t)smp * kCnnInput;
      for (int ks = 0; ks < 2; ks++)
#pragma unroll
        for (int side = 0; side < 2; side++) {
          const int z = 4 * ks + g;
          Pack8 a, b;
#pragma unroll
          for (int e = 0; e < 8; e++) a.h[e] = hs[(z * So + e) * kTRow + 8 * c + 7 * side];
#pragma unroll
          for (int dy = 0; dy < 3; dy++) {
#pragma unroll
            for (int e = 0; e < 8; e++) b.h[e] = xb[(((z + dz) * S + e + dy) * S + 9 * side) * CH + c];
            acc[3 * dy + 2 * side] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, acc[3 * dy + 2 * side], 0, 0, 0);
          }
        }
    }
    __syncthreads();
  }
  // D[i = co][j = ci]: lane holds ci = lane%16, co = 4*(lane/16) + r
#pragma unroll
  for (int t = 0; t < 9; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) out[(4 * g + r) * K + (9 * dz + t) * CH + c] = acc[t][r];
  if (dz == 0 && c == 0) {
#pragma unroll
    for (int r = 0; r < 4; r++) out[CH * K + 4 * g + r] = accb[r];
  }
}

__global__ void __launch_bounds__(kWThreads) weight_grad_kernel(GradInputs in, const u16* __restrict__ dH, int n,
                                                                float* __restrict__ part) {
  __shared__ __align__(16) u16 xs[kXRows * kTRow];
  __shared__ __align__(16) u16 hs[kHRows * kTRow];
  const int l = blockIdx.y;
  const u16* h = dH + (size_t)l * n * kCnnVox * CH;
  float* out = part + ((size_t)l * gridDim.x + blockIdx.x) * kCnnLayerParams;
  if (l == 0)
    weight_grad_block<true>(in.x[0], h, n, out, xs, hs);
  else
    weight_grad_block<false>(in.x[l], h, n, out, xs, hs);
}

// Sum of the partials of every layer ([6][parts][kCnnLayerParams]) into the gradient vector, in a fixed order: 16
// threads per column, each over every 16th partial, then a tree.  Reads at most 6 * 128 partials (21 MB); one wave of
// serial loops over 1024 (weights) and 4096 (biases) partials took 4.7 of the 5.15 ms of a 256-sample step.
constexpr int kRCols = 16, kRGroups = 16;
__global__ void __launch_bounds__(kRCols * kRGroups) grad_reduce_kernel(const float* __restrict__ part, int parts,
                                                                        float* __restrict__ g) {
  __shared__ float red[kRGroups][kRCols];
  const int c = threadIdx.x % kRCols, q = threadIdx.x / kRCols;
  const int col = blockIdx.x * kRCols + c, l = col / kCnnLayerParams;
  static_assert(kCnnLayerParams % kRCols == 0, "whole blocks per layer");
  const float* p = part + (size_t)l * parts * kCnnLayerParams + col % kCnnLayerParams;
  float s = 0.0f;
#pragma unroll 4
  for (int i = q; i < parts; i += kRGroups) s += p[(size_t)i * kCnnLayerParams];
  red[q][c] = s;
  __syncthreads();
#pragma unroll
  for (int o = kRGroups / 2; o > 0; o >>= 1) {
    if (q < o) red[q][c] += red[q + o][c];
    __syncthreads();
  }
  if (q == 0) g[col] = red[0][c];
}

// Adam on the FP32 master weights.
__global__ void adam_kernel(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                            float* __restrict__ v, int n, float lr, float b1, float b2, float eps, float c1, float c2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// BF16 copies of the six weight matrices: the forward layout Wb[l][co][c*32 + kk] (step c = dz*5 + s,
// position 2s + kk/16, channel kk%16; zero at the pad position 9), the same values lane-major
// WL[l][c][lane][8] (lane = co + 16*(kk/8) reads kk%8 = 0..7 of its row: one contiguous 1 KB load per step),
// and lane-major WT: rows and channels exchanged, taps reversed (W[l][kk%16][26 - tap][row]), for the input gradient.
__global__ void weight_copies_kernel(const float* __restrict__ P, u16* __restrict__ Wb, u16* __restrict__ WT,
                                     u16* __restrict__ WL) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= kCnnLayers * 16 * KF) return;
  const int l = i / (16 * KF), r = i % (16 * KF);
  const int row = r / KF, k = r % KF, c = k / 32, kk = k % 32;
  const int dz = c / 5, pos = 2 * (c % 5) + (kk >> 4), tap = dz * 9 + pos, ch = kk & 15;
  const float* W = P + (size_t)l * kCnnLayerParams;
  const u16 v = pos < 9 ? f2bf(W[row * K + tap * CH + ch]) : (u16)0;
  const size_t lm = (((size_t)l * KZ + c) * 64 + row + 16 * (kk >> 3)) * 8 + (kk & 7);
  Wb[i] = v;
  WL[lm] = v;
  WT[lm] = pos < 9 ? f2bf(W[ch * K + (26 - tap) * CH + row]) : (u16)0;
}

// ---- input preparation and guess assembly -------------------------------------------------------------

constexpr float kResScale = 64.0f;   // q1 = kResScale * r / s

// SOR residual of the interpolated cube at interior cube cell (X, Y, Z) (1..R), reference operand order.
template <int N>
__device__ __forceinline__ float interp_residual(const float* cube, int X, int Y, int Z, float crho) {
  const float* c = cube + (Z * N + Y) * N + X;
  return c[N * N] + c[-N * N] + c[N] + c[-N] + c[1] + c[-1] - 6.0f * c[0] - crho;
}

// Interpolated solve cube of one patch into LDS (N^3 floats).
template <int GS>
__device__ void interp_cube(const float* __restrict__ cpot, int int_scheme, float* cube) {
  constexpr Geo g = geo_of(GS);
  constexpr int N = g.N, C = g.C, U = g.U, NC = C - 2;
  for (int q = threadIdx.x; q < NC * NC * NC; q += kThreads) {
    const int i = q % NC + 1, j = (q / NC) % NC + 1, k = q / (NC * NC) + 1;
    float v[3][3][3];
    for (int dk = 0; dk < 3; dk++)
      for (int dj = 0; dj < 3; dj++)
        for (int di = 0; di < 3; di++) v[dk][dj][di] = cpot[((k + dk - 1) * C + (j + dj - 1)) * C + (i + di - 1)];
    float ch[2][2][2];
    interp_children(v, int_scheme, ch);
    for (int cz = 0; cz < 2; cz++)
      for (int cy = 0; cy < 2; cy++)
        for (int cx = 0; cx < 2; cx++) {
          const int X = 2 * (i - 1) + cx - U, Y = 2 * (j - 1) + cy - U, Z = 2 * (k - 1) + cz - U;
          if (X >= 0 && X < N && Y >= 0 && Y < N && Z >= 0 && Z < N) cube[(Z * N + Y) * N + X] = ch[cz][cy][cx];
        }
  }
  __syncthreads();
}

// One workgroup per patch: interpolate, take s = max|interp|, write the packed input (zero outside the solve
// interior, so every voxel with a coordinate 0 or 9 is zero).
template <int GS>
__device__ void prep_patch(const float* __restrict__ rho, const float* __restrict__ cpot, float cst, int int_scheme,
                           u16* __restrict__ x, float* __restrict__ scale, float* cube) {
  constexpr Geo g = geo_of(GS);
  constexpr int N = g.N, R = g.R, OFF = 5 - GS;
  __shared__ float red[kThreads];
  interp_cube<GS>(cpot, int_scheme, cube);
  float mx = 0.0f;
  for (int t = threadIdx.x; t < N * N * N; t += kThreads) mx = fmaxf(mx, fabsf(cube[t]));
  red[threadIdx.x] = mx;
  __syncthreads();
  for (int o = kThreads / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + o]);
    __syncthreads();
  }
  const float s = red[0] > 0.0f ? red[0] : 1.0f;
  const float inv = 1.0f / s;
  if (threadIdx.x == 0) *scale = s;
  // one thread per (coarse voxel, sub-cell): 1000 x 8 items, 2 channels each
  for (int t = threadIdx.x; t < S * S * S * 8; t += kThreads) {
    const int vox = t >> 3, d = t & 7;
    const int cx = vox % S, cy = (vox / S) % S, cz = vox / (S * S);
    const int dz = d >> 2, dy = (d >> 1) & 1, dx = d & 1;
    // frame index f = 2c - 1 + d, cube index f - OFF
    const int X = 2 * cx - 1 + dx - OFF, Y = 2 * cy - 1 + dy - OFF, Z = 2 * cz - 1 + dz - OFF;
    float c0 = 0.0f, c1 = 0.0f;
    if (X >= 1 && X <= R && Y >= 1 && Y <= R && Z >= 1 && Z <= R) {   // the solve interior only
      c0 = cube[(Z * N + Y) * N + X] * inv;
      c1 = (interp_residual<N>(cube, X, Y, Z, cst * rho[((Z - 1) * R + (Y - 1)) * R + (X - 1)]) * inv) * kResScale;
    }
    reinterpret_cast<uint32_t*>(x)[t] = (uint32_t)f2bf(c0) | ((uint32_t)f2bf(c1) << 16);
  }
  __syncthreads();
}

__global__ void __launch_bounds__(kThreads) prep_kernel(const float* __restrict__ rho, const float* __restrict__ cpot,
                                                        int gs, float cst, int int_scheme, u16* __restrict__ x,
                                                        float* __restrict__ scale) {
  extern __shared__ float cube[];
  const int p = blockIdx.x;
  const Geo g = geo_of(gs);
  const float* r = rho + (size_t)p * g.R * g.R * g.R;
  const float* c = cpot + (size_t)p * g.C * g.C * g.C;
  u16* xp = x + (size_t)p * kCnnInput;
  switch (gs) {
    case 1: prep_patch<1>(r, c, cst, int_scheme, xp, scale + p, cube); break;
    case 2: prep_patch<2>(r, c, cst, int_scheme, xp, scale + p, cube); break;
    case 3: prep_patch<3>(r, c, cst, int_scheme, xp, scale + p, cube); break;
    case 4: prep_patch<4>(r, c, cst, int_scheme, xp, scale + p, cube); break;
    default: prep_patch<5>(r, c, cst, int_scheme, xp, scale + p, cube); break;
  }
}

// Guess of the interior: interp + s * D at interior frame index i = 2o + p.
template <int GS>
__device__ void guess_patch(const float* __restrict__ cpot, const float* __restrict__ d, float s, int int_scheme,
                            float* __restrict__ guess, float* cube) {
  constexpr Geo g = geo_of(GS);
  constexpr int N = g.N, R = g.R, OFF = 5 - GS;
  interp_cube<GS>(cpot, int_scheme, cube);
  for (int t = threadIdx.x; t < R * R * R; t += kThreads) {
    const int x = t % R, y = (t / R) % R, z = t / (R * R);   // interior-local; cube index +1
    // interior frame index: cube index + OFF - 1 = interior-local + OFF
    const int ix = x + OFF, iy = y + OFF, iz = z + OFF;
    const int o = ((iz >> 1) * So + (iy >> 1)) * So + (ix >> 1);
    const int p = ((iz & 1) * 2 + (iy & 1)) * 2 + (ix & 1);
    guess[t] = cube[((z + 1) * N + y + 1) * N + x + 1] + s * d[o * kCnnOut + p];
  }
  __syncthreads();
}

__global__ void __launch_bounds__(kThreads) guess_kernel(const float* __restrict__ cpot, const float* __restrict__ D,
                                                         const float* __restrict__ scale, int gs, int int_scheme,
                                                         float* __restrict__ guess) {
  extern __shared__ float cube[];
  const int p = blockIdx.x;
  const Geo g = geo_of(gs);
  const float* c = cpot + (size_t)p * g.C * g.C * g.C;
  const float* d = D + (size_t)p * kCnnOutputs;
  float* out = guess + (size_t)p * g.R * g.R * g.R;
  switch (gs) {
    case 1: guess_patch<1>(c, d, scale[p], int_scheme, out, cube); break;
    case 2: guess_patch<2>(c, d, scale[p], int_scheme, out, cube); break;
    case 3: guess_patch<3>(c, d, scale[p], int_scheme, out, cube); break;
    case 4: guess_patch<4>(c, d, scale[p], int_scheme, out, cube); break;
    default: guess_patch<5>(c, d, scale[p], int_scheme, out, cube); break;
  }
}

// ---- fused inference: one workgroup per patch, activations resident in LDS ------------------------------
// interpolation -> packing -> six convolutions ping-ponging between two LDS buffers -> guess written by the
// output layer's epilogue.  Each output value goes through the MFMA sequence of
// conv_fwd_kernel with the products of the all-zero input planes (padded z = 0 and 9) left out (adding those
// zero products to an accumulator that started at +0 leaves it bitwise unchanged), so the guess is bitwise
// that of prep + forward + guess with the layer-by-layer kernels.
//
// * An activation buffer holds only the 8 planes of the output grid, each [half][10 x 10 voxels][8 channels]
//   BF16 with a zero ring (y or x = 0 or 9), 26.6 KB.
// * The packed input (the solve interior only; its border voxels are zero like the activations' padding)
//   has the same layout, so the first layer is a layer like the others.
// * Wave w owns output rows w and w + 4 of every plane and sweeps the 8 input planes once; every A operand
//   read from LDS feeds up to three MFMAs, and the next plane's operands are requested before the current
//   plane's MFMAs.
// * Two buffers only: the coarse staging, the packed input and the activations share them with the FP32
//   interpolated cube.  The interpolated values the guess adds to are written to the guess array while the
//   input is packed; the output layer's epilogue reads them back (same lane, same address: L2), adds s * D and
//   stores the guess.  LDS per workgroup 53.3 KB: three workgroups per CU.
constexpr int kActVec = So * kPlaneV / 8;   // uint4 per buffer (8 planes)
constexpr int kCoarseMax = 12 * 12 * 12;    // C^3 at ghost size 5
constexpr int kCubeMax = 18 * 18 * 18;      // N^3 at ghost size 5
constexpr int kInteriorMax = 16 * 16 * 16;  // R^3 at ghost size 5
constexpr int kFT = 256;                    // threads of a fused workgroup (4 waves)
constexpr int kRing = 4 * S - 4;            // ring voxels of a half-plane (36)

constexpr int kFusedBlocksPerCU = 3;

struct FusedLds {
  uint4 X[kActVec];   // coarse staging -> packed input -> activations
  uint4 C[kActVec];   // interpolated cube (FP32, unpadded N^3) -> activations
  float red[kFT / 64];
};
static_assert(kCoarseMax * 4 <= kActVec * 16 && kInteriorMax * 4 <= kActVec * 16 && kCubeMax * 4 <= kActVec * 16,
              "staging must fit a buffer");
static_assert(kFusedBlocksPerCU * sizeof(FusedLds) <= 160 * 1024, "workgroups per CU");

// The biases of layer l for this lane's output channels 4*(lane/16)..+3.
__device__ __forceinline__ void load_bias(const float* __restrict__ P, int l, float4& b) {
  b = *reinterpret_cast<const float4*>(P + (size_t)l * kCnnLayerParams + 16 * K + 4 * ((threadIdx.x & 63) >> 4));
}

// Layer l's weights (A operand, from the lane-major copy WL) and the biases of this lane's output channels
// 4*(lane/16)..+3.
__device__ __forceinline__ void load_layer(const u16* __restrict__ WL, const float* __restrict__ P, int l,
                                           bf16x8 (&w)[KZ], float4& b) {
#pragma unroll
  for (int c = 0; c < KZ; c++) w[c] = load_weight_step(WL + (size_t)l * 16 * KF, c);
  load_bias(P, l, b);
}

// This lane's A-operand offsets (bf16 elements, relative to its row voxel in an input plane) for the five
// position pairs: position fwd_pos(s, g) of the plane, channel half g & 1 (g = lane/16).
__device__ __forceinline__ void pair_offsets(int (&off)[5]) {
  const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int s = 0; s < 5; s++) {
    const int pos = fwd_pos(s, g);
    off[s] = (g & 1) * kHalfV + ((pos / 3) * S + pos % 3) * 8;
  }
}

// Zero the ring voxels (y or x = 0 or 9) of both half-planes of the 8 planes of a buffer.
__device__ __forceinline__ void zero_ring(uint4* buf) {
  for (int i = threadIdx.x; i < 2 * So * kRing; i += kFT) {
    const int hp = i / kRing, k = i % kRing;
    int vox;
    if (k < S) {
      vox = k;                                   // row 0
    } else if (k < 2 * S) {
      vox = (S - 1) * S + k - S;                 // row 9
    } else {
      const int r = k - 2 * S;                   // rows 1..8, x = 0 or 9
      vox = (1 + (r >> 1)) * S + (r & 1) * (S - 1);
    }
    buf[hp * (kHalfV / 8) + vox] = make_uint4(0, 0, 0, 0);
  }
}

// What the output layer's epilogue needs: the scale, the interpolated interior (LDS) and where the guess goes.
struct GuessOut {
  float s;
  float* sd;         // s * D on the solve interior, [R^3] FP32 in the LDS buffer the output layer does not read
};

// Epilogue of output plane o for this wave's row pair: output channels co0..co0+3 (co0 = 4*(lane/16)) of voxel
// lane%16 of the tile.  MODE 0/1: 4 consecutive channels of one half-plane (8 bytes), y = relu(h) (+ the
// layer input at the same voxel, MODE 1).  MODE 2: channels 0..7 are the 2^3 sub-cells of the voxel; the
// guess interp + s * h of those fine cells is stored.
template <int GS, bool CUBE, int MODE>
__device__ __forceinline__ void conv_store(const u16* in, u16* out, const floatx4& acc, const float4& b, int o,
                                           const GuessOut& go) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int co0 = 4 * (lane >> 4);
  const int row = wave + tile_dy(lane), xv = tile_x(lane);
  const float h0 = acc[0] + b.x, h1 = acc[1] + b.y, h2 = acc[2] + b.z, h3 = acc[3] + b.w;
  if (MODE == 2) {
    if (co0 < kCnnOut) {
      constexpr int R = geo_of(GS).R, OFF = 5 - GS;
      const int lz = 2 * o + (co0 >> 2) - OFF, ly0 = 2 * row - OFF, lx0 = 2 * xv - OFF;
      const float h[4] = {h0, h1, h2, h3};
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int ly = ly0 + (k >> 1), lx = lx0 + (k & 1);
        if (lz >= 0 && lz < R && ly >= 0 && ly < R && lx >= 0 && lx < R) go.sd[(lz * R + ly) * R + lx] = go.s * h[k];
      }
    }
  } else {
    const int c0 = o * kPlaneV + (co0 >> 3) * kHalfV + ((row + 1) * S + xv + 1) * 8 + (co0 & 7);
    float o0 = fmaxf(h0, 0.0f), o1 = fmaxf(h1, 0.0f), o2 = fmaxf(h2, 0.0f), o3 = fmaxf(h3, 0.0f);
    if (MODE == 1) {
      const uint2 rx = *reinterpret_cast<const uint2*>(in + c0);
      o0 += bf_lo(rx.x);
      o1 += bf_hi(rx.x);
      o2 += bf_lo(rx.y);
      o3 += bf_hi(rx.y);
    }
    *reinterpret_cast<uint2*>(out + c0) = pack4_bf16(o0, o1, o2, o3);
  }
}

// One convolution layer (in != out).  Input plane z (0..7) feeds output plane z + 1 (dz = 0), z (dz = 1) and
// z - 1 (dz = 2); output plane o accumulates its steps in the order of conv_fwd_kernel (dz = 0, 1, 2; s = 0..4
// within each) without the steps of the zero planes z = -1 and 8.  The operands of plane z + 1 are requested
// before the MFMAs of plane z, so their LDS latency hides behind those.
// Wn (not null): the next layer's weights are requested into w as the current ones die: the dz = 0 steps before
// the last input plane (which feeds no plane z + 1), the others after its MFMAs.  The next layer then does not
// start with the whole round trip, and no extra registers are needed: 4% of the kernel, measured.  (Leaving
// the reloads out of a timing copy saves 11%: the rest is the bandwidth of 15 KB of weights per wave and layer.)
template <int GS, bool CUBE, int MODE>
__device__ __forceinline__ void conv_layer(const u16* in, u16* out, bf16x8 (&w)[KZ], const float4& b,
                                           const int (&off)[5], const GuessOut& go, const u16* __restrict__ Wn) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const u16* col = in + ((wave + tile_dy(lane)) * S + tile_x(lane)) * 8;   // padded row = output row + dy
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  floatx4 a0 = zero, a1 = zero;   // output planes z - 1 and z
  Pack8 nx[5];
#pragma unroll
  for (int s = 0; s < 5; s++) nx[s].u = *reinterpret_cast<const uint4*>(col + off[s]);
#pragma unroll
  for (int z = 0; z < So; z++) {
    Pack8 a[5];
#pragma unroll
    for (int s = 0; s < 5; s++) a[s] = nx[s];
    if (z + 1 < So) {
#pragma unroll
      for (int s = 0; s < 5; s++) nx[s].u = *reinterpret_cast<const uint4*>(col + (z + 1) * kPlaneV + off[s]);
    }
    floatx4 a2 = zero;            // output plane z + 1
    if (z + 1 == So && Wn) {
#pragma unroll
      for (int c = 0; c < 5; c++) w[c] = load_weight_step(Wn, c);
    }
#pragma unroll
    for (int s = 0; s < 5; s++) {
      if (z + 1 < So) a2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[s], a[s].v, a2, 0, 0, 0);
      a1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[5 + s], a[s].v, a1, 0, 0, 0);
      if (z >= 1) a0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[10 + s], a[s].v, a0, 0, 0, 0);
    }
    if (z + 1 == So && Wn) {
#pragma unroll
      for (int c = 5; c < KZ; c++) w[c] = load_weight_step(Wn, c);
    }
    if (z >= 1) conv_store<GS, CUBE, MODE>(in, out, a0, b, z - 1, go);
    a0 = a1;
    a1 = a2;
  }
  conv_store<GS, CUBE, MODE>(in, out, a0, b, So - 1, go);   // its dz = 2 input is the zero plane z = 8
}

// Interpolated solve cube from a coarse cube staged in LDS (the arithmetic of interp_cube) into an unpadded
// N^3 cube.  Returns this thread's max |value| (the cube's max once reduced over the workgroup).
template <int GS>
__device__ __forceinline__ float interp_cube_lds(const float* cs, int int_scheme, float* cube) {
  constexpr Geo g = geo_of(GS);
  constexpr int N = g.N, C = g.C, U = g.U, NC = C - 2;
  float mx = 0.0f;
  for (int q = threadIdx.x; q < NC * NC * NC; q += kFT) {
    const int i = q % NC + 1, j = (q / NC) % NC + 1, k = q / (NC * NC) + 1;
    float v[3][3][3];
    for (int dk = 0; dk < 3; dk++)
      for (int dj = 0; dj < 3; dj++)
        for (int di = 0; di < 3; di++) v[dk][dj][di] = cs[((k + dk - 1) * C + (j + dj - 1)) * C + (i + di - 1)];
    float ch[2][2][2];
    interp_children(v, int_scheme, ch);
    const int X0 = 2 * (i - 1) - U, Y0 = 2 * (j - 1) - U, Z0 = 2 * (k - 1) - U;
#pragma unroll
    for (int cz = 0; cz < 2; cz++)
#pragma unroll
      for (int cy = 0; cy < 2; cy++)
#pragma unroll
        for (int cx = 0; cx < 2; cx++) {
          const int X = X0 + cx, Y = Y0 + cy, Z = Z0 + cz;
          if (X >= 0 && X < N && Y >= 0 && Y < N && Z >= 0 && Z < N) {
            cube[(Z * N + Y) * N + X] = ch[cz][cy][cx];
            mx = fmaxf(mx, fabsf(ch[cz][cy][cx]));
          }
        }
  }
  return mx;
}

template <int GS, bool CUBE, bool KEEP>
__device__ void fused_patch(const float* __restrict__ rho, const float* __restrict__ cpot, const u16* __restrict__ WL,
                            const float* __restrict__ P, float cst, int int_scheme, float* __restrict__ guess,
                            FusedLds& L) {
  constexpr Geo g = geo_of(GS);
  constexpr int N = g.N, R = g.R, C = g.C, OFF = 5 - GS;
  constexpr int C3 = C * C * C;
  static_assert(C3 % 4 == 0, "float4 staging");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float* cs = reinterpret_cast<float*>(L.X);      // coarse staging
  float* cube = reinterpret_cast<float*>(L.C);
  u16* X0 = reinterpret_cast<u16*>(L.X);
  u16* A = reinterpret_cast<u16*>(L.C);
  // the coarse cube and this thread's density column are requested together.  Thread t owns the frame-interior
  // column (fx, fy) = (t % 16, t / 16); its solve-interior column is (fx, fy) - OFF.
  for (int t = threadIdx.x; t < C3 / 4; t += kFT)
    reinterpret_cast<float4*>(cs)[t] = reinterpret_cast<const float4*>(cpot)[t];
  const int fx = threadIdx.x & 15, fy = threadIdx.x >> 4;
  const int x = fx - OFF, y = fy - OFF;
  const bool colv = x >= 0 && x < R && y >= 0 && y < R;
  float rcol[R];
#pragma unroll
  for (int z = 0; z < R; z++) rcol[z] = colv ? rho[(z * R + y) * R + x] : 0.0f;
  __syncthreads();
  float mx = interp_cube_lds<GS>(cs, int_scheme, cube);
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  if (lane == 0) L.red[wave] = mx;
  __syncthreads();   // the cube is complete and the coarse staging is dead
  mx = L.red[0];
#pragma unroll
  for (int k = 1; k < kFT / 64; k++) mx = fmaxf(mx, L.red[k]);
  const float s = mx > 0.0f ? mx : 1.0f;
  const float inv = 1.0f / s;
  // The whole-cube guess takes the Dirichlet layer from the interpolation (its interior is the epilogue's).
  if (CUBE) {
    constexpr int NSHELL = 2 * N * N + 4 * (N - 1) * (N - 2);
    for (int q = threadIdx.x; q < NSHELL; q += kFT) {
      int X, Y, Z;
      shell_cell<N>(q, X, Y, Z);
      const int t = (Z * N + Y) * N + X;
      guess[t] = cube[t];
    }
  }
  // Packed input on the 16^3 frame interior (the solve interior, centred; zero elsewhere): fine cell
  // (fx, fy, fz) is sub-cell ((fz&1)*2 + (fy&1))*2 + (fx&1) of voxel (fx, fy, fz)/2, i.e. half-plane fz&1 and
  // 32-bit word (fy&1)*2 + (fx&1) of the voxel; the word is (q0, q1) = (interp/s, 64 r/s) with r the SOR
  // residual of the interpolated cube.  The column owner sweeps z with the column's cube values in registers
  // and keeps the column's interpolated values for the guess.
  uint32_t* X32 = reinterpret_cast<uint32_t*>(X0);
  const int colw = (((fy >> 1) + 1) * S + (fx >> 1) + 1) * 4 + (fy & 1) * 2 + (fx & 1);
  auto word = [&](int fz) -> uint32_t& { return X32[(fz >> 1) * (kPlaneV / 2) + (fz & 1) * (kHalfV / 2) + colw]; };
  zero_ring(L.X);
#pragma unroll
  for (int fz = 0; fz < OFF; fz++) word(fz) = 0u;
#pragma unroll
  for (int fz = OFF + R; fz < 16; fz++) word(fz) = 0u;
  // The column's interpolated values are kept for the guess: in registers in the uniform-batch instances (KEEP;
  // 164 VGPRs for the whole-cube guess, 168 for the interior guess), parked in the guess array in the
  // mixed-batch instance, whose five ghost sizes would spill.
  float icol[R];
  float* gcol = guess + (CUBE ? N * N + (y + 1) * N + (x + 1) : y * R + x);   // interior column, z = 0
  if (colv) {
    const float* cc = cube + (y + 1) * N + (x + 1);   // cube column, stride N^2
    float cm = cc[0], c = cc[N * N];
#pragma unroll
    for (int z = 0; z < R; z++) {
      const float* cz = cc + (z + 1) * N * N;
      const float cp = cz[N * N];
      const float r = cp + cm + cz[N] + cz[-N] + cz[1] + cz[-1] - 6.0f * c - cst * rcol[z];
      word(z + OFF) = pack2_bf16(c * inv, (r * inv) * kResScale);
      if (KEEP)
        icol[z] = c;
      else
        gcol[z * R * R] = c;
      cm = c;
      c = cp;
    }
  } else {
#pragma unroll
    for (int z = 0; z < R; z++) word(z + OFF) = 0u;
  }
  bf16x8 w[KZ];
  float4 b;
  load_layer(WL, P, 0, w, b);
  __syncthreads();   // the packed input is complete; the cube is dead
  zero_ring(L.C);
  int off[5];
  pair_offsets(off);
  __syncthreads();
  GuessOut go{s, reinterpret_cast<float*>(L.X)};   // X is free during the output layer (layer 5 read it)
  // each layer requests the next one's weights into w as it finishes; the bias follows it (first used after
  // the next layer's first plane of MFMAs)
  auto wnext = [&](int l) { return WL + (size_t)l * 16 * KF; };
  conv_layer<GS, CUBE, 0>(X0, A, w, b, off, go, wnext(1));   // layer 1: packed input -> A
  load_bias(P, 1, b);
  __syncthreads();   // every wave is done reading the packed input
  u16* Bb = X0;
  conv_layer<GS, CUBE, 1>(A, Bb, w, b, off, go, wnext(2));   // layers 2-5: A -> B -> A -> B -> A
  load_bias(P, 2, b);
  __syncthreads();
  conv_layer<GS, CUBE, 1>(Bb, A, w, b, off, go, wnext(3));
  load_bias(P, 3, b);
  __syncthreads();
  conv_layer<GS, CUBE, 1>(A, Bb, w, b, off, go, wnext(4));
  load_bias(P, 4, b);
  __syncthreads();
  conv_layer<GS, CUBE, 1>(Bb, A, w, b, off, go, wnext(5));
  load_bias(P, 5, b);
  __syncthreads();
  conv_layer<GS, CUBE, 2>(A, nullptr, w, b, off, go, nullptr);   // layer 6: s * D into X
  __syncthreads();
  // the guess, interp + s * D, by interior columns (whole rows per wave)
  if (colv) {
    const float* sd = reinterpret_cast<const float*>(L.X) + y * R + x;
#pragma unroll
    for (int z = 0; z < R; z++) {
      constexpr int ZS = CUBE ? N * N : R * R;
      const float base = KEEP ? icol[z] : gcol[z * ZS];
      gcol[z * ZS] = base + sd[z * R * R];
    }
  }
}

template <bool CUBE, bool KEEP>
__device__ __forceinline__ void fused_dispatch(int gs, const float* r, const float* c, const u16* WL, const float* P,
                                               float cst, int int_scheme, float* out, FusedLds& L) {
  switch (gs) {
    case 1: fused_patch<1, CUBE, KEEP>(r, c, WL, P, cst, int_scheme, out, L); break;
    case 2: fused_patch<2, CUBE, KEEP>(r, c, WL, P, cst, int_scheme, out, L); break;
    case 3: fused_patch<3, CUBE, KEEP>(r, c, WL, P, cst, int_scheme, out, L); break;
    case 4: fused_patch<4, CUBE, KEEP>(r, c, WL, P, cst, int_scheme, out, L); break;
    default: fused_patch<5, CUBE, KEEP>(r, c, WL, P, cst, int_scheme, out, L); break;
  }
}

// CUBE: the guess is the whole solve cube [n][N^3] (Dirichlet layer included), else the interior [n][R^3].
template <bool CUBE>
__global__ void __launch_bounds__(kFT, kFusedBlocksPerCU) fused_guess_kernel(const float* __restrict__ rho,
                                                             const float* __restrict__ cpot,
                                                             const u16* __restrict__ WL, const float* __restrict__ P,
                                                             int npatch, int gs, float cst, int int_scheme,
                                                             float* __restrict__ guess) {
  __shared__ FusedLds L;
  const int p = blockIdx.x;
  if (p >= npatch) return;
  const Geo g = geo_of(gs);
  const float* r = rho + (size_t)p * g.R * g.R * g.R;
  const float* c = cpot + (size_t)p * g.C * g.C * g.C;
  float* out = guess + (size_t)p * (CUBE ? g.N * g.N * g.N : g.R * g.R * g.R);
  fused_dispatch<CUBE, true>(gs, r, c, WL, P, cst, int_scheme, out, L);
}

// Mixed ghost sizes: patch p reads its ghost size and packed offsets from the plan's descriptors; the
// guess is packed like the density (offset rho_off).
__global__ void __launch_bounds__(kFT, kFusedBlocksPerCU) fused_guess_mixed_kernel(const float* __restrict__ rho,
                                                                   const float* __restrict__ cpot,
                                                                   const PatchDesc* __restrict__ desc,
                                                                   const u16* __restrict__ WL,
                                                                   const float* __restrict__ P, int npatch, float cst,
                                                                   int int_scheme, float* __restrict__ guess) {
  __shared__ FusedLds L;
  const int p = blockIdx.x;
  if (p >= npatch) return;
  const PatchDesc d = desc[p];
  fused_dispatch<false, false>(d.gs, rho + d.rho_off, cpot + d.cpot_off, WL, P, cst, int_scheme, guess + d.rho_off, L);
}

}  // namespace cnn

// ---- host launchers ----------------------------------------------------------------------------------------

using namespace cnn;

hipError_t cnn_conv_fwd(const uint16_t* X, const uint16_t* W, const float* b, uint16_t* Y, float* D, int n, int mode,
                        hipStream_t s) {
  const dim3 grid(n * kSlabs), block(kThreads);
  if (mode == 0)
    hipLaunchKernelGGL(conv_fwd_kernel<0>, grid, block, 0, s, X, W, b, Y, D);
  else if (mode == 1)
    hipLaunchKernelGGL(conv_fwd_kernel<1>, grid, block, 0, s, X, W, b, Y, D);
  else if (mode == 2)
    hipLaunchKernelGGL(conv_fwd_kernel<2>, grid, block, 0, s, X, W, b, Y, D);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

int cnn_train_blocks(int n) { return n < kCnnTrainBlocks ? n : kCnnTrainBlocks; }

hipError_t cnn_train_pass(const uint16_t* x0, const uint16_t* WL, const uint16_t* WT, const float* P, const float* T,
                          uint16_t* const (&y)[kCnnLayers], uint16_t* dH, float* lossp, int n, float res_weight,
                          hipStream_t s) {
  TrainOut out;
  for (int l = 1; l < kCnnLayers; l++) out.y[l] = y[l];
  out.y[0] = nullptr;
  out.dh = dH;
  out.loss = lossp;
  hipLaunchKernelGGL(train_pass_kernel, dim3(cnn_train_blocks(n)), dim3(kTrainThreads), 0, s, x0, WL, WT, P, T, n,
                     res_weight, out);
  return hipGetLastError();
}

// One partial per block and layer: 6 * 128 blocks are three per CU.
int cnn_grad_parts(int n) { return n < 128 ? n : 128; }

hipError_t cnn_weight_grad(const uint16_t* const (&x)[kCnnLayers], const uint16_t* dH, int n, float* part, float* g,
                           hipStream_t s) {
  GradInputs in;
  for (int l = 0; l < kCnnLayers; l++) in.x[l] = x[l];
  const int parts = cnn_grad_parts(n);
  hipLaunchKernelGGL(weight_grad_kernel, dim3(parts, kCnnLayers), dim3(kWThreads), 0, s, in, dH, n, part);
  hipLaunchKernelGGL(grad_reduce_kernel, dim3(kCnnParams / kRCols), dim3(kRCols * kRGroups), 0, s, part, parts, g);
  return hipGetLastError();
}

hipError_t cnn_adam(float* p, const float* g, float* m, float* v, int n, float lr, float b1, float b2, float eps,
                    float c1, float c2, hipStream_t s) {
  hipLaunchKernelGGL(adam_kernel, dim3((n + 255) / 256), dim3(256), 0, s, p, g, m, v, n, lr, b1, b2, eps, c1, c2);
  return hipGetLastError();
}

hipError_t cnn_weight_copies(const float* P, uint16_t* Wb, uint16_t* WT, uint16_t* WL, hipStream_t s) {
  const int n = kCnnLayers * 16 * KF;
  hipLaunchKernelGGL(weight_copies_kernel, dim3((n + 255) / 256), dim3(256), 0, s, P, Wb, WT, WL);
  return hipGetLastError();
}

hipError_t cnn_prep(const float* rho, const float* cpot, int n, int gs, float cst, int int_scheme, uint16_t* x,
                    float* scale, hipStream_t s) {
  const Geo g = geo_of(gs);
  hipLaunchKernelGGL(prep_kernel, dim3(n), dim3(kThreads), sizeof(float) * g.N * g.N * g.N, s, rho, cpot, gs, cst,
                     int_scheme, x, scale);
  return hipGetLastError();
}

hipError_t cnn_fused_guess(const float* rho, const float* cpot, const uint16_t* WL, const float* P, int n, int gs,
                           float cst, int int_scheme, float* guess, int cube, hipStream_t s) {
  if (cube)
    hipLaunchKernelGGL(fused_guess_kernel<true>, dim3(n), dim3(kFT), 0, s, rho, cpot, WL, P, n, gs, cst, int_scheme,
                       guess);
  else
    hipLaunchKernelGGL(fused_guess_kernel<false>, dim3(n), dim3(kFT), 0, s, rho, cpot, WL, P, n, gs, cst, int_scheme,
                       guess);
  return hipGetLastError();
}

hipError_t cnn_fused_guess_mixed(const float* rho, const float* cpot, const PatchDesc* desc, const uint16_t* WL,
                                 const float* P, int n, float cst, int int_scheme, float* guess, hipStream_t s) {
  hipLaunchKernelGGL(fused_guess_mixed_kernel, dim3(n), dim3(kFT), 0, s, rho, cpot, desc, WL, P, n, cst,
                     int_scheme, guess);
  return hipGetLastError();
}

hipError_t cnn_guess(const float* cpot, const float* D, const float* scale, int n, int gs, int int_scheme,
                     float* guess, hipStream_t s) {
  const Geo g = geo_of(gs);
  hipLaunchKernelGGL(guess_kernel, dim3(n), dim3(kThreads), sizeof(float) * g.N * g.N * g.N, s, cpot, D, scale, gs,
                     int_scheme, guess);
  return hipGetLastError();
}

}  // namespace pgamd
