// Learned subgrid form: a small periodic 3-D CNN on a coarse grid, trained and
// run with hand-written bf16 MFMA kernels (FP32 accumulation).  No
// counterpart in the reference.
//
// Layouts of the bf16 activations, C a multiple of 16:
//   N < 16: channels-last, A[node][C], node = (x N + y) N + z;
//   N >= 16: per z-line, segments of 16 NT nodes (NT = min(4, N / 16)), in each
//   C/8 planes of 8 channels, in each the nodes z = NT l + t ordered [t][l]
//   (tiled_at()).  Tile t of a segment is then 16 consecutive 16-byte cells per
//   channel plane, which the 16 lanes of an MFMA operand row read as 256
//   consecutive bytes: channels-last rows put neighbouring lanes 64 bytes
//   apart, and the cache lines a load then touched bounded the convolutions
//   (32 -> 32 channels at 128^3, inference: 192 us, 603 TFLOP/s; 122 us, 950
//   TFLOP/s now, against 1200 TFLOP/s that the instruction reaches by itself).
// Weights per layer W[tap][co][ci] (and the transposed copy Wt[tap][ci][co] for
// the data gradient), tap = (dx+1) 9 + (dy+1) 3 + (dz+1) for offsets in
// {-1, 0, 1}; periodic neighbours.
//
// A 3x3x3 convolution is an implicit GEMM: M = nodes, K = 27 taps x CI,
// N = CO.  One wavefront computes 16 nodes x CO outputs with
// __builtin_amdgcn_mfma_f32_16x16x16bf16_1k, whose operand layout is
//   A (16x16, M x K): lane l holds A[l % 16][4 (l / 16) + i], i = 0..3
//   B (16x16, K x N): lane l holds B[4 (l / 16) + i][l % 16]
//   D (16x16):        lane l holds D[4 (l / 16) + i][l % 16]
// so a lane reads 4 consecutive channels (8 bytes) of one node.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace ld {
namespace cnn {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t bf16;

// FP32 -> bf16, round to nearest even (NaN kept quiet).
__device__ __forceinline__ bf16 f2b(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16)((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16)(u >> 16);
}
__device__ __forceinline__ float b2f(bf16 b) { return __uint_as_float((uint32_t)b << 16); }

// element offset of (z, channel c) in a tiled line of C channels
template <int NT> __device__ __forceinline__ int tiled_at(int z, int c, int C) {
  const int seg = z / (16 * NT), r = z % (16 * NT);
  return ((seg * (C / 8) + c / 8) * (16 * NT) + (r % NT) * 16 + r / NT) * 8 + c % 8;
}

__device__ __forceinline__ int nbr(int node, int tap, int N, bool flip) {
  int dx = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dz = tap % 3 - 1;
  if (flip) { dx = -dx; dy = -dy; dz = -dz; }
  const int z = node & (N - 1), y = (node / N) & (N - 1), x = node / (N * N);
  return (((x + dx) & (N - 1)) * N + ((y + dy) & (N - 1))) * N + ((z + dz) & (N - 1));
}

// out[node][co] = bias[co] + sum_{tap, ci} X[nbr(node, tap)][ci] W[tap][co][ci]
// FLIP: neighbours at -offset (the data gradient, with Wt);
// RELU: max(., 0); MASK: times (mask[node][co] > 0) (ReLU derivative of the
// layer below); Yb: bf16 output, Yf: FP32 rows of cout channels (either may be null).
// 256 threads = 4 wavefronts x 16 nodes; N^3 must be a multiple of 64.
template <int CI, int CO, bool FLIP, bool RELU, bool MASK>
__global__ void __launch_bounds__(256)
k_conv(const bf16* __restrict__ X, const bf16* __restrict__ W, const float* __restrict__ bias,
       const bf16* __restrict__ mask, bf16* __restrict__ Yb, float* __restrict__ Yf, int cout, int N) {
  static_assert(CI % 16 == 0 && CO % 16 == 0, "channels: multiples of 16");
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int node0 = blockIdx.x * 64 + wv * 16;
  const int row = lane & 15, kq = 4 * (lane >> 4);
  f32x4 acc[CO / 16];
#pragma unroll
  for (int t = 0; t < CO / 16; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int tap = 0; tap < 27; ++tap) {
    const bf16* xa = X + (size_t)nbr(node0 + row, tap, N, FLIP) * CI + kq;
    const bf16* wb = W + ((size_t)tap * CO + row) * CI + kq;
#pragma unroll
    for (int cb = 0; cb < CI / 16; ++cb) {
      const bf16x4 a = *reinterpret_cast<const bf16x4*>(xa + cb * 16);
#pragma unroll
      for (int t = 0; t < CO / 16; ++t) {
        const bf16x4 b = *reinterpret_cast<const bf16x4*>(wb + (size_t)t * 16 * CI + cb * 16);
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[t], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < CO / 16; ++t) {
    const int co = t * 16 + row;
    const float bv = bias ? bias[co] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const size_t o = (size_t)(node0 + kq + i) * CO + co;
      float v = acc[t][i] + bv;
      if (RELU) v = v > 0.f ? v : 0.f;
      if (MASK) v = b2f(mask[o]) > 0.f ? v : 0.f;
      if (Yb) Yb[o] = f2b(v);
      if (Yf && co < cout) Yf[(size_t)(node0 + kq + i) * cout + co] = v;
    }
  }
}

// The same convolution with the gfx950 double-rate instruction
// __builtin_amdgcn_mfma_f32_16x16x32_bf16, oriented M = output channels,
// N = nodes, K = (tap, input channel) pairs in steps of 32:
//   A (16x32): lane l holds W[tap][co0 + l % 16][ci0 + i]       (8 bf16, 16 B)
//   B (32x16): lane l holds X[nbr(node(l % 16), tap)][ci0 + i]   (8 bf16, 16 B)
//   D (16x16): lane l holds Y[node(l % 16)][co0 + 4 (l / 16) + i], i < 4
// with (tap, ci0) = divmod(32 ks + 8 (l / 16), CI) for K-step ks (CI = 16: a
// step covers two taps; the 28th tap of the last step has zero weights).
// The layer's weights are staged in LDS once per block; a wavefront computes
// a z-line segment of 16 NT nodes for all CO as NT tiles of 16 nodes, so each
// weight fragment feeds NT instructions and each input fragment CO/16.
//
// Tile t holds the nodes z0 + NT n + t (n = lane % 16), not 16 consecutive
// ones: the z neighbour of a node then lies in the next or previous tile of
// the same lane, and only one tile per direction needs a lane shift (64
// instructions per neighbour line with consecutive nodes, 16 now); and a
// lane's NT nodes are consecutive, so the node-blocked copy needs no transpose
// through LDS.  Inputs and outputs are in the tiled layout.
// Blocks loop over segments (persistent grid: two blocks fill a CU's LDS),
// XCD-aware: each XCD takes a contiguous run of blocks, so neighbouring lines
// share its L2.  The K order of a sum (taps, then channels) is part of the
// result: the hidden layers round it to bf16.
// Needs N a multiple of 16 * NT.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

template <unsigned CTRL>
__device__ __forceinline__ uint32_t dpp_u(uint32_t old, uint32_t src) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)src, CTRL, 0xf, 0xf, false);
}
// lanes of a 16-lane row take the next lane's fragment; lane 15 takes its own of `edge`
__device__ __forceinline__ uint4 shift_up(const uint4& a, const uint4& edge) {
  return make_uint4(dpp_u<0x101>(edge.x, a.x), dpp_u<0x101>(edge.y, a.y), dpp_u<0x101>(edge.z, a.z),
                    dpp_u<0x101>(edge.w, a.w));
}
// the previous lane's fragment; lane 0 takes its own of `edge`
__device__ __forceinline__ uint4 shift_down(const uint4& a, const uint4& edge) {
  return make_uint4(dpp_u<0x111>(edge.x, a.x), dpp_u<0x111>(edge.y, a.y), dpp_u<0x111>(edge.z, a.z),
                    dpp_u<0x111>(edge.w, a.w));
}

// Where a convolution's results go; each may be null.
struct ConvOut {
  bf16* Yb;            // tiled
  float* Yf;           // FP32 rows of cout channels
  int cout, vec;       // vec: 16-byte stores into the rows (cout % 4 == 0, Yf aligned)
  bf16* Yblk;          // node-blocked channel-major copy (blocked_at()): runs of 8 nodes x 1 channel
};
__device__ __forceinline__ size_t blocked_at(size_t node, int c, int C) { return ((node >> 3) * C + c) * 8 + (node & 7); }

// Bias, ReLU / mask and stores of a segment's accumulators: tile t's lane node
// z0 + NT n16 + t of z-line `line`, channels 16 m + 4 q + i.  With NT = 4 a lane
// holds half a run of each of its channels of the blocked copy; neighbouring
// lanes exchange two channels each and store whole runs.
template <int CO, bool RELU, bool MASK, int NT>
__device__ __forceinline__ void conv_out(const f32x4 (&acc)[NT][CO / 16], const float4 (&bv)[CO / 16], int N, int line,
                                         int z0, const bf16* __restrict__ mask, const ConvOut& O) {
  const int lane = threadIdx.x & 63, n16 = lane & 15, q = lane >> 4;
  const size_t node0 = (size_t)line * N + z0 + NT * n16;
  const size_t cell0 = (size_t)line * N * CO + z0 * CO;       // the segment's cells
#pragma unroll
  for (int m = 0; m < CO / 16; ++m) {
    const int co = m * 16 + 4 * q;
    const size_t tb = cell0 + ((2 * m + (q >> 1)) * (16 * NT) + n16) * 8 + 4 * (q & 1);
    uint32_t pk[NT][2];                // channels (0, 1) and (2, 3) of each node
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const size_t o = tb + t * 128;
      const float b4[4] = {bv[m].x, bv[m].y, bv[m].z, bv[m].w};
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] = acc[t][m][i] + b4[i];
        if (RELU) v[i] = v[i] > 0.f ? v[i] : 0.f;
      }
      if (MASK) {
        const uint2 mk = *reinterpret_cast<const uint2*>(mask + o);
        const bf16 mb[4] = {(bf16)(mk.x & 0xffff), (bf16)(mk.x >> 16), (bf16)(mk.y & 0xffff), (bf16)(mk.y >> 16)};
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = b2f(mb[i]) > 0.f ? v[i] : 0.f;
      }
      if (O.Yf) {
        float* row = O.Yf + (node0 + t) * O.cout + co;
        if (O.vec) {
          if (co < O.cout) *reinterpret_cast<float4*>(row) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (co + i < O.cout) row[i] = v[i];
        }
      }
      pk[t][0] = (uint32_t)f2b(v[0]) | ((uint32_t)f2b(v[1]) << 16);
      pk[t][1] = (uint32_t)f2b(v[2]) | ((uint32_t)f2b(v[3]) << 16);
      if (O.Yb) *reinterpret_cast<uint2*>(O.Yb + o) = make_uint2(pk[t][0], pk[t][1]);
    }
    if (!O.Yblk) continue;
    if constexpr (NT == 4) {
      // c[i]: nodes 0..3 of channel i
      uint2 c[4];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        c[2 * h] = make_uint2((pk[0][h] & 0xffffu) | (pk[1][h] << 16), (pk[2][h] & 0xffffu) | (pk[3][h] << 16));
        c[2 * h + 1] = make_uint2((pk[0][h] >> 16) | (pk[1][h] & 0xffff0000u), (pk[2][h] >> 16) | (pk[3][h] & 0xffff0000u));
      }
      const bool odd = n16 & 1;
#pragma unroll
      for (int e = 0; e < 2; ++e) {    // even lanes store channels 0, 1; odd lanes 2, 3
        const uint2 mine = odd ? c[2 + e] : c[e], theirs = odd ? c[e] : c[2 + e];
        const uint2 got = make_uint2(dpp_u<0xb1>(0u, theirs.x), dpp_u<0xb1>(0u, theirs.y));   // quad_perm 1,0,3,2
        const uint4 run = odd ? make_uint4(got.x, got.y, mine.x, mine.y) : make_uint4(mine.x, mine.y, got.x, got.y);
        *reinterpret_cast<uint4*>(O.Yblk + ((node0 >> 3) * CO + co + (odd ? 2 : 0) + e) * 8) = run;
      }
    } else {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          O.Yblk[blocked_at(node0 + t, co + i, CO)] = (bf16)(pk[t][i >> 1] >> (16 * (i & 1)));
    }
  }
}
template <int CO> __device__ __forceinline__ void load_bias(const float* __restrict__ bias, float4 (&bv)[CO / 16]) {
  const int q = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int m = 0; m < CO / 16; ++m)
    bv[m] = bias ? *reinterpret_cast<const float4*>(bias + m * 16 + 4 * q) : make_float4(0.f, 0.f, 0.f, 0.f);
}

// CI = 16: every K-step covers two taps, lanes q < 2 the even one and q >= 2
// the odd one.  The K-steps are unrolled, so a lane's tap offsets are selects
// between constants and the tiles' addresses differ by constants (only the
// first and last tile can reach past the lane's nodes).
template <int CI, int CO, bool FLIP, bool RELU, bool MASK, int NT, int WPB>
__global__ void __launch_bounds__(64 * WPB)
k_conv2(const bf16* __restrict__ X, const bf16* __restrict__ W, const float* __restrict__ bias,
        const bf16* __restrict__ mask, ConvOut O, int N, int nseg) {
  static_assert(CI == 16 && CO % 16 == 0, "16 input channels");
  constexpr int MT = CO / 16;
  constexpr int KS = (27 * CI + 31) / 32;
  constexpr int WN = 27 * CO * CI;
  __shared__ __attribute__((aligned(16))) bf16 sW[WN];
  for (int e = threadIdx.x; e < WN / 8; e += 64 * WPB)
    reinterpret_cast<uint4*>(sW)[e] = reinterpret_cast<const uint4*>(W)[e];
  __syncthreads();
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n16 = lane & 15, q = lane >> 4;
  const bool hi = q >= 2;
  const int ci0 = 8 * (q & 1);
  const int G = gridDim.x;
  const int lb = (G % 8 == 0) ? (blockIdx.x % 8) * (G / 8) + blockIdx.x / 8 : blockIdx.x;
  const int spl = N / (16 * NT);                  // segments per z-line
  const int msk = N - 1;
  float4 bv[MT];
  load_bias<CO>(bias, bv);
  for (int seg = lb * WPB + wv; seg < nseg; seg += G * WPB) {
    const int line = seg / spl, z0 = (seg % spl) * 16 * NT;
    const int x = line / N, y = line & msk;
    // element offsets inside a line: tile 0 of the lane's nodes (tile t 128 t
    // further), the node before tile 0's and the one after tile NT - 1's
    const int zl = z0 + NT * n16;
    const int own = tiled_at<NT>(zl, ci0, CI), prev = tiled_at<NT>((zl - 1) & msk, ci0, CI),
              next = tiled_at<NT>((zl + NT) & msk, ci0, CI);
    f32x4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      constexpr int S = FLIP ? -1 : 1;
      const int tA = 2 * ks, tB = 2 * ks + 1 < 27 ? 2 * ks + 1 : 26;
      const bool valid = 2 * ks + 1 < 27 || !hi;
      const size_t rA = ((size_t)((x + S * (tA / 9 - 1)) & msk) * N + ((y + S * ((tA / 3) % 3 - 1)) & msk)) * N;
      const size_t rB = ((size_t)((x + S * (tB / 9 - 1)) & msk) * N + ((y + S * ((tB / 3) % 3 - 1)) & msk)) * N;
      const int dA = S * (tA % 3 - 1), dB = S * (tB % 3 - 1);      // z offsets of the two taps
      const bf16* row = X + (hi ? rB : rA) * CI;
      const bf16* mid = row + own + (hi ? dB : dA) * 128;
      bf16x8 wf[MT], xf[NT];
      // opaque to the compiler, so the weight fragments are re-read from LDS
      // per segment instead of being hoisted into registers for all K-steps
      int wofs = ((hi ? tB : tA) * CO + n16) * CI + ci0;
      asm volatile("" : "+v"(wofs));
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const uint4 v = *reinterpret_cast<const uint4*>(sW + wofs + m * 16 * CI);
        wf[m] = valid ? __builtin_bit_cast(bf16x8, v) : bf16x8{};
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        // only the first and last tile can reach past the lane's nodes
        auto far = [&](int d) { return t + d < 0 || t + d >= NT; };
        auto at = [&](int d) { return t + d < 0 ? prev : t + d >= NT ? next : own + (t + d) * 128; };
        const bf16* src = far(dA) || far(dB) ? row + (hi ? at(dB) : at(dA)) : mid + t * 128;
        const uint4 v = *reinterpret_cast<const uint4*>(src);
        xf[t] = valid ? __builtin_bit_cast(bf16x8, v) : bf16x8{};
      }
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[m], xf[t], acc[t][m], 0, 0, 0);
    }
    conv_out<CO, RELU, MASK, NT>(acc, bv, N, line, z0, mask, O);
  }
}

// CI = 32: the input fragments of a neighbour line (dx, dy) serve its three dz
// taps: a wavefront loads its NT tiles once plus the node before and after the
// segment (one load: lane 0 the one before, lane 15 the one after).  The next
// line's loads are issued before this line's products.
template <int CO, bool FLIP, bool RELU, bool MASK, int NT, int WPB>
__global__ void __launch_bounds__(64 * WPB)
k_conv3(const bf16* __restrict__ X, const bf16* __restrict__ W, const float* __restrict__ bias,
        const bf16* __restrict__ mask, ConvOut O, int N, int nseg) {
  constexpr int CI = 32, MT = CO / 16;
  constexpr int WN = 27 * CO * CI;
  __shared__ __attribute__((aligned(16))) bf16 sW[WN];
  for (int e = threadIdx.x; e < WN / 8; e += 64 * WPB)
    reinterpret_cast<uint4*>(sW)[e] = reinterpret_cast<const uint4*>(W)[e];
  __syncthreads();
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n16 = lane & 15, q = lane >> 4, ci0 = 8 * q;
  const int G = gridDim.x;
  const int lb = (G % 8 == 0) ? (blockIdx.x % 8) * (G / 8) + blockIdx.x / 8 : blockIdx.x;
  const int spl = N / (16 * NT);
  const int msk = N - 1;
  float4 bv[MT];
  load_bias<CO>(bias, bv);
  for (int seg = lb * WPB + wv; seg < nseg; seg += G * WPB) {
    const int line = seg / spl, z0 = (seg % spl) * 16 * NT;
    const int x = line / N, y = line & msk;
    const int zl = z0 + NT * n16;
    // element offsets inside a line: the lane's first node; the node before or
    // after the segment for the end lanes
    const int own = tiled_at<NT>(zl, ci0, CI);         // tile t 128 t further
    const int end = n16 == 0 ? tiled_at<NT>((z0 - 1) & msk, ci0, CI)
                             : n16 == 15 ? tiled_at<NT>((z0 + 16 * NT) & msk, ci0, CI) : own;
    f32x4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint4 xc[NT], edge;
    auto fetch = [&](int dxy, uint4 (&f)[NT], uint4& e) {
      const bf16* row = X + ((size_t)((x + dxy / 3 - 1) & msk) * N + ((y + dxy % 3 - 1) & msk)) * N * CI;
#pragma unroll
      for (int t = 0; t < NT; ++t) f[t] = *reinterpret_cast<const uint4*>(row + own + t * 128);
      e = *reinterpret_cast<const uint4*>(row + end);
    };
    fetch(0, xc, edge);
#pragma unroll
    for (int dxy = 0; dxy < 9; ++dxy) {
      const int ndx = dxy / 3 - 1, ndy = dxy % 3 - 1;     // neighbour line offset
      uint4 xn[NT], en;
      if (dxy < 8) fetch(dxy + 1, xn, en);
#pragma unroll
      for (int ndz = -1; ndz <= 1; ++ndz) {
        // weight tap of this neighbour offset (mirrored for the data gradient)
        const int tap = FLIP ? (1 - ndx) * 9 + (1 - ndy) * 3 + (1 - ndz) : (ndx + 1) * 9 + (ndy + 1) * 3 + (ndz + 1);
        int wofs = (tap * CO + n16) * CI + ci0;
        asm volatile("" : "+v"(wofs));
        bf16x8 wf[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m)
          wf[m] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(sW + wofs + m * 16 * CI));
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          uint4 v;
          if (t + ndz < 0) v = shift_down(xc[NT - 1], edge);
          else if (t + ndz >= NT) v = shift_up(xc[0], edge);
          else v = xc[t + ndz];
          const bf16x8 xf = __builtin_bit_cast(bf16x8, v);
#pragma unroll
          for (int m = 0; m < MT; ++m)
            acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[m], xf, acc[t][m], 0, 0, 0);
        }
      }
      if (dxy < 8) {
#pragma unroll
        for (int t = 0; t < NT; ++t) xc[t] = xn[t];
        edge = en;
      }
    }
    conv_out<CO, RELU, MASK, NT>(acc, bv, N, line, z0, mask, O);
  }
}

// Weight and bias gradients of one layer, per block over `chunk` nodes:
//   part[blk][(tap CO + co) CI + ci] = sum_node dZ[node][co] X[nbr(node, tap)][ci]
//   part[blk][27 CO CI + co]         = sum_node dZ[node][co]
// (M = co, N = ci, K = nodes).  The dZ rows of 64 nodes are staged in LDS for
// the block, the X neighbour rows per wavefront (wavefront w does taps
// w, w + 4, ...).  chunk is a multiple of 64.
template <int CI, int CO>
__global__ void __launch_bounds__(256)
k_wgrad(const bf16* __restrict__ X, const bf16* __restrict__ dZ, float* __restrict__ part, int N, int chunk) {
  constexpr int NT = 7;                       // taps per wavefront (27 = 7 + 7 + 7 + 6)
  __shared__ bf16 sdz[64 * CO];
  __shared__ bf16 sx[4][64 * CI];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int row = lane & 15, kq = 4 * (lane >> 4);
  f32x4 acc[NT][CO / 16][CI / 16];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int a = 0; a < CO / 16; ++a)
#pragma unroll
      for (int b = 0; b < CI / 16; ++b) acc[j][a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  float db = 0.f;
  const size_t nbase = (size_t)blockIdx.x * chunk;
  for (int s = 0; s < chunk; s += 64) {
    __syncthreads();
    for (int e = threadIdx.x; e < 64 * CO; e += 256) sdz[e] = dZ[(nbase + s) * CO + e];
    __syncthreads();
    if (threadIdx.x < CO) {
      for (int n = 0; n < 64; ++n) db += b2f(sdz[n * CO + threadIdx.x]);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int tap = wv + 4 * j;
      if (tap >= 27) break;
      // this lane's node: neighbour row of X
      const int node = (int)(nbase + s) + lane;
      const bf16* src = X + (size_t)nbr(node, tap, N, false) * CI;
#pragma unroll
      for (int c = 0; c < CI; c += 4)
        *reinterpret_cast<bf16x4*>(&sx[wv][lane * CI + c]) = *reinterpret_cast<const bf16x4*>(src + c);
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
#pragma unroll
        for (int a = 0; a < CO / 16; ++a) {
          bf16x4 fa;
#pragma unroll
          for (int i = 0; i < 4; ++i) fa[i] = (short)sdz[(kk * 16 + kq + i) * CO + a * 16 + row];
#pragma unroll
          for (int b = 0; b < CI / 16; ++b) {
            bf16x4 fb;
#pragma unroll
            for (int i = 0; i < 4; ++i) fb[i] = (short)sx[wv][(kk * 16 + kq + i) * CI + b * 16 + row];
            acc[j][a][b] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(fa, fb, acc[j][a][b], 0, 0, 0);
          }
        }
      }
    }
  }
  float* out = part + (size_t)blockIdx.x * (27 * CO * CI + CO);
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int tap = wv + 4 * j;
    if (tap >= 27) break;
#pragma unroll
    for (int a = 0; a < CO / 16; ++a)
#pragma unroll
      for (int b = 0; b < CI / 16; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          out[((size_t)tap * CO + a * 16 + kq + i) * CI + b * 16 + row] = acc[j][a][b][i];
  }
  if (threadIdx.x < CO) out[27 * CO * CI + threadIdx.x] = db;
}

// Weight and bias gradients from node-blocked channel-major operands
// (blocked_at()) on the 16x16x32 bf16 MFMA (M = output channels, N = input
// channels, K = nodes):
//   A (16x32): lane l holds dZ[node k0 + 8 (l / 16) + i][co0 + l % 16]  (one 16-byte run)
//   B (32x16): lane l holds X[nbr(node k0 + 8 (l / 16) + i, tap)][ci0 + l % 16]
// so the 16 lanes of a row read 256 consecutive bytes.
// Eight consecutive nodes of a lane lie on one z-line, so their neighbours for
// tap (dx, dy, dz) are eight consecutive z on the neighbour line, shifted by
// dz: the lane loads the aligned 16 bytes at z plus one dword on each side
// (periodic in z) and forms the dz = -1 and +1 operands with v_alignbyte.
struct XRun {
  uint4 c;
  uint32_t pv, nv;           // the dwords before and after the run
  // the line's runs of this lane's channel: own at o, before at op, after at on
  // (byte offsets; a uniform line pointer plus 32-bit lane offsets)
  __device__ __forceinline__ void load(const bf16* __restrict__ line, uint32_t o, uint32_t op, uint32_t on) {
    const char* l = reinterpret_cast<const char*>(line);
    c = *reinterpret_cast<const uint4*>(l + o);
    pv = *reinterpret_cast<const uint32_t*>(l + op + 12);
    nv = *reinterpret_cast<const uint32_t*>(l + on);
  }
  __device__ __forceinline__ void taps(bf16x8 f[3]) const {      // dz = -1, 0, 1
    const uint32_t s1 = __builtin_amdgcn_alignbyte(c.y, c.x, 2), s2 = __builtin_amdgcn_alignbyte(c.z, c.y, 2),
                   s3 = __builtin_amdgcn_alignbyte(c.w, c.z, 2);
    f[0] = __builtin_bit_cast(bf16x8, make_uint4(__builtin_amdgcn_alignbyte(c.x, pv, 2), s1, s2, s3));
    f[1] = __builtin_bit_cast(bf16x8, c);
    f[2] = __builtin_bit_cast(bf16x8, make_uint4(s1, s2, s3, __builtin_amdgcn_alignbyte(nv, c.w, 2)));
  }
};

// N >= 32.  A unit of work is a run of y-lines of one x and one 32-node z chunk;
// wavefront (dx, t) of a block owns the nine taps of one dx and 16 input
// channels, and walks the unit's X lines in y: each X run it loads meets the
// dZ runs of the three lines around it, which it keeps in registers (one new
// dZ line per step), so a step's loads (one X run, CO/16 dZ runs, the next
// step's issued before this step's products) feed 9 CO/16 instructions.  One
// neighbour line per wavefront, nine wavefronts reading the same dZ, fed 3 per
// X run and was bound by the loads.  Twelve wavefronts fill a CU (three per
// SIMD): two (32 input channels) or four shares of the unit's lines, which add
// up through LDS.
// Blocks take consecutive units and write one partial each:
//   part[b][(tap CO + co) CI + ci],  part[b][27 CO CI + co] (bias: products
// with a run of ones).  128^3: 32 -> 32 channels 315 -> 119 us (980 TFLOP/s),
// 32 -> 16 213 -> 97, 16 -> 32 204 -> 70.  Blocks of six wavefronts took 189 us
// (SIMDs unevenly filled), a scheduling barrier after the loads 180 (spills).
template <int CI, int CO>
__global__ void __launch_bounds__(768, 3)
k_wgrad3(const bf16* __restrict__ XB, const bf16* __restrict__ dZB, float* __restrict__ part, int N, int units,
         int ysplit) {
  constexpr int MT = CO / 16, TI = CI / 16, H = 4 / TI;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n16 = lane & 15, q = lane >> 4, msk = N - 1, G8 = N >> 3;
  const int role = w % (3 * TI), h = w / (3 * TI);       // taps and channels; share of the unit's lines
  const int dxi = role % 3, t = role / 3;
  const bool bias = role == 1;
  f32x4 acc[9][MT], db[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    db[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < 9; ++d) acc[d][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const bf16x8 ones = __builtin_bit_cast(bf16x8, make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u));
  const int G = gridDim.x, per = (units + G - 1) / G;
  const int lb = (G % 8 == 0) ? (blockIdx.x % 8) * (G / 8) + blockIdx.x / 8 : blockIdx.x;
  const int zcs = N / 32, len = N / ysplit / H;
  const size_t xs = (size_t)N * CI, zs = (size_t)N * CO;            // elements per line
  for (int u = lb * per; u < units && u < (lb + 1) * per; ++u) {
    const int zc = u % zcs, ys = (u / zcs) % ysplit, x = u / zcs / ysplit;
    const int y0 = (ys * H + h) * len;
    const int g = zc * 4 + q;
    const int ci = t * 16 + n16;
    const uint32_t xo = (uint32_t)(g * CI + ci) * 16, xp = (uint32_t)((g ? g - 1 : G8 - 1) * CI + ci) * 16,
                   xn = (uint32_t)((g + 1 < G8 ? g + 1 : 0) * CI + ci) * 16, zo = (uint32_t)(g * CO + n16) * 16;
    const bf16* xb = XB + (size_t)((x + dxi - 1) & msk) * N * xs;
    const bf16* zb = dZB + (size_t)x * N * zs;
    auto loadz = [&](int y, uint4 (&d)[MT]) {
      const char* line = reinterpret_cast<const char*>(zb + (size_t)(uint32_t)(y & msk) * zs);
#pragma unroll
      for (int m = 0; m < MT; ++m) d[m] = *reinterpret_cast<const uint4*>(line + zo + m * 256);
    };
    // four steps per turn: dZ lines y - 1 .. y + 2 rotate through d[0..3], X lines
    // y and y + 1 through xr[0..1], without register moves (len is a multiple of 4)
    uint4 d[4][MT];
    XRun xr[2];
#pragma unroll
    for (int k = 0; k < 3; ++k) loadz(y0 - 1 + k, d[k]);
    xr[0].load(xb + (size_t)y0 * xs, xo, xp, xn);
#pragma unroll 1
    for (int s4 = 0; s4 < len; s4 += 4) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int y = y0 + s4 + k;
        loadz(y + 2, d[(k + 3) & 3]);
        xr[(k + 1) & 1].load(xb + (size_t)(uint32_t)((y + 1) & msk) * xs, xo, xp, xn);
        bf16x8 f[3];
        xr[k & 1].taps(f);
        // X line y is the neighbour dy = 1, 0, -1 of dZ lines y - 1, y, y + 1
#pragma unroll
        for (int e = 0; e < 3; ++e)
#pragma unroll
          for (int dz = 0; dz < 3; ++dz)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
              const int a = 3 * (2 - e) + dz;
              acc[a][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, d[(k + e) & 3][m]), f[dz],
                                                                  acc[a][m], 0, 0, 0);
            }
        if (bias) {
#pragma unroll
          for (int m = 0; m < MT; ++m)
            db[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, d[(k + 1) & 3][m]), ones, db[m], 0, 0, 0);
        }
      }
    }
  }
  // the shares add up in order, CO/16 parts of the accumulators at a time
  __shared__ f32x4 sum[3 * TI][10][64];
#pragma unroll
  for (int k = 1; k < H; ++k)
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      __syncthreads();
      if (h == k) {
        sum[role][9][lane] = db[m];
#pragma unroll
        for (int d = 0; d < 9; ++d) sum[role][d][lane] = acc[d][m];
      }
      __syncthreads();
      if (h == 0) {
        db[m] += sum[role][9][lane];
#pragma unroll
        for (int d = 0; d < 9; ++d) acc[d][m] += sum[role][d][lane];
      }
    }
  if (h) return;
  float* out = part + (size_t)blockIdx.x * (27 * CO * CI + CO);
#pragma unroll
  for (int m = 0; m < MT; ++m) {
#pragma unroll
    for (int d = 0; d < 9; ++d)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        out[((size_t)(dxi * 9 + d) * CO + m * 16 + 4 * q + i) * CI + t * 16 + n16] = acc[d][m][i];
    if (bias && n16 == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) out[27 * CO * CI + m * 16 + 4 * q + i] = db[m][i];
    }
  }
}

// N = 16: a K-step of 32 nodes covers two z-lines.  Wavefront w owns neighbour
// line (dx, dy) = (w / 3 - 1, w % 3 - 1) and its three taps; block b sums nodes
// [b chunk, (b + 1) chunk) and writes its partial as above.
template <int CI, int CO>
__global__ void __launch_bounds__(576)
k_wgrad2(const bf16* __restrict__ XB, const bf16* __restrict__ dZB, float* __restrict__ part, int N, int chunk) {
  constexpr int MT = CO / 16, NT = CI / 16;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int n16 = lane & 15, q = lane >> 4, msk = N - 1, G = N >> 3;
  f32x4 acc[3][MT][NT];
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[d][m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float db[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) db[m] = 0.f;
  for (int ks = 0; ks < chunk / 32; ++ks) {
    const size_t node = (size_t)blockIdx.x * chunk + 32 * ks + 8 * q, line = node / N;
    const int g = (int)(node & msk) >> 3, x = (int)(line / N), y = (int)(line & msk);
    bf16x8 a[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const uint4 v = *reinterpret_cast<const uint4*>(dZB + ((node >> 3) * CO + m * 16 + n16) * 8);
      a[m] = __builtin_bit_cast(bf16x8, v);
      if (w == 0) {
        const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) db[m] += b2f((bf16)(u[i] & 0xffff)) + b2f((bf16)(u[i] >> 16));
      }
    }
    const bf16* nl = XB + ((size_t)((x + w / 3 - 1) & msk) * N + ((y + w % 3 - 1) & msk)) * N * CI;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int ci = t * 16 + n16;
      XRun r;
      r.load(nl, (uint32_t)(g * CI + ci) * 16, (uint32_t)((g ? g - 1 : G - 1) * CI + ci) * 16,
             (uint32_t)((g + 1 < G ? g + 1 : 0) * CI + ci) * 16);
      bf16x8 f[3];
      r.taps(f);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int d = 0; d < 3; ++d)
          acc[d][m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], f[d], acc[d][m][t], 0, 0, 0);
    }
  }
  float* out = part + (size_t)blockIdx.x * (27 * CO * CI + CO);
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          out[((size_t)(3 * w + d) * CO + m * 16 + 4 * q + i) * CI + t * 16 + n16] = acc[d][m][t][i];
  if (w == 0) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      float v = db[m];
      v += __shfl_xor(v, 16, 64);
      v += __shfl_xor(v, 32, 64);
      if (q == 0) out[27 * CO * CI + m * 16 + n16] = v;
    }
  }
}

// out[i] = sum over blocks of part[b][i], i < n, in a fixed order: thread group
// k of a block's 8 sums the partials b = k (mod 8), loads in batches of 8 ahead
// of their additions, and the eight sums are added in order.  The four layers
// of 3-32-32-32-3 at 128^3: 75 us over 512 partials with one thread per entry,
// 34 us like this, 23 us over k_wgrad3's 256.
static __global__ void __launch_bounds__(256)
k_reduce_parts(const float* __restrict__ part, int nblk, int n, float* __restrict__ out) {
  __shared__ float sh[8][32];
  const int e = threadIdx.x & 31, k = threadIdx.x >> 5;
  const int i = blockIdx.x * 32 + e;
  float s = 0.f;
  if (i < n) {
    int b = k;
    for (; b + 56 < nblk; b += 64) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = part[(size_t)(b + 8 * u) * n + i];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += v[u];
    }
    for (; b < nblk; b += 8) s += part[(size_t)b * n + i];
  }
  sh[k][e] = s;
  __syncthreads();
  if (k == 0 && i < n) {
#pragma unroll
    for (int u = 1; u < 8; ++u) s += sh[u][e];
    out[i] = s;
  }
}

// Rows of bf16 values of EN nodes staged in LDS (sh[node][c], c < cn real
// channels) -> an activation of CP channels (the others zero) in the layout of
// N (channels-last for N < 16, else tiled), and with AB its node-blocked copy;
// 16-byte stores.  Nodes node0 .. node0 + n - 1 (n a multiple of 8).
constexpr int EN = 256;
__device__ __forceinline__ void emit_rows(const bf16* sh, int cn, int CP, size_t node0, int n, int N,
                                          bf16* __restrict__ A, bf16* __restrict__ AB) {
  const int G = CP / 8;
  for (int e = threadIdx.x; e < n * G; e += blockDim.x) {
    const int k = e % n, g = e / n;                       // node fastest
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = 8 * g + 2 * i;
      const uint32_t lo = c < cn ? sh[k * cn + c] : 0u, hi = c + 1 < cn ? sh[k * cn + c + 1] : 0u;
      w[i] = lo | (hi << 16);
    }
    const size_t node = node0 + k;
    size_t o;
    if (N < 16) {
      o = node * CP + 8 * g;
    } else {
      const int z = (int)(node & (N - 1));
      o = (node - z) * CP + (N >= 64 ? tiled_at<4>(z, 8 * g, CP) : N == 32 ? tiled_at<2>(z, 8 * g, CP)
                                                                     : tiled_at<1>(z, 8 * g, CP));
    }
    *reinterpret_cast<uint4*>(A + o) = make_uint4(w[0], w[1], w[2], w[3]);
  }
  if (!AB) return;
  for (int e = threadIdx.x; e < n / 8 * CP; e += blockDim.x) {
    const int c = e % CP, g = e / CP;                     // channel fastest
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t lo = c < cn ? sh[(8 * g + 2 * i) * cn + c] : 0u, hi = c < cn ? sh[(8 * g + 2 * i + 1) * cn + c] : 0u;
      w[i] = lo | (hi << 16);
    }
    *reinterpret_cast<uint4*>(AB + ((node0 / 8 + g) * CP + c) * 8) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// Input rows x[node][cin] FP32 -> bf16 activation of CP channels (and blocked copy).
static __global__ void __launch_bounds__(256)
k_pack_input(const float* __restrict__ x, int cin, int CP, size_t nodes, int N, bf16* __restrict__ A,
             bf16* __restrict__ AB) {
  __shared__ bf16 sh[EN * 32];
  const size_t node0 = (size_t)blockIdx.x * EN;
  const int n = nodes - node0 < EN ? (int)(nodes - node0) : EN;
  for (int e = threadIdx.x; e < n * cin; e += 256) sh[e] = f2b(x[node0 * cin + e]);
  __syncthreads();
  emit_rows(sh, cin, CP, node0, n, N, A, AB);
}

// Master FP32 weights w[tap][co][ci] -> bf16 W[tap][co][ci] and Wt[tap][ci][co].
static __global__ void k_pack_weights(const float* __restrict__ w, int CI, int CO, bf16* __restrict__ Wb,
                                      bf16* __restrict__ Wt) {
  const int n = 27 * CO * CI;
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < n; e += gridDim.x * blockDim.x) {
    const int tap = e / (CO * CI), co = (e / CI) % CO, ci = e % CI;
    const bf16 b = f2b(w[e]);
    Wb[e] = b;
    Wt[((size_t)tap * CI + ci) * CO + co] = b;
  }
}

// Mean squared error over nodes x cout: dY[node][co] = 2 (y - t) / (nodes cout)
// for co < cout (0 for padding channels) as an activation and its blocked copy,
// per-block sums of (y - t)^2.  y and t are rows of cout channels.
static __global__ void __launch_bounds__(256)
k_mse(const float* __restrict__ y, const float* __restrict__ t, int cout, int CP, size_t nodes, int N,
      bf16* __restrict__ dY, bf16* __restrict__ dYB, double* __restrict__ part) {
  __shared__ bf16 rows[EN * 32];
  __shared__ double sh[256];
  double s = 0.0;
  const double scale = 2.0 / ((double)nodes * cout);
  for (size_t node0 = (size_t)blockIdx.x * EN; node0 < nodes; node0 += (size_t)gridDim.x * EN) {
    const int n = nodes - node0 < EN ? (int)(nodes - node0) : EN;
    for (int e = threadIdx.x; e < n * cout; e += 256) {
      const double d = (double)y[node0 * cout + e] - (double)t[node0 * cout + e];
      s += d * d;
      rows[e] = f2b((float)(scale * d));
    }
    __syncthreads();
    emit_rows(rows, cout, CP, node0, n, N, dY, dYB);
    __syncthreads();
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (threadIdx.x < k) sh[threadIdx.x] += sh[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// Adam on the FP32 master parameters (Kingma & Ba 2015), step t >= 1.
static __global__ void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                              float* __restrict__ v, int n, float lr, float b1, float b2, float eps, int t) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float mh = mi / (1.f - powf(b1, (float)t)), vh = vi / (1.f - powf(b2, (float)t));
  w[i] -= lr * mh / (sqrtf(vh) + eps);
}

}  // namespace cnn
}  // namespace ld
