// Droplet kernels: cosine-kernel gather/deposit (particles.py:6-35, 435-577),
// droplet RHS (particles.py:817-837) and its RK4 stage update
// (forced-dns-sm.py:337-362 for the droplet rows).
//
// Engine state is structure-of-arrays: positions in FP64 (pos[c*cap + p],
// unwrapped, as the reference accumulates them), velocity and mass in PT
// (vm[c*cap + p], c = vx, vy, vz, m/M0).  The step's stage kernel takes 4 or 8
// lanes per droplet, the gathers of sorted rows four lanes or one thread per
// row, the rest one thread per row.
#pragma once
#include "ld_kernels.hpp"
#include <type_traits>

namespace ld {

// The 4-point cosine weights of one axis: nodes i-1..i+2 with i = floor(x/dx),
// w = (1 + cos((x - X_j) pi / (2 dx))) / 4 (particles.py:12, 16, 456).  X_j is
// taken unwrapped (j*dx), which equals the reference's wrapped X[j mod N]
// through the period 4*dx of the kernel (N % 4 == 0).
template <int N> __device__ __forceinline__ int wrapIdx(int j) {
  int jj = j % N;
  return jj < 0 ? jj + N : jj;
}
// The four weights of one axis from one sincos: with
// theta = (x - i0 dx) pi / (2 dx), i0 = floor(x/dx) - 1, node i0 + a has the
// argument theta - a pi/2, so its weight is (1 + {cos, sin, -cos, -sin}(theta))/4.
// The four weights then sum to 1 in exact arithmetic.  Returns i0.
__device__ __forceinline__ int cosW4(double x, double dx, double pi_2dx, double w[4]) {
  const int i0 = (int)floor(x / dx) - 1;
  double sn, cs;
  sincos((x - (double)i0 * dx) * pi_2dx, &sn, &cs);
  w[0] = 0.25 * (1.0 + cs);
  w[1] = 0.25 * (1.0 + sn);
  w[2] = 0.25 * (1.0 - cs);
  w[3] = 0.25 * (1.0 - sn);
  return i0;
}
template <int N>
__device__ __forceinline__ void cosWeights(double x, double dx, double pi_2dx, int idx[4], double w[4]) {
  const int i0 = cosW4(x, dx, pi_2dx, w);
#pragma unroll
  for (int a = 0; a < 4; ++a) idx[a] = wrapIdx<N>(i0 + a);
}

// sin and cos of an FP64 angle in precision G (FP32: of the angle rounded to FP32).
template <typename G> __device__ __forceinline__ void sincosGT(double th, G& s, G& c) {
  if constexpr (sizeof(G) == 4) {
    sincosf((float)th, &s, &c);
  } else {
    sincos(th, &s, &c);
  }
}

// sin and cos of the stencil angle (x - i0 dx) pi / (2 dx), which lies in
// [pi/2, pi).  FP64: as sincospi of the angle over pi (no reduction of large
// arguments, whose code costs registers and scratch memory).
template <typename G>
__device__ __forceinline__ void sincosStencil(double x, int i0, double dx, double inv_dx, double pi_2dx, G& s, G& c) {
#pragma clang fp contract(off)
  const double d = fma(-(double)i0, dx, x);
  if constexpr (sizeof(G) == 4) sincosGT<G>(d * pi_2dx, s, c);
  else sincospi(d * (0.5 * inv_dx), &s, &c);
}

// Periodic wrap of one coordinate, x mod L with numpy's sign convention
// (particles.py:269 `x[:, :d] %= L`).
__device__ __forceinline__ double wrapL(double x, double L) {
  double r = fmod(x, L);
  if (r < 0.0) r += L;
  // a non-finite position must not become an out-of-range stencil index
  if (!(r >= 0.0 && r <= L)) r = 0.0;
  return r;
}

// The step's droplet kernels (stage gather, sort bins, brick and fallback
// deposits) wrap and bin positions with multiplications by 1/L and 1/dx
// instead of fmod and divisions; all of them use these same three functions,
// so their cells agree.  The wrapped position can differ from fmod's in the
// last bit, and a stencil origin can differ by one cell when x/dx is within
// an ulp of an integer; the cosine kernel gives the node at distance 2 dx
// zero weight, so both stencils give the same interpolant.
__device__ __forceinline__ double wrapFast(double x, double L, double invL) {
  double r = fma(-L, floor(x * invL), x);
  r = r < 0.0 ? r + L : r;
  r = r >= L ? r - L : r;
  if (!(r >= 0.0 && r < L)) r = 0.0;   // a non-finite position must not become an out-of-range index
  return r;
}
// cell of a wrapped position, clamped to [0, N)
template <int N> __device__ __forceinline__ int cellOf(double xw, double inv_dx) {
  const int c = (int)(xw * inv_dx);
  return c < 0 ? 0 : (c > N - 1 ? N - 1 : c);
}
// stencil origin i0 = floor(x / dx) - 1 (nodes i0 .. i0 + 3)
__device__ __forceinline__ int originOf(double x, double inv_dx) { return (int)floor(x * inv_dx) - 1; }

// cosW4 with the origin from originOf, the sines and cosines taken in precision G
// (the angle in FP64).
template <typename G>
__device__ __forceinline__ int cosW4F(double x, double dx, double inv_dx, double pi_2dx, G w[4]) {
  const int i0 = originOf(x, inv_dx);
  G sn, cs;
  sincosStencil<G>(x, i0, dx, inv_dx, pi_2dx, sn, cs);
  const G q = (G)0.25;
  w[0] = q * ((G)1 + cs);
  w[1] = q * ((G)1 + sn);
  w[2] = q * ((G)1 - cs);
  w[3] = q * ((G)1 - sn);
  return i0;
}

// Geometry of one droplet's stencil.
template <int N> struct Stencil {
  int i0;
  int iy[4], iz[4];
  double wx[4], wy[4], wz[4];
  __device__ __forceinline__ void set(const double xw[3], double dx, double pi_2dx) {
    i0 = cosW4(xw[0], dx, pi_2dx, wx);
    cosWeights<N>(xw[1], dx, pi_2dx, iy, wy);
    cosWeights<N>(xw[2], dx, pi_2dx, iz, wz);
  }
  __device__ __forceinline__ int xa(int a) const { return wrapIdx<N>(i0 + a); }
  __device__ __forceinline__ double wxa(int a) const { return wx[a]; }
};

// Gather of NC fields f[c*R + idx] (particles.py:6-20, 454-509): for each x
// node a, sum over the (y, z) nodes, then weight by w_x(a).
template <typename T, int N, int NC>
__device__ __forceinline__ void gatherN(const Stencil<N>& s, const T* __restrict__ f, size_t R, double out[NC]) {
#pragma unroll
  for (int c = 0; c < NC; ++c) out[c] = 0.0;
#pragma unroll 1
  for (int a = 0; a < 4; ++a) {
    double t[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) t[c] = 0.0;
    const size_t plane = (size_t)s.xa(a) * N;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const size_t row = (plane + s.iy[b]) * N;
#pragma unroll
      for (int cc = 0; cc < 4; ++cc) {
        const double wyz = s.wy[b] * s.wz[cc];
        const size_t o = row + s.iz[cc];
#pragma unroll
        for (int c = 0; c < NC; ++c) t[c] += (double)f[c * R + o] * wyz;
      }
    }
    const double wx = s.wxa(a);
#pragma unroll
    for (int c = 0; c < NC; ++c) out[c] += t[c] * wx;
  }
}

// Gather of the stage density with the lazy clip (nStage) applied per node.
template <typename T, int N>
__device__ __forceinline__ double gatherDensity(const Stencil<N>& s, const T* __restrict__ n, const double* __restrict__ clip) {
  double out = 0.0;
  const bool doclip = clip[2] != 0.0;
#pragma unroll 1
  for (int a = 0; a < 4; ++a) {
    double t = 0.0;
    const size_t plane = (size_t)s.xa(a) * N;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const size_t row = (plane + s.iy[b]) * N;
#pragma unroll
      for (int cc = 0; cc < 4; ++cc) {
        double v = (double)n[row + s.iz[cc]];
        if (doclip && v < 0.0) v = 0.0;
        t += v * (s.wy[b] * s.wz[cc]);
      }
    }
    out += t * s.wxa(a);
  }
  if (doclip) out = (out * clip[0]) / clip[1];
  return out;
}

// Deposit W into c with the same kernel, divided by the cell volume
// (particles.py:23-35, 529-575).  Atomic adds (the reference's prange loop
// races on the same updates).
template <typename T, int N>
__device__ __forceinline__ void deposit(const Stencil<N>& s, double W, double inv_vol, T* c) {
#pragma unroll 1
  for (int a = 0; a < 4; ++a) {
    const double wa = W * s.wxa(a);
    const size_t plane = (size_t)s.xa(a) * N;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const double wab = wa * s.wy[b];
      const size_t row = (plane + s.iy[b]) * N;
#pragma unroll
      for (int cc = 0; cc < 4; ++cc) {
        unsafeAtomicAdd(&c[row + s.iz[cc]], (T)(wab * s.wz[cc] * inv_vol));
      }
    }
  }
}

struct DropPhys {
  double L, dx, pi_2dx, inv_vol;
  double factor, growth, st_s, tau_eta, g;
  double invL, inv_dx, inv_factor;
};

// Growth rate W (= mdot / M0) and St tau_eta of a droplet at one stage
// coordinate (particles.py:823-828).  vp: velocity, m: mass/M0.  I: the 7
// interpolated components [u, v, n].
__device__ __forceinline__ double dropletGrowth(const DropPhys& P, const double vp[3], double m, const double I[7],
                                                double& W) {
#pragma clang fp contract(off)
  const double st = pow(m / P.factor, 2.0 / 3.0);                          // :823
  const double d0 = vp[0] - I[3], d1 = vp[1] - I[4], d2 = vp[2] - I[5];
  const double nrm = sqrt(fma(d2, d2, fma(d1, d1, d0 * d0)));
  const double q = 1.0 + sqrt(P.st_s / st);
  W = P.growth * (q * q) * I[6] * nrm;                                      // :828
  return st * P.tau_eta;
}
// Droplet RHS at one stage coordinate (particles.py:823-835): rhs[7] and W.
__device__ __forceinline__ void dropletRhs(const DropPhys& P, const double vp[3], double m, const double I[7],
                                           double rhs[7], double& W) {
  const double den = dropletGrowth(P, vp, m, I, W);
  rhs[0] = vp[0]; rhs[1] = vp[1]; rhs[2] = vp[2];                           // :831
  rhs[3] = (I[0] - vp[0]) / den;                                            // :832
  rhs[4] = (I[1] - vp[1]) / den;
  rhs[5] = (I[2] - vp[2]) / den - P.g;                                      // :834
  rhs[6] = W;                                                               // :835
}

// The growth rate in single precision for the FP32 form (velocities and masses
// are FP32 there); St from exp2(2/3 log2(m / factor)).
__device__ __forceinline__ float dropletGrowth(const DropPhys& P, const float vp[3], float m, const float I[7],
                                               float& W) {
#pragma clang fp contract(off)
  const float st = exp2f((2.0f / 3.0f) * log2f(m * (float)P.inv_factor));   // :823
  const float d0 = vp[0] - I[3], d1 = vp[1] - I[4], d2 = vp[2] - I[5];
  const float nrm = sqrtf(fmaf(d2, d2, fmaf(d1, d1, d0 * d0)));
  const float q = 1.0f + sqrtf((float)P.st_s / st);
  W = (float)P.growth * (q * q) * I[6] * nrm;                                // :828
  return st * (float)P.tau_eta;
}
// x / den (FP32: by the reciprocal), less g
__device__ __forceinline__ double dragTerm(double x, double den, double g) { return x / den - g; }
__device__ __forceinline__ float dragTerm(float x, float den, float g) { return fmaf(x, 1.0f / den, -g); }
__device__ __forceinline__ double fmaG(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float fmaG(float a, float b, float c) { return fmaf(a, b, c); }

// ------------------------------------------------------------ lane quads
// v of the lane L of the caller's quad of lanes (all four active), and of the
// lane whose number in the quad differs in the bits X: DPP moves, no LDS.
template <int CTRL, typename G> __device__ __forceinline__ G dppMove(G v) {
  if constexpr (sizeof(G) == 4) {
    return __builtin_bit_cast(G, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
  } else {
    const long long b = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(G, ((long long)hi << 32) | (unsigned int)lo);
  }
}
template <int L, typename G> __device__ __forceinline__ G quadLane(G v) { return dppMove<L * 0x55>(v); }
template <int X, typename G> __device__ __forceinline__ G quadXor(G v) { return dppMove<X == 1 ? 0xB1 : 0x4E>(v); }

// ------------------------------------------------------------ spatial sort
// Droplets are reordered by spatial bin once per step (counting sort), so
// that lanes of a wavefront gather from and deposit into the same cache
// lines.  Bins are cubes of BS = max(2, N/128) grid cells; bins are numbered
// tile-major (tiles of TS^3 bins = TC^3 cells, the deposit bricks), so the
// droplets of one tile are contiguous; tiles run along z in columns (long
// contiguous z-runs of the fields), and the columns follow a Morton (Z-order)
// curve in (x, y), so the columns a run of gather blocks covers are mostly
// neighbours and share their halo nodes in one L2.
template <int N> struct Bins {
  static constexpr int BS = (N / 128 > 2) ? N / 128 : 2;
  static constexpr int B = N / BS;
  static constexpr int NB = B * B * B;
  static constexpr int TC = (N >= 32) ? 16 : 8;     // tile side in cells
  static constexpr int TS = TC / BS;                 // tile side in bins
  static constexpr int NTt = B / TS;                 // tiles per side
  static_assert(TC % BS == 0 && B % TS == 0, "bin tiles");
  static_assert((NTt & (NTt - 1)) == 0 && NTt <= 256, "tiles per side: a power of two");
  // bits of v spread to every second position (v < 256)
  static __device__ __forceinline__ int spread2(int v) {
    int r = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) r |= ((v >> i) & 1) << (2 * i);
    return r;
  }
  // every second bit of v, packed (the inverse of spread2)
  static __device__ __forceinline__ int pack2(int v) {
    int r = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) r |= ((v >> (2 * i)) & 1) << i;
    return r;
  }
  // first cell of tile number `tile` (key / TS^3)
  static __device__ __forceinline__ void tileCell(int tile, int& cx, int& cy, int& cz) {
    const int col = tile / NTt;
    cx = pack2(col >> 1) * TC; cy = pack2(col) * TC; cz = (tile % NTt) * TC;
  }
  // key of bin (bx, by, bz): tile columns along z, the columns in Morton order
  // of (tile x, tile y); x-major inside the tile
  static __device__ __forceinline__ int key(int bx, int by, int bz) {
    const int tile = ((spread2(bx / TS) << 1) | spread2(by / TS)) * NTt + bz / TS;
    return tile * (TS * TS * TS) + ((bx % TS) * TS + by % TS) * TS + bz % TS;
  }
};

// ------------------------------------------------------------ fused RK stage
template <typename T, typename PT> struct PStage {
  int np, cap, stage;          // stage 0..3
  double* x0; PT* v0;          // RK base (unwrapped); final stage writes the new state here
  double* sx; PT* sv;          // sump accumulator
  PT* kx; PT* kv;              // stage rhs (read: previous stage, write: this stage); dx/dt is
                               // the stage velocity, which PT holds exactly
  const V4<T>* gu; const V4<T>* gv;   // gather records {u, 0} (recU) and {v, n_stage} (recV); one array
  double4* dep;                // out: wrapped stage position and W per slot (brick deposit input)
  int* flist; int* fcount;     // out: slots whose stage bin moved > 1 bin since the sort
  unsigned long long* wmax;    // out: largest W > 0 of the launch (bits of positive doubles, WSLOTS slots); zero before
  double ah, wh;               // a_s * h, w_s * h
  DropPhys P;
  size_t rs;                   // realization stride in bytes (batched launches)
  __device__ PStage shifted() const {
    PStage a = *this;
    a.x0 = rsel1(x0, rs); a.v0 = rsel1(v0, rs); a.sx = rsel1(sx, rs); a.sv = rsel1(sv, rs);
    a.kx = rsel1(kx, rs); a.kv = rsel1(kv, rs); a.gu = rsel1(gu, rs); a.gv = rsel1(gv, rs);
    a.dep = rsel1(dep, rs); a.flist = rsel1(flist, rs); a.fcount = rsel1(fcount, rs); a.wmax = rsel1(wmax, rs);
    return a;
  }
};

// One RK4 stage of every droplet: stage coordinate X0 + a h k_prev
// (forced-dns-sm.py:347, 352, 357), wrap (particles.py:269), gather of
// [u, v, n] (:826), growth rate and deposit (:828-829), RHS (:831-835) and
// sump accumulation (forced-dns-sm.py:342-358).
//
// NL = 4 or 8 lanes per droplet.  Lane c of a quad owns z-node c of the 4x4x4
// stencil, so a load touches one 64-byte run of each droplet; with 8 lanes the
// first quad takes the u records and the second the v records, which lie on the
// same 128-byte lines, so a line is asked for once instead of twice, by half as
// many droplets at a time.  Around the gather the lanes of a quad split the
// droplet's components instead of repeating each other: lane c forms axis c's
// wrap, cell and sincos (lane 3 repeats z) and loads, updates and stores
// component c of the position and of (velocity, mass); what all need moves by
// DPP.  Both give the same bits: products and sums are fused as written, not by
// the compiler, which does it differently in the two.
// Measured per launch (one lane forming everything, one slot for the largest W
// -> 4 lanes -> 8 lanes): 10^6 droplets at 256^3 FP32 288 -> 300 -> 278 us (8
// lanes, four blocks per CU: 267); 10^7 at 512^3 FP32 2470 -> 2562 -> 2358
// (2262); 10^5 in each of 64 times 64^3 FP32 895 -> 871 -> 929 (4 lanes, four
// blocks: 834); 10^5 at 64^3 FP32 26.2 -> 15.0 -> 17.7; 123457 at 128^3 FP64
// 79.5 -> 83.7 -> 72.7.  Sparse droplets (each of the 28 lines of a stencil
// serves few of them) are bound by the lines, dense ones by instructions:
// Engine::eight_lanes.
// BAT: batched launch (blockIdx.z = realization); the single-realization
// instantiation skips the pointer offsets and their registers.
template <typename T, typename PT, int N, bool BAT, int NL>
__global__ void __launch_bounds__(256)
k_particles_stage(PStage<T, PT> A0) {
#pragma clang fp contract(off)
  const PStage<T, PT> A = BAT ? A0.shifted() : A0;
  // XCD-aware mapping: the 8 XCDs take consecutive blocks round-robin; give
  // each XCD one contiguous range of (spatially sorted) droplets so its L2
  // sees one region of the fields.
  const int nb = gridDim.x, per = nb / 8;
  const int lb = (blockIdx.x % 8) * per + blockIdx.x / 8;
  static_assert(NL == 4 || NL == 8, "one or two quads per droplet");
  const int p = lb * (256 / NL) + threadIdx.x / NL, c = threadIdx.x & 3;
  const bool hi = NL == 8 && (threadIdx.x & 4);         // second quad: v records
  const bool live = p < A.np;
  const int pp = live ? p : 0;
  constexpr size_t R = (size_t)N * N * N;
  const int cap = A.cap;
  // Loads are grouped into two round trips (stage position; the gather with
  // velocity, mass and the sump inputs), with uniform pointer selects or
  // branches (stage 0 takes k = 0 and the sump inputs from the RK base).
  const bool s0 = A.stage == 0;
  const double ah = s0 ? 0.0 : A.ah;
  const int ax = c < 3 ? c : 2;
  const double x0c = A.x0[ax * cap + pp];
  double kxc = 0.0;
  if (!s0) kxc = (double)A.kx[ax * cap + pp];
  const double L = A.P.L, dx = A.P.dx, pi_2dx = A.P.pi_2dx, invL = A.P.invL, inv_dx = A.P.inv_dx;
  const double xw = wrapFast(fma(ah, kxc, x0c), L, invL);
  // one sincos per axis (cosW4); node i0 + a has weight (1 +- {cos, sin})/4.
  // The angles and the sincos are FP64; the weights and the gather sums are
  // kept in the field precision GT (FP32 fields: FP32 sums of 64 terms).
  using GT = std::conditional_t<sizeof(T) == 4, float, double>;
  // deposit input for the brick pass (k_brick_deposit), written before the
  // gather so the wrapped position holds no registers across it: the wrapped
  // stage position now, W after the RHS.  Slots whose stage bin left the
  // +-1-bin window around their sorted bin go to the fallback list.
  bool far;
  {
    // bins exactly as k_bin_count forms them
    const int cs = cellOf<N>(xw, inv_dx), c0 = cellOf<N>(wrapFast(x0c, L, invL), inv_dx);
    const int d = ((cs / Bins<N>::BS - c0 / Bins<N>::BS) % Bins<N>::B + Bins<N>::B) % Bins<N>::B;
    int f = d > 1 && d < Bins<N>::B - 1;
    f |= quadXor<1>(f);
    f |= quadXor<2>(f);
    far = f != 0;
  }
  if (live) {
    if (c < 3 && !hi) reinterpret_cast<double*>(A.dep + p)[c] = xw;
    if (far && c == 0 && !hi) A.flist[atomicAdd(A.fcount, 1)] = p;
  }
  const int o0 = originOf(xw, inv_dx);
  // the angles are formed in FP64; their sines and cosines are taken in the
  // weight precision GT (the FP32 form rounds the angle in [pi/2, pi) to FP32)
  GT snc, csc;
  sincosStencil<GT>(xw, o0, dx, inv_dx, pi_2dx, snc, csc);
  const int i0 = quadLane<0>(o0), j0 = quadLane<1>(o0), k0 = quadLane<2>(o0);
  const GT xsn = quadLane<0>(snc), xcs = quadLane<0>(csc), ysn = quadLane<1>(snc), ycs = quadLane<1>(csc),
           zsn = quadLane<2>(snc), zcs = quadLane<2>(csc);
  const GT q = (GT)0.25;
  const GT wy[4] = {q * ((GT)1 + ycs), q * ((GT)1 + ysn), q * ((GT)1 - ycs), q * ((GT)1 - ysn)};
  int iy[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) iy[b] = wrapIdx<N>(j0 + b);
  const GT wz = q * ((GT)1 + ((c & 2) ? (GT)-1 : (GT)1) * ((c & 1) ? zsn : zcs));
  const GT gxs = xsn, gxc = xcs;
  const int iz = wrapIdx<N>(k0 + c);
  // stage velocity and mass (v0 + a h kv) and the sump inputs (x0, v0 at
  // stage 0, else the accumulators), issued before the gather so that their
  // round trip overlaps its loads (measured 0.320 -> 0.306 ms per launch at
  // 256^3 with 10^6 droplets, though occupancy drops from 5 to 4 waves/SIMD)
  const PT* kvp = s0 ? A.v0 : A.kv;
  const double* sxp = s0 ? A.x0 : A.sx;
  const PT* svp = s0 ? A.v0 : A.sv;
  const PT v0c = A.v0[c * cap + pp], kvc = kvp[c * cap + pp], prv = svp[c * cap + pp];
  const double prx = sxp[ax * cap + pp];
  // gather: this lane's z node, all (x, y) nodes; two 16-byte records per node
  PT I[7];
  if constexpr (NL == 8) {
    // this quad's record of each node, all 16 loads ahead of the sums
    GT Ig[4] = {(GT)0, (GT)0, (GT)0, (GT)0};
    if (live) {
      V4<T> U[16];
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const uint32_t plane = (uint32_t)wrapIdx<N>(i0 + a) * N;
#pragma unroll
        for (int b = 0; b < 4; ++b)
          U[a * 4 + b] = ldRec<T, N>(A.gu, recU((plane + (uint32_t)iy[b]) * N + (uint32_t)iz) | (hi ? 4u : 0u));
      }
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const GT wx = (GT)0.25 * ((GT)1 + ((a & 2) ? (GT)-1 : (GT)1) * ((a & 1) ? gxs : gxc));
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const GT w = wy[b] * wx;
          const V4<T>& u = U[a * 4 + b];
          Ig[0] = fmaG((GT)u.x, w, Ig[0]);
          Ig[1] = fmaG((GT)u.y, w, Ig[1]);
          Ig[2] = fmaG((GT)u.z, w, Ig[2]);
          Ig[3] = fmaG((GT)u.w, w, Ig[3]);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      GT v = Ig[k] * wz;
      v += quadXor<1>(v);
      v += quadXor<2>(v);
      const GT o = dppMove<0x141>(v);          // the other quad's sum (mirrored half row)
      if (k < 3) I[k] = (PT)(hi ? o : v);
      I[3 + k] = (PT)(hi ? v : o);
    }
  } else {
    GT Ig[7];
#pragma unroll
    for (int k = 0; k < 7; ++k) Ig[k] = (GT)0;
    // FP32 fields: all 32 record loads are written ahead of the sums, so the
    // compiler keeps about a dozen in flight per lane (at 5 waves per SIMD);
    // this measured faster than a plane-by-plane loop at 8 waves per SIMD.
    // FP64 records are twice the size; they keep the loop.
    if (sizeof(T) == 4 && live) {
      V4<T> U[16], V[16];
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const uint32_t plane = (uint32_t)wrapIdx<N>(i0 + a) * N;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const uint32_t o = (plane + (uint32_t)iy[b]) * N + (uint32_t)iz;
          U[a * 4 + b] = ldRec<T, N>(A.gu, recU(o));
          V[a * 4 + b] = ldRec<T, N>(A.gv, recV(o));
        }
      }
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const GT wx = (GT)0.25 * ((GT)1 + ((a & 2) ? (GT)-1 : (GT)1) * ((a & 1) ? gxs : gxc));
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const GT w = wy[b] * wx;
          const V4<T>& u = U[a * 4 + b];
          const V4<T>& v = V[a * 4 + b];
          Ig[0] = fmaG((GT)u.x, w, Ig[0]);
          Ig[1] = fmaG((GT)u.y, w, Ig[1]);
          Ig[2] = fmaG((GT)u.z, w, Ig[2]);
          Ig[3] = fmaG((GT)v.x, w, Ig[3]);
          Ig[4] = fmaG((GT)v.y, w, Ig[4]);
          Ig[5] = fmaG((GT)v.z, w, Ig[5]);
          Ig[6] = fmaG((GT)v.w, w, Ig[6]);
        }
      }
    } else if (live) {
#pragma unroll 1
      for (int a = 0; a < 4; ++a) {
        const GT wx = (GT)0.25 * ((GT)1 + ((a & 2) ? (GT)-1 : (GT)1) * ((a & 1) ? gxs : gxc));
        const uint32_t plane = (uint32_t)wrapIdx<N>(i0 + a) * N;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const uint32_t o = (plane + (uint32_t)iy[b]) * N + (uint32_t)iz;   // < N^3 <= 2^27
          const GT w = wy[b] * wx;
          const V4<T> U = ldRec<T, N>(A.gu, recU(o));
          const V4<T> V = ldRec<T, N>(A.gv, recV(o));
          Ig[0] = fmaG((GT)U.x, w, Ig[0]);
          Ig[1] = fmaG((GT)U.y, w, Ig[1]);
          Ig[2] = fmaG((GT)U.z, w, Ig[2]);
          Ig[3] = fmaG((GT)V.x, w, Ig[3]);
          Ig[4] = fmaG((GT)V.y, w, Ig[4]);
          Ig[5] = fmaG((GT)V.z, w, Ig[5]);
          Ig[6] = fmaG((GT)V.w, w, Ig[6]);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < 7; ++k) {
      GT v = Ig[k] * wz;
      v += quadXor<1>(v);
      v += quadXor<2>(v);
      I[k] = (PT)v;
    }
  }
  // lane c's velocity component or, c == 3, the mass, and the droplet's four
  const PT vc = fmaG((PT)ah, kvc, v0c);
  const PT vp[3] = {quadLane<0>(vc), quadLane<1>(vc), quadLane<2>(vc)};
  PT W = (PT)0;
  const PT den = dropletGrowth(A.P, vp, quadLane<3>(vc), I, W);
  const PT Ic = c == 0 ? I[0] : c == 1 ? I[1] : I[2];
  const PT drag = dragTerm(Ic - vc, den, c == 2 ? (PT)A.P.g : (PT)0);      // :832-834
  const PT rc = c < 3 ? drag : W;                                          // :835
  // largest growth rate of the launch: the bound of the deposits' fixed-point
  // scale.  A NaN or negative W (not a growth) makes it infinite, so the
  // deposit writes NaN everywhere, as the reference's would spread it.
  {
    __shared__ PT wm[4];
    PT v = !live ? (PT)0 : (W > (PT)0 ? W : (W == (PT)0 ? (PT)0 : (PT)INFINITY));
#pragma unroll
    for (int off = 32; off > NL / 2; off >>= 1) {      // a droplet's lanes hold one W
      const PT o = __shfl_xor(v, off, 64);
      v = o > v ? o : v;
    }
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
      const PT a = wm[0] > wm[1] ? wm[0] : wm[1], b = wm[2] > wm[3] ? wm[2] : wm[3], m = a > b ? a : b;
      if (m > (PT)0) atomicMax(A.wmax + wslot(blockIdx.x), (unsigned long long)__double_as_longlong((double)m));
    }
  }
  if (!live || hi) return;
  // sump (forced-dns-sm.py:337, 342-358); the last stage writes the new state
  double* dxp = A.stage == 3 ? A.x0 : A.sx;
  PT* dvp = A.stage == 3 ? A.v0 : A.sv;
  dvp[c * cap + p] = fmaG((PT)A.wh, rc, prv);
  if (A.stage < 3) A.kv[c * cap + p] = rc;
  if (c < 3) {
    dxp[c * cap + p] = fma(A.wh, (double)vc, prx);                           // :831
    if (A.stage < 3) A.kx[c * cap + p] = vc;
  } else {
    // a fallback slot stores -W so the brick pass (which takes W > 0) skips it
    reinterpret_cast<double*>(A.dep + p)[3] = far ? -(double)W : (double)W;
  }
}

// ------------------------------------------------------------ fallback deposit
// Fallback deposit of the slots that moved more than one bin since the sort, by
// extra blocks of the brick launch (one launch instead of three: on small grids
// the density chain is a sequence of launches of a few microseconds each: with
// the counters' two fills gone as well, ten steps at 64^3 FP64 went from 4.85
// to 4.40 ms; at 256^3 and above the step is unchanged).
// Deterministic like the bricks: each slot's 64 node values are added as 64-bit
// fixed-point integers to the scratch field fx (zero between stages; integer
// sums do not depend on the order of the additions), with the scale 2^e of the
// largest value any node can reach (slots x Wmax / dx^3 / 8); the z pass that
// reads the deposit adds fx to it and clears it (OpZFwdFc).
template <typename T, int N>
__device__ __forceinline__ void fallbackAccum(const double4* __restrict__ dep, const int* __restrict__ flist, int nf,
                                              unsigned long long wmax_bits, unsigned long long* fx, const DropPhys& P,
                                              int first, int stride) {
  const FallbackScale sc(nf, wmax_bits, P.inv_vol);
  if (!sc.finite) return;
  using GT = std::conditional_t<sizeof(T) == 4, float, double>;
  for (int f = first; f < nf; f += stride) {
    const double4 d = dep[flist[f]];
    const double w = -d.w;                       // fallback slots carry -W
    if (!(w > 0.0)) continue;
    GT wx[4], wy[4], wz[4];
    const int i0 = cosW4F<GT>(d.x, P.dx, P.inv_dx, P.pi_2dx, wx), j0 = cosW4F<GT>(d.y, P.dx, P.inv_dx, P.pi_2dx, wy),
              k0 = cosW4F<GT>(d.z, P.dx, P.inv_dx, P.pi_2dx, wz);
    const double W = w * P.inv_vol * sc.scale;
#pragma unroll 1
    for (int a = 0; a < 4; ++a) {
      const double wa = W * (double)wx[a];
      const size_t plane = (size_t)wrapIdx<N>(i0 + a) * N;
#pragma unroll 1
      for (int b = 0; b < 4; ++b) {
        const double wab = wa * (double)wy[b];
        const size_t row = (plane + wrapIdx<N>(j0 + b)) * N;
#pragma unroll
        for (int c = 0; c < 4; ++c)
          atomicAdd(&fx[row + wrapIdx<N>(k0 + c)], (unsigned long long)llrint(wab * (double)wz[c]));
      }
    }
  }
}

// ------------------------------------------------------------ brick deposit
// Deposit of W with the cosine kernel / dx^3 (particles.py:23-35, 529-575),
// organised by output: one workgroup per brick of S^3 grid nodes accumulates
// in a 64-bit fixed-point LDS tile and writes each node of the brick exactly
// once.  Integer sums do not depend on the order of the additions, so the
// deposit is bitwise reproducible, and ds_add_u64 is the fastest LDS atomic
// wide enough (gfx950: u64 15, f64 27, f32 196 cycles per wavefront).  The
// scale 2^e is the largest power of two with  total * Wmax / dx^3 / 8 * 2^e
// < 2^62, 2^52 for FP32 fields  (total = candidates of the brick, Wmax =
// largest W of the launch, 1/8 = largest product of three weights), so no sum
// can overflow; one unit is ~2^-62 (2^-52) of that bound.
//
// The droplets that can reach the brick are those whose stage cell lies in
// [c0 - 2, c0 + S] per axis; their sorted bins (bins of the position at the
// last sort) lie in that cell range's bins widened by one bin of motion
// (slots that moved further are on the fallback list and skipped here).  For
// each (bin x, bin y) of that window the z-run of bins is one contiguous range
// of sorted slots per bin tile it crosses, so the candidates form at most
// NZS * NBX^2 ranges.  Per round, CH candidates are tested for overlap with the
// brick; those that overlap are compacted into an LDS list, and each listed
// droplet is then deposited by one lane.
template <int N> struct Brick {
  static constexpr int S = Bins<N>::TC;              // nodes per side (one bin tile)
  static constexpr int NB = N / S;                   // bricks per side
  // threads: 512 measured against 256 and 1024 (deposit 0.143 / 0.130 / 0.335 ms per
  // stage at 256^3 with 10^6 droplets; 64^3 ensemble step 10.99 / 10.67 / 10.68 ms)
  static constexpr int NT = 512;
  // bins spanned by S + 3 stage cells from a bin-aligned start, +-1 bin of motion
  static constexpr int W0 = (S + 2 + Bins<N>::BS - 1) / Bins<N>::BS + 1 + 2;
  static constexpr int NBX = W0 < Bins<N>::B ? W0 : Bins<N>::B;
  // z-runs of NBX bins split at tile boundaries into at most NZS key ranges
  static constexpr int NZS = (NBX + Bins<N>::TS - 1) / Bins<N>::TS + 1;
  static constexpr int NR = NZS * NBX * NBX;         // slot ranges
  static constexpr int CH = 2 * NT;                  // candidates tested per round (LDS fits 4 blocks per CU)
  static constexpr int CROWD = 8 * CH, PARTS = 64;   // DEP_ROWS: candidates that one block takes, most shares
  static_assert(N % S == 0 && (NB * NB * NB) % 8 == 0, "brick grid");
};

//
// MODE: DEP_STEP sums growth rates in 64-bit fixed point; DEP_WIDE (RK4 on a
// caller's rows) the same with a 2^62 range in FP32 contexts too, as that call's
// fallback deposit has it.  DEP_ROWS (the API's deposits, whose weights may be
// negative, of any range or not finite): the tile is FP64 and added to in FP64
// (ds_add_f64, 27 against 15 cycles), every candidate with W != 0 deposits, and
// the stencil weights are FP64 as the API's are.
//
// DEP_ROWS, more than CROWD candidates in a brick (rows that cluster: 10^6 in a
// box of side L/20 took 21 ms when a brick's workgroup took them all): the
// brick's block only lists up to PARTS shares of them, and a second launch of
// persistent blocks (k_brick_crowd, DEP_SHARE) takes the shares, adds each one's
// tile to the FP64 scratch field `sums` (zero between calls), and the block that
// adds a brick's last share rounds the sums into fc and clears them.
enum { DEP_STEP, DEP_WIDE, DEP_ROWS, DEP_SHARE };
struct CrowdShare { int brick, part, parts, pad; };
struct Crowd {
  int* count;                  // shares listed (zero before the DEP_ROWS launch)
  int* done;                   // shares added, per brick
  CrowdShare* list;            // at most np / 512 of them: a slot is a candidate of at most 8 bricks
  double* sums;
};
template <typename T, int N, int MODE>
__device__ __forceinline__ void brickDeposit(const double4* __restrict__ dep, const int* __restrict__ start, int np,
                                             const unsigned long long* __restrict__ wmax, T* __restrict__ fc,
                                             const DropPhys& P, const CrowdShare& it, const Crowd& crowd) {
  constexpr bool FIX = MODE == DEP_STEP || MODE == DEP_WIDE;
  using Bk = Brick<N>;
  constexpr int S = Bk::S, NBr = Bk::NB, NBX = Bk::NBX, NR = Bk::NR, NT = Bk::NT, NZS = Bk::NZS, CH = Bk::CH;
  constexpr int TS = Bins<N>::TS;
  constexpr int BS = Bins<N>::BS, B = Bins<N>::B;
  constexpr int NBIN = B * B * B;
  __shared__ std::conditional_t<FIX, unsigned long long, double> tile[S * S * S];
  __shared__ int rb[NR], rn[NR], rl[NR + 1];
  __shared__ int list[CH];
  __shared__ int cnt;
  __shared__ unsigned long long wtop;
  const int tid = threadIdx.x, lane = tid & 63;
  const int br = it.brick;
  const int c0x = (br / (NBr * NBr)) * S, c0y = ((br / NBr) % NBr) * S, c0z = (br % NBr) * S;
  for (int i = tid; i < S * S * S; i += NT) tile[i] = 0;
  if (tid == 0) cnt = 0;
  if (FIX && tid < WSLOTS) {
    unsigned long long v = wmax[wslot(tid)];
#pragma unroll
    for (int off = WSLOTS / 2; off > 0; off >>= 1) {
      const unsigned long long o = __shfl_xor(v, off, 64);
      v = o > v ? o : v;
    }
    if (tid == 0) wtop = v;
  }
  // slot ranges of the window's z-runs
  const int lo = (NBX == B) ? 0 : 1;
  const int blx = ((c0x - 2 + N) % N) / BS - lo, bly = ((c0y - 2 + N) % N) / BS - lo;
  const int z0 = (NBX == B) ? 0 : (((c0z - 2 + N) % N) / BS - lo + B) % B;
  for (int r = tid; r < NBX * NBX; r += NT) {
    const int bx = (blx + r / NBX + B) % B, by = (bly + r % NBX + B) % B;
    int bz = z0, rem = NBX;
#pragma unroll
    for (int sgm = 0; sgm < NZS; ++sgm) {
      int b0 = 0, len = 0;
      if (rem > 0) {
        const int l = bz % TS;
        const int nz = (TS - l < rem) ? TS - l : rem;   // bins of this run inside one tile
        const int k0 = Bins<N>::key(bx, by, bz);        // keys k0 .. k0 + nz - 1 are consecutive
        b0 = start[k0];
        len = ((k0 + nz < NBIN) ? start[k0 + nz] : np) - b0;
        bz = (bz + nz) % B;
        rem -= nz;
      }
      rb[NZS * r + sgm] = b0; rn[NZS * r + sgm] = len;
    }
  }
  __syncthreads();
  // exclusive prefix of the range lengths (wavefront 0)
  if (tid < 64) {
    constexpr int PER = (NR + 63) / 64;
    int loc[PER];
    int sum = 0;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int idx = tid * PER + k;
      loc[k] = sum;
      sum += (idx < NR) ? rn[idx] : 0;
    }
    int inc = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int t = __shfl_up(inc, off, 64);
      if (tid >= off) inc += t;
    }
    const int ex = inc - sum;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int idx = tid * PER + k;
      if (idx < NR) rl[idx] = ex + loc[k];
    }
    if (tid == 63) rl[NR] = inc;
  }
  __syncthreads();
  const int all = rl[NR];
  if constexpr (MODE == DEP_ROWS) {
    if (all > Bk::CROWD) {
      int parts = (all + Bk::CROWD - 1) / Bk::CROWD;
      parts = parts < Bk::PARTS ? parts : Bk::PARTS;
      if (tid == 0) { cnt = atomicAdd(crowd.count, parts); crowd.done[br] = 0; }
      __syncthreads();
      if (tid < parts) crowd.list[cnt + tid] = CrowdShare{br, tid, parts, 0};
      return;
    }
  }
  // the candidates [first, total): all of them, or the share
  const int share = MODE == DEP_SHARE ? (all + it.parts - 1) / it.parts : all;
  const int first = MODE == DEP_SHARE ? it.part * share : 0;
  const int total = MODE == DEP_SHARE && first + share < all ? first + share : all;
  const double dx = P.dx, pi_2dx = P.pi_2dx, inv_dx = P.inv_dx;
  const double bound = FIX ? (double)total * __longlong_as_double((long long)wtop) * P.inv_vol * 0.125 : 0.0;
  const bool finite = isfinite(bound);
  // FP32 steps: sums below 2^52, so a value converts to its integer by one
  // addition of 2^52 (round to nearest even, as llrint); FP64 fields and
  // DEP_WIDE keep the 2^62 range and llrint
  constexpr bool F32 = sizeof(T) == 4 && MODE == DEP_STEP;
  constexpr int EMAX = F32 ? 51 : 61;
  const int e = (bound > 0.0 && finite) ? EMAX - ilogb(bound) : 0;
  const double scale = ldexp(1.0, e), unit = ldexp(1.0, -e);
  for (int base = first; base < total && finite; base += CH) {
    // test and compact: growing candidates whose stencil meets the brick
#pragma unroll 1
    for (int k = 0; k < CH / NT; ++k) {
      const int f = base + k * NT + tid;
      bool take = false;
      int t = 0;
      if (f < total) {
        int a = 0, b = NR;                                  // rl[a] <= f < rl[b]
        while (b - a > 1) {
          const int mid = (a + b) >> 1;
          if (rl[mid] <= f) a = mid; else b = mid;
        }
        t = rb[a] + (f - rl[a]);
        const double4 d = dep[t];
        if (FIX ? d.w > 0.0 : d.w != 0.0) {
          const int rx = ((originOf(d.x, inv_dx) - c0x) % N + N) % N;
          const int ry = ((originOf(d.y, inv_dx) - c0y) % N + N) % N;
          const int rz = ((originOf(d.z, inv_dx) - c0z) % N + N) % N;
          take = (rx < S || rx > N - 4) && (ry < S || ry > N - 4) && (rz < S || rz > N - 4);
        }
      }
      const unsigned long long m = __ballot(take);
      const int nw = __popcll(m);
      int wbase = 0;
      if (lane == 0 && nw) wbase = atomicAdd(&cnt, nw);
      wbase = __shfl(wbase, 0, 64);
      if (take)
        list[wbase + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] = t;
    }
    __syncthreads();
    const int n = cnt;
    for (int i = tid; i < n; i += NT) {
      const double4 d = dep[list[i]];
      // stencil weights in the field precision (FP32 fields: FP32 sines and cosines)
      using GT = std::conditional_t<FIX && sizeof(T) == 4, float, double>;
      GT wx[4], wy[4], wz[4];
      const int i0 = cosW4F<GT>(d.x, dx, inv_dx, pi_2dx, wx), j0 = cosW4F<GT>(d.y, dx, inv_dx, pi_2dx, wy),
                k0 = cosW4F<GT>(d.z, dx, inv_dx, pi_2dx, wz);
      const int rx = ((i0 - c0x) % N + N) % N, ry = ((j0 - c0y) % N + N) % N, rz = ((k0 - c0z) % N + N) % N;
      // scale is a power of two, so W * scale is exact and the products below
      // round as (W wx wy wz) scale would
      const double W = d.w * P.inv_vol * scale;
      const double wzd[4] = {(double)wz[0], (double)wz[1], (double)wz[2], (double)wz[3]};
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const int nx = (rx + a) % N;
        if (nx >= S) continue;
        const double wa = W * (double)wx[a];
#pragma unroll
        for (int bb = 0; bb < 4; ++bb) {
          const int ny = (ry + bb) % N;
          if (ny >= S) continue;
          const double wab = wa * (double)wy[bb];
#pragma unroll
          for (int cc = 0; cc < 4; ++cc) {
            const int nz = (rz + cc) % N;
            if (nz >= S) continue;
            const double v = wab * wzd[cc];
            if constexpr (!FIX) {
              atomicAdd(&tile[(nx * S + ny) * S + nz], v);
              continue;
            }
            unsigned long long q;
            if constexpr (F32)
              q = (unsigned long long)(__double_as_longlong(v + 0x1p52) - __double_as_longlong(0x1p52));
            else
              q = (unsigned long long)llrint(v);
            if constexpr (FIX) atomicAdd(&tile[(nx * S + ny) * S + nz], q);
          }
        }
      }
    }
    __syncthreads();
    if (tid == 0) cnt = 0;
    __syncthreads();
  }
  auto node = [&](int i) {
    const int nx = i / (S * S), ny = (i / S) % S, nz = i % S;
    return ((size_t)(c0x + nx) * N + (c0y + ny)) * N + (c0z + nz);
  };
  if constexpr (MODE != DEP_SHARE) {
    for (int i = tid; i < S * S * S; i += NT) fc[node(i)] = finite ? (T)((double)tile[i] * unit) : (T)NAN;
  } else {
    for (int i = tid; i < S * S * S; i += NT)
      if (tile[i] != 0.0) unsafeAtomicAdd(crowd.sums + node(i), tile[i]);
    __threadfence();                     // this share's additions before its count
    __syncthreads();
    if (tid == 0) cnt = atomicAdd(crowd.done + br, 1);
    __syncthreads();
    if (cnt == it.parts - 1) {
      __threadfence();                   // all counts before the loads
      for (int i = tid; i < S * S * S; i += NT) {
        double* v = crowd.sums + node(i);
        fc[node(i)] = (T)__hip_atomic_load(v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *v = 0.0;
      }
    }
  }
}

template <typename T, int N, int MODE = DEP_STEP>
__global__ void __launch_bounds__(Brick<N>::NT)
k_brick_deposit(const double4* __restrict__ dep0, const int* __restrict__ start0, int np,
                const unsigned long long* __restrict__ wmax0, T* __restrict__ fc0, DropPhys P, size_t rs,
                const int* __restrict__ flist0, const int* __restrict__ fcount0, unsigned long long* fx0, Crowd crowd) {
  const double4* __restrict__ dep = rsel1(dep0, rs);
  const unsigned long long* __restrict__ wmax = rsel1(wmax0, rs);
  constexpr int NBRICK = Brick<N>::NB * Brick<N>::NB * Brick<N>::NB;
  if constexpr (MODE != DEP_ROWS) {
    if (blockIdx.x >= NBRICK) {          // the extra blocks: fallback slots
      const int nf = *rsel1(fcount0, rs), b = (int)blockIdx.x - NBRICK;
      if (nf)
        fallbackAccum<T, N>(dep, rsel1(flist0, rs), nf, maxOfSlots(wmax), rsel1(fx0, rs), P, b * Brick<N>::NT + (int)threadIdx.x,
                            ((int)gridDim.x - NBRICK) * Brick<N>::NT);
      return;
    }
  }
  // XCD-aware: each of the 8 XCDs takes a contiguous run of bricks
  constexpr int per = NBRICK / 8;
  const int br = (blockIdx.x % 8) * per + blockIdx.x / 8;
  brickDeposit<T, N, MODE>(dep, rsel1(start0, rs), np, wmax, rsel1(fc0, rs), P, CrowdShare{br, 0, 1, 0}, crowd);
}
template <typename T, int N>
__global__ void __launch_bounds__(Brick<N>::NT)
k_brick_crowd(const double4* __restrict__ dep, const int* __restrict__ start, int np, T* __restrict__ fc, DropPhys P,
              Crowd crowd) {
  const int n = *crowd.count;
  for (int i = blockIdx.x; i < n; i += gridDim.x) {
    const CrowdShare it = crowd.list[i];
    brickDeposit<T, N, DEP_SHARE>(dep, start, np, nullptr, fc, P, it, crowd);
    __syncthreads();                     // the shared arrays of the next share
  }
}

// ------------------------------------------------------------ tile gather
// Gather of several planar fields at bin-sorted slots, one field of one bin
// tile per workgroup: the field's nodes that the stencils of the tile's S^3
// cells reach are staged in LDS and one thread per slot sums its 64 nodes from
// there.
//
// A gather straight from global memory reads a 128-byte line of L2 for every
// 16 (planar FP32) or 64 bytes (node records) of a stencil row, which bounds
// it; a tile of a field is 35 KB (FP32) for all of the tile's slots.  One field
// per workgroup, not all of them in turn: blocks run field by field over groups
// of 64 neighbouring tiles, so that neighbours read a field's halo while it is
// in their L2 (seven fields per block: 357 us for 10^6 rows at 256^3 FP32, the
// same with 256, 384 and 512 threads; 222 us like this, against 737 us for four
// lanes per row on planar fields, k_prhs_sorted).
//
// A tile's block takes its first PART slots at most.  Slots crowd where droplets
// cluster (10^6 rows in a box of side L/20: 3.7 ms for seven fields when one
// block per field took a tile's slots).  So behind the tiles' blocks there is one
// per aligned run of PART slots, which takes those of the run that lie beyond
// the first PART of their tile, all fields: they are of one tile, that of the
// run's first slot, because a tile that starts inside the run has no such slots
// in it.
template <typename T> struct GatherFields {
  const T *a, *b, *c;          // fields 0 .. na - 1 of a, na .. na + nb - 1 of b (N^3 apart), then c
  int na, nb, n;               // n fields in all
  __device__ __forceinline__ const T* field(int k, size_t R) const {
    return k < na ? a + k * R : k < na + nb ? b + (k - na) * R : c;
  }
};
template <int N> struct GatherTile {
  static constexpr int S = Bins<N>::TC;
  static constexpr int RX = S + 3;                               // nodes per side in x and y
  static constexpr int QZ = S / 4 + 2, PZ = 4 * QZ;              // along z: aligned quads from 4 nodes before
  static constexpr int NQ = RX * RX * QZ;
  static constexpr int TSB = Bins<N>::TS * Bins<N>::TS * Bins<N>::TS, NTILE = Bins<N>::NB / TSB;
  static constexpr int XT = NTILE / 8, GS = XT < 64 ? XT : 64;   // tiles per XCD and per group
  static constexpr int NT = 256, PART = 1024;
  static constexpr int IT = (NQ + NT - 1) / NT;                  // staged quads per thread (the last ones are padding)
  static_assert(RX <= N && PZ <= N && NTILE % 8 == 0 && XT % GS == 0, "gather tile");
};
// Field f, number k of n, at the slots [s0, s1) of the tile with first cell
// (cx, cy, cz); FP64 weights and sums.  rowmap null: out[k cap + slot]; else
// out[rowmap[slot] n + k].
template <typename T, int N>
__device__ __forceinline__ void gatherTile(T* lds, const T* __restrict__ f, int k, int n, int cx, int cy, int cz, int s0,
                                           int s1, const double4* __restrict__ dep, int cap,
                                           const int* __restrict__ rowmap, double* __restrict__ out, const DropPhys& P) {
  using GT = GatherTile<N>;
  constexpr int RX = GT::RX, QZ = GT::QZ, PZ = GT::PZ, NT = GT::NT, IT = GT::IT;
  {
    V4<T> q[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int e = (int)threadIdx.x + it * NT, z4 = e % QZ, row = e / QZ;
      const uint32_t x = (uint32_t)(cx - 1 + row / RX) & (N - 1), y = (uint32_t)(cy - 1 + row % RX) & (N - 1),
                     z = (uint32_t)(cz - 4 + 4 * z4) & (N - 1);
      q[it] = ld32(reinterpret_cast<const V4<T>*>(f), ((x * N + y) * N + z) / 4);
    }
    // the writes wait for one load each, in order (mixed with the loads by the
    // scheduler, 237 instead of 222 us for 10^6 rows at 256^3 FP32)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int it = 0; it < IT; ++it) *reinterpret_cast<V4<T>*>(lds + 4 * ((int)threadIdx.x + it * NT)) = q[it];
  }
  __syncthreads();
  for (int s = s0 + (int)threadIdx.x; s < s1; s += NT) {
    const double4 d = dep[s];
    const int i0 = originOf(d.x, P.inv_dx), j0 = originOf(d.y, P.inv_dx), k0 = originOf(d.z, P.inv_dx);
    double xs, xc, ys, yc, zs, zc;
    sincosStencil<double>(d.x, i0, P.dx, P.inv_dx, P.pi_2dx, xs, xc);
    sincosStencil<double>(d.y, j0, P.dx, P.inv_dx, P.pi_2dx, ys, yc);
    sincosStencil<double>(d.z, k0, P.dx, P.inv_dx, P.pi_2dx, zs, zc);
    const double wx[4] = {0.25 * (1.0 + xc), 0.25 * (1.0 + xs), 0.25 * (1.0 - xc), 0.25 * (1.0 - xs)};
    const double wy[4] = {0.25 * (1.0 + yc), 0.25 * (1.0 + ys), 0.25 * (1.0 - yc), 0.25 * (1.0 - ys)};
    const double wz[4] = {0.25 * (1.0 + zc), 0.25 * (1.0 + zs), 0.25 * (1.0 - zc), 0.25 * (1.0 - zs)};
    // the slot's cell is one of the tile's (k_row_bin takes it from the same
    // wrapped position), so its stencil starts at 0 .. S - 1 of the staged nodes
    const T* o = lds + ((i0 - cx + 1) * RX + (j0 - cy + 1)) * PZ + (k0 - cz + 4);
    double sum = 0.0;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      // the plane's 16 values are read ahead of their sum
      T v[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] = o[(a * RX + (e >> 2)) * PZ + (e & 3)];
      double sa = 0.0;
#pragma unroll
      for (int b = 0; b < 4; ++b)
        sa += wy[b] * ((double)v[4 * b] * wz[0] + (double)v[4 * b + 1] * wz[1] + (double)v[4 * b + 2] * wz[2] +
                       (double)v[4 * b + 3] * wz[3]);
      sum += wx[a] * sa;
    }
    if (rowmap) out[(size_t)rowmap[s] * n + k] = sum;
    else out[(size_t)k * cap + s] = sum;
  }
}
template <typename T, int N>
__global__ void __launch_bounds__(GatherTile<N>::NT)
k_tile_gather(GatherFields<T> F, const double4* __restrict__ dep, const int* __restrict__ start, int np, int cap,
              const int* __restrict__ rowmap, double* __restrict__ out, DropPhys P) {
  using GT = GatherTile<N>;
  constexpr int PART = GT::PART;
  constexpr size_t R = (size_t)N * N * N;
  __shared__ __attribute__((aligned(32))) T lds[4 * GT::IT * GT::NT];
  int cx, cy, cz;
  auto end = [&](int tile) { return tile + 1 < GT::NTILE ? start[(tile + 1) * GT::TSB] : np; };
  const int extra = (int)blockIdx.x - GT::NTILE * F.n;
  if (extra < 0) {
    const int j = blockIdx.x / 8, r = j % (GT::GS * F.n);
    const int tile = (blockIdx.x % 8) * GT::XT + j / (GT::GS * F.n) * GT::GS + r % GT::GS, k = r / GT::GS;
    const int s0 = start[tile * GT::TSB], s1 = end(tile);
    if (s0 == s1) return;
    Bins<N>::tileCell(tile, cx, cy, cz);
    gatherTile<T, N>(lds, F.field(k, R), k, F.n, cx, cy, cz, s0, s1 - s0 < PART ? s1 : s0 + PART, dep, cap, rowmap, out, P);
    return;
  }
  const int run = (extra + 1) * PART;
  const double4 d = dep[run];
  const int tile = Bins<N>::key(cellOf<N>(d.x, P.inv_dx) / Bins<N>::BS, cellOf<N>(d.y, P.inv_dx) / Bins<N>::BS,
                                cellOf<N>(d.z, P.inv_dx) / Bins<N>::BS) / GT::TSB;
  const int first = start[tile * GT::TSB] + PART, last = end(tile);
  const int s0 = first > run ? first : run, s1 = last < run + PART ? last : run + PART;
  if (s0 >= s1) return;
  Bins<N>::tileCell(tile, cx, cy, cz);
#pragma unroll 1
  for (int k = 0; k < F.n; ++k) {
    if (k) __syncthreads();              // the sums of the field before
    gatherTile<T, N>(lds, F.field(k, R), k, F.n, cx, cy, cz, s0, s1, dep, cap, rowmap, out, P);
  }
}

// ------------------------------------------------------------ API kernels
// interp_cosine (particles.py:435-511) of NC fields at rows of coord (Np, 7).
template <typename T, int N>
__global__ void __launch_bounds__(256)
k_interp(const double* __restrict__ coord, int np, const T* __restrict__ f, int ncomp, double* __restrict__ out,
         DropPhys P) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  constexpr size_t R = (size_t)N * N * N;
  double xw[3];
  for (int c = 0; c < 3; ++c) xw[c] = wrapL(coord[(size_t)p * 7 + c], P.L);
  Stencil<N> s;
  s.set(xw, P.dx, P.pi_2dx);
  for (int c = 0; c < ncomp; ++c) {
    double v;
    gatherN<T, N, 1>(s, f + (size_t)c * R, R, &v);
    out[(size_t)p * ncomp + c] = v;
  }
}

// exterp_cosine_scalar (particles.py:514-577): deposit w[p] into c (c must be zeroed).
template <typename T, int N>
__global__ void __launch_bounds__(256)
k_exterp(const double* __restrict__ coord, int np, const double* __restrict__ w, T* c, DropPhys P) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  double xw[3];
  for (int k = 0; k < 3; ++k) xw[k] = wrapL(coord[(size_t)p * 7 + k], P.L);
  Stencil<N> s;
  s.set(xw, P.dx, P.pi_2dx);
  deposit<T, N>(s, w[p], P.inv_vol, c);
}

// pRHS (particles.py:817-837) on rows of a stage coordinate (Np, 7): writes
// rhs (Np, 7), interpmat (Np, 7), exterpmat (Np) and deposits into fc (zeroed).
// n is used as given (clip = nullptr) or through the lazy clip.
template <typename T, int N>
__global__ void __launch_bounds__(256)
k_prhs(const double* __restrict__ coord, int np, const T* __restrict__ u, const T* __restrict__ us,
       const T* __restrict__ n, const double* __restrict__ clip, T* fc, double* __restrict__ rhs,
       double* __restrict__ interp, double* __restrict__ exterp, DropPhys P) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  constexpr size_t R = (size_t)N * N * N;
  const double* row = coord + (size_t)p * 7;
  double xw[3], vp[3];
  for (int c = 0; c < 3; ++c) { xw[c] = wrapL(row[c], P.L); vp[c] = row[3 + c]; }
  Stencil<N> s;
  s.set(xw, P.dx, P.pi_2dx);
  double I[7];
  gatherN<T, N, 3>(s, u, R, I);
  gatherN<T, N, 3>(s, us, R, I + 3);
  I[6] = gatherDensity<T, N>(s, n, clip);
  double r[7], W;
  dropletRhs(P, vp, row[6], I, r, W);
  deposit<T, N>(s, W, P.inv_vol, fc);
  for (int c = 0; c < 7; ++c) { rhs[(size_t)p * 7 + c] = r[c]; interp[(size_t)p * 7 + c] = I[c]; }
  exterp[p] = W;
}

// ------------------------------------------------------------ sorted API path
// With enough rows the API's gathers and deposits work on rows sorted by bin
// (Engine::rows_sorted): k_row_bin counts the rows of each bin, the scans of
// the step's sort give the bin starts, k_row_scatter writes each row's wrapped
// position, weight and row number to its slot.  The gather then runs four
// lanes per row (lane c owns z node c of the stencil), so one load touches 16
// rows that lie in neighbouring cells, and the deposit takes the bricks.
// Positions, weights and sums stay FP64.
// wrapped coordinate whose cell is below N (a position that rounds to L is 0)
template <int N> __device__ __forceinline__ double wrapRow(double x, double L, double inv_dx) {
  const double r = wrapL(x, L);
  return r * inv_dx < (double)N ? r : 0.0;
}
// Rows are counted per block first (an open-addressed table of the block's bins
// in LDS), then one global atomic per bin and block: atomics that meet at one
// cache line take turns, and clustered rows meet at few.
template <int N, int NT>
__global__ void __launch_bounds__(NT)
k_row_bin(const double* __restrict__ rows, int np, double L, double inv_dx, int* __restrict__ key,
          int* __restrict__ rank, int* __restrict__ hist) {
  constexpr int SLOTS = 2 * NT;              // never full: each probe ends
  __shared__ int bin[SLOTS], count[SLOTS];
  for (int i = threadIdx.x; i < SLOTS; i += NT) { bin[i] = -1; count[i] = 0; }
  __syncthreads();
  const int p = blockIdx.x * NT + threadIdx.x;
  int h = 0, local = 0;
  if (p < np) {
    int b[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) b[c] = cellOf<N>(wrapRow<N>(rows[(size_t)p * 7 + c], L, inv_dx), inv_dx) / Bins<N>::BS;
    const int k = Bins<N>::key(b[0], b[1], b[2]);
    key[p] = k;
    h = (int)(((uint32_t)k * 2654435761u) >> 21) & (SLOTS - 1);
    for (;;) {
      const int old = atomicCAS(&bin[h], -1, k);
      if (old == -1 || old == k) break;
      h = (h + 1) & (SLOTS - 1);
    }
    local = atomicAdd(&count[h], 1);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < SLOTS; i += NT)
    if (bin[i] >= 0) count[i] = atomicAdd(&hist[bin[i]], count[i]);
  __syncthreads();
  if (p < np) rank[p] = count[h] + local;
}
template <int N>
__global__ void __launch_bounds__(256)
k_row_scatter(const double* __restrict__ rows, int np, double L, double inv_dx, const double* __restrict__ w,
              const int* __restrict__ key, const int* __restrict__ rank, const int* __restrict__ start,
              double4* __restrict__ dep, int* __restrict__ row, int* __restrict__ crowd_count) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p == 0) *crowd_count = 0;          // of the deposit that follows
  if (p >= np) return;
  const double* r = rows + (size_t)p * 7;
  double4 d;
  d.x = wrapRow<N>(r[0], L, inv_dx); d.y = wrapRow<N>(r[1], L, inv_dx); d.z = wrapRow<N>(r[2], L, inv_dx);
  d.w = w ? w[p] : 0.0;
  const int s = start[key[p]] + rank[p];
  dep[s] = d;
  row[s] = p;
}

// One slot's stencil, four lanes per slot: this lane's z node and weight, all
// x and y nodes.  Lane c takes the sine and cosine of axis c (FP64) and the
// four lanes share them.
template <int N> struct QuadStencil {
  int i0, j0, iz;
  double wx[4], wy[4], wz;
  __device__ __forceinline__ QuadStencil(const double4& d, int c, const DropPhys& P) {
    i0 = originOf(d.x, P.inv_dx); j0 = originOf(d.y, P.inv_dx);
    const int k0 = originOf(d.z, P.inv_dx);
    const double x = c == 0 ? d.x : c == 1 ? d.y : d.z;
    const int o = c == 0 ? i0 : c == 1 ? j0 : k0;
    double sn, cs;
    sincosStencil<double>(x, o, P.dx, P.inv_dx, P.pi_2dx, sn, cs);
    const double xs = __shfl(sn, 0, 4), xc = __shfl(cs, 0, 4), ys = __shfl(sn, 1, 4), yc = __shfl(cs, 1, 4),
                 zs = __shfl(sn, 2, 4), zc = __shfl(cs, 2, 4);
    wx[0] = 0.25 * (1.0 + xc); wx[1] = 0.25 * (1.0 + xs); wx[2] = 0.25 * (1.0 - xc); wx[3] = 0.25 * (1.0 - xs);
    wy[0] = 0.25 * (1.0 + yc); wy[1] = 0.25 * (1.0 + ys); wy[2] = 0.25 * (1.0 - yc); wy[3] = 0.25 * (1.0 - ys);
    const double zt = (c & 1) ? zs : zc;
    wz = 0.25 * (1.0 + ((c & 2) ? -zt : zt));
    iz = wrapIdx<N>(k0 + c);
  }
  // node index of x node a, y node b and this lane's z node (< N^3 <= 2^27)
  __device__ __forceinline__ uint32_t node(int a, int b) const {
    return ((uint32_t)wrapIdx<N>(i0 + a) * N + (uint32_t)wrapIdx<N>(j0 + b)) * N + (uint32_t)iz;
  }
  // sum over the four lanes of v times this lane's z weight
  __device__ __forceinline__ double sum(double v) const {
    v *= wz;
    v += __shfl_xor(v, 1, 4);
    v += __shfl_xor(v, 2, 4);
    return v;
  }
};
// this lane's slot: blocks map XCD-aware (each XCD one contiguous range of slots)
__device__ __forceinline__ int quadSlot() {
  const int per = gridDim.x / 8, lb = (blockIdx.x % 8) * per + blockIdx.x / 8;
  return (lb * (int)blockDim.x + (int)threadIdx.x) >> 2;
}

// pRHS (particles.py:817-837) on sorted rows: rhs, interpolants and growth
// rate in row order, W to the slot's deposit record.  Bound by the stencil
// loads (112 per lane, each one 16-byte (FP32) run per row).
template <typename T, int N>
__global__ void __launch_bounds__(256)
k_prhs_sorted(const double* __restrict__ coord, int np, const T* __restrict__ u, const T* __restrict__ us,
              const T* __restrict__ n, double4* __restrict__ dep, const int* __restrict__ row0,
              double* __restrict__ rhs, double* __restrict__ interp, double* __restrict__ exterp, DropPhys P) {
  constexpr size_t R = (size_t)N * N * N;
  const int s = quadSlot(), c = threadIdx.x & 3;
  const bool live = s < np;
  const double4 d = dep[live ? s : 0];
  const size_t p = (size_t)row0[live ? s : 0];
  const QuadStencil<N> q(d, c, P);
  double I[7];
#pragma unroll
  for (int k = 0; k < 7; ++k) I[k] = 0.0;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    T f[4][7];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const uint32_t o = q.node(a, b);
#pragma unroll
      for (int k = 0; k < 3; ++k) { f[b][k] = ld32(u + k * R, o); f[b][3 + k] = ld32(us + k * R, o); }
      f[b][6] = ld32(n, o);
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const double w = q.wx[a] * q.wy[b];
#pragma unroll
      for (int k = 0; k < 7; ++k) I[k] += (double)f[b][k] * w;
    }
  }
#pragma unroll
  for (int k = 0; k < 7; ++k) I[k] = q.sum(I[k]);
  if (!live) return;
  double vp[3], r[7], W;
  const double* rw = coord + p * 7;
#pragma unroll
  for (int k = 0; k < 3; ++k) vp[k] = rw[3 + k];
  dropletRhs(P, vp, rw[6], I, r, W);
  // the four lanes write the row's 56 bytes together
#pragma unroll
  for (int k = 0; k < 7; ++k)
    if ((k & 3) == c) { rhs[p * 7 + k] = r[k]; interp[p * 7 + k] = I[k]; }
  if (c == 0) {
    exterp[p] = W;
    dep[s].w = W;
  }
}

// The droplet side of pRHS on sorted rows whose interpolants k_tile_gather left
// in I[k cap + slot].  Bound by the scattered rows (10^6: 110 us; moving them
// through LDS with neighbouring lanes took the same).
static __global__ void __launch_bounds__(256)
k_prhs_finish(const double* __restrict__ coord, int np, int cap, const double* __restrict__ I0,
              double4* __restrict__ dep, const int* __restrict__ row0, double* __restrict__ rhs,
              double* __restrict__ interp, double* __restrict__ exterp, DropPhys P) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= np) return;
  const size_t p = (size_t)row0[s];
  const double* rw = coord + p * 7;
  double I[7], vp[3], r[7], W;
#pragma unroll
  for (int k = 0; k < 7; ++k) I[k] = I0[(size_t)k * cap + s];
#pragma unroll
  for (int k = 0; k < 3; ++k) vp[k] = rw[3 + k];
  dropletRhs(P, vp, rw[6], I, r, W);
#pragma unroll
  for (int k = 0; k < 7; ++k) { rhs[p * 7 + k] = r[k]; interp[p * 7 + k] = I[k]; }
  exterp[p] = W;
  dep[s].w = W;
}

// interp_cosine (particles.py:435-511) of sorted rows, one component at a time.
template <typename T, int N>
__global__ void __launch_bounds__(256)
k_interp_sorted(int np, const T* __restrict__ f, int ncomp, const double4* __restrict__ dep,
                const int* __restrict__ row0, double* __restrict__ out, DropPhys P) {
  constexpr size_t R = (size_t)N * N * N;
  const int s = quadSlot(), c = threadIdx.x & 3;
  const bool live = s < np;
  const double4 d = dep[live ? s : 0];
  const size_t p = (size_t)row0[live ? s : 0];
  const QuadStencil<N> q(d, c, P);
  for (int k = 0; k < ncomp; ++k) {
    const T* fk = f + (size_t)k * R;
    T v[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = ld32(fk, q.node(e >> 2, e & 3));
    double t = 0.0;
#pragma unroll
    for (int e = 0; e < 16; ++e) t += (double)v[e] * (q.wx[e >> 2] * q.wy[e & 3]);
    t = q.sum(t);
    if (live && c == (k & 3)) out[p * ncomp + k] = t;
  }
}

// AoS (Np, 7) rows <-> engine SoA state, the rows of the realizations
// (blockIdx.z) back to back.  rid[p]: the input row of engine slot p (slots are
// permuted by the spatial sort).
template <typename PT>
__global__ void k_rows_to_soa(const double* __restrict__ rows0, int np, int cap, double* pos0, PT* vm0, int64_t* rid0,
                              size_t rs) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  const double* __restrict__ rows = rows0 + (size_t)blockIdx.z * np * 7;
  double* pos = rsel1(pos0, rs);
  PT* vm = rsel1(vm0, rs);
  for (int c = 0; c < 3; ++c) pos[c * cap + p] = rows[(size_t)p * 7 + c];
  for (int c = 0; c < 4; ++c) vm[c * cap + p] = (PT)rows[(size_t)p * 7 + 3 + c];
  rsel1(rid0, rs)[p] = p;
}
template <typename PT>
__global__ void k_soa_to_rows(const double* __restrict__ pos0, const PT* __restrict__ vm0,
                              const int64_t* __restrict__ rid0, int np, int cap, double* rows0, size_t rs) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  const double* __restrict__ pos = rsel1(pos0, rs);
  const PT* __restrict__ vm = rsel1(vm0, rs);
  const size_t r = (size_t)rsel1(rid0, rs)[p];
  double* rows = rows0 + (size_t)blockIdx.z * np * 7;
  for (int c = 0; c < 3; ++c) rows[r * 7 + c] = pos[c * cap + p];
  for (int c = 0; c < 4; ++c) rows[r * 7 + 3 + c] = (double)vm[c * cap + p];
}

// n 16-byte units of every realization (blockIdx.z), the realizations ss and ds
// bytes apart.  One launch for an ensemble's field instead of a copy per
// realization, which is mostly launch: with the row moves and the band check
// batched alike, setting and reading the state of an ensemble takes 10 launches
// (64 times 64^3 FP32 with 10^5 droplets, four steps and both moves 44.5 ->
// 43.4 ms; with 2 10^4 droplets 10.2 -> 9.4 ms).
static __global__ void __launch_bounds__(256)
k_copy_fields(const char* __restrict__ src, size_t ss, char* __restrict__ dst, size_t ds, size_t n) {
  const uint4* __restrict__ a = reinterpret_cast<const uint4*>(src + blockIdx.z * ss);
  uint4* __restrict__ b = reinterpret_cast<uint4*>(dst + blockIdx.z * ds);
  for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += gridDim.x * (size_t)256) b[i] = a[i];
}

template <int N>
__global__ void __launch_bounds__(256)
k_bin_count(const double* __restrict__ pos0, int np, int cap, double L, double invL, double inv_dx, int* __restrict__ key0,
            int* __restrict__ rank0, int* __restrict__ hist0, size_t rs) {
  const double* __restrict__ pos = rsel1(pos0, rs);
  int* __restrict__ key = rsel1(key0, rs);
  int* __restrict__ rank = rsel1(rank0, rs);
  int* __restrict__ hist = rsel1(hist0, rs);
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const bool valid = p < np;
  int k = -1 - lane;                        // invalid lanes: keys no other lane has
  if (valid) {
    int b[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) b[c] = cellOf<N>(wrapFast(pos[c * cap + p], L, invL), inv_dx) / Bins<N>::BS;
    k = Bins<N>::key(b[0], b[1], b[2]);
    key[p] = k;
  }
  // The slots are in last step's bin order, so lanes with one key mostly form
  // runs: the first lane of each run of equal keys adds the run's length to
  // the bin count and the run takes consecutive ranks from the old count
  // (one atomic per run instead of one per droplet).
  const int kprev = __shfl_up(k, 1, 64);     // every lane takes part in the shuffle
  const bool head = lane == 0 || kprev != k;
  const unsigned long long hm = __ballot(head);
  const unsigned long long upto = (2ull << lane) - 1ull;         // bits 0 .. lane
  const int start = 63 - __clzll(hm & upto);
  const unsigned long long after = hm & ~upto;
  const int next = after ? __ffsll((long long)after) - 1 : 64;
  int base = 0;
  if (head && valid) base = atomicAdd(&hist[k], next - lane);
  base = __shfl(base, start, 64);
  if (valid) rank[p] = base + (lane - start);
}

// Exclusive scan of 4096 ints per block (1024 threads x 4); block totals to bsum.
__device__ __forceinline__ int blockExclusiveScan1024(int v, int* sh, int& total) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63) sh[wid] = x;
  __syncthreads();
  if (wid == 0) {
    int w = lane < 16 ? sh[lane] : 0;
#pragma unroll
    for (int d = 1; d < 16; d <<= 1) {
      const int y = __shfl_up(w, d, 64);
      if (lane >= d) w += y;
    }
    if (lane < 16) sh[16 + lane] = w;   // inclusive wave prefix
  }
  __syncthreads();
  const int wpre = wid > 0 ? sh[16 + wid - 1] : 0;
  total = sh[16 + 15];
  __syncthreads();
  return wpre + x - v;
}

// chunk number `chunk` of 4096 entries
__device__ __forceinline__ void scanChunk(int* __restrict__ data, int n, int* __restrict__ bsum, int chunk, int* sh) {
  const int base = chunk * 4096 + threadIdx.x * 4;
  int v[4], s = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) { v[i] = (base + i < n) ? data[base + i] : 0; s += v[i]; }
  int total;
  int pre = blockExclusiveScan1024(s, sh, total);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (base + i < n) data[base + i] = pre;
    pre += v[i];
  }
  if (threadIdx.x == 0) bsum[chunk] = total;
}
static __global__ void __launch_bounds__(1024)
k_scan_local(int* __restrict__ data, int n, int* __restrict__ bsum, size_t rs) {
  __shared__ int sh[32];
  scanChunk(rsel1(data, rs), n, rsel1(bsum, rs), blockIdx.x, sh);
}

// += the sums of the 4096-entry chunks before the block's, which each block adds
// up itself (one launch of 5 us less than with a scan of the sums between the two).
__device__ __forceinline__ void scanAddChunk(int* __restrict__ data, int n, const int* __restrict__ bsum, int chunk,
                                             int* sh) {
  data += (size_t)chunk * 4096;
  const int left = n - chunk * 4096, tid = threadIdx.x;
  int v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = tid + k * 1024 < left ? data[tid + k * 1024] : 0;
  int s = 0;
  for (int i = tid; i < chunk; i += 1024) s += bsum[i];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if ((tid & 63) == 0) sh[tid >> 6] = s;
  __syncthreads();
  int base = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) base += sh[w];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (tid + k * 1024 < left) data[tid + k * 1024] = v[k] + base;
}
static __global__ void __launch_bounds__(1024)
k_scan_add(int* __restrict__ data, int n, const int* __restrict__ bsum, size_t rs) {
  __shared__ int sh[16];
  if (blockIdx.x) scanAddChunk(rsel1(data, rs), n, rsel1(bsum, rs), blockIdx.x, sh);
}

// Scatter the droplet state to its sorted slot.
template <typename PT>
__global__ void __launch_bounds__(256)
k_bin_scatter(int np, int cap, const int* __restrict__ key0, const int* __restrict__ rank0,
              const int* __restrict__ start0, const double* __restrict__ pos0, const PT* __restrict__ vm0,
              const int64_t* __restrict__ id0, double* __restrict__ pos20, PT* __restrict__ vm20,
              int64_t* __restrict__ id20, size_t rs) {
  const int* __restrict__ key = rsel1(key0, rs);
  const int* __restrict__ rank = rsel1(rank0, rs);
  const int* __restrict__ start = rsel1(start0, rs);
  const double* __restrict__ pos = rsel1(pos0, rs);
  const PT* __restrict__ vm = rsel1(vm0, rs);
  const int64_t* __restrict__ id = rsel1(id0, rs);
  double* __restrict__ pos2 = rsel1(pos20, rs);
  PT* __restrict__ vm2 = rsel1(vm20, rs);
  int64_t* __restrict__ id2 = rsel1(id20, rs);
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  const int d = start[key[p]] + rank[p];
#pragma unroll
  for (int c = 0; c < 3; ++c) pos2[c * cap + d] = pos[c * cap + p];
#pragma unroll
  for (int c = 0; c < 4; ++c) vm2[c * cap + d] = vm[c * cap + p];
  id2[d] = id[p];
}

}  // namespace ld
