// Diagnostics of the reference's save() and plot.py, on the device:
//   shell spectrum  e3d_to_e1d(w * sum_c |f_c|^2 * normalize)   (forced-dns-sm.py:232-233, 423, 431; plot.py:37-38)
//   energy flux     e3d_to_e1d(Re(conj(uk) . ku) * dealias * normalize), cumulated from high k
//                                                                   (forced-dns-sm.py:425-428)
//   field stats     sum, min, max, sum of squares of a real field  (forced-dns-sm.py:467-471)
// Shell binning follows np.histogram with bins [0, 0.5), [0.5, 1.5), ...,
// [N/2 - 0.5, N/2 + 0.5]: bin s holds |k| in [s - 1/2, s + 1/2) (s >= 1) and
// |k| < 1/2 for s = 0; modes with |k| > N/2 + 1/2 are not counted.
// Reductions are deterministic: per-block partial sums, then a fixed-order
// final sum.
#pragma once
#include "ld_kernels.hpp"

namespace ld {

// mode: 0 -> w * sum_c |f_c|^2 * normalize (nf fields); 1 -> Re(conj(a).b) * mask * normalize (3 fields each);
// 2 -> w * |k|^2 * sum_c |f_c|^2 * normalize (nf fields: the dissipation spectrum for w = nu)
//
// Bound by the fields' reads.  A thread takes four consecutive modes (32 or 64
// bytes of each field, loaded as 16-byte vectors before the first use; the
// fields are 32-byte aligned and hold a multiple of four modes), and adds the
// modes of one shell together before its LDS atomic: neighbours along kz mostly
// share a shell.  1024 threads keep the chip's loads in flight with the 256
// blocks that the scratch holds.  256^3 FP32, three fields: 173 us with 256
// threads of one mode each and 64-bit index arithmetic, 46 us now (4.4 TB/s).
constexpr int DIAG_NT = 1024;
template <typename T, int N>
__global__ void __launch_bounds__(DIAG_NT)
k_shell_partial(const C<T>* __restrict__ a, const C<T>* __restrict__ b, int nf, size_t fs, int mode, double w,
                double norm0, double* __restrict__ part) {
  constexpr int Nf = N / 2 + 1, NW = DIAG_NT / 64;
  // one set of bins per wavefront, summed in a fixed order at the end:
  // additions into one bin come only from the lanes of one instruction, whose
  // order the hardware fixes, so the sums are reproducible
  __shared__ double bins[NW][Nf];
  for (int i = threadIdx.x; i < NW * Nf; i += DIAG_NT) bins[i / Nf][i % Nf] = 0.0;
  __syncthreads();
  double* wbins = bins[threadIdx.x >> 6];
  const uint32_t nq = (uint32_t)(fs / 4), per = (nq + gridDim.x - 1) / gridDim.x;
  const uint32_t q0 = blockIdx.x * per, q1 = (q0 + per < nq) ? q0 + per : nq;
  for (uint32_t q = q0 + threadIdx.x; q < q1; q += DIAG_NT) {
    const uint32_t i = 4 * q;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    auto pairs = [&](const C<T>* f, V4<T>* z) {
      const V4<T>* p = reinterpret_cast<const V4<T>*>(f + i);
      z[0] = p[0]; z[1] = p[1];
    };
    if (mode != 1) {
      for (int c = 0; c < nf; ++c) {
        V4<T> z[2];
        pairs(a + c * fs, z);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          v[2 * e] += (double)z[e].x * (double)z[e].x + (double)z[e].y * (double)z[e].y;
          v[2 * e + 1] += (double)z[e].z * (double)z[e].z + (double)z[e].w * (double)z[e].w;
        }
      }
    } else {
      for (int c = 0; c < 3; ++c) {
        V4<T> x[2], y[2];
        pairs(a + c * fs, x);
        pairs(b + c * fs, y);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          v[2 * e] += (double)x[e].x * (double)y[e].x + (double)x[e].y * (double)y[e].y;
          v[2 * e + 1] += (double)x[e].z * (double)y[e].z + (double)x[e].w * (double)y[e].w;
        }
      }
    }
    int iz = (int)(i % Nf), iy = (int)((i / Nf) % N), ix = (int)(i / Nf / N);
    int cur = -1;
    double sum = 0.0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int kx = kwave(ix, N), ky = kwave(iy, N);
      const int k2 = kx * kx + ky * ky + iz * iz;
      const int ki = kround(k2);
      // outside the last bin; outside the dealias mask (flux)
      const bool in = ki <= N / 2 && (mode != 1 || 3 * ki <= N);
      if (in) {
        const double val = v[e] * ((iz == 0 || iz == N / 2) ? norm0 : 2.0 * norm0) *
                           (mode == 1 ? 1.0 : mode == 2 ? w * (double)k2 : w);
        if (ki != cur) {
          if (cur >= 0) atomicAdd(&wbins[cur], sum);
          cur = ki;
          sum = 0.0;
        }
        sum += val;
      }
      if (++iz == Nf) {
        iz = 0;
        if (++iy == N) { iy = 0; ++ix; }
      }
    }
    if (cur >= 0) atomicAdd(&wbins[cur], sum);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < Nf; i += DIAG_NT) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < NW; ++k) t += bins[k][i];
    part[(size_t)blockIdx.x * Nf + i] = t;
  }
}

// out[s] = sum over blocks (fixed order), one wavefront per shell (256^3: 64
// us with one block's threads each summing a shell, 4.4 us now).
template <int N>
__global__ void __launch_bounds__(64) k_shell_final(const double* __restrict__ part, int nblk, double* __restrict__ out) {
  constexpr int Nf = N / 2 + 1;
  const int s = blockIdx.x;
  double acc = 0.0;
  for (int b = threadIdx.x; b < nblk; b += 64) acc += part[(size_t)b * Nf + s];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (threadIdx.x == 0) out[s] = acc;
}
// out[s] <- sum of out[s'] over s' >= s (one wavefront; lane l owns a run of shells)
template <int N>
__global__ void __launch_bounds__(64) k_shell_cumulate(double* __restrict__ out) {
  constexpr int Nf = N / 2 + 1, PER = (Nf + 63) / 64;
  double v[PER], sum = 0.0;
#pragma unroll
  for (int k = PER - 1; k >= 0; --k) {
    const int s = (int)threadIdx.x * PER + k;
    sum += s < Nf ? out[s] : 0.0;
    v[k] = sum;
  }
  double inc = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double t = __shfl_down(inc, off, 64);
    if (threadIdx.x + off < 64) inc += t;
  }
  double above = __shfl_down(inc, 1, 64);      // the runs above this lane's
  if (threadIdx.x == 63) above = 0.0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int s = (int)threadIdx.x * PER + k;
    if (s < Nf) out[s] = v[k] + above;
  }
}

// Spectral divergence i (kx u_x + ky u_y + kz u_z) of a vector field, with the
// derivative of each axis's Nyquist mode taken as zero: the reference's
// diff_x / diff_y / diff_z (forced-dns-sm.py:216-229) differentiate with a
// 1-D rfft along the axis, multiply by i k (k = 0..N/2) and irfft, which drops
// the imaginary Nyquist coefficient that i (N/2) times a real one makes.
template <typename T, int N>
__global__ void __launch_bounds__(256)
k_div_spec(const C<T>* __restrict__ u, size_t fs, C<T>* __restrict__ out) {
  constexpr int Nf = N / 2 + 1;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < fs; i += (size_t)gridDim.x * blockDim.x) {
    const int iz = (int)(i % Nf);
    const size_t rem = i / Nf;
    const int ix = (int)(rem / N), iy = (int)(rem % N);
    const T kx = ix == N / 2 ? (T)0 : (T)kwave(ix, N);
    const T ky = iy == N / 2 ? (T)0 : (T)kwave(iy, N);
    const T kz = iz == N / 2 ? (T)0 : (T)iz;
    const C<T> a = u[i], b = u[fs + i], c = u[2 * fs + i];
    const T re = kx * a.x + ky * b.x + kz * c.x, im = kx * a.y + ky * b.y + kz * c.y;
    out[i] = mkc<T>(-im, re);      // i (k . u)
  }
}

// per block: sum, min, max, sum of squares.  Bound by the read: 16-byte (FP32)
// loads, four in flight per thread, when x is aligned for them (fields are;
// the droplets' mass column need not be), else one entry at a time.  256^3
// FP32, a pass over three fields and one over one field: 428 us with one entry
// per thread and load, 64 us now (4.2 TB/s).
template <typename T>
__global__ void __launch_bounds__(DIAG_NT)
k_stats_partial(const T* __restrict__ x, size_t n, double* __restrict__ part) {
  __shared__ double sh[DIAG_NT];
  double s = 0.0, q = 0.0, mn = INFINITY, mx = -INFINITY;
  auto one = [&](T e) {
    const double v = (double)e;
    s += v; q += v * v; mn = fmin(mn, v); mx = fmax(mx, v);
  };
  const size_t nv = (reinterpret_cast<uintptr_t>(x) % sizeof(V4<T>) == 0) ? n / 4 : 0;
  const size_t per = (nv + gridDim.x - 1) / gridDim.x;
  const size_t i0 = blockIdx.x * per, i1 = (i0 + per < nv) ? i0 + per : nv;
  const V4<T>* xv = reinterpret_cast<const V4<T>*>(x);
  constexpr int U = 4;
  for (size_t i = i0 + threadIdx.x; i < i1; i += U * DIAG_NT) {
    V4<T> v[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i + u * DIAG_NT < i1) v[u] = xv[i + u * DIAG_NT];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i + u * DIAG_NT < i1) { one(v[u].x); one(v[u].y); one(v[u].z); one(v[u].w); }
  }
  // the entries not taken in quads
  const size_t t0 = 4 * nv, tper = (n - t0 + gridDim.x - 1) / gridDim.x;
  const size_t j0 = t0 + blockIdx.x * tper, j1 = (j0 + tper < n) ? j0 + tper : n;
  for (size_t j = j0 + threadIdx.x; j < j1; j += DIAG_NT) one(x[j]);
  const double a = blockSum<DIAG_NT>(s, sh);
  __syncthreads();
  const double b = blockSum<DIAG_NT>(q, sh);
  __syncthreads();
  const double c = -blockMax<DIAG_NT>(-mn, sh);
  __syncthreads();
  const double d = blockMax<DIAG_NT>(mx, sh);
  if (threadIdx.x == 0) { part[4 * blockIdx.x] = a; part[4 * blockIdx.x + 1] = c; part[4 * blockIdx.x + 2] = d; part[4 * blockIdx.x + 3] = b; }
}

// One wavefront over the blocks (fixed order): 32 us with one thread, 4.9 us now.
static __global__ void __launch_bounds__(64) k_stats_final(const double* __restrict__ part, int nblk, double* __restrict__ out) {
  double s = 0.0, q = 0.0, mn = INFINITY, mx = -INFINITY;
  for (int b = threadIdx.x; b < nblk; b += 64) {
    s += part[4 * b]; mn = fmin(mn, part[4 * b + 1]); mx = fmax(mx, part[4 * b + 2]); q += part[4 * b + 3];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    s += __shfl_xor(s, off, 64); q += __shfl_xor(q, off, 64);
    mn = fmin(mn, __shfl_xor(mn, off, 64)); mx = fmax(mx, __shfl_xor(mx, off, 64));
  }
  if (threadIdx.x == 0) { out[0] = s; out[1] = mn; out[2] = mx; out[3] = q; }
}

}  // namespace ld
