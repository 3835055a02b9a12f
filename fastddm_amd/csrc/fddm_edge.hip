// FP64 edge correction of the compensated FP32 path.
//
// A lag dt with n = L - dt frame pairs sums n squared differences.  For n = 1
// the single difference |F(L-1) - F(0)|^2 can be arbitrarily small compared
// with |F|^2 (the two frames happen to agree at that q), and the float
// rounding of the spatial transform -- about 1e-6 of the spectrum's rms --
// then dominates it: at 1024^2 x 4000 about one q in 10^6 misses rtol 1e-3.
// For n >= 2 all n differences would have to be small at once, which does
// not happen at these sizes.  So the first and last kEdgeFrames frames are
// transformed once more in FP64 (a child plan over those frames, frame-0
// subtracted like the main pass, whose rows read them where they lie; the raw
// first frame is transformed beside them, for PS), and the lags with n <= kEdgeFrames are
// recomputed from them by direct sums in FP64, after the time / diff kernel
// has written its own values.
//
// The time kernel's Wiener-Khinchin values carry an absolute error of a few
// 1e-7 of sum_t |G|^2 in (L - dt) D.  Where (L - dt) D is small against that
// sum -- slow low-q modes and chance near-recurrences -- the kernel marks the
// q, and k_fix recomputes the affected lags of the marked q by direct
// differences of the stored float series in double: each workgroup lists its
// marked columns (flags read in parallel), each marked one's lags are shared
// by the workgroup's waves, lanes run over t and a wave sum closes each lag.
#include <algorithm>

#include "fddm_kernels.hpp"
#include "fddm_wave.hpp"

namespace fddm {
namespace {

constexpr int kThreads = 256;

// Two threads per output column o (y-shifted q), comp = 0 and 1: for every lag
// index i >= i0 (those with n = L - lags[i] <= E), D = sum_{t < n}
// |F(t + dt) - F(t)|^2 / n from the FP64 edge spectra S64[q][c] (row pitch lp),
// where frame f sits in column f if f < E or the stack is short (L <= 2E), else
// f - (L - 2E).  For E = kEdgeFrames and L > 2E the 2E values are loaded once
// (16 loads in flight) and D depends on n alone: frame t + dt = L - n + t sits
// in column 2E - n + t, so the E sums run over registers with compile-time
// indices, a thread taking one component, and are then stored to the lag rows
// they belong to, the two threads in turn.  (One thread for both components
// took 98 VGPRs, which left the marked columns 4 waves per SIMD.)
template <typename OutT>
__device__ __forceinline__ void edge_fix(const TimeArgs& a, const double2* __restrict__ S64, uint64_t lp, int E, int i0,
                                         int c, int comp) {
  const int q = col_q(a, c), L = a.L, nl = a.nl;
  const uint32_t* __restrict__ lags = a.lags;
  OutT* __restrict__ out = static_cast<OutT*>(a.out);
  const size_t o = col_out(a, c), ldo = a.ldo;
  const double2* __restrict__ f = S64 + static_cast<size_t>(q) * lp;
  if (E == kEdgeFrames && L > 2 * kEdgeFrames) {
    constexpr int EE = kEdgeFrames;
    const double* __restrict__ fc = reinterpret_cast<const double*>(f) + comp;
    double v[2 * EE];
#pragma unroll
    for (int k = 0; k < 2 * EE; ++k) v[k] = fc[2 * k];
    double dn[EE] = {};  // dn[n - 1]: n D of the lag with n pairs
#pragma unroll
    for (int t = 0; t < EE; ++t)
#pragma unroll
      for (int n = t + 1; n <= EE; ++n) {
        const double d = v[2 * EE - n + t] - v[t];
        dn[n - 1] += d * d;
      }
#pragma unroll
    for (int n = 0; n < EE; ++n) dn[n] += __shfl_xor(dn[n], 1, 64);
    for (int i = i0 + comp; i < nl; i += 2) {
      const int n = L - static_cast<int>(lags[i]);  // 1 <= n <= EE
      double D = dn[0];
#pragma unroll
      for (int k = 1; k < EE; ++k)
        if (n == k + 1) D = dn[k];
      out[static_cast<size_t>(i) * ldo + o] = static_cast<OutT>(D / n);
    }
    return;
  }
  const int shift = L <= 2 * E ? 0 : L - 2 * E;
  for (int i = i0 + comp; i < nl; i += 2) {
    const int d = static_cast<int>(lags[i]), n = L - d;
    double acc = 0.0;
    for (int t = 0; t < n; ++t) {
      const int e = t + d;
      const double2 x = f[e < E ? e : e - shift];
      const double2 y = f[t];  // t < n <= E
      const double dr = x.x - y.x, di = x.y - y.y;
      acc += dr * dr + di * di;
    }
    out[static_cast<size_t>(i) * ldo + o] = static_cast<OutT>(acc / n);
  }
}

// Both corrections in one launch: they write different lags (at most E pairs;
// more than 32).  S64 null: no edge lags; a.flags null: no marked columns.
template <typename OutT>
__global__ void __launch_bounds__(kThreads, 8)
    k_fix(TimeArgs a, const double2* __restrict__ S64, uint64_t lp, int E, int i0) {
  if (S64)  // (both threads of a column are inside or outside the loop)
    for (int c = static_cast<int>((blockIdx.x * kThreads + threadIdx.x) / 2); c < a.cols; c += static_cast<int>(gridDim.x) * (kThreads / 2))
      edge_fix<OutT>(a, S64, lp, E, i0, c, threadIdx.x & 1);
  if (!a.flags) return;
  // workgroup g owns the columns g + m G (G workgroups); their flags are read
  // at once, one per thread, the marked columns listed in LDS, and the
  // waves of the workgroup share the lags of each listed column
  __shared__ int list[kThreads];
  __shared__ int count;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int L = a.L, nl = a.nl, G = static_cast<int>(gridDim.x), g = static_cast<int>(blockIdx.x);
  const uint32_t* __restrict__ lags = a.lags;
  OutT* __restrict__ out = static_cast<OutT*>(a.out);
  const size_t ldo = a.ldo;
  const int M = (a.cols - g + G - 1) / G;  // columns of this workgroup (g < cols)
  for (int m0 = 0; m0 < M; m0 += kThreads) {
    if (threadIdx.x == 0) count = 0;
    __syncthreads();
    const int m = m0 + static_cast<int>(threadIdx.x);
    if (m < M) {
      const int c = g + m * G;
      if (a.flags[col_q(a, c)] != 0) list[atomicAdd(&count, 1)] = c;
    }
    __syncthreads();
    const int nmark = count;
    for (int k = 0; k < nmark; ++k) {
      const int c = list[k];
      const int q = col_q(a, c);
      const size_t oq = col_out(a, c);
      const double var = static_cast<double>(out[static_cast<size_t>(nl + 1) * ldo + oq]);
      const double thr = kWkFlag * static_cast<double>(L) * var;
      const float2* __restrict__ f = static_cast<const float2*>(a.S) + static_cast<size_t>(q - a.s_q0) * a.Lp;
      for (int b = wave * 64; b < nl; b += kThreads) {
        const int i = b + lane;
        bool need = false;
        if (i < nl) {
          const int n = L - static_cast<int>(lags[i]);
          need = n > 32 && static_cast<double>(n) * static_cast<double>(out[static_cast<size_t>(i) * ldo + oq]) < thr;
        }
        uint64_t todo = __ballot(need);
        while (todo) {
          const int ii = b + __ffsll(static_cast<long long>(todo)) - 1;
          todo &= todo - 1;
          const int d = static_cast<int>(lags[ii]), n = L - d;
          double acc = 0.0;
          for (int t = lane; t < n; t += 64) {
            const float2 x = f[t + d], y = f[t];
            const double dr = static_cast<double>(x.x) - static_cast<double>(y.x);
            const double di = static_cast<double>(x.y) - static_cast<double>(y.y);
            acc += dr * dr + di * di;
          }
          acc = wave::incl_scan(acc);
          if (lane == 63) out[static_cast<size_t>(ii) * ldo + oq] = static_cast<OutT>(acc / n);
        }
      }
    }
    __syncthreads();  // list and count are rewritten by the next round
  }
}

}  // namespace

hipError_t launch_fix(const TimeArgs& a, const void* S64, uint64_t lp, int E, int i0, int out_dtype, hipStream_t s) {
  if (i0 >= a.nl) S64 = nullptr;
  if (a.nl <= 0 || a.cols <= 0 || (!S64 && !a.flags)) return hipSuccess;
  // two threads per column for the edge lags; 2048 workgroups, which the chip
  // holds at once, share the marked columns (and the edge lags then)
  const unsigned edge = (static_cast<unsigned>(a.cols) + kThreads / 2 - 1) / (kThreads / 2);
  const dim3 grid(a.flags ? static_cast<unsigned>(std::min(a.cols, 2048)) : edge);
  if (out_dtype == OUT_F32) {
    hipLaunchKernelGGL(k_fix<float>, grid, dim3(kThreads), 0, s, a, static_cast<const double2*>(S64), lp, E, i0);
  } else {
    hipLaunchKernelGGL(k_fix<double>, grid, dim3(kThreads), 0, s, a, static_cast<const double2*>(S64), lp, E, i0);
  }
  return hipGetLastError();
}

}  // namespace fddm
