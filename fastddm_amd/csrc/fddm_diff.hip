// Stages (d) + (e): direct differences, D(q, d) = sum_t |F(t + d) - F(t)|^2 / (L - d).
//
// Three forms, chosen by diff_l:
//
// k_diff: one column (q) per workgroup.  The series is staged once in LDS,
// the workgroup's waves take batches of four lags in turn: 64 lanes walk t,
// each F(t) read serves four differences, and the main loop, over the t for
// which all four lags are inside the series, needs no mask.  The four sums of
// a batch are reduced together (halves of the wave, then rows, are traded
// while adding, so the last four steps work on four lags at once).
// Bound: LDS reads, 1.25 per difference (a read of sizeof(F) bytes per lane),
// and in compensated FP32 VALU issue (6.5 instructions per difference,
// widening included).
//
// k_diff_short: four, two or one column per wave, one per 16, 32 or 64 lanes,
// each series in its own LDS slice: with short series fewer lanes per column
// leave less of them idle in the last step over t and share one reduction, and
// with few lags a workgroup works on four columns or more at once.
//
// k_diff_long: one column per wave, for series beyond the LDS.
//
// Differences are formed after widening to Acc, so they are exact on the
// compensated paths.
//
// Kernel time against one wave per column or segment with masked loops and a
// scan per lag (131584 columns of 1200 FP64 samples, 60 lags, read from L2
// there): 7.40 -> 2.1 ms; 33024 columns, 50 lags: 600 samples compensated FP32
// 0.435 -> 0.297 ms, 300 samples 0.220 -> 0.153 ms (a column per workgroup
// takes 0.211 there), FP64 0.250 -> 0.148 ms.
#include <algorithm>
#include <type_traits>

#include "fddm_kernels.hpp"
#include "fddm_wave.hpp"

namespace fddm {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kLagBatch = 4;

template <int PREC>
using acc_t = std::conditional_t<PREC == PREC_FP32, float, double>;

// a: rows or halves [a0 | b0], b: [a1 | b1] of two values' halves (permlane
// swaps); then a + b holds a's sum in the first and b's in the second ones.
template <bool ROWS>
__device__ __forceinline__ void trade(unsigned& a, unsigned& b) {
  const auto r = ROWS ? __builtin_amdgcn_permlane16_swap(a, b, false, false)
                      : __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
template <bool ROWS>
__device__ __forceinline__ float add_traded(float x, float y) {
  unsigned a = __float_as_uint(x), b = __float_as_uint(y);
  trade<ROWS>(a, b);
  return __uint_as_float(a) + __uint_as_float(b);
}
template <bool ROWS>
__device__ __forceinline__ double add_traded(double x, double y) {
  const uint64_t u = static_cast<uint64_t>(__double_as_longlong(x)), v = static_cast<uint64_t>(__double_as_longlong(y));
  unsigned al = static_cast<unsigned>(u), ah = static_cast<unsigned>(u >> 32);
  unsigned bl = static_cast<unsigned>(v), bh = static_cast<unsigned>(v >> 32);
  trade<ROWS>(al, bl);
  trade<ROWS>(ah, bh);
  return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(ah) << 32) | al)) +
         __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(bh) << 32) | bl));
}
// Inclusive scan inside 16-lane rows.
template <typename A>
__device__ __forceinline__ A row_scan(A v) {
  v += wave::dpp_zero<wave::kRowShr1, 0xf>(v);
  v += wave::dpp_zero<wave::kRowShr2, 0xf>(v);
  v += wave::dpp_zero<wave::kRowShr4, 0xf>(v);
  v += wave::dpp_zero<wave::kRowShr8, 0xf>(v);
  return v;
}

// PS and VAR of one column from its sums.
template <typename Acc, typename C, typename OutT>
__device__ __forceinline__ void store_moments(const TimeArgs& a, int q, size_t oq, Acc sr, Acc si, Acc s2) {
  OutT* __restrict__ out = static_cast<OutT*>(a.out);
  const int L = a.L;
  const Acc mr = sr / L, mi = si / L;
  Acc ps, var;
  if (a.S0) {
    // spectra hold F(t) - F(0): VAR is shift invariant, PS adds |F(0) + mean|^2
    var = s2 / L - (mr * mr + mi * mi);
    const C z = frame0_spectrum<C>(a, q);
    const Acc fr = mr + static_cast<Acc>(z.x), fi = mi + static_cast<Acc>(z.y);
    ps = var + fr * fr + fi * fi;
  } else {
    ps = s2 / L;
    var = ps - mr * mr - mi * mi;
  }
  out[static_cast<size_t>(a.nl) * a.ldo + oq] = static_cast<OutT>(ps);
  out[static_cast<size_t>(a.nl + 1) * a.ldo + oq] = static_cast<OutT>(var);
}

// Lags i0 .. i0 + K - 1 of the series in LDS by one wave.
template <typename C, typename Acc, typename OutT, int K>
__device__ __forceinline__ void wave_lags(const TimeArgs& a, const C* ser, int i0, size_t oq, int lane) {
  const int L = a.L;
  int d[K], dmin = L, dmax = 0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    d[k] = __builtin_amdgcn_readfirstlane(static_cast<int>(a.lags[i0 + k]));
    dmin = min(dmin, d[k]);
    dmax = max(dmax, d[k]);
  }
  Acc acc[K] = {};
  const int whole = (L - dmax) & ~63;  // t below it: inside the series for every lag
  const C* const p = ser + lane;
#pragma unroll 2
  for (int t = 0; t < whole; t += 64) {
    const C v = p[t];
    C u[K];
#pragma unroll
    for (int k = 0; k < K; ++k) u[k] = p[t + d[k]];
    const Acc vx = static_cast<Acc>(v.x), vy = static_cast<Acc>(v.y);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const Acc dr = static_cast<Acc>(u[k].x) - vx, di = static_cast<Acc>(u[k].y) - vy;
      acc[k] += dr * dr + di * di;
    }
  }
  for (int t0 = whole; t0 < L - dmin; t0 += 64) {
    const int t = t0 + lane;
    const C v = ser[min(t, L - 1)];
    const Acc vx = static_cast<Acc>(v.x), vy = static_cast<Acc>(v.y);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const C u = ser[min(t + d[k], L - 1)];
      const Acc dr = static_cast<Acc>(u.x) - vx, di = static_cast<Acc>(u.y) - vy;
      acc[k] += t + d[k] < L ? dr * dr + di * di : Acc(0);
    }
  }
  OutT* __restrict__ out = static_cast<OutT*>(a.out) + static_cast<size_t>(i0) * a.ldo + oq;
  if constexpr (K == 4) {
    // rows 0 .. 3 end with the sums of lags 0, 2, 1, 3
    const Acc s = row_scan(add_traded<true>(add_traded<false>(acc[0], acc[1]), add_traded<false>(acc[2], acc[3])));
    const int row = lane >> 4, k = (row >> 1) | ((row & 1) << 1);
    const int dk = k == 0 ? d[0] : k == 1 ? d[1] : k == 2 ? d[2] : d[3];
    if ((lane & 15) == 15) out[static_cast<size_t>(k) * a.ldo] = static_cast<OutT>(s / static_cast<Acc>(L - dk));
  } else {
    static_assert(K == 1, "batches of four, the rest one by one");
    const Acc s = wave::incl_scan(acc[0]);
    if (lane == 63) out[0] = static_cast<OutT>(s / static_cast<Acc>(L - d[0]));
  }
}

template <typename T, typename OutT, int PREC>
__global__ void __launch_bounds__(1024) k_diff(TimeArgs a, int wg_per_xcd, int nb) {
  using C = cplx_t<T>;
  using Acc = acc_t<PREC>;
  extern __shared__ __align__(16) unsigned char smem[];
  // contiguous ranges of columns per XCD, so neighbouring outputs meet in one L2
  const int c = (blockIdx.x & 7) * wg_per_xcd + (blockIdx.x >> 3);
  if (c >= a.cols) return;  // whole workgroup: before any barrier
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int NT = blockDim.x, NW = NT >> 6, L = a.L;
  Acc* const red = reinterpret_cast<Acc*>(smem);
  C* const ser = reinterpret_cast<C*>(smem + 3 * 16 * sizeof(double));
  const int q = __builtin_amdgcn_readfirstlane(col_q(a, c));
  const C* __restrict__ src = static_cast<const C*>(a.S) + static_cast<size_t>(q - a.s_q0) * a.Lp;
  Acc sr = 0, si = 0, s2 = 0;
  for (int t0 = tid; t0 < L; t0 += 4 * NT) {  // four loads in flight per lane
    C v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = src[min(t0 + k * NT, L - 1)];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (t0 + k * NT < L) {
        ser[t0 + k * NT] = v[k];
        const Acc fx = static_cast<Acc>(v[k].x), fy = static_cast<Acc>(v[k].y);
        sr += fx;
        si += fy;
        s2 += fx * fx + fy * fy;
      }
  }
  sr = wave::incl_scan(sr);
  si = wave::incl_scan(si);
  s2 = wave::incl_scan(s2);
  if (lane == 63) {
    red[3 * wid] = sr;
    red[3 * wid + 1] = si;
    red[3 * wid + 2] = s2;
  }
  __syncthreads();
  const size_t oq = col_out(a, c);
  if (tid == NT - 1) {  // (the last wave has the fewest lags)
    sr = si = s2 = 0;
    for (int w = 0; w < NW; ++w) {
      sr += red[3 * w];
      si += red[3 * w + 1];
      s2 += red[3 * w + 2];
    }
    store_moments<Acc, C, OutT>(a, q, oq, sr, si, s2);
  }
  for (int b = wid; b < nb; b += NW) wave_lags<C, Acc, OutT, kLagBatch>(a, ser, b * kLagBatch, oq, lane);
  // the remaining lags, one by one, on the waves that had a batch less
  for (int i = nb * kLagBatch + (wid - nb % NW + NW) % NW; i < a.nl; i += NW)
    wave_lags<C, Acc, OutT, 1>(a, ser, i, oq, lane);
}

// a's sum over the lanes i and MIRROR(i) in the lanes without BIT, b's in
// those with it (the mirror of a lane without it has it).
template <int MIRROR, int BIT, typename A>
__device__ __forceinline__ A add_mirrored(A a, A b, int lane) {
  const bool hi = (lane & BIT) != 0;
  return (hi ? b : a) + wave::dpp_zero<MIRROR, 0xf>(hi ? a : b);
}
constexpr int kRowMirror = 0x140, kHalfMirror = 0x141, kQuadSwap1 = 0xb1, kQuadSwap2 = 0x4e;

// The segment's last lane ends with its sum.
template <int SEG, typename A>
__device__ __forceinline__ A segment_scan(A v) {
  if constexpr (SEG == 64) return wave::incl_scan(v);
  v = row_scan(v);
  if constexpr (SEG == 32) v += wave::dpp_zero<wave::kRowBcast15, 0xa>(v);
  return v;
}

// Lags i0 .. i0 + K - 1 of a segment's series; lane l of a segment takes
// t = l, l + SEG, ...
template <typename C, typename Acc, typename OutT, int SEG, int K>
__device__ __forceinline__ void segment_lags(const TimeArgs& a, const C* ser, int i0, size_t oq, int lane, bool valid) {
  const int L = a.L, sl = lane & (SEG - 1);
  const C* const p = ser + sl;
  OutT* __restrict__ const out = static_cast<OutT*>(a.out) + oq;
  int d[K];
#pragma unroll
  for (int k = 0; k < K; ++k) d[k] = __builtin_amdgcn_readfirstlane(static_cast<int>(a.lags[i0 + k]));
  Acc acc[K] = {};
  const int whole = (L - d[K - 1]) & ~(SEG - 1);  // (lags ascend) t below it: inside the series for every lag
#pragma unroll 2
  for (int t = 0; t < whole; t += SEG) {
    const C v = p[t];
    C u[K];
#pragma unroll
    for (int k = 0; k < K; ++k) u[k] = p[t + d[k]];
    const Acc vx = static_cast<Acc>(v.x), vy = static_cast<Acc>(v.y);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const Acc dr = static_cast<Acc>(u[k].x) - vx, di = static_cast<Acc>(u[k].y) - vy;
      acc[k] += dr * dr + di * di;
    }
  }
  for (int t0 = whole; t0 < L - d[0]; t0 += SEG) {
    const int t = t0 + sl;
    const C v = ser[min(t, L - 1)];
    const Acc vx = static_cast<Acc>(v.x), vy = static_cast<Acc>(v.y);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const C u = ser[min(t + d[k], L - 1)];
      const Acc dr = static_cast<Acc>(u.x) - vx, di = static_cast<Acc>(u.y) - vy;
      acc[k] += t + d[k] < L ? dr * dr + di * di : Acc(0);  // (not a product: the frames may hold NaN)
    }
  }
  if constexpr (K == 4) {
    // the four sums of every segment, traded while adding; k: the lag this lane ends with
    Acc s;
    int k;
    if constexpr (SEG == 16) {
      s = add_mirrored<kHalfMirror, 4>(add_mirrored<kRowMirror, 8>(acc[0], acc[1], lane),
                                       add_mirrored<kRowMirror, 8>(acc[2], acc[3], lane), lane);
      k = ((lane >> 3) & 1) | ((lane >> 1) & 2);
    } else {
      s = add_mirrored<kRowMirror, 8>(add_traded<true>(acc[0], acc[1]), add_traded<true>(acc[2], acc[3]), lane);
      s += wave::dpp_zero<kHalfMirror, 0xf>(s);
      k = ((lane >> 4) & 1) | ((lane >> 2) & 2);
    }
    s += wave::dpp_zero<kQuadSwap1, 0xf>(s);
    s += wave::dpp_zero<kQuadSwap2, 0xf>(s);
    const int dk = k == 0 ? d[0] : k == 1 ? d[1] : k == 2 ? d[2] : d[3];
    const bool writer = SEG == 16 ? (lane & 3) == 0 : (lane & 7) == 0;
    if (writer && valid)
      out[static_cast<size_t>(i0 + k) * a.ldo] = static_cast<OutT>(s / static_cast<Acc>(L - dk));
  } else {
    static_assert(K == 1, "batches of four, the rest one by one");
    const Acc s = segment_scan<SEG>(acc[0]);
    if (valid && sl == SEG - 1) out[static_cast<size_t>(i0) * a.ldo] = static_cast<OutT>(s / static_cast<Acc>(L - d[0]));
  }
}

// A wave works on 64 / SEG columns, one per segment of SEG lanes, four lags at
// a time and the rest one by one (with stand-ins for a last batch of four, one
// lag took as long as four: 300 x 512^2 in compensated FP32 113 us, now 95).
// Nothing of one column waits for another wave.
template <typename T, typename OutT, int PREC, int SEG>
__global__ void __launch_bounds__(kThreads) k_diff_short(TimeArgs a, int wg_per_xcd, int pitch) {
  using C = cplx_t<T>;
  using Acc = acc_t<PREC>;
  static_assert(SEG == 16 || SEG == 32 || SEG == 64, "segment");
  constexpr int QPW = 64 / SEG;
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int sl = lane & (SEG - 1), seg = lane / SEG;
  // columns of the launch: cw is this wave's first
  const int cw = ((blockIdx.x & 7) * wg_per_xcd + (blockIdx.x >> 3)) * kWaves * QPW + wid * QPW;
  if (cw >= a.cols) return;  // whole waves: nothing below synchronises the workgroup
  const bool valid = cw + seg < a.cols;
  const int c = valid ? cw + seg : a.cols - 1;  // (idle segments repeat the last column and store nothing)
  int q = col_q(a, c);
  if constexpr (SEG == 64) q = __builtin_amdgcn_readfirstlane(q);
  const int L = a.L, nl = a.nl;
  const C* __restrict__ src = static_cast<const C*>(a.S) + static_cast<size_t>(q - a.s_q0) * a.Lp;
  C* const ser = reinterpret_cast<C*>(smem) + static_cast<size_t>(wid * QPW + seg) * pitch;
  Acc sr = 0, si = 0, s2 = 0;
  for (int t0 = sl; t0 < L; t0 += 4 * SEG) {  // four loads in flight per lane
    C v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = src[min(t0 + SEG * k, L - 1)];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (t0 + SEG * k < L) {
        ser[t0 + SEG * k] = v[k];
        const Acc fx = static_cast<Acc>(v[k].x), fy = static_cast<Acc>(v[k].y);
        sr += fx;
        si += fy;
        s2 += fx * fx + fy * fy;
      }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  sr = segment_scan<SEG>(sr);
  si = segment_scan<SEG>(si);
  s2 = segment_scan<SEG>(s2);
  const size_t oq = col_out(a, c);
  if (valid && sl == SEG - 1) store_moments<Acc, C, OutT>(a, q, oq, sr, si, s2);

  const int nb = nl / kLagBatch;
  if constexpr (SEG == 64) {
    for (int b = 0; b < nb; ++b) wave_lags<C, Acc, OutT, kLagBatch>(a, ser, b * kLagBatch, oq, lane);
    for (int i = nb * kLagBatch; i < nl; ++i) wave_lags<C, Acc, OutT, 1>(a, ser, i, oq, lane);
  } else {
    for (int b = 0; b < nb; ++b) segment_lags<C, Acc, OutT, SEG, kLagBatch>(a, ser, b * kLagBatch, oq, lane, valid);
    for (int i = nb * kLagBatch; i < nl; ++i) segment_lags<C, Acc, OutT, SEG, 1>(a, ser, i, oq, lane, valid);
  }
}

// Series too long for the LDS: one column per wave, read from L2.
template <typename T, typename OutT, int PREC>
__global__ void __launch_bounds__(kThreads) k_diff_long(TimeArgs a, int wg_per_xcd) {
  using C = cplx_t<T>;
  using Acc = acc_t<PREC>;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int c = ((blockIdx.x & 7) * wg_per_xcd + (blockIdx.x >> 3)) * kWaves + wid;
  if (c >= a.cols) return;
  const int q = __builtin_amdgcn_readfirstlane(col_q(a, c)), L = a.L;
  const C* __restrict__ src = static_cast<const C*>(a.S) + static_cast<size_t>(q - a.s_q0) * a.Lp;
  Acc sr = 0, si = 0, s2 = 0;
  for (int t = lane; t < L; t += 64) {
    const Acc fx = static_cast<Acc>(src[t].x), fy = static_cast<Acc>(src[t].y);
    sr += fx;
    si += fy;
    s2 += fx * fx + fy * fy;
  }
  sr = wave::incl_scan(sr);
  si = wave::incl_scan(si);
  s2 = wave::incl_scan(s2);
  const size_t oq = col_out(a, c);
  if (lane == 63) store_moments<Acc, C, OutT>(a, q, oq, sr, si, s2);
  const int nb = a.nl / kLagBatch;
  for (int b = 0; b < nb; ++b) wave_lags<C, Acc, OutT, kLagBatch>(a, src, b * kLagBatch, oq, lane);
  for (int i = nb * kLagBatch; i < a.nl; ++i) wave_lags<C, Acc, OutT, 1>(a, src, i, oq, lane);
}

template <typename K, typename... Args>
hipError_t launch(K kernel, unsigned grid, unsigned threads, size_t lds, hipStream_t s, Args... args) {
  if (grid == 0) return hipSuccess;
  if (lds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), lds, s, args...);
  return hipGetLastError();
}

// Four or two columns per wave while their series leave four workgroups per
// CU, or eight with a few lags, where loading the series is most of the time
// (300 x 512^2 in compensated FP32: one lag 105 -> 95 us, five 124 -> 118, six
// 129 -> 138; 500 x 256^2, four lags: two columns per wave 54 us, one 48).  Plain
// FP32, with the least work per value read, takes eight and six (300 x 256^2,
// 24 lags: four columns 55 us, two 44; 500 x 256^2: two 79, one 69).
// Then, with few lags, a column per wave: a workgroup per column leaves most of
// its waves without a lag (256^2 columns, kernel time with a workgroup and with
// a wave per column: 700 samples in compensated FP32, 1 lag 66 and 50 us, 24
// lags 175 and 161, 60 lags 302 and 301; 400 in FP64, 1 lag 65 and 49 us, 24 lags
// 119 and 100; longer series want more waves per LDS: 1200 in compensated FP32, 1
// lag 86 and 99 us).
// Then a column per workgroup, with as many waves as keep 16 per CU or more
// beside the series' LDS, every lag by itself where there is a wave for each
// (4000 samples, 4 lags: as one batch 1145 us in FP64, by themselves 457);
// beyond the LDS, a wave per column.
template <typename T, typename OutT, int PREC>
hipError_t diff_l(const TimeArgs& a, hipStream_t s) {
  constexpr size_t csz = sizeof(cplx_t<T>);
  const int nq = a.cols;
  auto per_xcd = [&](int cols) { return ((nq + cols - 1) / cols + 7) / 8; };
  // slices: an odd multiple of 128 bytes apart, so the segments of 16 FP32 lanes read different banks
  const int pitch = ((a.L + 15) / 16 | 1) * 16;
  auto segments = [&](auto kernel, int qpw) {
    const int wpx = per_xcd(kWaves * qpw);
    return launch(kernel, 8u * wpx, kThreads, csz * pitch * kWaves * qpw, s, a, wpx, pitch);
  };
  constexpr bool plain = PREC == PREC_FP32;
  const size_t lds1 = csz * pitch * kWaves;  // of a workgroup with one column per wave
  const bool few = a.nl < 6;
  if (4 * lds1 <= (few || plain ? 20 : 40) << 10) return segments(k_diff_short<T, OutT, PREC, 16>, 4);
  if (2 * lds1 <= (few ? 20 : plain ? 28 : 40) << 10) return segments(k_diff_short<T, OutT, PREC, 32>, 2);
  if (lds1 <= (csz == 16 ? 34 : 28) << 10 && a.nl < 32) return segments(k_diff_short<T, OutT, PREC, 64>, 1);
  const size_t lds = csz * a.L + 3 * 16 * sizeof(double);
  if (lds <= 159 * 1024) {
    const unsigned threads = lds <= 40 * 1024 ? 256 : lds <= 80 * 1024 ? 512 : 1024;
    // a launch holds less than 2^32 threads: larger planes (16.7 M columns of
    // 256 threads) in several
    const int nb = a.nl <= static_cast<int>(threads / 64) ? 0 : a.nl / kLagBatch;
    const int64_t most = static_cast<int64_t>((uint64_t(1) << 32) / threads) - 8;
    for (int64_t c = 0; c < nq; c += most) {
      TimeArgs part = a;
      part.c0 += static_cast<int>(c);
      part.cols = static_cast<int>(std::min<int64_t>(most, nq - c));
      if (a.local) part.out = static_cast<OutT*>(a.out) + c;  // (stored by column of the launch)
      const int wpx = (part.cols + 7) / 8;
      const hipError_t e = launch(k_diff<T, OutT, PREC>, 8u * wpx, threads, lds, s, part, wpx, nb);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  const int wpx = per_xcd(kWaves);
  return launch(k_diff_long<T, OutT, PREC>, 8u * wpx, kThreads, 0, s, a, wpx);
}

}  // namespace

hipError_t launch_diff(const TimeArgs& a, int precision, int out_dtype, hipStream_t s) {
  const bool f32 = out_dtype == OUT_F32;
  switch (precision) {
    case PREC_FP64: return f32 ? diff_l<double, float, PREC_FP64>(a, s) : diff_l<double, double, PREC_FP64>(a, s);
    case PREC_FP32: return f32 ? diff_l<float, float, PREC_FP32>(a, s) : diff_l<float, double, PREC_FP32>(a, s);
    case PREC_FP32C: return f32 ? diff_l<float, float, PREC_FP32C>(a, s) : diff_l<float, double, PREC_FP32C>(a, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace fddm
