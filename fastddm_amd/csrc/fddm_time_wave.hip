// Stages (c) + (e), fft mode, for series of up to 2048 frames: every
// transform held in the registers of one wave.  (Planes of few columns take
// fddm_time_p2.hip, see short_columns in fddm_capi.hip.)
//
// D(q, dt) does not depend on the zero-padded length N >= 2L - 1, so the
// time stage runs at N = 2M, M = max(128, 2^ceil(log2 L)).  With the upper
// half of the input zero, the N-point transform G of the M samples x splits
// into two M-point ones, G(2k) = FFT_M(x)(k) and G(2k + 1) = FFT_M(x W_N^t)(k),
// and Re C(d) = Re IFFT_N(|G|^2) needs one more, Z = FFT_M(z) of
// z(k) = |G(2k)|^2 + i |G(2k + 1)|^2.
//
// A wave holds 64 / P columns (fddm_time_wave.hpp) and nothing waits at a
// workgroup barrier until the results of the workgroup's columns are written.
//
// What bounds it: VALU issue (74 % busy at M = 2048; 5400 instructions per
// column against 9600 of the workgroup form, k_time_p2, which spent 62 % of
// them on addresses, moves and conversions and met at two barriers per pass).
// All M lags are evaluated and staged, however few are written, and the series is
// read three times (7.25 GB of traffic for 131584 columns of 2000 samples, 5.07
// for the workgroup form); the requests mostly hit caches.
// Kernel time, before and after: 3.06 -> 1.85 ms for 131584 columns of 2000
// samples in compensated FP32, 1.58 -> 1.15 ms for 154080 of 997, 0.142 ->
// 0.088 ms for 15456 of 271 in FP64.
// Waves per workgroup: four, so that two or more workgroups per CU overlap;
// eight at M = 1024 in FP32, whose lag rows then leave in 32-byte pieces
// (1.35 -> 1.05 ms with all of 1002 lags); at M = 2048 and 512 and in FP64
// eight measured slower.
// Every batch of global loads is issued well before its use (issued()): with
// two to four waves per SIMD the latency is not hidden otherwise (the same
// kernel with the loads left to the scheduler: 3.7 ms at M = 2048).
#include <vector>

#include "fddm_time_wave.hpp"

namespace fddm {
namespace {
using namespace tw;

// Waves per SIMD: what the LDS of M = 2^10 and 2^11 allows in FP32, 3 where
// the registers of the others fit, 2 in double.
template <typename T, int R, int P>
constexpr int wave_occ() {
  return sizeof(T) == 8 ? (R == 8 ? 3 : 2) : R == 32 ? 2 : P == 64 || R == 8 ? 4 : 3;
}

template <typename T, typename OutT, int R, int P, int W>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(wave_occ<T, R, P>(), wave_occ<T, R, P>())))
    k_time_wave(TimeArgs a, int wg_per_xcd, int wgs, int subtract_mean) {
  using C = cplx_t<T>;
  using Lay = WaveLay<R, P, W>;
  constexpr int M = Lay::M, Q = Lay::Q;
  constexpr bool F64 = sizeof(T) == 8;

  extern __shared__ __align__(16) unsigned char smem[];

  // contiguous ranges of columns per XCD, so neighbouring output columns meet in one L2
  const int wgi = (blockIdx.x & 7) * wg_per_xcd + (blockIdx.x >> 3);
  if (wgi >= wgs) return;  // whole workgroup: before any barrier
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane / P, p = lane % P;
  const int qi = wave * Lay::GROUPS + g;  // column of the workgroup
  const int c0 = wgi * Q;
  const bool active = c0 + qi < a.cols;
  const int c = active ? c0 + qi : a.cols - 1;  // (idle groups repeat the last column and store nothing)
  int q = col_q(a, c);
  if constexpr (P == 64) q = __builtin_amdgcn_readfirstlane(q);
  const int L = a.L;
  const C* __restrict__ src = static_cast<const C*>(a.S) + static_cast<size_t>(q - a.s_q0) * a.Lp;
  const C* __restrict__ tab = static_cast<const C*>(a.twt);
  const double* __restrict__ inv = reinterpret_cast<const double*>(tab + Lay::TW_END);
  double* const wlds = reinterpret_cast<double*>(smem) + wave * Lay::WAVE;
  double* const xlds = wlds + g * Lay::GS;  // exchange
  double* const clds = wlds + g * Lay::CG;  // chunks
  double* const tlds = wlds + Lay::BUF + g * kLast;  // last samples

  // samples t = p + P r, zero from L on.  L > M / 2 except at the smallest M, so the first half needs no check.
  constexpr int FULL = M > 128 ? R / 2 : 0;
  auto load = [&](C(&x)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r) x[r] = r < FULL ? entry(src, P * r, p) : entry(src, 0, min(p + P * r, L - 1));
    issued();
  };
  auto center = [&](C(&x)[R], T mr, T mi) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const C f{x[r].x - mr, x[r].y - mi};
      x[r] = r < FULL || p + P * r < L ? f : C{0, 0};
    }
  };

  // 1. the series and its mean
  C v[R], x[R];
  load(v);
  const double rl = inv[0];
  const C first = frame0_spectrum<C>(a, q);  // F(0) of the raw first frame
  T m_r = 0, m_i = 0;
  center(v, T(0), T(0));
  double sr = 0, si = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    sr += static_cast<double>(v[r].x);
    si += static_cast<double>(v[r].y);
  }
  sr = group_last<P>(group_scan<P>(sr, p));
  si = group_last<P>(group_scan<P>(si, p));
  if (subtract_mean) {
    m_r = static_cast<T>(sr * rl);
    m_i = static_cast<T>(si * rl);
  }
  // sum of the subtracted series, for VAR and PS
  const double fsr = sr - static_cast<double>(L) * static_cast<double>(m_r);
  const double fsi = si - static_cast<double>(L) * static_cast<double>(m_i);
  center(v, m_r, m_i);

  // 2. power spectrum of the padded series, even and odd bins, then Z.  The
  // series is read again (from the caches) rather than held.
  C cs[R / 2];
  {
    T pe[R];
    wave_fft<T, Lay>(v, xlds, tab + Lay::TW_E, tab + Lay::TW_2, p, std::false_type{}, [&] { load(x); });
#pragma unroll
    for (int r = 0; r < R; ++r) pe[r] = v[r].x * v[r].x + v[r].y * v[r].y;
    center(x, m_r, m_i);
    wave_fft<T, Lay>(x, xlds, tab + Lay::TW_O, tab + Lay::TW_2, p, std::true_type{}, [] {});
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = C{pe[r], x[r].x * x[r].x + x[r].y * x[r].y};
  }
  wave_fft<T, Lay>(v, xlds, tab + Lay::TW_E, tab + Lay::TW_2, p, std::false_type{}, [&] {
#pragma unroll
    for (int r = 0; r < R / 2; ++r) cs[r] = entry(tab, Lay::TW_CS + P * r, p);
    issued();
  });
  load(x);

  // 3. 2 N Re C(d) and 2 N Re C(M - d) for d = p + P r < M / 2, from Z(d),
  // Z(M - d) and (c, s) = (cos, sin)(2 pi d / N):
  //   A.x + B.x +- (c (A.y + B.y) - s (A.x - B.x)).
  // Z(M - d) sits in lane P - p, register R - 1 - r (lane 0: register R - r).
  // Lane 0, r = 0 takes d = M / 2 in place of M - d (and of d = 0, unused).
  double ca[R / 2], cb[R / 2];
  {
    const int other = ((lane - p) + ((P - p) & (P - 1))) * 4;
    constexpr int B = 4;  // values fetched from other lanes at once
#pragma unroll
    for (int rb = 0; rb < R / 2; rb += B) {
      C o[B];
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const int r = rb + i, r0 = r == 0 ? R / 2 : R - r;
        o[i].x = from_lane(p == 0 ? v[r0].x : v[R - 1 - r].x, other);
        o[i].y = from_lane(p == 0 ? v[r0].y : v[R - 1 - r].y, other);
      }
      issued();
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const int r = rb + i;
        double ax = v[r].x, ay = v[r].y;
        const double bx = o[i].x;
        double by = o[i].y;
        if (r == 0) {
          ax = p == 0 ? bx : ax;
          ay = p == 0 ? 0.0 : ay;
          by = p == 0 ? 0.0 : by;
        }
        const double s = ax + bx;
        const double w = static_cast<double>(cs[r].x) * (ay + by) - static_cast<double>(cs[r].y) * (ax - bx);
        ca[r] = s + w;
        cb[r] = s - w;
      }
    }
  }

  // 4. prefix sums of |x|^2 and the lags with few pairs.  The samples go to
  // LDS, each lane sums its R consecutive ones, a scan over the lanes
  // offsets them, and the exclusive sums take the samples' place.
  // Direct sums: 32 n-pair lags spread over the P lanes (P = 64: two lanes
  // share one lag's pairs; fewer lanes: 32 / P lags each).
  constexpr int NE = P >= kEdge ? 1 : kEdge / P, SPL = P > kEdge ? P / kEdge : 1;
  double de[NE];
  double ptot;
  double ia[R / 2], ib[R / 2];  // 1 / (L - d)
  {
    double s[R];
    center(x, m_r, m_i);
    auto reciprocals = [&] {
#pragma unroll
      for (int r = 0; r < R / 2; ++r) {
        ia[r] = entry(inv, P * r, p);
        ib[r] = entry(inv, 0, r == 0 && p == 0 ? M / 2 : M - p - P * r);
      }
      issued();
    };
    // adds the squared differences of one component, or of both (eight pairs in
    // flight: a block of t from a multiple of 8 on shares a chunk)
    auto direct = [&](const auto* first, auto* last, auto square) {
      for (int i = p; i < kLast; i += P)
        last[i] = i < kEdge ? first[chunk_pos<R>(max(L - kEdge + i, 0))] : std::decay_t<decltype(*last)>{};
      wave_sync();
#pragma unroll
      for (int e = 0; e < NE; ++e)
        few_pairs<SPL, 8>(de[e], p / SPL + e * P + 1, p % SPL, min((e + 1) * P, kEdge), last, first,
                          [](int t0) { return chunk_pos<R>(t0); }, square);
    };
#pragma unroll
    for (int e = 0; e < NE; ++e) de[e] = 0;
    const int wb = chunk_pos<R>(p), rb = p * Lay::CS;
    if constexpr (!F64) {
      float2* const b = reinterpret_cast<float2*>(clds);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        b[wb + Lay::chunk_row(r)] = x[r];
      }
      wave_sync();
      direct(b, reinterpret_cast<float2*>(tlds), [](float2 u, float2 w) {
        const double dr = static_cast<double>(u.x) - static_cast<double>(w.x);
        const double di = static_cast<double>(u.y) - static_cast<double>(w.y);
        return dr * dr + di * di;
      });
#pragma unroll
      for (int i = 0; i < R; i += 2) {
        const f32x4 f = *reinterpret_cast<const f32x4*>(b + rb + i);
        const double f0 = f[0], f1 = f[1], f2 = f[2], f3 = f[3];
        s[i] = f0 * f0 + f1 * f1;
        s[i + 1] = f2 * f2 + f3 * f3;
      }
      wave_sync();
    } else {
      sfor<0, 2>([&](auto compc) {
        constexpr int comp = decltype(compc)::value;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          clds[wb + Lay::chunk_row(r)] = comp ? x[r].y : x[r].x;
        }
        wave_sync();
        direct(clds, tlds, [](double u, double w) { return (u - w) * (u - w); });
#pragma unroll
        for (int i = 0; i < R; i += 2) {
          const f64x2 f = *reinterpret_cast<const f64x2*>(clds + rb + i);
          s[i] = comp ? s[i] + f[0] * f[0] : f[0] * f[0];
          s[i + 1] = comp ? s[i + 1] + f[1] * f[1] : f[1] * f[1];
        }
        wave_sync();
      });
    }
    if constexpr (R == 32) reciprocals();
    double run = 0;
#pragma unroll
    for (int i = 0; i < R; ++i) run += s[i];
    const double inc = group_scan<P>(run, p);
    ptot = group_last<P>(inc);
    double acc = inc - run;
#pragma unroll
    for (int i = 0; i < R; i += 2) {
      const double e0 = acc, e1 = e0 + s[i];
      acc = e1 + s[i + 1];
      *reinterpret_cast<f64x2*>(clds + rb + i) = f64x2{e0, e1};
    }
    wave_sync();
    if constexpr (R != 32) reciprocals();  // (no registers for them earlier)
    if constexpr (SPL == 2) de[0] += __shfl_xor(de[0], 1, 64);
  }

  // 5. D(d) = (psum(L - d) + psum(L) - psum(d) - 2 C(d)) / (L - d); lags at
  // or beyond L give values that nothing reads.  Compensated FP32: a lag
  // whose (L - d) D is small against sum |x|^2 marks the column for the
  // direct recomputation (launch_fix).
  bool flag = false;
  {
    const double thr = ptot * kWkFlag;
    constexpr double k = -0.5 / M;  // -2 / (2 N)
    // positions of p + P r, L - p - P r, M - p - P r = (P - p) + P (R - 1 - r)
    // and L - (M - p - P r): one base (NB where a chunk holds several register
    // rows) plus whole chunks; where the sample would be below 0 (lags beyond
    // L) position 0 stands in
    constexpr int NB = Lay::NB;
    int pd[NB], pl[NB], qd[NB], ql[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      pd[i] = chunk_pos<R>(p + P * i);
      pl[i] = chunk_pos<R>(L - p - P * i);
      qd[i] = chunk_pos<R>(P - p + P * i);
      ql[i] = chunk_pos<R>(L - M + p + P * i);
    }
    auto row = [&](int r) { return P >= R ? r * (P / R) * Lay::CS : (r / NB) * Lay::CS; };
    auto value = [&](double cc, int d, double tail, double head, double rn, bool first) {
      const double num = head + (ptot - tail) + k * cc;
      if constexpr (!F64) flag |= num < thr && (!first || d >= 1) && d < L - kEdge;
      return num * rn;
    };
    constexpr int B = 4;  // lag pairs whose sums are read at once
#pragma unroll
    for (int rb = 0; rb < R / 2; rb += B) {
      double ta[B], ha[B], tb[B], hb[B];
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const int r = rb + i;
        int tail = qd[(R - 1 - r) % NB] + row(R - 1 - r), head = max(ql[r % NB] + row(r), 0);
        if (r == 0) {
          tail = p == 0 ? chunk_pos<R>(M / 2) : tail;
          head = p == 0 ? chunk_pos<R>(max(L - M / 2, 0)) : head;
        }
        ta[i] = clds[pd[r % NB] + row(r)];
        ha[i] = clds[min(max(pl[r % NB] - row(r), 0), Lay::CG - 1)];
        tb[i] = clds[tail];
        hb[i] = clds[head];
      }
      issued();
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const int r = rb + i, d = p + P * r;
        ca[r] = value(ca[r], d, ta[i], ha[i], ia[r], r == 0);
        cb[r] = value(cb[r], r == 0 && p == 0 ? M / 2 : M - d, tb[i], hb[i], ib[r], false);
      }
    }
  }
  if constexpr (!F64) {
    const uint64_t any = __ballot(flag);
    const uint64_t mine = P == 64 ? ~uint64_t(0) : ((uint64_t(1) << (P & 63)) - 1) << (g * P);
    if (a.flags && active && p == 0) a.flags[q] = (any & mine) != 0;
  }
  OutT* __restrict__ out = static_cast<OutT*>(a.out);
  const size_t ldo = a.ldo;
  if (active && p == 0) {
    const size_t oq = col_out(a, c);
    const double mr2 = fsr * rl, mi2 = fsi * rl;
    const double var = ptot * rl - (mr2 * mr2 + mi2 * mi2);
    const double fr = static_cast<double>(m_r) + mr2 + static_cast<double>(first.x);
    const double fi = static_cast<double>(m_i) + mi2 + static_cast<double>(first.y);
    const double ps = var + fr * fr + fi * fi;
    out[static_cast<size_t>(a.nl) * ldo + oq] = static_cast<OutT>(ps);
    out[static_cast<size_t>(a.nl + 1) * ldo + oq] = static_cast<OutT>(var);
  }

  using Rows = LagRows<OutT, 64 * W, Q, M>;
  static_assert(Q * Rows::SS * sizeof(OutT) <= Lay::bytes, "results fit the exchange buffers");

  // 6. results to LDS by column and lag (over the exchange buffers), then
  // every requested lag's row of Q neighbouring columns to the output
  __syncthreads();
  OutT* const stage = reinterpret_cast<OutT*>(smem);
  {
    OutT* const st = stage + qi * Rows::SS;
#pragma unroll
    for (int r = 0; r < R / 2; ++r) st[p + P * r] = static_cast<OutT>(ca[r]);
#pragma unroll
    for (int r = 0; r < R / 2; ++r) {
      int d = M - p - P * r;
      if (r == 0) d = p == 0 ? M / 2 : d;
      st[d] = static_cast<OutT>(cb[r]);
    }
    wave_sync();
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const int n = p / SPL + e * P + 1;
      if (n < L && p % SPL == 0) st[L - n] = static_cast<OutT>(de[e] / n);
    }
  }
  __syncthreads();
  Rows::write(a, stage, c0, tid);
}

template <typename T, typename OutT, int R, int P, int W = 4>
hipError_t launch_one(const TimeArgs& a, bool subtract_mean, hipStream_t s) {
  using Lay = WaveLay<R, P, W>;
  const int wgs = (a.cols + Lay::Q - 1) / Lay::Q;
  const int wpx = (wgs + 7) / 8;
  auto kernel = k_time_wave<T, OutT, R, P, W>;
  if (Lay::bytes > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(Lay::bytes));
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kernel, dim3(8u * wpx), dim3(64 * W), Lay::bytes, s, a, wpx, wgs, subtract_mean ? 1 : 0);
  return hipGetLastError();
}

template <typename T, typename OutT>
hipError_t launch_logm(const TimeArgs& a, int logm, bool sub, hipStream_t s) {
  if (a.cols <= 0) return hipSuccess;
  switch (logm) {
    case 7: return launch_one<T, OutT, 8, 16>(a, sub, s);
    case 8: return launch_one<T, OutT, 16, 16>(a, sub, s);
    case 9: return launch_one<T, OutT, 16, 32>(a, sub, s);
    case 10: return launch_one<T, OutT, 16, 64, sizeof(T) == 4 ? 8 : 4>(a, sub, s);
    case 11:
      if constexpr (sizeof(T) == 4) return launch_one<T, OutT, 32, 64>(a, sub, s);
      return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

int time_wave_max_log(int precision) { return precision == PREC_FP64 ? 10 : 11; }

std::vector<unsigned char> time_wave_tables(int logm, int precision, uint64_t L) {
  const long long M = 1ll << logm;
  const int R = logm == 7 ? 8 : logm <= 10 ? 16 : 32;
  const bool f64 = precision == PREC_FP64;
  std::vector<unsigned char> out;
  put_transform(out, M, M / R, f64, true);
  for (long long d = 0; d < M / 2; ++d) put_root(out, -d, 2 * M, f64);
  put_reciprocals(out, M, L);
  return out;
}

hipError_t launch_time_wave(const TimeArgs& a, int logm, int precision, int out_dtype, hipStream_t s) {
  const bool f32 = out_dtype == OUT_F32;
  switch (precision) {
    case PREC_FP64:
      return f32 ? launch_logm<double, float>(a, logm, true, s) : launch_logm<double, double>(a, logm, true, s);
    case PREC_FP32:
    case PREC_FP32C: {
      const bool sub = precision == PREC_FP32C;
      return f32 ? launch_logm<float, float>(a, logm, sub, s) : launch_logm<float, double>(a, logm, sub, s);
    }
    default: return hipErrorInvalidValue;
  }
}

}  // namespace fddm
