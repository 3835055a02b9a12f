// Stages (c) + (e), fft mode, for series of up to 2048 frames: every
// transform held in the registers of one wave.
//
// D(q, dt) does not depend on the zero-padded length N >= 2L - 1, so the
// time stage runs at N = 2M, M = max(128, 2^ceil(log2 L)).  With the upper
// half of the input zero, the N-point transform G of the M samples x splits
// into two M-point ones, G(2k) = FFT_M(x)(k) and G(2k + 1) = FFT_M(x W_N^t)(k),
// and Re C(d) = Re IFFT_N(|G|^2) needs one more, Z = FFT_M(z) of
// z(k) = |G(2k)|^2 + i |G(2k + 1)|^2.
//
// An M-point transform is worked on by P lanes of one wave holding R points
// each (M = P R, sample t = p + P r in register r of lane p; 64 / P columns
// per wave): a radix-R DFT in registers, the twiddles W_M^(p k1), one exchange
// through the wave's own LDS, and a second DFT in registers (P points, or R
// points after one radix-2 step between the wave's halves when P = 2R).  The
// result is again in natural order, bin k = p + P r in register r of lane p.
// All LDS addresses are one base per lane plus immediate offsets, so next to
// no integer arithmetic is left, and nothing waits at a workgroup barrier
// until the results of the workgroup's columns are written out.
//
// What bounds it: VALU issue (74 % busy at M = 2048; 5400 instructions per
// column against 9600 of the workgroup form, k_time_p2, which spent 62 % of
// them on addresses, moves and conversions and met at two barriers per pass).
// Kernel time, before and after: 3.06 -> 1.89 ms for 131584 columns of 2000
// samples in compensated FP32, 1.58 -> 1.15 ms for 154080 of 997, 0.142 ->
// 0.088 ms for 15456 of 271 in FP64.
// Every batch of global loads is issued well before its use (issued()): with
// two to four waves per SIMD the latency is not hidden otherwise (the same
// kernel with the loads left to the scheduler: 3.7 ms at M = 2048).
#include <vector>

#include "fddm_kernels.hpp"
#include "fddm_p2.hpp"
#include "fddm_wave.hpp"

namespace fddm {
namespace {
using namespace p2;

constexpr int kWaves = 4;  // waves per workgroup
constexpr int kEdge = 32;  // lags of at most this many pairs: direct sums (compensated paths)

// Shape and LDS layout of M = P R.  Elements are 8 bytes: a float complex
// value, or one component of a double one (exchanged one after the other).
template <int R_, int P_>
struct WaveLay {
  static constexpr int R = R_, P = P_, M = R * P, GROUPS = 64 / P, Q = kWaves * GROUPS;
  // second stage, P points per k1: one pass (P <= R), a radix-2 step between
  // the halves of the wave and one pass (P = 2R = 64), or two passes R R3
  static constexpr bool LANE2 = P == 64 && R == 32;
  static constexpr int R3 = P > R && !LANE2 ? P / R : 1;
  static_assert(LANE2 || (P <= R ? R % P == 0 : R % R3 == 0), "plan");
  // exchange: rows of NC elements, read back 16 bytes at a time; blocks of
  // NC + 2 put eight such reads in distinct banks (three passes: R3 blocks
  // of R a row, then R3 rows of R^2)
  static constexpr int NC = LANE2 || R3 > 1 ? R : P, RS = R3 > 1 ? R3 * (R + 2) + 2 : NC + 2;
  static constexpr int ROWS = R3 > 1 ? R : M / NC, RS3 = R * R + 16;
  static constexpr int GS0 = ROWS * RS > R3 * RS3 || R3 == 1 ? ROWS * RS : R3 * RS3;
  static constexpr int GS = GS0 + (GROUPS > 2 ? P : 0);  // groups start in distinct banks
  // chunks of R consecutive samples, stride R + 2
  static constexpr int CS = R + 2, CG = P * CS;
  static constexpr int NB = P >= R ? 1 : R / P;  // register rows per chunk, where a chunk is longer than a row
  static constexpr int chunk_row(int r) { return P >= R ? r * (P / R) * CS : (r / NB) * CS + (r % NB) * P; }
  // the exchange buffer or the chunks, then the last kEdge samples of each group
  static constexpr int BUF = GROUPS * (GS > CG ? GS : CG), WAVE = BUF + GROUPS * kEdge;
  // results of one column, by lag; the columns' strides spread over the banks
  static constexpr int SS = M + 32 / Q;
  static_assert(Q <= 32 && Q * SS <= kWaves * WAVE, "results fit the exchange buffers");
  static constexpr size_t bytes = sizeof(double) * kWaves * WAVE;
  // tables, complex of the compute type: W_M^(p k1) at [k1][p],
  // W_M^(p (k1 + 1/2)) at [k1][p], then W_P^j (j < R; LANE2) or W_P^(p0 k2) at
  // [k2][p0] (R3 > 1), (cos, sin)(2 pi d / N) for d < M / 2; in double
  // 1 / (L - d) for d < M
  static constexpr int TW_E = 0, TW_O = M, TW_2 = 2 * M, TW_CS = TW_2 + (LANE2 ? R : R3 > 1 ? P : 0);
  static constexpr int TW_END = TW_CS + M / 2;
};

// Position of sample t in the chunk layout.
template <int R>
__device__ __forceinline__ int chunk_pos(int t) {
  constexpr int LR = R == 32 ? 5 : R == 16 ? 4 : 3;
  static_assert(R == 1 << LR, "R");
  return t + ((t >> LR) << 1);
}

// Orders this wave's LDS writes before its later reads (the hardware keeps a
// wave's LDS accesses in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

// a: [a of lanes 0..31 | b of lanes 0..31], b: [a of 32..63 | b of 32..63]
__device__ __forceinline__ void swap32(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap32(double& a, double& b) {
  const uint64_t ua = static_cast<uint64_t>(__double_as_longlong(a)), ub = static_cast<uint64_t>(__double_as_longlong(b));
  const auto lo = __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(ua), static_cast<unsigned>(ub), false, false);
  const auto hi =
      __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(ua >> 32), static_cast<unsigned>(ub >> 32), false, false);
  a = __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi[0]) << 32) | lo[0]));
  b = __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi[1]) << 32) | lo[1]));
}

__device__ __forceinline__ float from_lane(float v, int addr) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute(addr, __float_as_int(v)));
}
__device__ __forceinline__ double from_lane(double v, int addr) {
  const uint64_t u = static_cast<uint64_t>(__double_as_longlong(v));
  const unsigned lo = static_cast<unsigned>(__builtin_amdgcn_ds_bpermute(addr, static_cast<int>(u & 0xffffffffull)));
  const unsigned hi = static_cast<unsigned>(__builtin_amdgcn_ds_bpermute(addr, static_cast<int>(u >> 32)));
  return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi) << 32) | lo));
}

// Inclusive scan over the P lanes of a group, and the group's total in every lane.
template <int P>
__device__ __forceinline__ double group_scan(double v, int p) {
  if constexpr (P == 64) return wave::incl_scan(v);
#pragma unroll
  for (int s = 1; s < P; s *= 2) {
    const double u = __shfl_up(v, s, P);
    v += p >= s ? u : 0.0;
  }
  return v;
}
template <int P>
__device__ __forceinline__ double group_last(double v) {
  if constexpr (P == 64) return wave::lane63(v);
  return __shfl(v, P - 1, P);
}

// Keeps what is written before it (a batch of loads) ahead of what follows:
// left alone, the scheduler sinks each load to its use to save registers and
// waits for them one by one.
__device__ __forceinline__ void issued() { __builtin_amdgcn_sched_barrier(0); }

// Element i + p of a table (i the same for all lanes).
template <typename E>
__device__ __forceinline__ E entry(const E* __restrict__ table, int i, unsigned p) {
  return *reinterpret_cast<const E*>(reinterpret_cast<const char*>(table + i) + p * static_cast<unsigned>(sizeof(E)));
}

// Exchange between two passes: register i written to position wpos(i), then
// runs of NC registers read from consecutive positions from rpos(run) on
// (16 bytes at a time where NC > 1).
template <int R, int NC, typename E, typename FR>
__device__ __forceinline__ void read_rows(const E* b, E (&x)[R], FR&& rpos) {
  if constexpr (NC == 1) {
#pragma unroll
    for (int i = 0; i < R; ++i) x[i] = b[rpos(i)];
  } else {
    struct alignas(16) Two {
      E a, b;
    };
#pragma unroll
    for (int i = 0; i < R; i += 2) {
      const Two t = *reinterpret_cast<const Two*>(b + rpos(i / NC) + i % NC);
      x[i] = t.a;
      x[i + 1] = t.b;
    }
  }
}
template <typename T, int R, int NC, typename FW, typename FR>
__device__ __forceinline__ void exchange(cplx_t<T> (&v)[R], double* lds, FW&& wpos, FR&& rpos) {
  if constexpr (sizeof(T) == 4) {
    float2* const b = reinterpret_cast<float2*>(lds);
#pragma unroll
    for (int i = 0; i < R; ++i) b[wpos(i)] = v[i];
    wave_sync();
    read_rows<R, NC>(b, v, rpos);
    wave_sync();
  } else {
    double x[R];
#pragma unroll
    for (int i = 0; i < R; ++i) lds[wpos(i)] = v[i].x;
    wave_sync();
    read_rows<R, NC>(lds, x, rpos);
    wave_sync();
#pragma unroll
    for (int i = 0; i < R; ++i) lds[wpos(i)] = v[i].y;
    wave_sync();
#pragma unroll
    for (int i = 0; i < R; ++i) v[i].x = x[i];
    read_rows<R, NC>(lds, x, rpos);
#pragma unroll
    for (int i = 0; i < R; ++i) v[i].y = x[i];
    wave_sync();
  }
}

// Forward M-point transform, natural order in and out.  ODD: of x(t) W_N^t,
// the odd bins of the N-point one (in the first DFT W_R^(r / 2), the rest in
// its twiddle table).  mid() runs after the exchange (the place to issue
// loads for what follows the transform).
template <typename T, typename Lay, bool ODD, typename F>
__device__ __forceinline__ void wave_fft(cplx_t<T> (&v)[Lay::R], double* lds, const cplx_t<T>* __restrict__ tw, int p,
                                         F&& mid) {
  using C = cplx_t<T>;
  constexpr int R = Lay::R, P = Lay::P, RS = Lay::RS, R3 = Lay::R3;
  C w[R];
#pragma unroll
  for (int k = ODD ? 0 : 1; k < R; ++k) w[k] = entry(tw, (ODD ? Lay::TW_O : Lay::TW_E) + k * P, p);
  C wl{};
  if constexpr (Lay::LANE2) wl = entry(tw, Lay::TW_2, p & (R - 1));
  issued();
  if constexpr (ODD) sfor<1, R>([&](auto rc) {
      constexpr int r = decltype(rc)::value;
      v[r] = mul_w<T, r, 2 * R>(v[r]);
    });
  dft<T, R>(v);
#pragma unroll
  for (int k = ODD ? 0 : 1; k < R; ++k) v[k] = cmul(v[k], w[k]);
  if constexpr (Lay::LANE2) {
    // bins k1 + R k2, k2 = 2 kappa + g: sums (g = 0) and differences (g = 1)
    // of samples j and j + R of the P-point transforms; lanes below 32 take
    // the even k1, the others the odd ones
    const int j = p & (R - 1), hi = p >> 5;
    static_assert(R == 32, "the halves of the wave");
#pragma unroll
    for (int i = 0; i < R; i += 2) {
      swap32(v[i].x, v[i + 1].x);
      swap32(v[i].y, v[i + 1].y);
      const C a = v[i], b = v[i + 1];
      v[i] = cadd(a, b);
      v[i + 1] = cmul(csub(a, b), wl);
    }
    const int wb = hi * RS + j, rb = p * RS;
    // register i + g holds (k1 = i + hi, g): row k1 + R g
    exchange<T, R, R>(v, lds, [&](int i) { return wb + ((i & ~1) + R * (i & 1)) * RS; }, [&](int) { return rb; });
    mid();
    dft<T, R>(v);
  } else if constexpr (R3 > 1) {
    // sample p = p0 + R3 p1 of the P-point transforms: radix R over p1 (lane
    // p0 R + k1), twiddles, then radix R3 over p0 of the bins j = k1 + R k2
    // = p + P i, which leaves bin j + R^2 k3 in register i + (R / R3) k3
    const int k1 = p & (R - 1), p0 = p / R;
    const int wb = (p & (R3 - 1)) * (R + 2) + p / R3, rb = k1 * RS + p0 * (R + 2);
    exchange<T, R, R>(v, lds, [&](int i) { return wb + i * RS; }, [&](int) { return rb; });
#pragma unroll
    for (int k = 1; k < R; ++k) w[k] = entry(tw, Lay::TW_2 + k * R3, p0);
    issued();
    dft<T, R>(v);
#pragma unroll
    for (int k = 1; k < R; ++k) v[k] = cmul(v[k], w[k]);
    const int wb3 = p0 * Lay::RS3 + k1;
    constexpr int NI = R / R3;
    exchange<T, R, 1>(v, lds, [&](int i) { return wb3 + i * R; },
                      [&](int i) { return p + (i % NI) * P + (i / NI) * Lay::RS3; });
    mid();
    // register i + NI p0 holds sample p0 of butterfly i
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      C u[R3];
#pragma unroll
      for (int k = 0; k < R3; ++k) u[k] = v[i + NI * k];
      dft<T, R3>(u);
#pragma unroll
      for (int k = 0; k < R3; ++k) v[i + NI * k] = u[k];
    }
  } else {
    constexpr int CN = R / P;
    const int rb = p * RS;
    exchange<T, R, P>(v, lds, [&](int i) { return p + i * RS; }, [&](int i) { return rb + i * P * RS; });
    mid();
    C o[R];
#pragma unroll
    for (int i = 0; i < CN; ++i) {
      C u[P];
#pragma unroll
      for (int k = 0; k < P; ++k) u[k] = v[i * P + k];
      dft<T, P>(u);
#pragma unroll
      for (int k = 0; k < P; ++k) o[i + CN * k] = u[k];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = o[r];
  }
}

// Waves per SIMD: what the LDS of M = 2^10 and 2^11 allows in FP32, 3 where
// the registers of the others fit, 2 in double.
template <typename T, int R, int P>
constexpr int wave_occ() {
  return sizeof(T) == 8 ? (R == 8 ? 3 : 2) : R == 32 ? 2 : P == 64 || R == 8 ? 4 : 3;
}

template <typename T, typename OutT, int R, int P>
__global__ void __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(wave_occ<T, R, P>(), wave_occ<T, R, P>())))
    k_time_wave(TimeArgs a, int wg_per_xcd, int wgs, int subtract_mean) {
  using C = cplx_t<T>;
  using Lay = WaveLay<R, P>;
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
  const C* __restrict__ tw = static_cast<const C*>(a.twt);
  const double* __restrict__ inv = reinterpret_cast<const double*>(tw + Lay::TW_END);
  double* const wlds = reinterpret_cast<double*>(smem) + wave * Lay::WAVE;
  double* const xlds = wlds + g * Lay::GS;  // exchange
  double* const clds = wlds + g * Lay::CG;  // chunks
  double* const tlds = wlds + Lay::BUF + g * kEdge;  // last samples

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
    wave_fft<T, Lay, false>(v, xlds, tw, p, [&] { load(x); });
#pragma unroll
    for (int r = 0; r < R; ++r) pe[r] = v[r].x * v[r].x + v[r].y * v[r].y;
    center(x, m_r, m_i);
    wave_fft<T, Lay, true>(x, xlds, tw, p, [] {});
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = C{pe[r], x[r].x * x[r].x + x[r].y * x[r].y};
  }
  wave_fft<T, Lay, false>(v, xlds, tw, p, [&] {
#pragma unroll
    for (int r = 0; r < R / 2; ++r) cs[r] = entry(tw, Lay::TW_CS + P * r, p);
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
#pragma unroll
    for (int r = 0; r < R / 2; ++r) {
      const int r0 = r == 0 ? R / 2 : R - r;
      C b;
      b.x = from_lane(p == 0 ? v[r0].x : v[R - 1 - r].x, other);
      b.y = from_lane(p == 0 ? v[r0].y : v[R - 1 - r].y, other);
      double ax = v[r].x, ay = v[r].y;
      const double bx = b.x;
      double by = b.y;
      if (r == 0) {
        ax = p == 0 ? bx : ax;
        ay = p == 0 ? 0.0 : ay;
        by = p == 0 ? 0.0 : by;
      }
      const double s = ax + bx, w = static_cast<double>(cs[r].x) * (ay + by) - static_cast<double>(cs[r].y) * (ax - bx);
      ca[r] = s + w;
      cb[r] = s - w;
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
    // adds the squared differences of one component, or of both: sample
    // L - n + t sits in place kEdge - n + t of the copied last ones, t < n in
    // the first chunks
    auto reciprocals = [&] {
#pragma unroll
      for (int r = 0; r < R / 2; ++r) {
        ia[r] = entry(inv, P * r, p);
        ib[r] = entry(inv, 0, r == 0 && p == 0 ? M / 2 : M - p - P * r);
      }
      issued();
    };
    auto direct = [&](const auto* first, auto* last, auto square) {
      for (int i = p; i < kEdge; i += P) last[i] = first[chunk_pos<R>(max(L - kEdge + i, 0))];
      wave_sync();
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int n = p / SPL + e * P + 1, s0 = p % SPL;
        const auto* const u = last + kEdge - n + s0;
        constexpr int B = 8;  // pairs in flight
#pragma nounroll
        for (int t0 = 0; t0 < min((e + 1) * P, kEdge); t0 += B * SPL) {
          std::decay_t<decltype(*first)> x1[B], x0[B];
#pragma unroll
          for (int b = 0; b < B; ++b) {  // (t0 a multiple of 8: B pairs share a chunk)
            x1[b] = u[t0 + b * SPL];
            x0[b] = first[s0 + b * SPL + chunk_pos<R>(t0)];
          }
          issued();
#pragma unroll
          for (int b = 0; b < B; ++b) de[e] += t0 + b * SPL + s0 < n ? square(x1[b], x0[b]) : 0.0;
        }
      }
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
  // direct recomputation (launch_wk_fix).
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
    auto value = [&](double cc, int d, int tail, int head, double rn, bool first) {
      const double num = clds[head] + (ptot - clds[tail]) + k * cc;
      if constexpr (!F64) flag |= num < thr && (!first || d >= 1) && d < L - kEdge;
      return num * rn;
    };
#pragma unroll
    for (int r = 0; r < R / 2; ++r)
      ca[r] = value(ca[r], p + P * r, pd[r % NB] + row(r), min(max(pl[r % NB] - row(r), 0), Lay::CG - 1), ia[r], r == 0);
#pragma unroll
    for (int r = 0; r < R / 2; ++r) {
      int d = M - p - P * r, tail = qd[(R - 1 - r) % NB] + row(R - 1 - r), head = max(ql[r % NB] + row(r), 0);
      if (r == 0) {
        d = p == 0 ? M / 2 : d;
        tail = p == 0 ? chunk_pos<R>(M / 2) : tail;
        head = p == 0 ? chunk_pos<R>(max(L - M / 2, 0)) : head;
      }
      cb[r] = value(cb[r], d, tail, head, ib[r], false);
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
    double fr = static_cast<double>(m_r) + mr2, fi = static_cast<double>(m_i) + mi2;
    if (a.S0) {
      const C z = static_cast<const C*>(a.S0)[static_cast<size_t>(q) * a.s0_stride];
      fr += static_cast<double>(z.x);
      fi += static_cast<double>(z.y);
    }
    const double ps = var + fr * fr + fi * fi;
    out[static_cast<size_t>(a.nl) * ldo + oq] = static_cast<OutT>(ps);
    out[static_cast<size_t>(a.nl + 1) * ldo + oq] = static_cast<OutT>(var);
  }

  // 6. results to LDS by column and lag (over the exchange buffers), then
  // every requested lag's row of Q neighbouring columns to the output
  __syncthreads();
  OutT* const stage = reinterpret_cast<OutT*>(smem);
  {
    OutT* const st = stage + qi * Lay::SS;
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
  {
    const int qq = tid % Q, i0 = tid / Q;
    constexpr int STEP = 64 * kWaves / Q, B = 8;  // lags per round of the workgroup, rounds in flight
    if (c0 + qq < a.cols) {
      const OutT* const st = stage + qq * Lay::SS;
      OutT* dst = out + static_cast<size_t>(i0) * ldo + col_out(a, c0 + qq);
      const size_t step = STEP * ldo;
      for (int ib = 0; ib < a.nl; ib += B * STEP) {
        const int left = a.nl - ib - i0;  // lags of this lane from here on: b STEP < left
        uint32_t d[B];
#pragma unroll
        for (int b = 0; b < B; ++b) d[b] = a.lags[min(ib + i0 + b * STEP, a.nl - 1)];
        issued();
        OutT r[B];
#pragma unroll
        for (int b = 0; b < B; ++b) r[b] = st[d[b]];
        if (ib + B * STEP <= a.nl) {
#pragma unroll
          for (int b = 0; b < B; ++b) dst[b * step] = r[b];
        } else {
#pragma unroll
          for (int b = 0; b < B; ++b)
            if (b * STEP < left) dst[b * step] = r[b];
        }
        dst += B * step;
      }
    }
  }
}

template <typename T, typename OutT, int R, int P>
hipError_t launch_one(const TimeArgs& a, bool subtract_mean, hipStream_t s) {
  using Lay = WaveLay<R, P>;
  const int wgs = (a.cols + Lay::Q - 1) / Lay::Q;
  const int wpx = (wgs + 7) / 8;
  auto kernel = k_time_wave<T, OutT, R, P>;
  if (Lay::bytes > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(Lay::bytes));
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kernel, dim3(8u * wpx), dim3(64 * kWaves), Lay::bytes, s, a, wpx, wgs, subtract_mean ? 1 : 0);
  return hipGetLastError();
}

template <typename T, typename OutT>
hipError_t launch_logm(const TimeArgs& a, int logm, bool sub, hipStream_t s) {
  if (a.cols <= 0) return hipSuccess;
  switch (logm) {
    case 7: return launch_one<T, OutT, 8, 16>(a, sub, s);
    case 8: return launch_one<T, OutT, 16, 16>(a, sub, s);
    case 9: return launch_one<T, OutT, 16, 32>(a, sub, s);
    case 10: return launch_one<T, OutT, 16, 64>(a, sub, s);
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
  const long long P = M / R;
  const long double two_pi = 6.283185307179586476925286766559005768L;
  const bool f64 = precision == PREC_FP64;
  std::vector<unsigned char> out;
  auto put = [&](long double v, bool dbl) {
    const double d = static_cast<double>(v);
    const float f = static_cast<float>(v);
    const unsigned char* b = dbl ? reinterpret_cast<const unsigned char*>(&d) : reinterpret_cast<const unsigned char*>(&f);
    out.insert(out.end(), b, b + (dbl ? 8 : 4));
  };
  auto w = [&](long double num, long double den) {
    const long double ang = -two_pi * num / den;
    put(cosl(ang), f64);
    put(sinl(ang), f64);
  };
  for (long long k = 0; k < R; ++k)
    for (long long p = 0; p < P; ++p) w(static_cast<long double>(p * k), static_cast<long double>(M));
  for (long long k = 0; k < R; ++k)
    for (long long p = 0; p < P; ++p) w(static_cast<long double>(p * (2 * k + 1)), static_cast<long double>(2 * M));
  if (R == 32) {
    for (long long j = 0; j < R; ++j) w(static_cast<long double>(j), static_cast<long double>(P));
  } else if (P > R) {
    for (long long k = 0; k < R; ++k)
      for (long long p0 = 0; p0 < P / R; ++p0) w(static_cast<long double>(p0 * k), static_cast<long double>(P));
  }
  for (long long d = 0; d < M / 2; ++d) {
    const long double ang = two_pi * static_cast<long double>(d) / static_cast<long double>(2 * M);
    put(cosl(ang), f64);
    put(sinl(ang), f64);
  }
  for (uint64_t d = 0; d < static_cast<uint64_t>(M); ++d) put(d < L ? 1.0L / static_cast<long double>(L - d) : 0.0L, true);
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
