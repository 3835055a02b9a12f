// The few-pair sums of the time kernels on the host, with arrays that check
// every index: the places the lanes of a wave read, and the sums.
#include <cstdio>
#include <cstdlib>
#include <random>

#include "fddm_time_wave.hpp"

using namespace fddm::tw;

static int bad = 0;

struct Checked {
  const double* p;
  int n;
  double operator[](int i) const {
    if (i < 0 || i >= n) {
      ++bad;
      return 0;
    }
    return p[i];
  }
};

// STEP lanes share a lag, lanes 0 .. P - 1 take NE lags each; early samples
// at pos(t0) + (t - t0) of `size` places.
template <int STEP, int B, typename Pos>
static void check(const char* name, int P, int NE, int size, Pos pos) {
  std::mt19937 rng(1);
  std::vector<double> x(2 * kEdge), early(size, -1e30), late(kLast, 0.0);
  for (auto& v : x) v = static_cast<double>(rng() % 1000);
  for (int t = 0; t < kEdge; ++t) early[pos(t)] = x[t], late[t] = x[kEdge + t];
  const auto square = [](double u, double w) { return (u - w) * (u - w); };
  int wrong = 0;
  bad = 0;
  for (int e = 0; e < NE; ++e)
    for (int lag = 0; lag < P / STEP; ++lag) {
      const int n = lag + e * P + 1;
      double sum = 0, ref = 0;
      for (int s0 = 0; s0 < STEP; ++s0)
        few_pairs<STEP, B>(sum, n, s0, NE > 1 && (e + 1) * P < kEdge ? (e + 1) * P : kEdge, Checked{late.data(), kLast},
                           Checked{early.data(), size}, pos, square);
      for (int t = 0; t < n; ++t) ref += square(x[2 * kEdge - n + t], x[t]);
      if (sum != ref) ++wrong;
    }
  std::printf("%s out_of_range=%d wrong=%d\n", name, bad, wrong);
}

template <int R, int P, int W>
static void wave(const char* name) {
  using Lay = WaveLay<R, P, W>;
  static_assert(Lay::WAVE >= Lay::BUF + Lay::GROUPS * kLast, "a slice of last samples for every group");
  static_assert(Lay::bytes >= sizeof(double) * W * Lay::WAVE, "every wave's slices are allocated");
  constexpr int SPL = P > kEdge ? P / kEdge : 1;
  check<SPL, 8>(name, P, P >= kEdge ? 1 : kEdge / P, Lay::CG, [](int t) { return chunk_pos<R>(t); });
}

int main() {
  wave<8, 16, 4>("M=128");
  wave<16, 16, 4>("M=256");
  wave<16, 32, 4>("M=512");
  wave<16, 64, 8>("M=1024");
  wave<32, 64, 4>("M=2048");
  check<4, 4>("pair", 128, 1, kEdge, [](int t) { return t; });
  return 0;
}
