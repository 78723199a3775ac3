// Host-side check of the bins of equal width of the merged selection (lvar_amd/csrc/score_bins.h), with the arithmetic the
// device code uses and the thread layout of its kernel:
//   * the bin never falls as the key rises, infinities, NaN, zeros of both signs and denormals among them,
//   * the bin that holds the k-th key from the top holds few enough keys to be resolved by direct comparison, for rows of
//     normal scores with columns that do not compete, with one score or a hundredth of all far from the others, and others,
//   * a row without a bulk, or with scores spread over many orders of magnitude, is refused.
// Prints "ok <cases>" or the first violation.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>
#include <string>
#include <vector>
#include "../../lvar_amd/csrc/score_bins.h"

using namespace lvar;

static constexpr int THREADS = 1024, CANDIDATES = 256;   // of the kernel

static uint32_t key_of(float x) {
  x += 0.f;
  uint32_t u;
  memcpy(&u, &x, 4);
  const uint32_t k = u ^ ((u >> 31) ? 0xffffffffu : 0x80000000u);
  return k > 1u ? k : 1u;
}

// smallest of the largest keys of a group's threads, over the groups the largest, and the other way round, of threads [t0, t1)
static void bulk(const std::vector<uint32_t>& keys, int t0, int t1, uint32_t& lo, uint32_t& hi) {
  const int n = (int)keys.size(), kpt = (n + THREADS - 1) / THREADS, G = score_group(kpt);
  lo = 0xffffffffu;
  hi = 0u;
  for (int g = t0; g < t1; g += G) {
    uint32_t gmax = 0xffffffffu, gmin = 0u;
    bool any = false;
    for (int t = g; t < g + G; t++) {
      uint32_t kmax = 0u, kmin = 0xffffffffu;
      for (int c = 0; c < kpt; c++) {
        const int j = ((t / 64) * kpt + c) * 64 + t % 64;
        if (j >= n) continue;
        kmax = std::max(kmax, keys[j]);
        if (keys[j] > KEY_NEG_INF) kmin = std::min(kmin, keys[j]);
      }
      if (kmin > kmax) continue;
      any = true;
      gmax = std::min(gmax, kmax);
      gmin = std::max(gmin, kmin);
    }
    if (!any) continue;
    hi = std::max(hi, gmax);
    lo = std::min(lo, gmin);
  }
}

static bool row_bins(const std::vector<uint32_t>& keys, ScoreBins& b) {
  uint32_t lo, hi;
  float narrow = std::numeric_limits<float>::infinity();
  const int n = (int)keys.size(), kpt = (n + THREADS - 1) / THREADS;
  for (int t = 0; t < THREADS; t += 64) {
    bulk(keys, t, t + 64, lo, hi);
    const float w = score_width(lo, hi);
    if (w > 0.f && (t / 64 + 1) * kpt * 64 <= n) narrow = std::min(narrow, w);
  }
  bulk(keys, 0, THREADS, lo, hi);
  return score_bins(lo, hi, narrow, b);
}

static std::vector<float> scores(const std::string& kind, int n, unsigned seed) {
  std::mt19937 rng(seed);
  std::normal_distribution<float> normal;
  std::uniform_real_distribution<float> uniform(0.f, 1.f);
  const float inf = std::numeric_limits<float>::infinity();
  std::vector<float> x(n);
  for (int j = 0; j < n; j++) {
    float v = normal(rng);
    const float u = uniform(rng);
    if (kind == "uniform") v = u;
    if (kind == "cauchy") v = std::tan((u - 0.5f) * 3.1415f);
    if (kind == "trend") v += 20.f * j / n;
    if (kind == "magnitudes") v = std::copysign(std::exp(12.f * std::fabs(v)), v);
    if (kind == "mostly equal") v = u < 0.01f ? v : 0.25f;
    if (kind == "offset") v += 1000.f;
    if (kind == "small") v *= 1e-20f;
    if (kind == "far hundredth" && u < 0.01f) v *= 100.f;
    x[j] = v;
  }
  if (kind == "pooled") {   // the largest of five neighbours, as a max pool leaves them
    const std::vector<float> y = x;
    for (int j = 0; j < n; j++)
      for (int i = std::max(0, j - 2); i <= std::min(n - 1, j + 2); i++) x[j] = std::max(x[j], y[i]);
  }
  if (kind == "one of 100") x[n / 2] = 100.f * *std::max_element(x.begin(), x.end());
  if (kind == "far") x[n / 2] = 1e30f, x[n / 3] = -1e30f;
  if (kind == "infinite") x[n / 2] = inf, x[0] = inf;
  if (kind == "nan") x[n / 2] = std::numeric_limits<float>::quiet_NaN();
  if (kind != "plain")
    for (int j = 0; j < n; j++)
      if (uniform(rng) < 0.024f) x[j] = -inf;   // the window's own columns
  return x;
}

int main() {
  long cases = 0;
  // order
  std::vector<uint32_t> edge = {0u, 1u, 0x007ffffeu, KEY_NEG_INF, 0x00800000u, 0x7fffffffu, 0x80000000u, 0x80000001u, KEY_POS_INF - 1, KEY_POS_INF, KEY_POS_INF + 1, 0xffffffffu};
  std::mt19937 rng(1);
  for (int i = 0; i < 20000; i++) edge.push_back(rng());
  for (float v : {-3.4e38f, -1e20f, -2.f, -1e-40f, 0.f, 1e-40f, 0.3f, 2.f, 1e20f, 3.4e38f}) edge.push_back(key_of(v));
  std::sort(edge.begin(), edge.end());
  const float ranges[][2] = {{-1.f, 1.f}, {0.f, 1e-3f}, {-1e30f, 2e30f}, {5.f, 5.001f}, {-1e-30f, 1e-30f}};
  for (auto& r : ranges) {
    ScoreBins b;
    if (!score_bins(key_of(r[0]), key_of(r[1]), 1e38f, b)) { printf("no bins for %g .. %g\n", r[0], r[1]); return 1; }
    int last = 0;
    for (uint32_t k : edge) {
      const int at = score_bin(b, k);
      if (at < last || at >= SCORE_BINS) { printf("bin %d after %d at key %08x\n", at, last, k); return 1; }
      last = at;
      cases++;
    }
  }
  ScoreBins b;
  if (score_bins(key_of(1.f), key_of(1.f), 1e38f, b) || score_bins(0xffffffffu, 0u, 1e38f, b) || score_bins(key_of(0.f), KEY_POS_INF, 1e38f, b) ||
      score_bins(key_of(-3e38f), key_of(3e38f), 1e38f, b) || score_bins(key_of(1e-42f), key_of(2e-42f), 1e38f, b)) { printf("bins without a bulk\n"); return 1; }
  // candidates of the threshold
  // every remainder of the last wave: a row whose bulk is that of normal scores has bins
  for (const char* kind : {"plain", "holes", "pooled", "trend"})
    for (int n = kind[0] == 't' ? 1025 : 200; n <= 16384; n += n < 2000 ? 1 : 7) {
      const std::vector<float> x = scores(kind, n, n);
      std::vector<uint32_t> keys(n);
      for (int j = 0; j < n; j++) keys[j] = key_of(x[j]);
      cases++;
      if (!row_bins(keys, b)) { printf("no bins for a row of %d %s scores\n", n, kind); return 1; }
    }
  for (const char* kind : {"plain", "holes", "pooled", "uniform", "cauchy", "trend", "offset", "small", "far hundredth", "one of 100", "far", "infinite", "nan"})
    for (int n : {700, 1497, 4121, 10521, 16384})
      for (unsigned seed = 0; seed < 3; seed++) {
        const std::vector<float> x = scores(kind, n, seed + n);
        std::vector<uint32_t> keys(n);
        for (int j = 0; j < n; j++) keys[j] = key_of(x[j]);
        // (few keys per thread: a group may consist of far scores, and the row goes to the digits)
        const bool far = kind[0] == 'f' || kind[0] == 'c' || std::string(kind) == "one of 100";
        if (n < 4121 && far && !row_bins(keys, b)) continue;
        if (!row_bins(keys, b)) { printf("no bins for a row of %d %s scores\n", n, kind); return 1; }
        std::vector<int> count(SCORE_BINS);
        for (uint32_t k : keys) count[score_bin(b, k)]++;
        std::sort(keys.rbegin(), keys.rend());
        for (int k : {n / 50, n / 8, n / 5, n / 2}) {
          if (kind[0] == 'c' && k == n / 50) continue;   // beyond the bins: Cauchy scores have no such bulk
          cases++;
          const int held = count[score_bin(b, keys[k - 1])];
          if (held > CANDIDATES) { printf("%d candidates: row of %d %s scores, %d kept\n", held, n, kind, k); return 1; }
        }
      }
  for (const char* kind : {"magnitudes", "mostly equal"})
    for (int n : {4121, 10521, 16384}) {
      const std::vector<float> x = scores(kind, n, n);
      std::vector<uint32_t> keys(n);
      for (int j = 0; j < n; j++) keys[j] = key_of(x[j]);
      cases++;
      if (row_bins(keys, b)) { printf("bins for a row of %d %s scores\n", n, kind); return 1; }
    }
  printf("ok %ld\n", cases);
  return 0;
}
