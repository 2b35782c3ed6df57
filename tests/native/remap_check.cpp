// Host check of the region-remap pick (c-saw_amd/csrc/remap.hpp): the first
// CDF entry reaching the threshold key of r must be the first i with
// fl32(fl64(C_i) / fl64(T)) > r, for uint32 and FP32 CDFs with repeated values
// and totals over the whole range, at random r, at every quotient and its
// float neighbours, at 0 and just below 1.  Exit status 0 = all equal.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "../../c-saw_amd/csrc/remap.hpp"

using namespace csaw;

static long bad = 0, checks = 0, unsettled = 0;

template <typename T>
static void one(const std::vector<T>& C, float r) {
  if (!(r >= 0.0f && r < 1.0f)) return;
  const T tot = C.back();
  size_t want = 0;
  while (want < C.size() && !((float)((double)C[want] / (double)tot) > r)) ++want;
  T key;
  ++checks;
  if (!remap_key(r, tot, &key)) {
    ++unsettled;
    return;
  }
  const T below = sizeof(T) == 4 && std::is_integral<T>::value ? (T)(key - 1) : key;
  const size_t got = std::upper_bound(C.begin(), C.end(), below) - C.begin();
  if (got != want) {
    if (bad < 5) std::printf("r=%.9g d=%zu T=%.9g want %zu got %zu\n", r, C.size(), (double)tot, want, got);
    ++bad;
  }
}

template <typename T>
static void all(const std::vector<T>& C, std::mt19937_64& g) {
  if (!(C.back() > T(0))) return;
  for (int k = 0; k < 64; ++k) one(C, (float)(g() >> 40) * 5.9604644775390625e-08f);
  for (int k = 0; k < 16; ++k) one(C, std::ldexp((float)(g() >> 40), -24 - (int)(g() % 60)));
  for (size_t i = 0; i < C.size(); i += 1 + C.size() / 97) {
    const float q = (float)((double)C[i] / (double)C.back());
    one(C, q);
    one(C, std::nextafterf(q, 0.0f));
    one(C, std::nextafterf(q, 2.0f));
  }
  one(C, 0.0f);
  one(C, std::nextafterf(1.0f, 0.0f));
}

int main() {
  std::mt19937_64 g(7);
  for (int t = 0; t < 3000; ++t) {
    const int d = 1 + (int)(g() % (t % 10 ? 90 : 3000));
    const uint32_t cap = (uint32_t)std::min<uint64_t>(0xffffffffull / d, 1ull << (g() % 33));
    std::vector<uint32_t> U;
    std::vector<float> F;
    uint32_t u = 0;
    float f = 0.0f;
    const float scale = std::ldexp(1.0f, (int)(g() % 120) - 60);
    for (int i = 0; i < d; ++i) {
      const bool zero = g() % 3 == 0;
      u += zero ? 0u : (uint32_t)(g() % ((uint64_t)cap + 1));
      f += zero ? 0.0f : (float)((g() >> 40) + 1) * 5.9604644775390625e-08f * scale;
      U.push_back(u);
      F.push_back(f);
    }
    all(U, g);
    all(F, g);
  }
  std::printf("checks=%ld mismatches=%ld unsettled=%ld\n", checks, bad, unsettled);
  return bad != 0 || unsettled * 1000 > checks;
}
