// bm::exact_sum (bitmamba.c_amd/csrc/bm_exact.h) against sums in several
// orders: where it says exact, every order gives the same double.  Prints, per
// kind of terms, how many sets there were, how many it called exact, and how
// many of those differed somewhere; then its answers at the rule's limit.
#include <stdint.h>
#include <stdio.h>

#include <algorithm>
#include <cmath>
#include <random>
#include <vector>

#include "bm_exact.h"

static double in_order(const std::vector<float>& v) {
  double s = 0.0;
  for (float x : v) s += (double)x;
  return s;
}

static double pairwise(const std::vector<float>& v, size_t a, size_t b) {
  if (b - a == 1) return (double)v[a];
  const size_t m = a + (b - a) / 2;
  return pairwise(v, a, m) + pairwise(v, m, b);
}

int main() {
  std::mt19937_64 g(7);
  for (int kind = 0; kind < 6; ++kind) {
    int sets = 0, exact = 0, bad = 0;
    for (int it = 0; it < 4000; ++it) {
      const int n = 1 + (int)(g() % (kind == 5 ? 3000 : 300));
      std::uniform_real_distribution<double> u(0.0, 1.0);
      std::normal_distribution<double> z;
      std::vector<float> v(n);
      for (float& x : v) switch (kind) {
          case 0: x = (float)(0.05 + 0.95 * u(g)); break;       // a min_p cut
          case 1: x = (float)std::exp(5.0 * z(g) - 15.0); break;  // a softmax's spread
          case 2: x = std::ldexp(1.0f, -(int)(g() % 60)); break;
          case 3: x = g() % 4 ? 0.0f : std::ldexp((float)u(g), -130); break;  // subnormals
          case 4: x = std::ldexp((float)u(g), -(int)(g() % 30)); break;
          default: x = (float)std::exp(-8.0 * u(g)); break;
        }
      float least = INFINITY;
      for (float x : v)
        if (x > 0.0f) least = std::min(least, x);
      const double s = in_order(v);
      ++sets;
      if (!bm::exact_sum(s, least)) continue;
      ++exact;
      std::vector<float> w = v;
      std::sort(w.begin(), w.end());
      bool same = in_order(w) == s && pairwise(v, 0, v.size()) == s;
      std::reverse(w.begin(), w.end());
      same = same && in_order(w) == s;
      for (int k = 0; k < 3; ++k) {
        std::shuffle(w.begin(), w.end(), g);
        same = same && in_order(w) == s && pairwise(w, 0, w.size()) == s;
      }
      bad += !same;
    }
    printf("%d %d %d\n", sets, exact, bad);
  }
  // 2^53 ulps of the smallest term and the next double above; the smallest
  // subnormal; no term at all; a NaN
  printf("%d %d %d %d %d\n", bm::exact_sum(0x1p30, 1.0f), bm::exact_sum(0x1.0000000000001p30, 1.0f),
         bm::exact_sum(0x1p-96, 0x1p-149f), bm::exact_sum(0.0, INFINITY),
         bm::exact_sum(NAN, 1.0f));
  return 0;
}
