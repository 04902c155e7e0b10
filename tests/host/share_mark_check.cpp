// The mark of handed-over vectors (onsas.jl_amd/csrc/share_mark.hpp): the words of one
// store are taken as a whole, mixtures of the words of two are not.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "share_mark.hpp"

using namespace onsas;

struct Words {
  uint32_t w[4];
};
Words make(const uint32_t (&p)[3], uint32_t epoch) {
  return {{p[0], p[1], p[2], share_mark(p[0], p[1], p[2], epoch)}};
}
bool taken(const Words& x, uint32_t epoch) {
  return share_mark(x.w[0], x.w[1], x.w[2], epoch) == x.w[3];
}
#define CHECK(c)                                             \
  do {                                                       \
    if (!(c)) {                                              \
      std::fprintf(stderr, "line %d: %s\n", __LINE__, #c);   \
      std::exit(1);                                          \
    }                                                        \
  } while (0)

int main() {
  std::mt19937_64 rng(7);
  std::uniform_real_distribution<double> u(-1, 1);
  // payloads as the solvers hand them over: three floats, or the words of doubles, from
  // one iteration to the next, some of them unchanged (fixed dofs are zero)
  auto payload = [&](uint32_t(&p)[3], bool f64, int fixed, double scale) {
    if (f64) {
      double v[2] = {scale * u(rng), scale * u(rng)};
      std::memcpy(p, v, 12);
    } else {
      float v[3] = {(float)(scale * u(rng)), (float)(scale * u(rng)), (float)(scale * u(rng))};
      std::memcpy(p, v, 12);
    }
    for (int c = 0; c < 3; ++c)
      if ((fixed >> c) & 1) p[c] = 0;
  };
  long mixtures = 0;
  for (int n = 0; n < 200000; ++n) {
    const bool f64 = n & 1;
    const int fixed = (n >> 1) & 7;
    const uint32_t e0 = 1 + (uint32_t)(rng() % 0xf0000000u), e1 = e0 + 1 + (uint32_t)(rng() % 3);
    uint32_t a[3], b[3];
    payload(a, f64, fixed, 1.0);
    payload(b, f64, fixed, n % 3 ? 1.0 : 1.0 + 1e-6);
    const Words x = make(a, e0), y = make(b, e1), zero = {{0, 0, 0, 0}};
    CHECK(taken(x, e0) && taken(y, e1));                    // a whole store
    CHECK(!taken(x, e1) && !taken(y, e0));                  // ... of another epoch
    CHECK(!taken(zero, e0) && !taken(zero, e1));            // memory never written
    for (int m = 1; m < 15; ++m) {  // word q from the new store where bit q of m is set
      Words mix;
      for (int q = 0; q < 4; ++q) mix.w[q] = ((m >> q) & 1) ? y.w[q] : x.w[q];
      if (std::memcmp(&mix, &x, 16) == 0 || std::memcmp(&mix, &y, 16) == 0) continue;
      ++mixtures;
      const bool whole = std::memcmp(mix.w, y.w, 12) == 0;  // payload complete: harmless
      CHECK(whole || !taken(mix, e1));
    }
  }
  std::printf("ok %d\n", mixtures > 1000000);
}
