// chq::div_by (numerics.hpp) against the IEEE division p / (gamma - 1), for the usual and for random
// adiabatic indices, over every positive p it accepts, and its refusals.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "common.hpp"
#include "numerics.hpp"

static uint64_t s = 0x9e3779b97f4a7c15ull;
static uint64_t next() { s ^= s << 13; s ^= s >> 7; s ^= s << 17; return s; }

int main(int argc, char **argv) {
  const long n = argc > 1 ? std::atol(argv[1]) : 20000000L;
  const double usual[] = {5.0 / 3.0, 2.0, 1.4, 7.0 / 5.0, 4.0 / 3.0, 1.01, 1.0001, 3.0};
  long bad = 0, taken = 0;
  double g = usual[0] - 1.0, y = 1.0 / g;
  for (long t = 0; t < n; ++t) {
    if (t % 1000 == 0) {
      const long q = t / 1000;
      g = (q % 2 ? 1.0 + double(next() >> 11) / 9007199254740992.0 * 2.0 : usual[(q / 2) % 8]) - 1.0;
      y = 1.0 / g;
    }
    const uint64_t b = next() & 0x7fffffffffffffffull;
    double p;
    if (t % 2) p = std::ldexp(1.0 + double(b >> 11) / 4503599627370496.0, int(b % 64) - 48);
    else std::memcpy(&p, &b, 8);
    bool ok = true;
    const double r = chq::div_by(p, g, y, ok);
    if (!ok) continue;
    ++taken;
    if (!(r == p / g)) { if (bad < 5) std::printf("mismatch %a / %a\n", p, g); ++bad; }
  }
  const double refused[] = {0.0, -1.0, 1e-300, 5e-324, INFINITY, NAN};
  for (double p : refused) {
    bool ok = true;
    (void)chq::div_by(p, 0.5, 2.0, ok);
    if (ok) { std::printf("not refused %a\n", p); ++bad; }
  }
  std::printf("taken %ld mismatches %ld\n", taken, bad);
  return bad || taken < n / 4;
}
