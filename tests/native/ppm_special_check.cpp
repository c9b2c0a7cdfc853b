// The FP64 PPM half-states of a cell, as the face kernels form them (numerics.hpp, with the division
// fallback), against the oracle's, bit for bit over every window of five special values: NaN,
// infinities, zeros of both signs, denormals, values that overflow, ordinary ones. NaN equals NaN.
#include <cmath>
#include <cstdio>
#include <cstring>

#include "../../oracle/numerics.hpp"
#include "common.hpp"
#include "numerics.hpp"

static bool same(double a, double b) { return (a != a && b != b) || !std::memcmp(&a, &b, 8); }

int main() {
  using R = chq::Rec<double>;
  const double S[] = {NAN,  INFINITY, -INFINITY, 0.0,    -0.0,    1.0,     -1.0,    3.0,
                      2.5,  1.7e308,  -1.7e308,  1e-320, -3e-320, 1e-170,  3e-162};
  constexpr long N = sizeof(S) / sizeof(S[0]);
  long n = 0, bad = 0;
  for (long t = 0; t < N * N * N * N * N; ++t) {
    double q[5];
    long r = t;
    for (double &x : q) { x = S[r % N]; r /= N; }
    const double dm = R::mc(q[0], q[1], q[2]), d0 = R::mc(q[1], q[2], q[3]), dp = R::mc(q[2], q[3], q[4]);
    bool ok = true;
    double lo = R::edge(q[1], q[2], dm, d0, ok), hi = R::edge(q[2], q[3], d0, dp, ok);
    R::mono(q[2], lo, hi, ok);
    if (!ok) {
      lo = R::edge<true>(q[1], q[2], dm, d0, ok);
      hi = R::edge<true>(q[2], q[3], d0, dp, ok);
      R::mono<true>(q[2], lo, hi, ok);
    }
    double a = orc::ppm_edge(q[1], q[2], orc::slope_mc(q[0], q[1], q[2]), orc::slope_mc(q[1], q[2], q[3]));
    double b = orc::ppm_edge(q[2], q[3], orc::slope_mc(q[1], q[2], q[3]), orc::slope_mc(q[2], q[3], q[4]));
    orc::ppm_mono(q[2], a, b);
    ++n;
    if (!same(lo, a) || !same(hi, b)) {
      if (++bad <= 5) std::printf("%g %g %g %g %g: %g %g, oracle %g %g\n", q[0], q[1], q[2], q[3], q[4], lo, hi, a, b);
    }
  }
  std::printf("windows %ld mismatches %ld\n", n, bad);
  return bad != 0;
}
