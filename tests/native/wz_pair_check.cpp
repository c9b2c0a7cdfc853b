// wz_pair against two wz calls (stencil and mirrored stencil), bit for bit in FP64.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "numerics.hpp"

int main(int argc, char **argv) {
  const long n = argc > 1 ? std::atol(argv[1]) : 1000000;
  std::mt19937_64 r(17);
  std::uniform_real_distribution<double> u(-1.0, 1.0);
  long bad = 0;
  for (long t = 0; t < n; ++t) {
    double q[5];
    const int kind = int(t % 5);
    for (int m = 0; m < 5; ++m) {
      if (kind == 0) q[m] = u(r);
      else if (kind == 1) q[m] = 1.0 + 1e-9 * u(r);                          // smooth: indicators near eps
      else if (kind == 2) q[m] = (u(r) > 0.0 ? 1.0 : 0.125);                 // steps and constants
      else if (kind == 3) q[m] = std::ldexp(u(r), int(200 * u(r)));          // wide range of magnitudes
      else q[m] = 0.5 * m * double(t % 7) - (t % 3 ? 0.0 : 1.0);             // linear, zeros
    }
    double lo, hi;
    using R = chq::Rec<double>;
    R::wz_pair(q[0], q[1], q[2], q[3], q[4], lo, hi);
    const double h = R::wz(q[0], q[1], q[2], q[3], q[4]), l = R::wz(q[4], q[3], q[2], q[1], q[0]);
    if (std::memcmp(&h, &hi, 8) || std::memcmp(&l, &lo, 8)) ++bad;
  }
  std::printf("samples %ld mismatches %ld\n", n, bad);
  return bad != 0;
}
