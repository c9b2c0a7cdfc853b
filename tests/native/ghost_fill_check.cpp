// The ghost-fill map of the device (ghost.hpp) against the boundary conditions applied one
// direction after the other, entry by entry: 1D to 3D meshes, every combination of boundary
// conditions, every array.
#include <cstdio>
#include <set>
#include <vector>

#include "ghost.hpp"

using namespace chq;

struct Arr {   // (nk+1) x (nj+1) x (ni+1)
  int w3, w2, w1;
  std::vector<double> v;
  double &at(int k, int j, int i) { return v[(size_t(k) * w2 + j) * w1 + i]; }
};

// sequential fill of array A (0: cell values whose normal component is `vec`, 1..3 face field)
static void fill(Arr &x, const Geom &g, const int *bc, int A, int vec) {
  for (int d = 0; d < 3; ++d) {
    if ((d == 1 && !g.two_d) || (d == 2 && !g.three_d)) continue;
    const int s = d == 0 ? g.is : d == 1 ? g.js : g.ks, e = d == 0 ? g.ie : d == 1 ? g.je : g.ke;
    const int n = e - s + 1;
    const bool face = A == d + 1;
    const Arr old = x;   // a direction's ghosts come from entries it does not fill
    auto get = [&](int k, int j, int i) { Arr &o = const_cast<Arr &>(old); return o.at(k, j, i); };
    // the entries across the direction that its fill covers
    const int K = d == 2 ? 1 : (face || (d == 0 && A == 1) || (d == 1 && A == 2)) ? g.nk + 1 : g.nk;
    const int J = d == 1 ? 1 : d == 0 ? (A == 1 ? g.nj + 1 : g.nj) : (A == 0 ? g.nj : g.nj + 1);
    const int I = d == 0 ? 1 : d == 1 ? (A == 1 || A == 2 ? g.ni + 1 : g.ni) : (A == 0 ? g.ni : g.ni + 1);
    for (int k = 0; k < K; ++k)
      for (int j = 0; j < J; ++j)
        for (int i = 0; i < I; ++i) {
          auto put = [&](int q, double val) { d == 0 ? x.at(k, j, q) = val : d == 1 ? x.at(k, q, i) = val : x.at(q, j, i) = val; };
          auto from = [&](int q) { return d == 0 ? get(k, j, q) : d == 1 ? get(k, q, i) : get(q, j, i); };
          const double sg = bc[d] == 2 && (face || (A == 0 && vec == d + 1)) ? -1.0 : 1.0;
          for (int q = 0; q < g.ng; ++q) {
            if (face) {
              const int lo = q, hi = e + 2 + q;
              put(lo, bc[d] == 0 ? from(lo + n) : bc[d] == 1 ? from(s) : sg * from(2 * s - lo));
              if (bc[d] == 0) put(hi, hi - n > e ? from(hi - 2 * n) : from(hi - n));
              else put(hi, bc[d] == 1 ? from(e + 1) : sg * from(2 * (e + 1) - hi));
            } else {
              const int lo = q, hi = e + 1 + q;
              put(lo, sg * from(bc[d] == 0 ? lo + n : bc[d] == 1 ? s : 2 * s - 1 - lo));
              put(hi, sg * from(bc[d] == 0 ? hi - n : bc[d] == 1 ? e : 2 * e + 1 - hi));
            }
          }
          if (face && bc[d] == 0) put(e + 1, from(s));
        }
  }
}

static Geom geom(int n1, int n2, int n3, int ng) {
  Geom g{};
  g.nx1 = n1; g.nx2 = n2; g.nx3 = n3; g.ng = ng;
  g.two_d = n2 > 1; g.three_d = n3 > 1;
  g.ni = n1 + 2 * ng; g.nj = g.two_d ? n2 + 2 * ng : 1; g.nk = g.three_d ? n3 + 2 * ng : 1;
  g.is = ng; g.ie = ng + n1 - 1;
  g.js = g.two_d ? ng : 0; g.je = g.two_d ? ng + n2 - 1 : 0;
  g.ks = g.three_d ? ng : 0; g.ke = g.three_d ? ng + n3 - 1 : 0;
  g.pitch = g.ni + 1; g.plane = (long long)g.pitch * (g.nj + 1); g.cstride = g.plane * (g.nk + 1);
  return g;
}

template <int A>
static long check(const Geom &g, const int *bc, int vec) {
  Arr x{g.nk + 1, g.nj + 1, g.ni + 1, {}};
  x.v.resize(size_t(x.w1) * x.w2 * x.w3);
  for (size_t q = 0; q < x.v.size(); ++q) x.v[q] = 1.0 + double(q);
  Arr want = x;
  fill(want, g, bc, A, vec);
  std::set<long long> pts;
  long bad = 0;
  const int np = ghost_points(g);
  int k, j, i;
  for (int t = 0; t < np; ++t) {
    if (!ghost_point(g, t, k, j, i)) { ++bad; continue; }
    pts.insert(((long long)k * x.w2 + j) * x.w1 + i);
  }
  if (ghost_point(g, np, k, j, i) || (long)pts.size() != np) ++bad;
  std::set<long long> src;
  for (int kk = 0; kk < x.w3; ++kk)
    for (int jj = 0; jj < x.w2; ++jj)
      for (int ii = 0; ii < x.w1; ++ii) {
        const long long p = ((long long)kk * x.w2 + jj) * x.w1 + ii;
        int sk = kk, sj = jj, si = ii;
        const int m = ghost_source<A>(g, bc, sk, sj, si);
        double v = x.at(sk, sj, si);
        const int bit = A ? A - 1 : vec - 1;
        if ((A || vec) && ((m >> bit) & 1)) v = -v;
        if (v != want.at(kk, jj, ii)) ++bad;
        const bool moved = sk != kk || sj != jj || si != ii;
        if (moved && !pts.count(p)) ++bad;    // every filled entry is a ghost point
        // a source is never filled itself
        int tk = sk, tj = sj, ti = si;
        ghost_source<A>(g, bc, tk, tj, ti);
        if (tk != sk || tj != sj || ti != si) ++bad;
      }
  return bad;
}

int main() {
  long bad = 0, cases = 0;
  const int sizes[][3] = {{7, 1, 1}, {3, 1, 1}, {2, 1, 1}, {5, 4, 1}, {3, 3, 1}, {6, 5, 4}, {3, 3, 3}, {4, 3, 7}};
  for (const auto &n : sizes)
    for (int ng = 2; ng <= 3; ++ng) {
      if (n[0] < ng || (n[1] > 1 && n[1] < ng) || (n[2] > 1 && n[2] < ng)) continue;
      const Geom g = geom(n[0], n[1], n[2], ng);
      for (int q = 0; q < 27; ++q) {
        const int bc[3] = {q % 3, q / 3 % 3, q / 9};
        for (int vec = 0; vec < 4; ++vec) bad += check<0>(g, bc, vec);
        bad += check<1>(g, bc, 0) + check<2>(g, bc, 0) + check<3>(g, bc, 0);
        ++cases;
      }
    }
  std::printf("cases %ld mismatches %ld\n", cases, bad);
  return bad != 0;
}
