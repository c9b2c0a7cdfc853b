// The ghost fill as a map: for every entry of an array the entry whose value the boundary
// conditions give it, over all directions at once.
//
// physics.hpp:354-432 fills x1, then x2, then x3, each over the entries the ones before left. An
// entry's final value is therefore that of one entry that no fill writes (an active one, or one
// of the rows and planes beyond the last cell), found by following the maps backwards: x3 first,
// then x2 where that fill covers the entry reached, then x1. One thread per ghost point reads
// from there, so all three directions are one launch and no thread reads what another writes.
#pragma once
#include <hip/hip_runtime.h>

#include "common.hpp"

namespace chq {

// one direction's map (periodic, outflow, reflecting): cells s..e of n, ghosts on both sides; the
// faces s..e+1, where a periodic fill also sets e+1 from s. True when the entry is a mirror image.
template <bool FACE>
__host__ __device__ __forceinline__ bool ghost_map(int &i, int s, int e, int n, int ng, int bc) {
  if (i < s) {
    if (bc == 0) i += n;
    else if (bc == 1) i = s;
    else { i = FACE ? 2 * s - i : 2 * s - 1 - i; return true; }
    return false;
  }
  if (FACE) {
    if (i <= e) return false;
    if (bc == 0) { i -= n; if (i > e) i -= n; }
    else if (bc == 1) i = e + 1;
    else if (i > e + 1) { i = 2 * (e + 1) - i; return true; }
    return false;
  }
  if (i <= e || i > e + ng) return false;
  if (bc == 0) i -= n;
  else if (bc == 1) i = e;
  else { i = 2 * e + 1 - i; return true; }
  return false;
}
// A = 0: cell values, 1..3: the face field of that direction. Each direction covers what the
// reference's fill covers: cells k < nk, j < nj, i < ni; the face field's own direction every
// entry; the other face fields the rows (x1: j < nj, x2: i < ni except b1) of their cells.
// Returns the mask of the directions with a mirror image.
template <int A>
__host__ __device__ __forceinline__ int ghost_source(const Geom &g, const int *bc, int &k, int &j, int &i) {
  int m = 0;
  if (g.three_d && (A != 0 || (j < g.nj && i < g.ni)))
    m |= ghost_map<A == 3>(k, g.ks, g.ke, g.nx3, g.ng, bc[2]) ? 4 : 0;
  if (g.two_d && (A == 2 || (k < g.nk && (A == 1 || i < g.ni))))
    m |= ghost_map<A == 2>(j, g.js, g.je, g.nx2, g.ng, bc[1]) ? 2 : 0;
  if (A == 1 || (k < g.nk && j < g.nj)) m |= ghost_map<A == 1>(i, g.is, g.ie, g.nx1, g.ng, bc[0]) ? 1 : 0;
  return m;
}
// the filled value of face field A at (k, j, i); `own`: the entry is not filled
template <int A>
__host__ __device__ __forceinline__ double ghost_face(const Geom &g, const int *bc, const double *b, int k, int j, int i,
                                             bool &own) {
  const long long c = g.at(k, j, i);
  const int m = ghost_source<A>(g, bc, k, j, i);
  const long long s = g.at(k, j, i);
  own = s == c;
  const double v = b[s];
  return (m >> (A - 1)) & 1 ? -v : v;
}
// ghost points: the entries of the (nk+1) x (nj+1) x (ni+1) box outside the active range of a
// direction the mesh has (in 1D and 2D every row and plane of the others counts as inside)
inline __host__ __device__ int ghost_points(const Geom &g) {
  const int w1 = g.ni + 1, w2 = g.nj + 1, w3 = g.nk + 1;
  return w1 * w2 * w3 - g.nx1 * (g.two_d ? g.nx2 : w2) * (g.three_d ? g.nx3 : w3);
}
inline __host__ __device__ int ghost_tiles(const Geom &g) { return div_up(ghost_points(g), 256); }
// ghost point t: the ghost planes, then the ghost rows of the other
// planes, then the ghosts of the other rows
__host__ __device__ __forceinline__ bool ghost_point(const Geom &g, int t, int &k, int &j, int &i) {
  const int w1 = g.ni + 1, w2 = g.nj + 1, w3 = g.nk + 1;
  const int n1 = g.nx1, n2 = g.two_d ? g.nx2 : w2, n3 = g.three_d ? g.nx3 : w3;
  const int x1 = w1 - n1, x2 = w2 - n2, x3 = w3 - n3;   // (js, ks are 0 where n2, n3 are whole)
  if (t < x3 * w2 * w1) {
    i = t % w1;
    const int r = t / w1;
    j = r % w2;
    k = r / w2;
    if (k >= g.ks) k += n3;
    return true;
  }
  t -= x3 * w2 * w1;
  if (t < n3 * x2 * w1) {
    i = t % w1;
    const int r = t / w1;
    j = r % x2;
    if (j >= g.js) j += n2;
    k = g.ks + r / x2;
    return true;
  }
  t -= n3 * x2 * w1;
  if (t >= n3 * n2 * x1) return false;
  i = t % x1;
  if (i >= g.is) i += n1;
  const int r = t / x1;
  j = g.js + r % n2;
  k = g.ks + r / n2;
  return true;
}

}  // namespace chq
