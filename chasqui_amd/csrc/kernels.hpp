// Kernel argument blocks and launch helpers shared by the stage kernels and the C-ABI.
//
// T is the type of the arrays the face-flux / corner-EMF side works in: double for the FP64
// drop-in, float for the mixed-precision path (FP32 primitives, fluxes and EMFs). Conserved
// variables and face-centred B are always double.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.hpp"
#include "ghost.hpp"

namespace chq {

// A face-flux launch: one direction, faces [il..iu] x [jl..ju] x [kl..ku] (inclusive).
// Division by a divisor fixed before launch, for numerators below 2^31 (Granlund and Montgomery,
// "Division by invariant integers using multiplication", 1994, Theorem 4.2): with
// l = ceil(log2 d) and m = ceil(2^(31+l) / d), 0 <= m d - 2^(31+l) < d <= 2^l, so
// floor(n / d) = floor(n m / 2^(31+l)) for every 0 <= n < 2^31, and m < 2^32. A 32 x 32 -> 64-bit
// multiply and a shift per lane instead of an integer division (about 100 instructions for a
// 64-bit one). 1 <= d < 2^31 (a d below 1 is taken as 1).
struct FastDiv {
  unsigned m;
  int s;
};
__host__ __device__ inline FastDiv fast_div(int d) {
  if (d < 1) d = 1;
  int l = 0;
  while ((1LL << l) < d) ++l;
  const unsigned long long p = 1ULL << (31 + l);
  return FastDiv{unsigned((p + (unsigned long long)d - 1) / (unsigned long long)d), 31 + l};
}
__host__ __device__ __forceinline__ unsigned fdiv(unsigned n, FastDiv f) {
  return unsigned(((unsigned long long)n * f.m) >> f.s);
}

template <class T>
struct FluxArgsT {
  Geom g;
  Eos eos;
  int flatten, low_mach;
  int entropy;        // reconstruct and flux the entropy variable (IENT)
  int charac;         // reconstruct in characteristic variables (FP64 single-mesh launches only)
  double lhlld_phi;
  int il, iu, jl, ju, kl, ku;
  int seg;            // faces per thread of the y/z march (fluxk::march_seg)
  FastDiv q1, q2;     // x faces: by the cells per row and by the rows per plane of the face
                      // range (x_shape); y/z faces: by nx and by nt (m_item)
  const T *w;         // primitives, 6 components (IENT used only when entropy is transported)
  const T *bcc;       // cell-centred B, 3 components
  const double *bn;   // face-normal field of this direction (the stage-input face B)
  T *flx;             // fluxes, 6 components
  T *et2, *et1;       // face EMFs: et2 = -F(B_t1), et1 = +F(B_t2)
  const int *flag;    // fofc flags (repair launches only)
  const Ctrl *ctrl;
};
using FluxArgs = FluxArgsT<double>;

template <class T>
struct CornerArgsT {
  Geom g;
  const T *f1, *f2, *f3;       // mass-flux components (IDN) of the face fluxes
  const T *e2x1, *e3x1, *e1x2, *e3x2, *e1x3, *e2x3;
  const T *ecc;
  T *e1, *e2, *e3;
  const Ctrl *ctrl;
  int only_if_bad;             // skip unless the current stage flagged cells (fofc re-run)
  int xg;                      // XCD tile grouping (xcd_tile)
};
using CornerArgs = CornerArgsT<double>;

// RK combine + divergence + CT: fluxes and edge EMFs of type T are widened to double and
// every sum, product and combination is done in double.
template <class T>
struct UpdateArgsT {
  Geom g;
  double g0, g1, beta;         // beta_dt = beta * dt, dt from ctrl (or beta_dt given)
  double beta_dt;              // used when use_ctrl_dt == 0
  int use_ctrl_dt;
  int nvar;                    // 5 (entropy not transported) or 6
  const T *f1, *f2, *f3;
  const double *ua, *ub;
  double *uo;
  const double *b1a, *b2a, *b3a, *b1b, *b2b, *b3b;
  double *b1o, *b2o, *b3o;
  const T *e1, *e2, *e3;
  const Ctrl *ctrl;
  int only_if_bad;
  // FP64 first pass of a stage that may re-update locally (output = ub, g1 = 0): count into
  // *zcount the points whose recomputation could differ from this pass, i.e. where g0 * ua is
  // -0 and the divergence (curl) term is 0, or where the result is not finite
  int zwatch;
  int *zcount;
  int xg;                      // XCD tile grouping (xcd_tile)
};
using UpdateArgs = UpdateArgsT<double>;

// the ghost fill of all directions (bc[d]: 0 periodic, 1 outflow, 2 reflecting)
struct BcArgs {
  Geom g;
  int bc[3], nvar;
  double *u, *b1, *b2, *b3;
  const Ctrl *ctrl;
  int only_if_bad;
};

// con2prim computes in double and stores primitives, cell B and cell EMF as T
template <class T>
struct C2pArgsT {
  Geom g;
  Eos eos;
  double *b1, *b2, *b3;        // (the fused ghost fill writes their ghost entries)
  double *u;
  T *w, *bcc, *ecc;
  int bc[3];                   // boundary conditions of the fused ghost fill
  int write_went;              // also store w[IENT] (needed when entropy is transported)
  int compute_dt;
  int slot;                    // which running minimum receives the CFL dt (0 or 1)
  int flag_mode;               // 0: none; 1: flag array + count; 2: append flagged cells to badlist
  int *flag;
  int *badlist;
  Ctrl *ctrl;
  int only_if_bad;
  int xg;                      // XCD tile grouping (xcd_tile)
};
using C2pArgs = C2pArgsT<double>;

// ---------------------------------------------------------------- work decomposition
// The memory-bound kernels walk "virtual blocks": chunks of 256 consecutive points of one
// (j, i) plane of an nx x ny box (rows are linearised, so rows of 257 or 262 points waste no
// lanes), times nz planes.
// XCD-grouped tile order: the dispatcher deals consecutive workgroups of a launch to the 8 XCDs
// in turn, so neighbouring tiles (rows that read each other's lines) land in different L2s.
// Block b of n takes tile xcd_tile(b, n, grp): each XCD gets runs of grp consecutive tiles,
// groups of 8 * grp tiles in launch order (the tail past the last whole group keeps b). A
// bijection on [0, n); grp <= 1 is the identity.
__host__ __device__ __forceinline__ int xcd_tile(int b, int n, int grp) {
  if (grp <= 1) return b;
  const int span = 8 * grp, full = (n / span) * span;
  if (b >= full) return b;
  const int l = b >> 3;
  return (l / grp) * span + (b & 7) * grp + l % grp;
}
// Group sizes of the fused stage's kernels, measured at 256^3 (ms per RK3 step, FP64 / mixed):
// con2prim 32 (1.65 -> 1.58 / 1.28 -> 1.16; 4, 8, 16 and 64 gain less), corner EMF 4 (1.47 ->
// 1.44 / 0.90 -> 0.88; 8 and 16 the same), the float update march 8 (2.62 -> 2.60); the FP64
// update keeps the launch order (runs of 2, 3, 4, 8 or 16 made it 0.4-1.2% slower).
// The update that forms the edge EMFs itself (1D, 2D): 32 (512^2 mixed 11.72 -> 11.59 ms per pass,
// 1000x1024 FP64 27.15 -> 26.96); the batched update: 8 (48 vortices FP64 135.0 -> 134.4 ms).
constexpr int XG_C2P = 32, XG_CORNER = 4, XG_UPDATE_F32 = 8, XG_UPDATE_CORN = 32, XG_UPDATE_BATCH = 8;

struct VB {
  int nx, ny, cpp, n;   // plane size, chunks per plane, total chunks
  __device__ __forceinline__ bool at(int vb, int &k, int &j, int &i) const {
    k = vb / cpp;
    const int t = (vb - k * cpp) * 256 + int(threadIdx.x);
    j = t / nx;
    i = t - j * nx;
    return t < nx * ny;
  }
};
inline __host__ __device__ VB vgrid(int nx, int ny, int nz) {
  VB v;
  v.nx = nx;
  v.ny = ny;
  v.cpp = div_up(nx * ny, 256);
  v.n = v.cpp * nz;
  return v;
}
// corner EMF: the union box [is..ie+1] x [js..je+1] x [ks..ke+1] (one k plane below 3D)
inline __host__ __device__ VB corner_vb(const Geom &g) {
  return vgrid(g.ie - g.is + 2, g.je - g.js + 2, g.three_d ? g.ke - g.ks + 2 : 1);
}
// update: active cells plus the upper faces of the present directions
inline __host__ __device__ VB update_vb(const Geom &g) {
  return vgrid(g.ie - g.is + 2, g.two_d ? g.je - g.js + 2 : 1, g.three_d ? g.ke - g.ks + 2 : 1);
}

// Whether the update launch forms the edge EMFs: below 3D, in FP64 up to 2048 tiles. Above that the
// 127 VGPRs of the FP64 form (96 without) cost more than the launch it saves: 1000x1024 26.96 ms
// per pass against 26.72 with a corner launch, 700x720 10.2 against 10.8, 150x129 7.3 against 7.8;
// mixed 512^2 11.5 against 12.0, 1024x1000 13.3 against 13.6.
inline bool update_has_corner(const Geom &g, bool fp64) {
  return !g.three_d && (!fp64 || update_vb(g).n <= 2048);
}
// con2prim: every cell, ghosts included
inline __host__ __device__ VB c2p_vb(const Geom &g) { return vgrid(g.ni, g.nj, g.nk); }
// con2prim with the fused ghost fill: the active cells, in tiles after those of the ghost points
inline __host__ __device__ VB active_vb(const Geom &g) {
  return vgrid(g.ie - g.is + 1, g.je - g.js + 1, g.ke - g.ks + 1);
}

// face-flux decomposition (flux_impl.hpp): x faces by wave64 windows over the rows' cells laid
// end to end, y/z faces by threads marching a.seg faces along the direction; both linearised so
// that no lane idles at the end of a row (a 258-wide row in 64-wide tiles would leave a fifth
// of the lanes idle)
namespace fluxk {
constexpr int BX = 64, BY = 4;
// Faces per thread in the y/z march. A thread of a segment of s faces reconstructs s + 1 cells and
// solves s faces one after the other: long segments save the extra reconstruction, short ones
// give a small launch more waves and a shorter serial chain. march_seg picks the candidate of
// least cost (s + 0.9) (0.15 + 0.85 m), where m is the launch's 256-thread blocks per CU (a block
// puts one wave on each SIMD of its CU, and the waves of a SIMD share its issue slots, so the
// second block of a CU adds 0.85 of the first one's time); a partial last block per CU counts
// half as such and half as a whole one. The three constants are fitted to sweeps over segments of
// 1 to 24 of the meshes whose directions have a launch each (dual energy, explicit diffusion, the
// sizes beyond flux_merge's limits): 64^3 .. 240^3 and 200^2 .. 2200^2, PLM, PPM, PPMX, WENO-Z,
// both precisions: the choice is within 0.5% of the best candidate on average (4.3% at worst, 600^2
// of PPMX LHLLD; else 2.5%). (s + 0.7) (0.1 + 0.9 m) with three quarters of a whole block for the
// partial one gave 0.8% and 6.6%: 144^3 took 3 faces (now 8; ms per step of dual energy PPMX 3.78 ->
// 3.61, WENO-Z 4.02 -> 3.86, PPM with explicit diffusion 4.65 -> 4.54; 4.62 with the 24 faces it had
// before any model). The choice moves work between threads only: every face is computed by the same
// expressions either way.
struct MarchShape {
  long long rows;   // threads per segment layer: the face range across the march direction
  int nd;           // faces along it
};
// the march of direction d (1 or 2) over a face range
inline MarchShape march_shape(int il, int iu, int jl, int ju, int kl, int ku, int d) {
  const long long nx = iu - il + 1;
  return d == 1 ? MarchShape{nx * (ku - kl + 1), ju - jl + 1} : MarchShape{nx * (ju - jl + 1), ku - kl + 1};
}
// the segment of a launch that marches `n` shapes (the runs of a batch; one for a single mesh)
inline int march_seg(const MarchShape *sh, int n) {
  static constexpr int cand[] = {1, 2, 3, 4, 6, 8, 12, 16, 24};
  int best = 1;
  double least = 1e300;
  for (const int s : cand) {
    long long blocks = 0;
    int len = 1;   // the longest serial march
    for (int q = 0; q < n; ++q) {
      blocks += (sh[q].rows * ((sh[q].nd + s - 1) / s) + 255) / 256;
      len = len > sh[q].nd ? len : sh[q].nd;
    }
    const double per = double(blocks) / 256.0;   // 256 CUs
    const double m = 0.5 * double((blocks + 255) / 256) + 0.5 * per;
    const double cost = ((s < len ? s : len) + 0.9) * (0.15 + 0.85 * (m > 1.0 ? m : 1.0));
    if (cost < least) { least = cost; best = s; }
  }
  return best;
}

template <Recon RC> constexpr bool wide_v = !(RC == Recon::dc || RC == Recon::plm);
inline __host__ __device__ int fpw_of(Recon rc) {
  const bool w = !(rc == Recon::dc || rc == Recon::plm);
  return 64 - (w ? 3 : 2) - (w ? 2 : 1);
}
template <Recon RC> constexpr int fpw_v = 64 - (wide_v<RC> ? 3 : 2) - (wide_v<RC> ? 2 : 1);   // faces per wave

// x-face work: the cells of all rows (ni per row, rows (j, k) of the face range) laid end to
// end; wave w holds cells w * fpw - H ... w * fpw - H + 63 and computes the faces of its middle
// fpw lanes; 4 waves per block. nseg = ni (cells per row).
template <class T>
__host__ __device__ inline void x_shape(const FluxArgsT<T> &a, int fpw, int &nseg, int &nwaves) {
  nseg = a.g.ni;
  const long long cells = (long long)nseg * (a.ju - a.jl + 1) * (a.ku - a.kl + 1);
  nwaves = int((cells + fpw - 1) / fpw);
}

// y/z-face work: one thread per (i, transverse row, segment of a.seg faces along DIR), i fastest,
// in blocks of BX x BY threads (gx blocks; gy = gz = 1).
template <class T, int DIR>
__host__ __device__ inline void m_shape(const FluxArgsT<T> &a, int &gx, int &gy, int &gz) {
  const int nx = a.iu - a.il + 1;
  const int nt = DIR == 1 ? a.ku - a.kl + 1 : a.ju - a.jl + 1;
  const int nd = DIR == 1 ? a.ju - a.jl + 1 : a.ku - a.kl + 1;
  gx = int(((long long)nx * nt * div_up(nd, a.seg) + BX * BY - 1) / (BX * BY));
  gy = 1;
  gz = 1;
}
// thread `lin` of the y/z decomposition: i, transverse index t and segment sg (false: no work)
template <class T, int DIR>
__host__ __device__ inline bool m_item(const FluxArgsT<T> &a, long long lin, int &i, int &t, int &sg) {
  const int nx = a.iu - a.il + 1;
  const int nt = DIR == 1 ? a.ku - a.kl + 1 : a.ju - a.jl + 1;
  const int nd = DIR == 1 ? a.ju - a.jl + 1 : a.ku - a.kl + 1;
  const unsigned r = fdiv(unsigned(lin), a.q1), rs = fdiv(r, a.q2);   // lin < 2^31 (mesh limit)
  i = a.il + int(unsigned(lin) - r * unsigned(nx));
  t = int(r - rs * unsigned(nt));
  sg = int(rs);
  return sg < div_up(nd, a.seg);
}

// Whether the face fluxes of all directions go in one launch (k_flux_all, k_fluxc_all). One launch
// saves the others' dispatch and tails and lets the x blocks fill the SIMDs that a small march
// leaves idle; but the x waves then run at the march's occupancy (two waves per SIMD in FP64
// instead of four, four instead of eight in FP32), which costs more once each launch fills the
// device by itself. The limits are on the march blocks at one face per thread, both sides measured
// (ms per RK3 step, separate -> one launch):
//   FP64   PPM    64x56x45 (1378 blocks) 0.336 -> 0.269; the whole pass at 128^3 (17032) -1.3%, 160^3 -1.2%, 208^3
//                 (72031) -0.6%, 256^3 (133648) +1.6%; 800^2 (2519) -2.8%, 1000^2 (3929) -0.3%, 1200^2 +0.4%; PLM and
//                 PPMX alike (PPMX 144^3 -3.4%, 208^3 -0.2%)
//          WENO-Z 64^3 -15%, 144^3 (24145) -4.3%, 192^3 (56748) -1.1%, 224^3 (89778) +1.4%; 400^2 -8%, 800^2
//                 -4.2%, 1000^2 -0.3%
//          characteristic PPMX (x kernel and march both at two waves): 80x72x64 (3083) 1.087 -> 1.009, 96^3 (7278)
//                 -8%, 112^3 -4%, 144^3 (24145) -7%; 200^2 -16%, 500^2 -11%: always
//   FP32   PPM    144^3 (24145) -3.5%, 192^3 (56748) -2.2% for a wave but 30 steps of a blast +0.6%, 240^3 -0.2%, PPMX
//                 there +1.3%; 1300^2 (6616) -1.9%, 1600^2 +0.6%; PLM 192^3 +0.3%. The 3D limit is what the
//                 blast allows: a wave alone would take one launch at 192^3 too.
//          WENO-Z 192^3 -2.1%, 256^3 (133648) 9.62 -> 9.41; 1600^2 (10022) -2%, 2000^2 (15648) 1.78 -> 1.76
// A batch counts the march blocks of all its runs (64 small mixed runs 28.4 -> 26.6 ms per 100 steps).
inline bool merge_blocks(bool fp32, bool charac, Recon rc, bool d3, long long blocks) {
  const bool weno = rc == Recon::wenoz;
  if (fp32) return weno ? (d3 || blocks <= 16000) : blocks <= (d3 ? 40000 : 8000);
  if (charac) return true;
  return blocks <= (d3 ? (weno ? 65000 : 75000) : 4500);
}
template <class T>
inline bool flux_merge(const FluxArgsT<T> *a, int ndir, Recon rc, bool entropy) {
  if (ndir < 2 || (entropy && !a[0].charac)) return false;
  long long blocks = 0;
  for (int d = 1; d < ndir; ++d) {
    const MarchShape m = march_shape(a[d].il, a[d].iu, a[d].jl, a[d].ju, a[d].kl, a[d].ku, d);
    blocks += m.rows * m.nd / 256;
  }
  return merge_blocks(sizeof(T) == 4, a[0].charac, rc, ndir == 3, blocks);
}
// The march segment of a joint launch: the candidate of least (s + 1.5) (0.5 + m), m the march
// blocks per CU. Blocks of all lengths share a CU here, so the work term has no steps at whole
// blocks per CU as march_seg's has; fitted to sweeps over the sizes above (1.2% from the best
// candidate on average).
inline int joint_seg(const MarchShape *sh, int n) {
  static constexpr int cand[] = {1, 2, 3, 4, 6, 8, 12, 16, 24};
  int best = 1;
  double least = 1e300;
  for (const int s : cand) {
    double blocks = 0.0;
    for (int q = 0; q < n; ++q) blocks += double(sh[q].rows) * ((sh[q].nd + s - 1) / s) / 256.0;
    const double cost = (s + 1.5) * (0.5 + blocks / 256.0);
    if (cost < least) { least = cost; best = s; }
  }
  return best;
}
template <class T>
inline void joint_seg(FluxArgsT<T> *a, int ndir) {
  MarchShape sh[2];
  for (int d = 1; d < ndir; ++d) sh[d - 1] = march_shape(a[d].il, a[d].iu, a[d].jl, a[d].ju, a[d].kl, a[d].ku, d);
  const int best = joint_seg(sh, ndir - 1);
  for (int d = 1; d < ndir; ++d) a[d].seg = best;
}

}  // namespace fluxk

// ---------------------------------------------------------------- batches
// Many independent meshes advanced by the same launches. Every run keeps its own arena and
// control block; the launches walk device-resident work lists of (run, tile) items, so a
// captured step graph stays valid while runs join and leave (only list contents change).
struct Item { int run, tile; };
struct ItemList {
  const Item *item;
  const int *n;        // number of items (device memory)
};

// every launch description of one run, for each (stage-input buffer, primitive set)
template <class T>
struct RunArgs {
  FluxArgsT<T> flux[2][2][3];    // [input buffer][primitive set][dir]
  CornerArgsT<T> corner[2];      // [primitive set]
  UpdateArgsT<T> update[2];      // [output buffer]; coefficients come with the launch
  C2pArgsT<T> c2p[2][2];         // [buffer][primitive set written]
  Ctrl *ctrl;
  int *badlist;                  // cells flagged by con2prim in the current stage
  int ndir;
  int cond_tiles[2];             // tiles of the whole-mesh fofc re-runs: update, ghost fill + con2prim
};

// The fofc branch of a batch: the runs that flagged cells in the current stage, compacted on
// the device, with per-class tile prefixes (classes below).
enum : int { CL_REPAIR = 0, CL_CORNER, CL_UPDATE, CL_C2P, CL_N };
struct CondList {
  int cap;             // capacity in runs
  int *base;           // [0] = number of flagged runs, then run[cap], then pre[CL_N][cap + 1], then done()
  __host__ __device__ int *nrun() const { return base; }
  __host__ __device__ int *run() const { return base + 1; }
  __host__ __device__ int *pre(int cls) const { return base + 1 + cap + cls * (cap + 1); }
  __host__ __device__ int *done() const { return pre(CL_N); }   // finished blocks of the last launch (0 between)
  static size_t ints(int cap) { return size_t(2) + cap + size_t(CL_N) * (cap + 1); }
};

// launches (defined in stage.hip / flux.hip / flux32.hip)
hipError_t launch_flux(const FluxArgsT<double> &a, int dir, Recon rc, RSolver rs, bool entropy, hipStream_t s);
hipError_t launch_flux(const FluxArgsT<float> &a, int dir, Recon rc, RSolver rs, bool entropy, hipStream_t s);
// characteristic-variable reconstruction (FP64; launch_flux forwards when a.charac is set)
hipError_t launch_flux_charac(const FluxArgsT<double> &a, int dir, Recon rc, RSolver rs, bool entropy, hipStream_t s);
hipError_t launch_flux_charac_all(const FluxArgsT<double> a[3], int ndir, Recon rc, RSolver rs, bool entropy, hipStream_t s);
// every direction in one launch (flux_merge says when; the march segments are joint_seg's)
hipError_t launch_flux_all(const FluxArgsT<double> a[3], int ndir, Recon rc, RSolver rs, bool entropy, hipStream_t s);
hipError_t launch_flux_all(const FluxArgsT<float> a[3], int ndir, Recon rc, RSolver rs, bool entropy, hipStream_t s);
hipError_t launch_repair(const FluxArgs &a, int dir, bool only_if_bad, hipStream_t s);
// with `marks`, also stamps the points of the local fofc re-update (k_update_near)
hipError_t launch_repair_list(const FluxArgsT<double> a[3], int ndir, const int *list, int *marks, hipStream_t s);
hipError_t launch_repair_list(const FluxArgsT<float> a[3], int ndir, const int *list, int *marks, hipStream_t s);
template <class T> hipError_t launch_corner(const CornerArgsT<T> &a, hipStream_t s);
template <class T> hipError_t launch_corner_list(const CornerArgsT<T> &a, const int *list, hipStream_t s);
// with `ca` (1D and 2D meshes, update_has_corner) the launch forms the edge EMFs itself
template <class T>
hipError_t launch_update(const UpdateArgsT<T> &a, hipStream_t s, const CornerArgsT<T> *ca = nullptr);
// u[IENT] = rho p / rho^gamma over every cell of buffer a.u with con2prim's expressions (the
// deferred resynchronisation of the fast path's last stage); writes nothing else
hipError_t launch_ient_sync(const C2pArgsT<double> &a, hipStream_t s);
// the local fofc re-update: recompute the points that launch_repair_list stamped with the control
// block's epoch (every point where the first pass counted one that needs it)
template <class T>
hipError_t launch_update_near(const UpdateArgsT<T> &a, const CornerArgsT<T> *ca, const int *marks, hipStream_t s);
hipError_t launch_fill(const BcArgs &a, hipStream_t s);

// explicit diffusion (FP64 single-mesh path), diffusion.hip
struct DiffArgs {
  Geom g;
  double nu, kappa, eta, gm1;
  const double *w, *bcc;                 // primitives, cell-centred B
  const double *b1, *b2, *b3;            // face B the current density is taken from
  double *f[3];                          // face fluxes (6 components each)
  double *e1, *e2, *e3;                  // edge EMFs
  const int *flag;                       // fofc flags (repair launches only)
  const Ctrl *ctrl;
  int only_if_bad;                       // skip unless the current stage flagged cells (fofc branch)
};
hipError_t launch_diff_flux(const DiffArgs &a, int dir, bool flagged_only, hipStream_t s);
hipError_t launch_resistive_emf(const DiffArgs &a, hipStream_t s);
// minimum of w[IDN] over the active cells into ctrl->rho_bits (reset first)
hipError_t launch_rho_min(const double *w, const Geom &g, Ctrl *c, bool reset, hipStream_t s);
// ctrl->min_dt = min(ctrl->min_dt, parabolic limit from ctrl->rho_bits) when the step ran
hipError_t launch_diff_dt_fold(Ctrl *c, const DiffArgs &a, hipStream_t s);
// super-time-stepping pieces
hipError_t launch_fill_zero(double *p, long long n, hipStream_t s);
hipError_t launch_sts_div(const Geom &g, const double *f1, const double *f2, const double *f3, const double *e1,
                          const double *e2, const double *e3, double *mu, double *mb1, double *mb2, double *mb3,
                          hipStream_t s);
struct StsTerm { const double *x; double a; };
hipError_t launch_sts_combine(const Geom &g, double *out, const StsTerm t[5], int ncomp, bool faces, hipStream_t s);
hipError_t launch_ctrl_take_min(Ctrl *c, int slot, hipStream_t s);   // ctrl->min_dt = running minimum `slot`

// positivity flux limiter and source terms (FP64 single-mesh path), srcterms.hip
struct SrcArgs {
  Geom g;
  Eos eos;
  double x1min, x2min, x3min;
  int grav_uniform, grav_point;
  double g1, g2, g3, gm, gx0, gy0, gz0, rsoft;
  double lambda0, cool_alpha, tfloor;
  double beta;                           // stage weight: beta * ctrl->dt, or beta itself
  int use_ctrl_dt;
  double *u;                             // conserved state the sources act on
  const double *w, *bcc;
  double *f[3];
  Ctrl *ctrl;
  int only_if_bad;                       // fofc branch: skip unless cells were flagged
};
hipError_t launch_limit_fluxes(const SrcArgs &a, int dir, hipStream_t s);
hipError_t launch_gravity(const SrcArgs &a, hipStream_t s);
hipError_t launch_cooling(const SrcArgs &a, hipStream_t s);
template <class T> hipError_t launch_c2p(const C2pArgsT<T> &a, hipStream_t s);
// The control work between two stages, in this order: end of a stage (`last` of its step), end
// of the step, begin of the next step, begin of a stage (`stage`, `reset` the CFL minima). One
// launch, or none where a conditional con2prim launch takes it along (launch_fill_c2p).
struct CtrlTurn {
  int end_stage, last, fused, end_step, begin_step, begin_stage, reset, stage;
};
hipError_t launch_ctrl_turn(Ctrl *c, const CtrlTurn &t, hipStream_t s);
// ghost fill and con2prim of every cell in one launch (u[IENT] neither transported nor stored).
// With `turn` (a launch whose gate is closed by nbad == 0, at most FILL_TURN_TILES tiles), the
// launch ends with that control turn.
constexpr int FILL_TURN_TILES = 2048;
inline int fill_c2p_tiles(const Geom &g) { return ((ghost_tiles(g) + 7) & ~7) + active_vb(g).n; }
// Whether a stage may flag early (Ctrl::early), in a launch of its own before the fill. The early
// order saves a firing stage its second con2prim and costs every stage a launch: on meshes up to
// EARLY_FLAG_TILES tiles the flag always stays inside con2prim. With this and the two launches that
// the local re-update lost, ms per pass: 50 steps of 150x129 6.02 -> 5.67, 50 of 512^2 mixed 10.19 ->
// 9.75, 40 of 64x56x45 (its first stage fires) 11.78 -> 11.43.
constexpr int EARLY_FLAG_TILES = 2048;
inline bool early_flag(const Geom &g) { return fill_c2p_tiles(g) > EARLY_FLAG_TILES; }
template <class T> hipError_t launch_fill_c2p(const C2pArgsT<T> &a, hipStream_t s, const CtrlTurn *turn = nullptr);
hipError_t launch_flag(const C2pArgs &a, hipStream_t s);   // standalone FlagBadCells
// control-block kernels
// outside the time loop (the per-kernel entry points and split steps)
hipError_t launch_ctrl_begin_stage(Ctrl *c, int reset_slots, hipStream_t s);

// batched launches: `grid` blocks walk the list (grid-stride); stage coefficients are
// launch arguments, everything per run comes from the RunArgs table
hipError_t launchb_flux(const RunArgs<double> *R, ItemList L, int dir, int cur, Recon rc, RSolver rs, int grid, hipStream_t s);
hipError_t launchb_flux(const RunArgs<float> *R, ItemList L, int dir, int cur, Recon rc, RSolver rs, int grid, hipStream_t s);
// the lists of all directions in one launch (the batch's march work is below flux_merge's limits)
hipError_t launchb_flux_all(const RunArgs<double> *R, const ItemList L[3], int cur, Recon rc, RSolver rs, int grid, hipStream_t s);
hipError_t launchb_flux_all(const RunArgs<float> *R, const ItemList L[3], int cur, Recon rc, RSolver rs, int grid, hipStream_t s);
hipError_t launchb_repair(const RunArgs<double> *R, CondList C, int cur, int grid, hipStream_t s);
hipError_t launchb_repair(const RunArgs<float> *R, CondList C, int cur, int grid, hipStream_t s);
// the fofc branch of a batch of small runs: one block per run (cap blocks), the repair, then the
// edge EMFs, re-update, boundaries and con2prim of the run, and the stage's control turn (launchb_ctrl's
// op, arg and live)
hipError_t launchb_repair_runs(const RunArgs<double> *R, const int *nruns, int cap, int cur, hipStream_t s);
hipError_t launchb_repair_runs(const RunArgs<float> *R, const int *nruns, int cap, int cur, hipStream_t s);
template <class T> hipError_t launchb_fofc_runs(const RunArgs<T> *R, const int *nruns, int cap, int out, double g0,
                                                double g1, double beta, int last, int op, int arg, int *live,
                                                hipStream_t s);
template <class T> hipError_t launchb_corner(const RunArgs<T> *R, ItemList L, int grid, hipStream_t s);
template <class T> hipError_t launchb_update(const RunArgs<T> *R, ItemList L, int out, double g0, double g1, double beta, int grid, hipStream_t s);
template <class T> hipError_t launchb_c2p(const RunArgs<T> *R, ItemList L, int buf, int last, int grid, hipStream_t s);
template <class T> hipError_t launchb_fofc_scan(const RunArgs<T> *R, const int *nruns, CondList C, hipStream_t s);
template <class T> hipError_t launchb_corner_cond(const RunArgs<T> *R, CondList C, int grid, hipStream_t s);
template <class T> hipError_t launchb_update_cond(const RunArgs<T> *R, CondList C, int out, double g0, double g1, double beta, int grid, hipStream_t s);
// ... which ends the stage of every run with the control work op, arg, live (launchb_ctrl)
template <class T> hipError_t launchb_c2p_cond(const RunArgs<T> *R, const int *nruns, CondList C, int buf, int last, int op,
                                               int arg, int *live, int grid, hipStream_t s);
// control-block step of every run (one thread per table slot, `cap` slots); the end of a step
// also writes live[r] = run r has not reached tlim / nlim
template <class T> hipError_t launchb_ctrl(const RunArgs<T> *R, const int *nruns, int cap, int op, int arg, int *live, hipStream_t s);
// CTRL_STEP_FIRST: begin step + begin stage 1; CTRL_TURN: end a stage + begin the next (arg:
// the next one is the last); CTRL_END_LAST: end the last stage + end step (+ live flags)
enum : int { CTRL_BEGIN_STEP = 0, CTRL_BEGIN_STAGE, CTRL_END_STAGE, CTRL_END_STEP, CTRL_LIVE, CTRL_STEP_FIRST,
             CTRL_TURN, CTRL_END_LAST };

// A batched kernel's item and its run's launch description are the same for every lane of a wave.
// Said so (and the tables __restrict__: nothing a kernel writes aliases them), they are read by
// scalar loads into SGPRs; as vector loads they held 45 to 60 VGPRs of each kernel (con2prim 90-102
// against 46 in the single-mesh form) and stood in front of every tile's own loads. 48 vortices of
// 64^2 to 512^2, FP64, 40 steps: 143.2 -> 136.0 ms.
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ Item uniform_item(const Item *__restrict__ item, int it) {
  return Item{uniform(item[it].run), uniform(item[it].tile)};
}

// position of `it` in an exclusive prefix pre[0..n] (largest p with pre[p] <= it)
__device__ __forceinline__ int locate(const int *pre, int n, int it) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (pre[mid] <= it) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

}  // namespace chq
