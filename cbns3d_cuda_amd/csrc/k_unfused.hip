// k_unfused.hip -- the reference's launcher decomposition, one entry point per
// block3d_cuda call: calc_numerical_flux (face fluxes to HBM),
// calc_viscous_flux_contribution (dfv to HBM, k_viscous.hip) and update_rk3.  The fused sweep kernels (k_fused.hip) replace this chain in
// cbns_rk3_stage; this path exists so callers of the reference API can swap
// it in call for call, and it cross-checks the fused path.
#include "cbns_internal.hpp"
#include "face_math.hpp"

namespace cbns {

namespace {

// How a box of faces or nodes, one thread each, is cut into workgroups of 256: 64 x
// 4 tiles of a plane, `tiles` of them along a row, or (tiles == 0) all rows end to
// end.  A tile's wavefronts begin with a row, so their loads are whole lines, and its
// four rows share the eta-stencils; end to end no lane idles past a row's end.
struct Cut {
  Box box;
  int tiles;
};
inline unsigned cut_groups(const Cut& u) {
  return u.tiles ? (unsigned)u.tiles * ((u.box.n[1] + 3) / 4) * u.box.n[2]
                 : box_blocks(u.box, 256);
}
__device__ __forceinline__ bool cut_node(const Cut& u, unsigned group, int& i, int& j, int& k) {
  const Box& b = u.box;
  if (!u.tiles) return box_node(b, (long)group * 256 + threadIdx.x, i, j, k);
  const unsigned nty = (unsigned)(b.n[1] + 3) / 4, r = group / (unsigned)u.tiles, q = r / nty;
  const int ti = (int)(group - r * (unsigned)u.tiles) * 64 + (int)(threadIdx.x & 63);
  const int tj = (int)(r - q * nty) * 4 + (int)(threadIdx.x >> 6);
  if (ti >= b.n[0] || tj >= b.n[1]) return false;
  i = b.lo[0] + ti;
  j = b.lo[1] + tj;
  k = b.lo[2] + (int)q;
  return true;
}

// The faces of one axis: end to end where rows of at most three tiles leave a fifth of
// their lanes idle.  All three axes, us, tiles / end to end (launched an axis at a
// time on tiles, as at first): rows of 32 faces 43 / 29 (52), 60 48 / 56 (58), 70 85 / 66
// (116), 96 85 / 72 (93), 112 89 / 93 (98), 150 133 / 122 (139), 200 178 / 190 (189), 250
// 196 / 253 (202) of 96 x 64 each; 255x255x128 1095 / 1340 (1108).
inline Cut face_cut(const Box& b) {
  const int t = (b.n[0] + 63) / 64;
  return {b, t <= 3 && 5 * b.n[0] < 4 * 64 * t ? 0 : t};
}
// The update's nodes, which share no stencils: end to end where a row's last tile holds
// at most 24 nodes, or none past its whole ones.  us, tiles / end to end: rows of 16 nodes
// 10.0 / 7.7, 40 11.6 / 13.2, 60 14.7 / 18.2, 66 22.9 / 19.4, 96 26.1 / 26.8, 120 28.5 /
// 32.8, 128 31.1 / 28.2, 200 55 / 55, 240 61 / 71.
inline Cut node_cut(const Box& b) { return {b, b.n[0] % 64 <= 24 ? 0 : (b.n[0] + 63) / 64}; }

// The faces of the three axes in one launch: axis d from workgroup first[d] on.
// (Three launches have three tails.)
struct FaceBoxes {
  Cut cut[3];
  unsigned first[3];
};

// src/rec_riemann_kernel.cu:15-247: one thread per face; the face between
// node m and m+1 along `d` is stored at the index of node m.
__global__ void __launch_bounds__(256) k_face_flux(Consts c, FaceBoxes fb,
                                                   const double* __restrict__ Q,
                                                   const double* __restrict__ prim,
                                                   const double* __restrict__ met,
                                                   double* __restrict__ flux) {
  const int d = blockIdx.x >= fb.first[2] ? 2 : (blockIdx.x >= fb.first[1] ? 1 : 0);
  int i, j, k;
  if (!cut_node(fb.cut[d], blockIdx.x - fb.first[d], i, j, k)) return;
  const long S = c.S;
  const int st = stride(c, d);
  const int a = idx(c, i, j, k), bb = a + st;
  const double Ja = met[JAC * S + a], Jb = met[JAC * S + bb];
  const double nx = 0.5 * (met[(3 * d + 0) * S + a] * Ja + met[(3 * d + 0) * S + bb] * Jb);
  const double ny = 0.5 * (met[(3 * d + 1) * S + a] * Ja + met[(3 * d + 1) * S + bb] * Jb);
  const double nz = 0.5 * (met[(3 * d + 2) * S + a] * Ja + met[(3 * d + 2) * S + bb] * Jb);
  double q[6][5], e[5][5], pl[5], pr[5], f[5];
#pragma unroll
  for (int s = 0; s < 6; s++)
#pragma unroll
    for (int n = 0; n < 5; n++) q[s][n] = Q[n * S + a + (s - 2) * st];
#pragma unroll
  for (int n = 0; n < 5; n++) {
    pl[n] = prim[n * S + a];
    pr[n] = prim[n * S + bb];
  }
  const GasT<double> g{c.gamma, c.gam1, c.gam1_inv};
  // the Roe average from the node primitives, as the reference reads them
  Basis<double> B;
  roe_basis(g, pl[0], pl[1], pl[2], pl[3], pl[4], pr[0], pr[1], pr[2], pr[3], pr[4], nx, ny, nz,
            B);
  stencil_diffs(q, e);
  face_flux_basis(g, e, q[2], q[3], B, nx, ny, nz, f);
#pragma unroll
  for (int n = 0; n < 5; n++) flux[(d * 5 + n) * S + a] = f[n];
}

// src/runge_kutta_kernel.cu:13-80
__global__ void k_update_rk3(Consts c, Cut cut, double dt, int stage, const double* __restrict__ met,
                             const double* __restrict__ flux, const double* __restrict__ dfv,
                             double* __restrict__ Q, double* __restrict__ Qp) {
  int i, j, k;
  if (!cut_node(cut, blockIdx.x, i, j, k)) return;
  const long S = c.S;
  const int o = idx(c, i, j, k);
  const double Jac_a = met[JAC * S + o];
  for (int n = 0; n < NEQ; n++) {
    const double* Ep = flux + (0 * 5 + n) * S;
    const double* Fp = flux + (1 * 5 + n) * S;
    const double* Gp = flux + (2 * 5 + n) * S;
    double df = Ep[o] - Ep[o - 1];
    df += Fp[o] - Fp[o - c.PX];
    df += Gp[o] - Gp[o - c.PXY];
    if (c.viscous && n > 0) df -= dfv[(n - 1) * S + o];
    df /= Jac_a;
    const long qi = n * S + o;
    if (1 == stage) Qp[qi] = Q[qi] - dt * df;
    else if (2 == stage) Qp[qi] = 0.75 * Q[qi] + 0.25 * (Qp[qi] - dt * df);
    else if (3 == stage) Q[qi] = (Q[qi] + 2.0 * (Qp[qi] - dt * df)) / 3.0;
  }
}

Box update_box(const Consts& c) {
  Box b;
  for (int a = 0; a < 3; a++) {
    b.lo[a] = upd_lo(c, a);
    b.n[a] = upd_hi(c, a) - upd_lo(c, a) + 1;
  }
  return b;
}

}  // namespace

int launch_numerical_flux(cbns_block* b, const double* Q) {
  const Consts& c = b->c;
  FaceBoxes fb;
  unsigned groups = 0;
  for (int d = 0; d < 3; d++) {
    Box box = update_box(c);
    box.lo[d] = periodic(c, d) ? -1 : 0;
    box.n[d] = axis_n(c, d) - 1 + (periodic(c, d) ? 2 : 0);  // faces -1..N-1 or 0..N-2
    fb.cut[d] = face_cut(box);
    fb.first[d] = groups;
    groups += cut_groups(fb.cut[d]);
  }
  k_face_flux<<<groups, 256, 0, b->stream>>>(c, fb, Q, b->prim, b->met, b->flux);
  CBNS_HIP(b, hipGetLastError());
  return CBNS_OK;
}

int launch_viscous_unfused(cbns_block* b) { return launch_viscous(b, b->vtmp, b->dfv, 0); }

int launch_update_rk3(cbns_block* b, double dt, int stage) {
  const Cut cut = node_cut(update_box(b->c));
  k_update_rk3<<<cut_groups(cut), 256, 0, b->stream>>>(b->c, cut, dt, stage, b->met, b->flux,
                                                      b->dfv, b->Q, b->qp);
  CBNS_HIP(b, hipGetLastError());
  return CBNS_OK;
}

}  // namespace cbns
