// k_bc.hip -- set_bc_calc_primitive: interior primitives and ghost/boundary
// fill (src/primitive_bc_kernel.cu:13-494).  The reference runs every rule in
// one kernel whose phases are ordered only by block-local barriers (:187,
// :414), so a thread can read a boundary value another block has not written
// yet.  The order the barriers intend is: interior -> xi faces -> eta=0 writes
// -> eta=0 primitives -> eta=JM-1 -> zeta faces -> periodic wraps.  Here one
// launch fills the whole shell: each target node evaluates what that sequence
// leaves in it, from nodes that no rule writes (the updated interior, and
// boundary nodes outside every rule), so there is nothing to wait for.  All of
// it is integer index work plus the reference's per-node formulas, and it is
// compared bit for bit with the oracle.
#include "cbns_internal.hpp"

namespace cbns {

namespace {

constexpr int NGR = CBNS_NG_REF;  // ghost depth the reference's rules write

__device__ inline void load_q(const Consts& c, const double* __restrict__ Q, int o,
                              double (&q)[NEQ]) {
#pragma unroll
  for (int n = 0; n < NEQ; n++) q[n] = Q[(long)n * c.S + o];
}

// primitives of a state, those of the mask (T on viscous blocks)
__device__ inline void store_prim(const Consts& c, const double (&q)[NEQ],
                                  double* __restrict__ prim, int o, int mask) {
  const long S = c.S;
  const double rr = q[0], uu = q[1] / rr, vv = q[2] / rr, ww = q[3] / rr;
  const double pp = c.gam1 * (q[4] - 0.5 * rr * (uu * uu + vv * vv + ww * ww));
  if (mask & 1) prim[o] = rr;
  if (mask & 2) prim[S + o] = uu;
  if (mask & 4) prim[2 * S + o] = vv;
  if (mask & 8) prim[3 * S + o] = ww;
  if (mask & 16) prim[4 * S + o] = pp;
  if (mask & 32) prim[5 * S + o] = c.gM2 * pp / rr;
}

// interior primitives, src/primitive_bc_kernel.cu:56-79
__global__ void k_prim_box(Consts c, Box box, const double* __restrict__ Q,
                           double* __restrict__ prim) {
  int i, j, k;
  if (!box_node3(box, i, j, k)) return;
  const int o = idx(c, i, j, k);
  double q[NEQ];
  load_q(c, Q, o, q);
  store_prim(c, q, prim, o, c.viscous ? 0x3F : 0x1F);
}

// State of node (i, j, k), j and k updated, once the xi faces are written: far
// field at xi = 0 and IM-1, :84-186 (density and momentum of the neighbour,
// p_inf); the ghosts beyond them hold the same.
__device__ inline void after_xi(const Consts& c, const double* __restrict__ Q, int i, int j, int k,
                                double (&q)[NEQ]) {
  const bool face = !periodic(c, 0) && (i <= 0 || i >= c.IM - 1);
  load_q(c, Q, idx(c, face ? (i <= 0 ? 1 : c.IM - 2) : i, j, k), q);
  if (face)
    q[4] = c.p_inf / c.gam1 + 0.5 * (q[1] * q[1] + q[2] * q[2] + q[3] * q[3]) / q[0];
}

// State that the eta = 0 rules leave at (i, -lj, k), :190-352; false where none
// writes.  Wake cut: columns i < i_begin - 1 and their mirror images; wall: the
// others below i_end, which come after the mirror images in the sequence.
__device__ inline bool after_eta0(const Consts& c, const double* __restrict__ Q,
                                  const double* __restrict__ met, int i, int lj, int k,
                                  double (&q)[NEQ]) {
  const long S = c.S, wake = (long)c.i_begin - 1;
  const double gam1 = c.gam1;
  const int im = c.IM - 1 - i;
  const bool wall = i >= wake && i < c.i_end;
  if (!wall && i >= wake && im >= wake) return false;
  if (!wall) {
    if (lj > 0) {  // the cut's other side
      after_xi(c, Q, im, lj, k, q);
      return true;
    }
    double m[NEQ];
    after_xi(c, Q, i, 1, k, q);
    after_xi(c, Q, im, 1, k, m);
    double rr = q[0], uu = q[1] / rr, vv = q[2] / rr, ww = q[3] / rr;
    double pp = gam1 * (q[4] - 0.5 * rr * (uu * uu + vv * vv + ww * ww));
    const double rr1 = m[0], uu1 = m[1] / rr1, vv1 = m[2] / rr1, ww1 = m[3] / rr1;
    const double pp1 = gam1 * (m[4] - 0.5 * rr1 * (uu1 * uu1 + vv1 * vv1 + ww1 * ww1));
    rr += rr1; uu += uu1; vv += vv1; ww += ww1; pp += pp1;
    rr *= 0.5; uu *= 0.5; vv *= 0.5; ww *= 0.5; pp *= 0.5;
    q[0] = rr;
    q[1] = rr * uu;
    q[2] = rr * vv;
    q[3] = rr * ww;
    q[4] = pp / gam1 + 0.5 * rr * (uu * uu + vv * vv + ww * ww);
    return true;
  }
  after_xi(c, Q, i, lj > 0 ? lj : 1, k, q);
  if (c.viscous) {
    // no-slip wall :264-295
    if (lj > 0) {
      q[1] = -q[1];
      q[2] = -q[2];
      q[3] = -q[3];
    } else {
      const double pp = gam1 * (q[4] - 0.5 * (q[1] * q[1] + q[2] * q[2] + q[3] * q[3]) / q[0]);
      q[1] = 0.0;
      q[2] = 0.0;
      q[3] = 0.0;
      q[4] = pp / gam1;
    }
    return true;
  }
  // slip wall :297-349 (energy formula exactly as the reference writes it)
  const int o = idx(c, i, 0, k);
  double t_x = met[ETA_Y * S + o];
  double t_y = -met[ETA_X * S + o];
  double t_abs = met[JAC * S + o];
  t_x *= t_abs;
  t_y *= t_abs;
  t_abs = sqrt(t_x * t_x + t_y * t_y);
  t_x /= t_abs;
  t_y /= t_abs;
  if (lj > 0) {
    const double s1 = q[1], s2 = q[2];
    t_abs = s1 * t_x + s2 * t_y;
    q[1] = 2 * t_abs * t_x - s1;
    q[2] = 2 * t_abs * t_y - s2;
    q[4] = q[4] - 0.5 * (s1 * s1 + s2 * s2 - q[1] * q[1] + q[2] * q[2]) / q[0];
  } else {
    const double rr = q[0];
    double uu = q[1] / rr, vv = q[2] / rr;
    const double ww = q[3] / rr;
    const double pp = gam1 * (q[4] - 0.5 * rr * (uu * uu + vv * vv + ww * ww));
    t_abs = uu * t_x + vv * t_y;
    uu = t_abs * t_x;
    vv = t_abs * t_y;
    q[1] = rr * uu;
    q[2] = rr * vv;
    q[3] = rr * ww;
    q[4] = pp / gam1 + 0.5 * rr * (uu * uu + vv * vv + ww * ww);
  }
  return true;
}

// State of node (i, j, k), k updated, before the zeta faces are written; false
// where no rule writes it.
__device__ inline bool before_zeta(const Consts& c, const double* __restrict__ Q,
                                   const double* __restrict__ met, int i, int j, int k,
                                   double (&q)[NEQ]) {
  const bool in_i = i >= 0 && i < c.IM;
  if (!periodic(c, 1) && (j <= 0 || j >= c.JM - 1)) {
    if (j <= 0 && j >= -NGR && in_i && after_eta0(c, Q, met, i, -j, k, q)) return true;
  } else if (!periodic(c, 0) && (i <= 0 || i >= c.IM - 1) && i >= -NGR && i <= c.IM - 1 + NGR) {
    after_xi(c, Q, i, j, k, q);
    return true;
  }
  load_q(c, Q, idx(c, i, j, k), q);
  return false;
}

__device__ inline void copy_node(const Consts& c, double* __restrict__ Q,
                                 double* __restrict__ prim, int d, int s, int pmask) {
#pragma unroll
  for (int n = 0; n < NEQ; n++) Q[(long)n * c.S + d] = Q[(long)n * c.S + s];
#pragma unroll
  for (int n = 0; n < 6; n++)
    if (pmask >> n & 1) prim[(long)n * c.S + d] = prim[(long)n * c.S + s];
}

// The shell: every node outside the updated box that a rule or a periodic wrap
// writes.  Along an axis it is w nodes deep on either side, from -e: the G
// ghosts of a periodic axis; otherwise the boundary node and the ghosts the
// rules write (e = NGR), or all of them if another axis is periodic (its wrap
// copies ghosts of this axis whether or not a rule wrote them).
struct Shell {
  int e, w[3];
  unsigned n[3];     // nodes of the zeta, eta and xi slabs
};

inline __host__ __device__ int outer(const Shell& s, int n) { return n + 2 * s.e; }
__device__ inline int layer(const Shell& s, int a, int n, int g) {
  return g < s.w[a] ? g - s.e : n + s.e - 2 * s.w[a] + g;
}

// A periodic ghost is the node at its coordinates wrapped on every periodic
// axis at once: what wrapping one axis after another over the full extent of
// the other two leaves, edges and corners included.  Its primitives are those
// of pmask.
// Launches bound it on small blocks and partial lines (the 8 doubles between
// two rows) on large ones.  A launch for each phase took 31 us on 193 x 61 x 33
// nodes without a periodic axis (five launches), 16 on 131 x 75 x 53 and 14.5 on
// 128 x 64 x 64 where xi alone is not; this one takes 9.5, 11 and 10.  RULES: some
// axis is not periodic.  Where all are, only the copies are left (128^3: 20 us;
// field by field, since all loads ahead of all stores take 23).
template <bool RULES>
__global__ void k_shell(Consts c, Shell sh, double* __restrict__ Q, double* __restrict__ prim,
                        const double* __restrict__ met, int pmask) {
  unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
  int i, j, k;
  if (t < sh.n[0]) {  // zeta slabs: full extent
    const unsigned X = outer(sh, c.IM), Y = outer(sh, c.JM);
    const unsigned r = t / X, g = r / Y;
    i = (int)(t - r * X) - sh.e;
    j = (int)(r - g * Y) - sh.e;
    k = layer(sh, 2, c.KM, (int)g);
  } else if ((t -= sh.n[0]) < sh.n[1]) {  // eta slabs: updated zeta
    const unsigned X = outer(sh, c.IM), Y = 2 * sh.w[1];
    const unsigned r = t / X, g = r / Y;
    i = (int)(t - r * X) - sh.e;
    j = layer(sh, 1, c.JM, (int)(r - g * Y));
    k = upd_lo(c, 2) + (int)g;
  } else if ((t -= sh.n[1]) < sh.n[2]) {  // xi slabs: updated eta and zeta
    const unsigned X = 2 * sh.w[0], Y = upd_hi(c, 1) - upd_lo(c, 1) + 1;
    const unsigned r = t / X, g = r / Y;
    i = layer(sh, 0, c.IM, (int)(t - r * X));
    j = upd_lo(c, 1) + (int)(r - g * Y);
    k = upd_lo(c, 2) + (int)g;
  } else {
    return;
  }
  const int d = idx(c, i, j, k);
  if (periodic(c, 0)) i = i < 0 ? i + c.IM : (i >= c.IM ? i - c.IM : i);
  if (periodic(c, 1)) j = j < 0 ? j + c.JM : (j >= c.JM ? j - c.JM : j);
  if (periodic(c, 2)) k = k < 0 ? k + c.KM : (k >= c.KM ? k - c.KM : k);
  const int s = idx(c, i, j, k);
  const bool image = s != d;
  if (!image) pmask = c.viscous ? 0x3F : 0x1F;

  // what the rules leave at the source, and what its primitives are those of
  const bool in_i = i >= 0 && i < c.IM, ref_eta = !periodic(c, 1);
  bool rule_q = false, rule_p = false, frozen = false;
  double q[NEQ];
  if (!RULES) {
    copy_node(c, Q, prim, d, s, pmask);
    return;
  }
  if (!periodic(c, 2) && (k <= 0 || k >= c.KM - 1)) {
    // zeta = 0 and KM-1 copy the next node, :417-492
    const bool zeta = in_i && j >= 0 && j < c.JM && k >= -NGR && k <= c.KM - 1 + NGR;
    if (!zeta && !image) return;
    if (zeta) before_zeta(c, Q, met, i, j, k <= 0 ? 1 : c.KM - 2, q);
    else load_q(c, Q, s, q);
    rule_q = rule_p = zeta;
  } else {
    rule_q = before_zeta(c, Q, met, i, j, k, q);
    // eta = 0 primitives whether or not a rule writes there, :354-376; those at
    // JM-1 and JM are of Q(JM-1), which stays as it is, :383-413
    const bool eta0 = ref_eta && in_i && j <= 0 && j >= -NGR;
    const bool etaN = ref_eta && in_i && j >= c.JM - 1 && j < c.JM - 1 + NGR;
    rule_p = rule_q || eta0 || etaN;
    if (!rule_p && !image) return;
    frozen = etaN;
  }
  if (!rule_p) {  // a periodic image of a node that no rule writes
    copy_node(c, Q, prim, d, s, pmask);
    return;
  }
  if (image || rule_q) {
#pragma unroll
    for (int n = 0; n < NEQ; n++) Q[(long)n * c.S + d] = q[n];
  }
  if (frozen) load_q(c, Q, idx(c, i, c.JM - 1, k), q);
  store_prim(c, q, prim, d, pmask);
}

}  // namespace

// Boundary rules and ghost fill for state Q whose interior primitives are
// already in b->prim (the fused stage writes them with the new state).
int launch_bc_only(cbns_block* b, double* Q, int pmask) {
  const Consts& c = b->c;
  if (pmask < 0) pmask = c.viscous ? 0x3F : 0x1F;
  Shell sh;
  sh.e = periodic(c, 0) || periodic(c, 1) || periodic(c, 2) ? G : NGR;
  for (int a = 0; a < 3; a++) sh.w[a] = periodic(c, a) ? G : sh.e + 1;
  const unsigned ny = upd_hi(c, 1) - upd_lo(c, 1) + 1, nz = upd_hi(c, 2) - upd_lo(c, 2) + 1;
  sh.n[0] = (unsigned)outer(sh, c.IM) * outer(sh, c.JM) * 2 * sh.w[2];
  sh.n[1] = (unsigned)outer(sh, c.IM) * 2 * sh.w[1] * nz;
  sh.n[2] = 2 * sh.w[0] * ny * nz;
  const unsigned cnt = sh.n[0] + sh.n[1] + sh.n[2];
  const bool rules = !(periodic(c, 0) && periodic(c, 1) && periodic(c, 2));
  (rules ? k_shell<true> : k_shell<false>)<<<(cnt + 255) / 256, 256, 0, b->stream>>>(
      c, sh, Q, b->prim, b->met, pmask);
  CBNS_HIP(b, hipGetLastError());
  return CBNS_OK;
}

int launch_bc_primitive(cbns_block* b, double* Q) {
  const Consts& c = b->c;
  Box box;
  for (int a = 0; a < 3; a++) {
    box.lo[a] = upd_lo(c, a);
    box.n[a] = upd_hi(c, a) - upd_lo(c, a) + 1;
  }
  k_prim_box<<<box_grid(box), box_block(), 0, b->stream>>>(c, box, Q, b->prim);
  CBNS_HIP(b, hipGetLastError());
  return launch_bc_only(b, Q);
}

}  // namespace cbns
