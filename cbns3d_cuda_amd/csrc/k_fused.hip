// k_fused.hip -- one RK3 stage (cbns_rk3_stage) as sweep kernels, or on small
// blocks (stage_shape) as one pass over tiles:
//
//   k_march<1>   lanes along i, each thread marches a chunk of nodes along
//                eta holding the 6-node stencil and the previous face flux in
//                registers: each node is loaded once per sweep and each face
//                is computed once.  Writes rhs = dF.
//   [viscous]    k_visc_fluxes (k_viscous.hip) writes the viscous node
//                fluxes before the marches; each march subtracts their
//                4th-order face values from its face fluxes (visc_face), so
//                the divergence needs no pass of its own
//   k_march<2>   the same march along zeta; at every node it also computes
//                the xi-face on its right, from the neighbouring lanes'
//                windows, and takes the left one from the lane below, all by
//                wavefront shuffles.  Adds dE + dG, divides by J and applies
//                the Shu-Osher stage combination, writing the stage output
//                and its primitives (the boundary pass then only fills
//                boundaries and ghosts).
//   k_tile4, k_tile16   the faces along all three axes of a tile of nodes and
//                its update, in place of both marches
//
// Node primitives for the Roe average are recomputed from Q (the
// primitive array holds exactly f(Q) at every node a face reads:
// boundary rules write Q first and derive the primitives from it).
#include <algorithm>

#include "cbns_internal.hpp"
#include "face_math.hpp"
#include "learned.hpp"

namespace cbns {

namespace {

constexpr int MARCH_X = 64;  // lanes along i
constexpr int MARCH_Y = 4;   // wavefronts of a workgroup
constexpr int CHUNK_MAX = 32;  // most nodes per thread along the march axis (march_cut)
#ifndef WPE_M
#define WPE_M 2  // waves per SIMD the march kernels are compiled for
#endif
#ifndef WPE_H
#define WPE_H 2  // the same for the hybrid marches (linear faces only; three
                 // waves per SIMD measured 2-4 % slower, four spilled)
#endif
// Halo lanes on either side of the nodes a march wavefront updates: none in
// the eta march, 3 in the zeta march, whose xi-stencils come from the
// neighbouring lanes.  (The zeta march has the xi-faces because its RK-update
// traffic overlaps the extra face work; the eta march alone is bound by its
// face arithmetic: +3 to +5 % of the FP64 step, +9 % of the FP32 step.)
template <int AX>
constexpr int march_halo() { return AX == 2 ? 3 : 0; }

// The lines of a march (rows along i of ni updated nodes, halo nodes on either
// side) are laid end to end and cut into wavefronts of 64 lanes; a wavefront
// updates the lanes between its own 3 halo lanes and repeats those of its
// neighbours.  A row's end then costs its 2 x 3 halo lanes instead of the rest
// of a wavefront: tiles of 58 nodes on each row took 5 wavefronts for 256
// nodes (4.5 here), 3 for 128 (2.3), 2 for 64 (1.2), and a last tile of one or
// two nodes (176 nodes) took the zeta march from 0.60 to 0.96 ms.
template <int AX>
long march_wavefronts(int ni, int rows) {
  constexpr int H = march_halo<AX>(), W = MARCH_X - 2 * H;
  return ((long)rows * (ni + 2 * H) - 2 * H + W - 1) / W;
}

template <class T>
__device__ __forceinline__ void load_q(const double* __restrict__ Q, long S, int o, T q[5]) {
#pragma unroll
  for (int n = 0; n < 5; n++) q[n] = (T)Q[n * S + o];
}

// The characteristic-WENO fluxes of a hybrid stage's troubled faces
// (k_weno_list): face m of the axis at slot[m], field n of slot s at
// flux[n * stride + s].
struct TroubledFaces {
  const int* slot;
  const double* flux;
  long stride;
};

// Viscous terms in face form.  The reference's viscous contribution is the
// 4th-order central difference (1/12, -2/3, 0, 2/3, -1/12) of each node flux
// along its axis (src/viscous_contribution_kernel.cu:44-67); that difference
// at node m equals h(m+1/2) - h(m-1/2) with the face value
// h(m+1/2) = 7/12 (v[m] + v[m+1]) - 1/12 (v[m-1] + v[m+2]), so the marches
// subtract h from the inviscid face fluxes they already difference: the eta
// march h of Fv, the zeta march h of Gv and, at its xi-faces, h of Ev.  The
// differences are taken on the reference's lines (offset by -1 in both
// transverse indices; 0 for the centred divergence).
template <class T>
__device__ __forceinline__ T visc_face(T vm1, T v0, T v1, T v2) {
  return fma(T(7.0 / 12.0), v0 + v1, -(T(1.0 / 12.0) * (vm1 + v2)));
}

// J grad xi of a face, from J and a metric term of its two nodes: the plain form
// rounds both products, the others node m+1's (LEFT) or node m's.
enum Rounding { BOTH, LEFT, RIGHT };
template <class F, bool HYB>
constexpr Rounding rounding(bool left) {
  return sizeof(F) == sizeof(double) && !HYB ? BOTH : (left ? LEFT : RIGHT);
}
__device__ __forceinline__ double face_normal(Rounding r, double m0, double j0, double m1,
                                              double j1) {
  return 0.5 * (r == BOTH ? m0 * j0 + m1 * j1
                          : (r == LEFT ? fma(m0, j0, m1 * j1) : fma(m1, j1, m0 * j0)));
}

// Face flux of the stage's form at face `face` (node offset).  HYB: the
// linear-weight reconstruction, replaced by the face's characteristic-WENO
// flux from tf where the face is troubled (its flag or a neighbour's along
// the axis: one-cell dilation); the marches hold no WENO arithmetic, so they
// run at the occupancy of the linear faces.  Slots read for faces outside
// the listed range (lanes whose faces no node uses) are clamped into tflux.
template <class F, bool HYB>
__device__ __forceinline__ void stage_face(const GasT<double>& g, const double q[6][5],
                                           double nx, double ny, double nz, bool troubled,
                                           const TroubledFaces& tf, int face, bool yz,
                                           double f[5], bool xi = false) {
  if constexpr (!HYB) {
    F e[5][5];
    stencil_diffs(q, e);
    if constexpr (sizeof(F) == sizeof(double)) {
      face_flux(g, e, q[2], q[3], nx, ny, nz, f);
    } else {
      F d[6][5];
      dev_from_diffs(e, d);
      face_flux_dev<true>(g, d, q[2], node_t<F>(g, q_to_side(g, q[2])), node_t<F>(g, q_to_side(g, q[3])),
                    nx, ny, nz, yz, f);
    }
    return;
  }
  face_linear<F>(g, q, nx, ny, nz, xi, f);
  if (troubled) {
    const long sl = min(max(tf.slot[face], 0), (int)(tf.stride - 1));
#pragma unroll
    for (int n = 0; n < 5; n++) f[n] = tf.flux[n * tf.stride + sl];
  }
}

struct StageArgs {
  double dt;
  const double* dtp;    // dt on the device (the folded time step) or null: use dt
  int stage;
  double* prim;         // primitives of the stage output (AX == 2)
  const double* Qn;     // level-n state (stages 2, 3)
  const double* Qin;    // stage input (stencil source)
  double* Qout;         // stage output
  double* rhs;          // dF
  const void* vf;       // viscous node fluxes Ev, Fv, Gv (12 fields of the face type) or null
  const uint8_t* flags; // troubled faces of the march axis (HYB)
  const uint8_t* flags_x;  // troubled xi-faces (HYB, AX == 2)
  int pmask;            // AX == 2: primitives to write (bit n: field n of rho, u, v, w, p, T)
  TroubledFaces tf;     // WENO fluxes of the march axis' troubled faces (HYB)
  TroubledFaces tf_x;   // and of the troubled xi-faces (HYB, AX == 2)
  int parts;            // chunks per CHUNK_MAX nodes of a line
};

// The Shu-Osher combination of node o = (i, j, k) from its flux differences
// along xi (de), eta (df) and zeta (dg), its state qin, level-n state qn and
// Jacobian; with `own` also its stores.  WRAP: the periodic ghosts too.
template <bool WRAP>
__device__ __forceinline__ void finish_node(const Consts& c, const StageArgs& sa,
                                            const GasT<double>& g, double dt, int i, int j, int k,
                                            int o, bool own, const double de[5],
                                            const double df[5], const double dg[5],
                                            const double qin[5], const double qn[5], double jac) {
  const long S = c.S;
  const double inv_j = fast_rcp(jac);
  double out[5];
#pragma unroll
  for (int n = 0; n < 5; n++) {
    const double euler = fma(-dt, (df[n] + dg[n] + de[n]) * inv_j, qin[n]);
    if (sa.stage == 1) out[n] = euler;
    else if (sa.stage == 2) out[n] = fma(0.25, euler, 0.75 * qn[n]);
    else out[n] = fma(2.0, euler, qn[n]) * (1.0 / 3.0);
  }
  if (!own) return;
  // primitives of the new state (src/primitive_bc_kernel.cu:63-76)
  double rr, uu, vv, ww, pp;
  q_to_prim(g, out, rr, uu, vv, ww, pp);
  const double tt = c.gM2 * pp * fast_rcp(rr);
  // all stores of a node together, after its arithmetic: with the state's
  // ahead of the primitives the 256^3 zeta march took 1610 us for 1531 (hybrid
  // 1203 for 1165)
  const auto put = [&](int d) {
#pragma unroll
    for (int n = 0; n < 5; n++) sa.Qout[n * S + d] = out[n];
    if (sa.pmask & 1) sa.prim[d] = rr;
    if (sa.pmask & 2) sa.prim[S + d] = uu;
    if (sa.pmask & 4) sa.prim[2 * S + d] = vv;
    if (sa.pmask & 8) sa.prim[3 * S + d] = ww;
    if (sa.pmask & 16) sa.prim[4 * S + d] = pp;
    if (sa.pmask & 32) sa.prim[5 * S + d] = tt;
  };
  put(o);
  if (WRAP) {
    // the node's images in the ghosts: along each axis at whose end it
    // lies, and along each pair and all three of them
    const int di = i < G ? c.IM : (i >= c.IM - G ? -c.IM : 0);
    const int dj = j < G ? c.JM : (j >= c.JM - G ? -c.JM : 0);
    const int dk = k < G ? c.KM : (k >= c.KM - G ? -c.KM : 0);
    if (di | dj | dk) {
#pragma unroll 1
      for (int im = 1; im < 8; im++) {
        const int ex = im & 1 ? di : 0, ey = im & 2 ? dj : 0, ez = im & 4 ? dk : 0;
        if ((im & 1 && !ex) || (im & 2 && !ey) || (im & 4 && !ez)) continue;
        put(o + ex + ey * c.PX + ez * c.PXY);
      }
    }
  }
}

// AX = 1: march along eta, rhs = dF.  AX = 2: march along zeta with the
// xi-faces, finish.
template <int AX, class F, bool HYB>
__global__ void __launch_bounds__(MARCH_X * MARCH_Y)
__attribute__((amdgpu_waves_per_eu(HYB ? WPE_H : WPE_M, HYB ? WPE_H : WPE_M)))
k_march(Consts c, StageArgs sa, const double* __restrict__ met) {
  constexpr bool XI = AX == 2;
  // the update's time step; a NaN step (non-physical state) leaves the
  // stage output unwritten, and the caller reports it
  const double dt = AX == 2 && sa.dtp ? *sa.dtp : sa.dt;
  if (AX == 2 && !(dt == dt)) return;
  const int ax_t = AX == 1 ? 2 : 1;  // transverse axis other than i
  const int lane = threadIdx.x;
  // the workgroup's wavefronts follow each other along the lines, so each
  // step of the march reads whole rows of the fields (against wavefronts on
  // adjacent lines -9 % for the FP64 eta march, -12 % FP32)
  constexpr int H = march_halo<AX>(), W = MARCH_X - 2 * H;
  const int ni = upd_hi(c, 0) - upd_lo(c, 0) + 1;
  const unsigned slot = (blockIdx.x * blockDim.y + threadIdx.y) * W + lane;
  const unsigned row = slot / (unsigned)(ni + 2 * H);
  const int at = (int)(slot - row * (unsigned)(ni + 2 * H)) - H;  // node of the row's updated ones
  const int i = upd_lo(c, 0) + at;
  const int t = upd_lo(c, ax_t) + (int)row;
  if (t > upd_hi(c, ax_t)) return;
  const bool own = lane >= H && lane < H + W && at >= 0 && at < ni;
  const int mlo = upd_lo(c, AX), mhi = upd_hi(c, AX);
  const int mseg = mlo + CHUNK_MAX * (int)blockIdx.z, part = blockIdx.y;
  const int m0 = mseg + CHUNK_MAX * part / sa.parts;
  if (m0 > mhi) return;
  const int m1 = min(mseg + CHUNK_MAX * (part + 1) / sa.parts, mhi + 1);
  const long S = c.S;
  const int st = AX == 1 ? c.PX : c.PXY;
  const int base = AX == 1 ? idx(c, i, 0, t) : idx(c, i, t, 0);  // node m at base + m*st
  const double* __restrict__ Q = sa.Qin;
  const double* __restrict__ nX = met + (3 * AX + 0) * S;
  const double* __restrict__ nY = met + (3 * AX + 1) * S;
  const double* __restrict__ nZ = met + (3 * AX + 2) * S;
  const double* __restrict__ J = met + JAC * S;
  const GasT<double> g{c.gamma, c.gam1, c.gam1_inv};

  double q[6][5];  // nodes m-2 .. m+3 for the face m+1/2, of the pass before
#pragma unroll
  for (int s = 0; s < 6; s++) load_q(Q, S, base + (m0 - 3 + s) * st, q[s]);
  // J grad xi_AX at the face's two nodes
  int o = base + (m0 - 1) * st;
  double jb = J[o + st];
  // metric terms of the face's right node; where both products of a face normal
  // are rounded, with J, since they are the next face's left ones
  constexpr bool PROD = rounding<F, HYB>(false) == BOTH;
  double mx = nX[o + st], my = nY[o + st], mz = nZ[o + st];
  if (PROD) { mx *= jb; my *= jb; mz *= jb; }
  const auto normal = [&](Rounding r, double a, double ja, double m, double jm) {
    return PROD ? 0.5 * (a + m) : face_normal(r, a, ja, m, jm);
  };
  double fprev[5];
  // troubled flags of faces m-1, m, m+1 (face m between nodes m and m+1)
  const uint8_t* __restrict__ fl = sa.flags;
  uint8_t t0 = 0, t1 = 0, t2 = 0;
  if (HYB) {
    t0 = fl[base + (m0 - 2) * st];
    t1 = fl[base + (m0 - 1) * st];
    t2 = fl[base + m0 * st];
  }
  // Precision form (float faces, not hybrid): the sweep carries the float
  // differences e[k] = q[k+1] - q[k] of the window's nodes and the Roe
  // inputs of nodes m (nl) and m+1 (nr), each formed once per node, instead
  // of five double differences and two double face states per face.
  constexpr bool DC = sizeof(F) != sizeof(double) && !HYB;
  F e[5][5];
  NodeT<F> nl{}, nr{};
  if constexpr (DC) {
#pragma unroll
    for (int k = 0; k < 5; k++)
#pragma unroll
      for (int n = 0; n < 5; n++) e[k][n] = (F)(q[k + 1][n] - q[k][n]);
    nl = node_t<F>(g, q_to_side(g, q[2]));
    nr = node_t<F>(g, q_to_side(g, q[3]));
  }
  // the face left of the chunk's first node
  {
    const double ja = J[o];
    double ax = nX[o], ay = nY[o], az = nZ[o];
    if (PROD) { ax *= ja; ay *= ja; az *= ja; }
    // (the first of a line's CHUNK_MAX nodes rounds the other product)
    const bool first = part == 0;
    const Rounding r = rounding<F, HYB>(first);
    const double sx = normal(r, ax, ja, mx, jb), sy = normal(r, ay, ja, my, jb);
    const double sz = normal(r, az, ja, mz, jb);
    if constexpr (DC) {
      F d[6][5];
      dev_from_diffs(e, d);
      face_flux_dev<true>(g, d, q[2], nl, nr, sx, sy, sz, AX == 1 && !first, fprev);
    } else {
      stage_face<F, HYB>(g, q, sx, sy, sz, t0 | t1 | t2, sa.tf, o, AX == 1 && !first,
                         fprev);
    }
  }
  // viscous node flux of the march axis (Fv or Gv) on its offset line,
  // nodes m-1, m, m+1 of the face m+1/2 (visc_face); Ev of the xi-faces on
  // the zeta march's offset line
  const bool VIS = sa.vf != nullptr;
  const int vsh = c.visc_centered ? 0 : -1;
  const F* __restrict__ ve = static_cast<const F*>(sa.vf);
  const F* __restrict__ va = VIS ? ve + (long)(4 * AX) * S : nullptr;
  const int vbase = AX == 1 ? idx(c, i + vsh, 0, t + vsh) : idx(c, i + vsh, t + vsh, 0);
  const int ebase = idx(c, i, t + vsh, vsh);  // Ev of node m at ebase + m*st (XI)
  // The window (nodes m-1, m, m+1) is held in registers, or, in the FP64
  // zeta march, whose registers the xi-faces take, in a per-thread LDS ring
  // (slot vr holds node m-1, the next two slots the others; no thread reads
  // another's entries, so no barrier).
  constexpr bool VRING = AX == 2 && sizeof(F) == sizeof(double) && !HYB;
  constexpr int RR = VRING ? MARCH_Y : 1;
  __shared__ F vring[VRING ? 3 : 1][4][RR][VRING ? MARCH_X : 1];
  const int ty = VRING ? threadIdx.y : 0, tl = VRING ? lane : 0;
  F vw[3][4];
  int vr = 0;
  if (VIS) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      F w[4];
#pragma unroll
      for (int s = 0; s < 4; s++) w[s] = va[e * S + vbase + (m0 - 2 + s) * st];
      fprev[e + 1] -= (double)visc_face(w[0], w[1], w[2], w[3]);
#pragma unroll
      for (int s = 0; s < 3; s++) {
        if constexpr (VRING) vring[s][e][ty][tl] = w[s + 1];
        else vw[s][e] = w[s + 1];
      }
    }
  }
  // eta march: the next node's state and the next face's metrics are
  // fetched one iteration ahead (nodes up to mhi + 4 lie in the ghosted
  // array): -1.6 % for the FP64 eta march; the hybrid's eta march, bound by
  // memory latency at its register count, ran 2 % slower with it
  constexpr bool PF = AX == 1 && !HYB;
  double qpf[5] = {0, 0, 0, 0, 0}, jpf = 0.0, xpf = 0.0, ypf = 0.0, zpf = 0.0;
  if constexpr (PF) {
    load_q(Q, S, base + (m0 + 3) * st, qpf);
    const int on = base + (m0 + 1) * st;
    jpf = J[on]; xpf = nX[on]; ypf = nY[on]; zpf = nZ[on];
  }
  for (int m = m0; m < m1; m++) {
    // shift the window by one node
#pragma unroll
    for (int s = 0; s < 5; s++)
#pragma unroll
      for (int n = 0; n < 5; n++) q[s][n] = q[s + 1][n];
    o = base + m * st;
    if constexpr (PF) {
#pragma unroll
      for (int n = 0; n < 5; n++) q[5][n] = qpf[n];
      load_q(Q, S, o + 4 * st, qpf);
    } else {
      load_q(Q, S, o + 3 * st, q[5]);
    }
    F vn[4], ev[4];  // viscous flux of node m+2 along the axis; Ev of node m (XI)
    if (VIS) {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        vn[e] = va[e * S + vbase + (m + 2) * st];
        if constexpr (XI) ev[e] = ve[e * S + ebase + m * st];
      }
    }
    if constexpr (DC) {
#pragma unroll
      for (int n = 0; n < 5; n++) {
#pragma unroll
        for (int k = 0; k < 4; k++) e[k][n] = e[k + 1][n];
        e[4][n] = (F)(q[5][n] - q[4][n]);
      }
      nl = nr;
      nr = node_t<F>(g, q_to_side(g, q[3]));
    }
    const double jo = jb;  // J at node m, loaded as the previous face's right node
    // the zeta sweep's update operands are fetched before the face work so
    // their latency overlaps it; with FP64 faces and the xi-faces in this
    // march they are fetched where they are used (hoisted they would push
    // the kernel past 256 VGPRs)
    constexpr bool HOIST = AX == 2 && sizeof(F) != sizeof(double) && !HYB;
    double rin[5], qnv[5];
    if (HOIST) {
#pragma unroll
      for (int n = 0; n < 5; n++) {
        rin[n] = sa.rhs[n * S + o];
        qnv[n] = sa.stage > 1 ? sa.Qn[n * S + o] : 0.0;
      }
    }
    const double ax = mx, ay = my, az = mz;
    if constexpr (PF) {
      jb = jpf;
      mx = xpf; my = ypf; mz = zpf;
      const int on = o + 2 * st;
      jpf = J[on]; xpf = nX[on]; ypf = nY[on]; zpf = nZ[on];
    } else {
      jb = J[o + st];
      mx = nX[o + st]; my = nY[o + st]; mz = nZ[o + st];
    }
    if (PROD) { mx *= jb; my *= jb; mz *= jb; }
    double f[5], fxr[5];
    double xmx = 0.0, xmy = 0.0, xmz = 0.0;  // xi metrics of node m
    if (XI) {
      xmx = met[XI_X * S + o];
      xmy = met[XI_Y * S + o];
      xmz = met[XI_Z * S + o];
    }
    if (XI) {
      // the xi-face between node (i, m) and (i+1, m): stencil i-2 .. i+3
      // (every lane takes part in the shuffles)
      double qx[2][5];
      if constexpr (HYB) {
        // linear xi-face from the neighbouring lanes' values, one
        // component at a time (six values live, not the whole stencil)
#pragma unroll
        for (int n = 0; n < 5; n++) {
          const double v = q[2][n];
          linear_lr<F>(__shfl(v, lane - 2), __shfl(v, lane - 1), v, __shfl(v, lane + 1),
                       __shfl(v, lane + 2), __shfl(v, lane + 3), qx[0][n], qx[1][n]);
        }
      }
      const double jx = xmx * jo, jy = xmy * jo, jz = xmz * jo;
      // (the neighbour's product is rounded: face_normal with j1 = 1)
      constexpr Rounding rx = rounding<F, HYB>(true);
      const double nxx = face_normal(rx, xmx, jo, __shfl(jx, lane + 1), 1.0);
      const double nxy = face_normal(rx, xmy, jo, __shfl(jy, lane + 1), 1.0);
      const double nxz = face_normal(rx, xmz, jo, __shfl(jz, lane + 1), 1.0);
      if constexpr (!HYB) {
        // lane+1's node, the difference to it and those of lanes -2..+2 (and,
        // in float, lane+1's Roe inputs), by shuffles
        double qr[5];
        F ec[5][5];
#pragma unroll
        for (int n = 0; n < 5; n++) {
          qr[n] = __shfl(q[2][n], lane + 1);
          const F ex = (F)(qr[n] - q[2][n]);
          ec[0][n] = __shfl(ex, lane - 2);
          ec[1][n] = __shfl(ex, lane - 1);
          ec[2][n] = ex;
          ec[3][n] = __shfl(ex, lane + 1);
          ec[4][n] = __shfl(ex, lane + 2);
        }
        if constexpr (DC) {
          const NodeT<F> xr{__shfl(nl.r, lane + 1), __shfl(nl.u, lane + 1), __shfl(nl.v, lane + 1),
                            __shfl(nl.w, lane + 1), __shfl(nl.H, lane + 1)};
          F dx[6][5];
          dev_from_diffs(ec, dx);
          face_flux_dev<true>(g, dx, q[2], nl, xr, nxx, nxy, nxz, false, fxr);
        } else {
          face_flux(g, ec, q[2], qr, nxx, nxy, nxz, fxr);
        }
      } else {
        const int fo = sa.flags_x[o];
        const bool tx = (__shfl(fo, lane - 1) | fo | __shfl(fo, lane + 1)) != 0;
        // qx[0], qx[1]: the reconstructed left and right states
        lf_flux(g, q_to_side(g, qx[1]), q_to_side(g, qx[0]), nxx, nxy, nxz, fxr);
        if (tx) {
          const long sl = min(max(sa.tf_x.slot[o], 0), (int)(sa.tf_x.stride - 1));
#pragma unroll
          for (int n = 0; n < 5; n++) fxr[n] = sa.tf_x.flux[n * sa.tf_x.stride + sl];
        }
      }
      if (VIS) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const F v = ev[e];
          fxr[e + 1] -= (double)visc_face(__shfl(v, lane - 1), v, __shfl(v, lane + 1),
                                          __shfl(v, lane + 2));
        }
      }
    }
    constexpr Rounding rnd = rounding<F, HYB>(false);
    const double sx = normal(rnd, ax, jo, mx, jb), sy = normal(rnd, ay, jo, my, jb);
    const double sz = normal(rnd, az, jo, mz, jb);
    if (HYB) {
      t0 = t1;
      t1 = t2;
      t2 = fl[o + st];
    }
    if constexpr (DC) {
      F d[6][5];
      dev_from_diffs(e, d);
      face_flux_dev<true>(g, d, q[2], nl, nr, sx, sy, sz, AX == 1, f);
    } else {
      stage_face<F, HYB>(g, q, sx, sy, sz, t0 | t1 | t2, sa.tf, o, AX == 1, f);
    }
    if (VIS) {
      const int s0 = vr, s1 = vr == 2 ? 0 : vr + 1, s2 = vr == 0 ? 2 : vr - 1;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        if constexpr (VRING) {
          f[e + 1] -= (double)visc_face(vring[s0][e][ty][tl], vring[s1][e][ty][tl],
                                        vring[s2][e][ty][tl], vn[e]);
          vring[s0][e][ty][tl] = vn[e];  // node m+2 takes node m-1's slot
        } else {
          f[e + 1] -= (double)visc_face(vw[0][e], vw[1][e], vw[2][e], vn[e]);
          vw[0][e] = vw[1][e];
          vw[1][e] = vw[2][e];
          vw[2][e] = vn[e];
        }
      }
      vr = s1;
    }
    if (AX == 1) {
#pragma unroll
      for (int n = 0; n < 5; n++) sa.rhs[n * S + o] = f[n] - fprev[n];
    } else {
      double dfx[5];  // xi-face difference
#pragma unroll
      for (int n = 0; n < 5; n++) dfx[n] = fxr[n] - __shfl_up(fxr[n], 1);
      if (!HOIST) {
#pragma unroll
        for (int n = 0; n < 5; n++) {
          rin[n] = sa.rhs[n * S + o];
          qnv[n] = sa.stage > 1 ? sa.Qn[n * S + o] : 0.0;
        }
      }
      double dg[5];
#pragma unroll
      for (int n = 0; n < 5; n++) dg[n] = f[n] - fprev[n];
      finish_node<false>(c, sa, g, dt, i, t, m, o, own, dfx, rin, dg, q[2], qnv, jo);
    }
#pragma unroll
    for (int n = 0; n < 5; n++) fprev[n] = f[n];
  }
}

// A whole stage's fluxes and update in one launch, over tiles of nodes: the
// workgroup loads the tile's nodes and the three on either side along each axis
// into LDS, forms every face of the tile, one a lane, into LDS too, and updates
// the tile's nodes from them.  The faces between tiles are formed twice, but no
// lane waits for another's faces and dF stays out of memory, so blocks that are
// small for the marches run this way (stage_shape).  A face's operations are the
// marches', so the stage has their bits (for that it also rounds the face at every
// 32nd node as the march that opens a chunk of CHUNK_MAX there: first_on_line).

// The tile of this workgroup (X x Y x Z nodes from lo on, nx x ny x nz of them in
// the block); false past the last.  Workgroups go to the 8 XCDs in turn; each XCD
// takes a run of neighbouring tiles, whose halos its L2 then holds (128^3 viscous
// step 1739 -> 1566 us, 64^3 259 -> 242).
constexpr int TILE_XCDS = 8;
constexpr int TILE_TPB = 256;
template <int X, int Y, int Z>
__device__ __forceinline__ bool tile_origin(const int hi[3], int lo[3], int n[3]) {
  const unsigned tx = (unsigned)(hi[0] - lo[0] + X) / X, ty = (unsigned)(hi[1] - lo[1] + Y) / Y;
  const unsigned nt = tx * ty * ((unsigned)(hi[2] - lo[2] + Z) / Z);
  const unsigned t =
      blockIdx.x % TILE_XCDS * ((nt + TILE_XCDS - 1) / TILE_XCDS) + blockIdx.x / TILE_XCDS;
  if (t >= nt) return false;
  const unsigned r = t / tx, q = r / ty;
  lo[0] += (int)(t - r * tx) * X;
  lo[1] += (int)(r - q * ty) * Y;
  lo[2] += (int)q * Z;
  n[0] = min(X, hi[0] - lo[0] + 1);
  n[1] = min(Y, hi[1] - lo[1] + 1);
  n[2] = min(Z, hi[2] - lo[2] + 1);
  return true;
}

// Field values by byte offset (below 2^32: stage_shape keeps to small blocks).
template <class T>
__device__ __forceinline__ T at_byte(const T* __restrict__ f, unsigned byte) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(f) + byte);
}

// What a tile's face takes from memory: metrics of its two nodes (o and o + gs,
// gs the stride of its axis a) and the viscous fluxes around it.
template <class F>
struct FaceIn {
  double j[2], m[3][2];
  F v[4][4];
};
template <class F>
__device__ __forceinline__ void fetch_face(const Consts& c, const StageArgs& sa,
                                           const double* __restrict__ met, int a, int gs, int o,
                                           FaceIn<F>& w) {
  const long S = c.S;
  const unsigned o8 = 8u * (unsigned)o, g8 = 8u * (unsigned)gs;
  const double* __restrict__ nm = met + 3 * a * S;
#pragma unroll
  for (int s = 0; s < 2; s++) {
    w.j[s] = at_byte(met + JAC * S, o8 + s * g8);
#pragma unroll
    for (int d = 0; d < 3; d++) w.m[d][s] = at_byte(nm + d * S, o8 + s * g8);
  }
  if (sa.vf) {
    const int vsh = c.visc_centered ? 0 : -1;
    const F* __restrict__ v = static_cast<const F*>(sa.vf) + 4 * a * S;
    const int vo = o + vsh * (1 + c.PX + c.PXY - gs);
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
      for (int s = 0; s < 4; s++)
        w.v[e][s] = at_byte(v + e * S, (unsigned)sizeof(F) * (unsigned)(vo + (s - 1) * gs));
  }
}
// Whether a tile's lines along axis a begin where a march's CHUNK_MAX nodes do.
__device__ __forceinline__ bool first_on_line(const Consts& c, const int lo[3], int a) {
  return (a == 1 ? lo[1] - upd_lo(c, 1) : lo[2] - upd_lo(c, 2)) % CHUNK_MAX == 0;
}
// The face's flux from its stencil q and `w`.  first: the face that opens a
// march's CHUNK_MAX nodes.
template <class F, bool HYB>
__device__ __forceinline__ void tile_face(const Consts& c, const StageArgs& sa,
                                          const GasT<double>& g, const double q[6][5],
                                          const FaceIn<F>& w, int a, bool first, int gs, int o,
                                          double f[5]) {
  // the products that the marches round
  const bool left = a == 0 || first;
  double nv[3];
#pragma unroll
  for (int d = 0; d < 3; d++)
    nv[d] = face_normal(rounding<F, HYB>(left), w.m[d][0], w.j[0], w.m[d][1], w.j[1]);
  bool troubled = false;
  TroubledFaces tf = sa.tf_x;
  if (HYB) {
    const uint8_t* __restrict__ fl = sa.flags_x + (long)a * c.S;
    troubled = (fl[o - gs] | fl[o] | fl[o + gs]) != 0;
    tf.slot += (long)a * c.S;
  }
  stage_face<F, HYB>(g, q, nv[0], nv[1], nv[2], troubled, tf, o, a == 1 && !left, f,
                     a == 0);
  if (sa.vf) {
#pragma unroll
    for (int e = 0; e < 4; e++)
      f[e + 1] -= (double)visc_face(w.v[e][0], w.v[e][1], w.v[e][2], w.v[e][3]);
  }
}

// Tiles of 4 x 4 x 4 nodes: 240 faces for 256 lanes, a single face long.
template <class F, bool HYB, bool WRAP>
__global__ void __launch_bounds__(TILE_TPB) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_tile4(Consts c, StageArgs sa, const double* __restrict__ met) {
  constexpr int X = 4, N = X * X * X, L = X * X;  // nodes; lines of an axis
  // nodes in LDS: the tile's, then each axis' halo, three positions below the
  // tile and three above, a position of all lines together
  constexpr int NQ = N + 3 * 6 * L, NF = 3 * (X + 1) * L;
  __shared__ double sq[5 * NQ], sf[5 * NF];
  const double dt = sa.dtp ? *sa.dtp : sa.dt;
  if (!(dt == dt)) return;
  const long S = c.S;
  const int tid = threadIdx.x;
  const int hi[3] = {upd_hi(c, 0), upd_hi(c, 1), upd_hi(c, 2)};
  int lo[3] = {upd_lo(c, 0), upd_lo(c, 1), upd_lo(c, 2)}, nn[3];
  if (!tile_origin<X, X, X>(hi, lo, nn)) return;
#pragma unroll
  for (int r = 0; r < (NQ + TILE_TPB - 1) / TILE_TPB; r++) {
    const int t = tid + r * TILE_TPB;
    int p[3];
    if (t < N) {
      p[0] = t % X; p[1] = t / X % X; p[2] = t / L;
    } else {
      const int h = t - N, a = h / (6 * L), s = h / L % 6, l = h % L;
      const int e = s < 3 ? s - 3 : s - 3 + X, u = l % X, v = l / X;
      p[0] = a == 0 ? e : u;
      p[1] = a == 1 ? e : (a == 0 ? u : v);
      p[2] = a == 2 ? e : v;
    }
    // nodes past the stencils of the last updated ones are read by no face
    const int o = idx(c, min(lo[0] + p[0], hi[0] + 3), min(lo[1] + p[1], hi[1] + 3),
                      min(lo[2] + p[2], hi[2] + 3));
    if (t < NQ) {
#pragma unroll
      for (int n = 0; n < 5; n++) sq[n * NQ + t] = sa.Qin[n * S + o];
    }
  }
  // the lane's face, between positions p - 1 and p of line (u, v) along axis a;
  // its node o at p - 1
  const GasT<double> g{c.gamma, c.gam1, c.gam1_inv};
  const int a = tid / ((X + 1) * L), p = tid / L % (X + 1), u = tid % X, v = tid / X % X;
  const int x = a == 0 ? p - 1 : u, y = a == 1 ? p - 1 : (a == 0 ? u : v), z = a == 2 ? p - 1 : v;
  const bool has = tid < NF && x < nn[0] && y < nn[1] && z < nn[2];
  const int o = idx(c, lo[0] + x, lo[1] + y, lo[2] + z);
  const int gs = a == 0 ? 1 : (a == 1 ? c.PX : c.PXY);
  FaceIn<F> w;
  if (has) fetch_face<F>(c, sa, met, a, gs, o, w);
  __syncthreads();
  if (has) {
    const int st = a == 0 ? 1 : (a == 1 ? X : L);
    const int core = a == 0 ? X * u + L * v : (a == 1 ? u + L * v : u + X * v);
    const int halo = N + 6 * L * a + tid % L;
    double q[6][5], f[5];
#pragma unroll
    for (int s = 0; s < 6; s++) {
      const int pos = p - 3 + s;
      const int at = pos < 0 ? halo + (pos + 3) * L : (pos >= X ? halo + (pos - X + 3) * L
                                                                : core + pos * st);
#pragma unroll
      for (int n = 0; n < 5; n++) q[s][n] = sq[n * NQ + at];
    }
    tile_face<F, HYB>(c, sa, g, q, w, a, p == 0 && first_on_line(c, lo, a), gs, o, f);
#pragma unroll
    for (int n = 0; n < 5; n++) sf[n * NF + tid] = f[n];
  }
  __syncthreads();
  if (tid < N) {
    const int x = tid % X, y = tid / X % X, z = tid / L;
    if (x >= nn[0] || y >= nn[1] || z >= nn[2]) return;
    const int i = lo[0] + x, j = lo[1] + y, k = lo[2] + z, o = idx(c, i, j, k);
    // face p of line (u, v) of axis a at (5 a + p) L + u + X v
    const int fe = x * L + y + X * z, ff = (5 + y) * L + x + X * z, fg = (10 + z) * L + x + X * y;
    double de[5], df[5], dg[5], qin[5], qn[5];
#pragma unroll
    for (int n = 0; n < 5; n++) {
      qn[n] = sa.stage > 1 ? sa.Qn[n * S + o] : 0.0;
      qin[n] = sq[n * NQ + tid];
      const double* s = sf + n * NF;
      de[n] = s[fe + L] - s[fe];
      df[n] = s[ff + L] - s[ff];
      dg[n] = s[fg + L] - s[fg];
    }
    finish_node<WRAP>(c, sa, g, dt, i, j, k, o, true, de, df, dg, qin, qn, met[JAC * S + o]);
  }
}

// Tiles of 16 x 4 x 4 nodes, a node a lane for the update.  Their faces are
// handed to the wavefronts by position: the 64 of one position along eta or zeta,
// 4 lines of 16 along xi, and the 17th of the 16 lines, so the axis, and along
// eta and zeta the position too, are the wavefront's and cost the lanes no
// arithmetic.
template <class F, bool HYB, bool WRAP>
__global__ void __launch_bounds__(TILE_TPB) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_tile16(Consts c, StageArgs sa, const double* __restrict__ met) {
  constexpr int X = 16, Y = 4, R = X + 6;  // a row's nodes in LDS, xi-halo included
  // nodes in LDS: the rows (y + 4 z), then 3 + 3 positions along eta, then along
  // zeta, 64 nodes each
  constexpr int HY = R * Y * Y, HZ = HY + 6 * 64, NQ = HZ + 6 * 64;
  constexpr int FZ = (Y + 1) * 64, FX = 2 * FZ, NF = FX + (X + 1) * Y * Y;
  constexpr int CHUNKS = 15;
  __shared__ double sq[5 * NQ], sf[5 * NF];
  const double dt = sa.dtp ? *sa.dtp : sa.dt;
  if (!(dt == dt)) return;
  const long S = c.S;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hi[3] = {upd_hi(c, 0), upd_hi(c, 1), upd_hi(c, 2)};
  int lo[3] = {upd_lo(c, 0), upd_lo(c, 1), upd_lo(c, 2)}, nn[3];
  if (!tile_origin<X, Y, Y>(hi, lo, nn)) return;
  // nodes past the stencils of the last updated ones are read by no face
  const auto node = [&](int x, int y, int z) {
    return idx(c, min(lo[0] + x, hi[0] + 3), min(lo[1] + y, hi[1] + 3), min(lo[2] + z, hi[2] + 3));
  };
  const int lx = lane % X, lv = lane / X;
  {
    double h[5][5];
    int to[5];
#pragma unroll
    for (int r = 0; r < 5; r++) {
      int x, y, z;
      if (r < 2) {
        const int t = tid + r * TILE_TPB;
        x = t % R - 3; y = t / R % Y; z = t / (R * Y);
        to[r] = t;
      } else {
        const int p = 4 * (r - 2) + wv, s = p % 6, e = s < 3 ? s - 3 : s - 3 + Y;
        x = lx;
        y = p < 6 ? e : lv;
        z = p < 6 ? lv : e;
        to[r] = HY + 64 * p + lane;
      }
      const unsigned o8 = 8u * (unsigned)node(x, y, z);
#pragma unroll
      for (int n = 0; n < 5; n++) h[r][n] = at_byte(sa.Qin + n * S, o8);
    }
#pragma unroll
    for (int r = 0; r < 5; r++)
#pragma unroll
      for (int n = 0; n < 5; n++)
        if (r != 1 || to[r] < HY) sq[n * NQ + to[r]] = h[r][n];
  }
  const GasT<double> g{c.gamma, c.gam1, c.gam1_inv};
  __syncthreads();
#pragma unroll 1
  for (int ch = wv; ch < CHUNKS; ch += TILE_TPB / 64) {
    // chunk 0-4: eta, position ch; 5-9: zeta, position ch - 5; 10-13: xi, lines of
    // plane ch - 10, positions 0-15; 14: xi, position 16
    const int a = ch < 5 ? 1 : (ch < 10 ? 2 : 0);
    const int p = a == 1 ? ch : ch - 5;  // eta and zeta: the faces' position
    int x = lx, y = lv, z = lv;
    if (a == 1) y = p - 1;
    else if (a == 2) z = p - 1;
    else if (ch < 14) { x = lx - 1; z = ch - 10; }
    else { x = X - 1; y = lane % Y; z = lane / Y; }
    if (x >= nn[0] || y >= nn[1] || z >= nn[2]) continue;
    const int gs = a == 0 ? 1 : (a == 1 ? c.PX : c.PXY);
    const int o = idx(c, lo[0] + x, lo[1] + y, lo[2] + z);
    FaceIn<F> w;
    fetch_face<F>(c, sa, met, a, gs, o, w);
    // position s of the stencil: in the rows at row + s (xi) or row + pos * st, or
    // in the halo of the axis
    const int row = a == 1 ? lx + 3 + R * Y * lv
                           : (a == 2 ? lx + 3 + R * lv : x + 1 + R * (y + Y * z));
    const int halo = (a == 1 ? HY : HZ) + lane, st = a == 1 ? R : R * Y;
    double q[6][5], f[5];
#pragma unroll
    for (int s = 0; s < 6; s++) {
      const int pos = p - 3 + s;
      const int at = a == 0 ? row + s
                            : ((unsigned)pos < (unsigned)Y
                                   ? row + pos * st
                                   : halo + 64 * (pos < 0 ? pos + 3 : pos - Y + 3));
#pragma unroll
      for (int n = 0; n < 5; n++) q[s][n] = sq[n * NQ + at];
    }
    tile_face<F, HYB>(c, sa, g, q, w, a, p == 0 && first_on_line(c, lo, a), gs, o, f);
    const int to = a == 0 ? FX + (X + 1) * (y + Y * z) + x + 1 : 64 * ch + lane;
#pragma unroll
    for (int n = 0; n < 5; n++) sf[n * NF + to] = f[n];
  }
  __syncthreads();
  const int x = lx, y = lv, z = wv;
  if (x >= nn[0] || y >= nn[1] || z >= nn[2]) return;
  const int i = lo[0] + x, j = lo[1] + y, k = lo[2] + z, o = idx(c, i, j, k);
  const int fe = FX + (X + 1) * (y + Y * z) + x, ff = 64 * y + x + X * z, fg = FZ + 64 * z + x + X * y;
  double de[5], df[5], dg[5], qin[5], qn[5];
#pragma unroll
  for (int n = 0; n < 5; n++) {
    qn[n] = sa.stage > 1 ? sa.Qn[n * S + o] : 0.0;
    qin[n] = sq[n * NQ + x + 3 + R * (y + Y * z)];
    const double* s = sf + n * NF;
    de[n] = s[fe + 1] - s[fe];
    df[n] = s[ff + 64] - s[ff];
    dg[n] = s[fg + 64] - s[fg];
  }
  finish_node<WRAP>(c, sa, g, dt, i, j, k, o, true, de, df, dg, qin, qn, met[JAC * S + o]);
}

// The troubled faces of axis AX in the flux kernels' face range fb: face m
// is troubled when its flag or a neighbour's along AX is set (the same
// one-cell dilation the marches apply).  Each is appended to list (node
// offset) and its slot (slot_base + position) recorded in slot[face].  A
// thread takes LIST_PLANES faces along k and a workgroup (64 x 4 threads)
// reserves the positions of all its faces with one atomic, so the counter
// sees one request per 4096 faces (one per wavefront and plane measured
// 70 ms per step at 512^3 with 60 % of the faces troubled: same-address
// atomics serialise).  Positions past cap are not written (the host then
// runs full WENO); once the count has passed cap, workgroups stop adding.
constexpr int LIST_PLANES = 16;

template <int AX>
__global__ void __launch_bounds__(256) k_face_list(Consts c, Box fb,
                                                   const uint8_t* __restrict__ fl,
                                                   int* __restrict__ slot, int* __restrict__ list,
                                                   unsigned* __restrict__ count, unsigned cap,
                                                   int slot_base) {
  const int lane = threadIdx.x, w = threadIdx.y;  // 64 x 4: one wavefront per row
  const int i = fb.lo[0] + (int)blockIdx.x * 64 + lane;
  const int j = fb.lo[1] + (int)blockIdx.y * 4 + w;
  const int k0 = fb.lo[2] + (int)blockIdx.z * LIST_PLANES;
  const int np = min(LIST_PLANES, fb.lo[2] + fb.n[2] - k0);
  const bool line = i < fb.lo[0] + fb.n[0] && j < fb.lo[1] + fb.n[1];
  const int st = stride(c, AX), sz = c.PXY;
  const int a0 = idx(c, i, j, k0);
  unsigned mine = 0;       // bit p: face (i, j, k0 + p) is troubled
  unsigned long long bal[LIST_PLANES];
  unsigned nwave = 0;
#pragma unroll
  for (int p = 0; p < LIST_PLANES; p++) {
    bool tr = false;
    if (line && p < np) {
      const int a = a0 + p * sz;
      tr = (fl[a - st] | fl[a] | fl[a + st]) != 0;
    }
    bal[p] = __ballot(tr);
    mine |= (unsigned)tr << p;
    nwave += (unsigned)__popcll(bal[p]);
  }
  __shared__ unsigned wn[4], wbase;
  if (lane == 0) wn[w] = nwave;
  __syncthreads();
  if (lane == 0 && w == 0) {
    const unsigned tot = wn[0] + wn[1] + wn[2] + wn[3];
    // past cap already (the count only grows): list nothing, positions from cap
    unsigned b = cap;
    if (tot && __hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <= cap)
      b = atomicAdd(count, tot);
    wbase = b;
  }
  __syncthreads();
  unsigned pos = wbase;
  for (int q = 0; q < w; q++) pos += wn[q];
  const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
  for (int p = 0; p < LIST_PLANES; p++) {
    if ((mine >> p) & 1u) {
      const unsigned at = pos + (unsigned)__popcll(bal[p] & below);
      if (at < cap) {
        const int a = a0 + p * sz;
        list[at] = a;
        slot[a] = slot_base + (int)at;
      }
    }
    pos += (unsigned)__popcll(bal[p]);
  }
}

// Characteristic-WENO flux (the stage's arithmetic form) of each listed face, from
// the stage input Q, into its slot: the lists of the three axes in one launch, n[a]
// faces of axis a from slot off[a] on, over workgroups from first[a] on (three
// launches left the chip idle between them: 92 -> 78 us on the 256x128x128
// shock-vortex block, 24 -> 16 on the 256^3 vortex; what is left is the gather of the
// stencils).
struct WenoLists {
  unsigned n[3], first[3];
  int off[3];
};
template <class F>
__global__ void __launch_bounds__(256) k_weno_list(Consts c, WenoLists wl,
                                                   const int* __restrict__ list,
                                                   const double* __restrict__ Q,
                                                   const double* __restrict__ met,
                                                   double* __restrict__ flux, long fstride) {
  const int ax = blockIdx.x >= wl.first[2] ? 2 : (blockIdx.x >= wl.first[1] ? 1 : 0);
  const unsigned t = (blockIdx.x - wl.first[ax]) * blockDim.x + threadIdx.x;
  if (t >= wl.n[ax]) return;
  const long S = c.S, slot = wl.off[ax] + (long)t;
  const int st = stride(c, ax);
  const int a = list[slot], bn = a + st;
  double q[6][5], f[5];
#pragma unroll
  for (int s = 0; s < 6; s++) load_q(Q, S, a + (s - 2) * st, q[s]);
  const double Ja = met[JAC * S + a], Jb = met[JAC * S + bn];
  const double* nX = met + (3 * ax + 0) * S;
  const double* nY = met + (3 * ax + 1) * S;
  const double* nZ = met + (3 * ax + 2) * S;
  const double nx = face_normal(LEFT, nX[a], Ja, nX[bn], Jb);
  const double ny = face_normal(LEFT, nY[a], Ja, nY[bn], Jb);
  const double nz = face_normal(LEFT, nZ[a], Ja, nZ[bn], Jb);
  const GasT<double> g{c.gamma, c.gam1, c.gam1_inv};
  if constexpr (sizeof(F) == sizeof(double)) {
    F e[5][5];
    stencil_diffs(q, e);
    face_flux(g, e, q[2], q[3], nx, ny, nz, f);
  } else {
    F d[6][5];
#pragma unroll
    for (int s = 0; s < 6; s++)
#pragma unroll
      for (int m = 0; m < 5; m++) d[s][m] = (F)(q[s][m] - q[2][m]);
    face_flux_dev<false>(g, d, q[2], node_t<F>(g, q_to_side(g, q[2])),
                         node_t<F>(g, q_to_side(g, q[3])), nx, ny, nz, false, f);
  }
#pragma unroll
  for (int m = 0; m < 5; m++) flux[m * fstride + slot] = f[m];
}

template <int AX>
void launch_face_list_axis(cbns_block* b, const Box& fb) {
  const dim3 grid((fb.n[0] + 63) / 64, (fb.n[1] + 3) / 4, (fb.n[2] + LIST_PLANES - 1) / LIST_PLANES);
  k_face_list<AX><<<grid, dim3(64, 4), 0, b->stream>>>(
      b->c, fb, b->flags + (long)AX * b->c.S, b->tslot + (long)AX * b->c.S, b->tlist + b->toff[AX],
      b->tcount + AX, (unsigned)b->tcap[AX], (int)b->toff[AX]);
}

template <class F>
int launch_weno_lists(cbns_block* b, const double* qin) {
  ProfScope ps(b, CBNS_K_WENO_LIST);
  WenoLists wl;
  unsigned groups = 0;
  for (int a = 0; a < 3; a++) {
    wl.n[a] = b->h_tcount[a];
    wl.first[a] = groups;
    wl.off[a] = (int)b->toff[a];
    groups += (wl.n[a] + 255) / 256;
  }
  if (groups == 0) return CBNS_OK;
  k_weno_list<F><<<groups, 256, 0, b->stream>>>(b->c, wl, b->tlist, qin, b->met, b->tflux,
                                                b->ttotal);
  CBNS_HIP(b, hipGetLastError());
  return CBNS_OK;
}

}  // namespace

int launch_face_lists(cbns_block* b) {
  CBNS_HIP(b, hipMemsetAsync(b->tcount, 0, 3 * sizeof(unsigned), b->stream));
  for (int a = 0; a < 3; a++) {
    const Box fb = face_box(b->c, a, 0);
    if (fb.count() == 0) continue;
    if (a == 0) launch_face_list_axis<0>(b, fb);
    else if (a == 1) launch_face_list_axis<1>(b, fb);
    else launch_face_list_axis<2>(b, fb);
    CBNS_HIP(b, hipGetLastError());
  }
  CBNS_HIP(b, hipMemcpyAsync(b->h_tcount, b->tcount, 3 * sizeof(unsigned), hipMemcpyDeviceToHost,
                             b->stream));
  CBNS_HIP(b, hipStreamSynchronize(b->stream));
  b->tfull = false;
  for (int a = 0; a < 3; a++)
    if ((long)b->h_tcount[a] > b->tcap[a]) b->tfull = true;
  return CBNS_OK;
}

// How a march over `lines` wavefronts and n nodes along its axis is cut: the
// chunks per CHUNK_MAX nodes.  A thread's chunk is a serial chain of about
// chunk + 1 faces (its first face and the window's loads come on top; one
// wavefront alone takes 2.1 us a node in the eta march, 4.2 in the zeta march),
// so a block that does not fill the chip (1024 SIMDs, two march wavefronts
// each) is cut into shorter chunks until it does, and a large one into long
// chunks, which repeat the fewest faces and window loads.  The cut with the
// least
//   (chunk + 1) x (rounds of 2048 wavefronts)
// is taken, a round costing 1.8 (two wavefronts on a SIMD slow each other) and
// the last one 1 if it leaves a wavefront per SIMD; since wavefronts start as
// others end, the rounds count half as whole ones and half as a fraction.  Of
// 15 cuts tried on each of 45 blocks (24^3 to 224^3, three forms) the rule's is
// 1.6 % off the best on average, 14 % at worst.  Measured (FP64, eta / zeta
// march, us, before: 32 nodes always): 24^3 58 / 110 -> 9 / 14, 64^3 58 / 152
// -> 18 / 38, 128x64x64 59 / 149 -> 28 / 63, 128^3 viscous 127 / 302 -> 101 /
// 215; 256^3 keeps 32.
struct MarchCut {
  int parts;   // chunks per CHUNK_MAX nodes
  long waves;  // wavefronts in all
};
static MarchCut march_cut(long lines, int n) {
  constexpr long SLOTS = 2048;
  constexpr double PAIR = 1.8;
  MarchCut best{1, 0};
  double least = 1e300;
  for (int p = 1; p <= CHUNK_MAX; p++) {
    const int len = std::min((CHUNK_MAX + p - 1) / p, n);
    long chunks = (long)(n / CHUNK_MAX) * p;
    for (int s = 0; s < p && CHUNK_MAX * s / p < n % CHUNK_MAX; s++) chunks++;
    const long w = lines * chunks, rest = w % SLOTS;
    const double whole = PAIR * (double)(w / SLOTS) +
                         (rest == 0 ? 0.0 : (rest <= SLOTS / 2 ? 1.0 : PAIR));
    const double cost = (len + 1) * (whole + std::max(1.0, PAIR * (double)w / SLOTS));
    if (cost < least) {
      least = cost;
      best = {p, w};
    }
  }
  return best;
}

template <int AX, class F, bool HYB>
int launch_march(cbns_block* b, StageArgs& sa) {
  const Consts& c = b->c;
  const int ax_t = AX == 1 ? 2 : 1;
  const int ni = upd_hi(c, 0) - upd_lo(c, 0) + 1;
  const int nt = upd_hi(c, ax_t) - upd_lo(c, ax_t) + 1;
  const int nm = upd_hi(c, AX) - upd_lo(c, AX) + 1;
  const long nw = march_wavefronts<AX>(ni, nt);
  const MarchCut cut = march_cut(nw, nm);
  sa.parts = cut.parts;
  // up to a wavefront per SIMD: workgroups of one, over all CUs (24^3 zeta
  // march 17.3 -> 15.8 us); above, neighbours along the lines share a CU's L1
  // (128^3 zeta march 215 us, 252 with single wavefronts)
  const int R = cut.waves <= 1024 ? 1 : MARCH_Y;
  const dim3 grid((unsigned)((nw + R - 1) / R), sa.parts, (nm + CHUNK_MAX - 1) / CHUNK_MAX);
  ProfScope ps(b, AX == 1 ? CBNS_K_MARCH_ETA : CBNS_K_MARCH_ZETA);
  k_march<AX, F, HYB><<<grid, dim3(MARCH_X, R), 0, b->stream>>>(c, sa, b->met);
  CBNS_HIP(b, hipGetLastError());
  return CBNS_OK;
}

template <class F, bool HYB>
int launch_tiles(cbns_block* b, const StageArgs& sa, int x, bool wrap) {
  const unsigned grid = (unsigned)((stage_tiles(b->c, x) + TILE_XCDS - 1) / TILE_XCDS * TILE_XCDS);
  ProfScope ps(b, CBNS_K_MARCH_ZETA);
  const auto kern = x == 4 ? (wrap ? k_tile4<F, HYB, true> : k_tile4<F, HYB, false>)
                           : (wrap ? k_tile16<F, HYB, true> : k_tile16<F, HYB, false>);
  kern<<<grid, TILE_TPB, 0, b->stream>>>(b->c, sa, b->met);
  CBNS_HIP(b, hipGetLastError());
  return CBNS_OK;
}

template <class F>
int viscous_fluxes(cbns_block* b, double* lam, const double* q) {
  return sizeof(F) == sizeof(double) ? launch_viscous(b, b->vtmp, b->rhs, 1, lam, 1, q)
                                     : launch_viscous_f32(b, b->vtmp, b->rhs, lam, 1, q);
}

constexpr int TFULL_EVERY = 8;  // steps between indicator passes while a list overflows

// One fused stage: [indicator and face lists (hybrid, when due)], viscous
// flux pass, then the tiles or the eta march and the zeta march.  The flux pass reads only the stage
// input's primitives, so it may run before the eta march; the marches
// difference its node fluxes along with the inviscid face fluxes.
template <class F>
int fused_stage(cbns_block* b, double dt, int stage, const double* qin, double* qout,
                bool hyb_form) {
  const Consts& c = b->c;
  int rc = CBNS_OK;
  if (hyb_form) {
    // once per step on the stage-1 input (or every ind_every steps, or at
    // every stage).  While a list has overflowed, every face takes WENO and
    // the flags go unused: the pass then runs every TFULL_EVERY steps, to
    // see whether the lists fit again.
    const int every = b->tfull ? std::max(b->ind_every, TFULL_EVERY) : b->ind_every;
    const bool due = !b->flags_valid || (b->ind_per_stage && !b->tfull) ||
                     (stage == 1 && b->ind_age >= every);
    if (due) {
      if ((rc = launch_indicator(b, qin)) || (rc = launch_face_lists(b))) return rc;
      b->ind_age = 0;
    }
    if (stage == 1) b->ind_age++;
  }
  // first stage of a folded step: the flux pass also forms dt
  double* lam = c.viscous && b->dt_fold && stage == 1 ? b->lam_part : nullptr;
  // inside a step the first two stages leave periodic blocks no primitives
  const bool from_q = b->step_internal && stage > 1 && flux_pass_from_q(c);
  if (c.viscous && (rc = viscous_fluxes<F>(b, lam, from_q ? qin : nullptr))) return rc;
  // more troubled faces than the lists hold: WENO at every face
  const bool hyb = hyb_form && !b->tfull;
  if (hyb && (rc = launch_weno_lists<F>(b, qin))) return rc;
  const long S = c.S;
  const uint8_t* fl = hyb ? b->flags : nullptr;
  const int pmask = stage_prim_mask(b, stage);
  StageArgs sa{dt, b->dt_fold ? b->red + 2 : nullptr, stage, b->prim, b->Q, qin, qout,
               b->rhs, c.viscous ? b->vtmp : nullptr,
               hyb ? fl + S : nullptr, hyb ? fl : nullptr, pmask,
               TroubledFaces{hyb ? b->tslot + S : nullptr, b->tflux, b->ttotal},
               TroubledFaces{hyb ? b->tslot : nullptr, b->tflux, b->ttotal}, 1};
  const int shape = stage_shape(c);
  if (!shape && (rc = hyb ? launch_march<1, F, true>(b, sa) : launch_march<1, F, false>(b, sa)))
    return rc;
  if (lam) {
    ProfScope ps(b, CBNS_K_DT);
    if ((rc = launch_dt_from_partials(b, lam, (int)visc_flux_blocks(c), b->dt_cap, b->red + 2, b->h_scalar + 2)))
      return rc;
  }
  if (shape)
    return hyb ? launch_tiles<F, true>(b, sa, shape, stage_wraps(c, dt))
               : launch_tiles<F, false>(b, sa, shape, stage_wraps(c, dt));
  if (hyb) {
    sa.flags = fl + 2 * S;
    sa.tf.slot = b->tslot + 2 * S;
  }
  return hyb ? launch_march<2, F, true>(b, sa) : launch_march<2, F, false>(b, sa);
}

int launch_fused_stage(cbns_block* b, double dt, int stage, const double* qin, double* qout) {
  const bool hyb = (b->form & CBNS_FORM_HYBRID) != 0;
  return (b->form & CBNS_FORM_FP32) ? fused_stage<float>(b, dt, stage, qin, qout, hyb)
                                    : fused_stage<double>(b, dt, stage, qin, qout, hyb);
}

}  // namespace cbns
