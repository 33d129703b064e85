// k_viscous.hip -- viscous terms in two passes instead of the reference's six
// (gradient_wg_kernel x4, viscous_terms_kernel, viscous_flux_kernel,
// viscous_contribution_kernel; src/calc_viscous_terms.cu:16-88 and
// src/calc_viscous_flux_contribution.cu:16-69):
//
//   k_visc_fluxes  per node of the viscous range [-2, N+1]^3: 4th-order
//                  derivatives of u,v,w,T along xi,eta,zeta, Sutherland mu,
//                  stress tau and heat flux q (from the Cartesian velocity
//                  and temperature gradients), contracted with J grad xi_d
//                  into the 12 values Ev,Fv,Gv (4 each).  The 12 gradients,
//                  6 stresses and 3 heat fluxes never reach HBM.
//   k_visc_div     4th-order central divergence of Ev,Fv,Gv at the update
//                  nodes, at the reference's transverse offset (-1) or
//                  centred; written to dfv (reference decomposition) or
//                  subtracted from a right-hand side.  The fused stage
//                  does without it: its marches subtract the fluxes' face
//                  values from their face fluxes (k_fused.hip, visc_face).
// Both walk along k in chunks (TileMarch): the five zeta-planes a 4th-order
// stencil needs (u,v,w,T in the flux pass, Gv in the divergence) stay in a
// register window, so each plane value is loaded once per chunk instead of
// five times (a plane of one field is 0.56 MB at 256^3: the +-2 planes of
// four fields do not fit a 4 MB XCD L2 and would be re-read from HBM).
// In the flux pass a wavefront holds its 60-node tile along i and two nodes
// on either side; the xi-derivatives take their neighbours from the adjacent
// lanes by wavefront shuffles (LDS crossbar) instead of 16 loads per node,
// and the eta-derivatives from a plane buffer in LDS that holds the
// workgroup's rows and two rows on either side.
// The flux pass streams 14 fields and writes 12: 0.78 ms at 256^3 for those
// alone (a probe of the same streams in the same order, 4.4 TB/s), 1.02 ms for
// the pass, FP32 0.82; what is left is the re-read of the halo rows and planes.
// Its loads are issued together, ahead of the plane's barrier and its
// shuffles: with a branch around each load and each one-sided stencil the
// compiler waited for them one by one, and for the previous plane's stores
// (us, before and now: 32^3 26 -> 11, 64^3 34 -> 25, 193x61x33 with reference
// axes 60 -> 37, 128^3 135 -> 134, 256^3 1036 -> 1023; FP32 131x75x53 50 -> 38,
// 128^3 119 -> 117, 256^3 815 -> 817).  Loading the metrics a plane ahead too
// took 182 VGPRs and was 5 % slower at 128^3; the workgroups of an XCD on
// neighbouring tiles (its L2 then holds their halos) made no difference.
// The divergence pass keeps its loads: there the shuffles cost 30 VGPRs, two of
// its six waves per SIMD and 20 % of its time, and a plane buffer for Fv saved
// nothing (it is bound by its HBM bytes).
#include "cbns_internal.hpp"
#include "face_math.hpp"

namespace cbns {

namespace {

#ifndef VISC_CHUNK
#define VISC_CHUNK 8  // divergence-pass nodes along k per thread
#endif
#ifndef VISC_ROWS
#define VISC_ROWS 8  // divergence-pass workgroup rows along j (64 x VISC_ROWS threads)
#endif
constexpr int VROWS = VISC_ROWS;
#ifndef VISC_FLUX_ROWS
#define VISC_FLUX_ROWS 4  // flux-pass workgroup rows along j
#endif
// Flux-pass nodes along k per thread.  A chunk is a chain of about one memory
// latency a plane (2 us on an idle chip, 4 planes of lead-in on top), so the
// best length is short: 5 of 1, 2, 3, 4, 5, 6, 8, 12, 16, 32 at 64^3 to 256^3
// (128^3 FP64 134 us, 137 at 4, 143 at 12; 256^3 1023, 1040 at 8, 1064 at 12),
// 2 where 5 would leave fewer than 448 workgroups (32^3: 11 us, 16 at 5; 64^3, 476
// of them, 26.5, 28.7 at 2), or, with reference axes, whose kernel runs two a CU,
// just over 512: a second round nearly empty (us at 5 / 2: FP32 456 of them 28.5 /
// 30.9, 520 34.6 / 29.8, FP64 520 38 / 34, 193x61x33 with 544 37 / 34, 130x100x30 with
// 546 39 / 39; from there to 576 nothing was measured, and a third round, past 1024,
// is a smaller part of the pass and left as it is).
constexpr int VISC_FLUX_CHUNK = 5, VISC_FLUX_CHUNK_SMALL = 2;
constexpr int FROWS = VISC_FLUX_ROWS;

// The sums below name their fused operations, so their last bits do not depend
// on how the compiler arranges the code around them (in the precision form a
// float's last bit shows in the step's result).

// 4th-order central difference from the values at -2, -1, +1, +2
__device__ __forceinline__ double central4(double a, double b, double d, double e) {
  return fma(-1.0 / 12.0, e, fma(2.0 / 3.0, d, fma(1.0 / 12.0, a, -(2.0 / 3.0 * b))));
}

// 4th-order derivatives of the four fields f at node offset o on one of the two
// outermost layers of a reference axis (one-sided, src/gradient_kernel.cu:
// 162-253): position p of the ne nodes of the viscous range along the axis, p
// = 0, 1, ne - 2 or ne - 1, st between neighbours.  All 20 values are loaded
// before any is used: one latency, not one per field.
__device__ __forceinline__ void dedge(const double* const f[4], int o, int p, int ne, int st,
                                      double d[4]) {
  const int first = p == 0 ? 0 : (p == 1 ? -1 : (p == ne - 2 ? -3 : -4));
  double v[4][5];
#pragma unroll
  for (int q = 0; q < 4; q++)
#pragma unroll
    for (int s = 0; s < 5; s++) v[q][s] = f[q][o + (first + s) * st];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const double* w = v[q];
    if (0 == p)
      d[q] = -25.0 / 12.0 * w[0] + 4.0 * w[1] - 3.0 * w[2] + (4.0 / 3.0) * w[3] - 0.25 * w[4];
    else if (1 == p)
      d[q] = -5.0 / 6.0 * w[1] - 0.25 * w[0] + 1.5 * w[2] - 0.5 * w[3] + (1.0 / 12.0) * w[4];
    else if (ne - 2 == p)
      d[q] = (5.0 / 6.0) * w[3] - 1.0 / 12.0 * w[0] + 0.5 * w[1] - 1.5 * w[2] + 0.25 * w[4];
    else
      d[q] = (25.0 / 12.0) * w[4] + 0.25 * w[0] - 4.0 / 3.0 * w[1] + 3.0 * w[2] - 4.0 * w[3];
  }
}

// xi-neighbours of a lane's value: n = v at i-2, i-1, i+1, i+2 (meaningful
// on the lanes that own their node; the shuffles wrap at the wave's ends)
template <class V>
__device__ __forceinline__ void xi_neighbours(V v, V n[4]) {
  const int lane = threadIdx.x;
  n[0] = __shfl(v, lane - 2);
  n[1] = __shfl(v, lane - 1);
  n[2] = __shfl(v, lane + 1);
  n[3] = __shfl(v, lane + 2);
}

// d/dxi of v at the node from the neighbouring lanes (every lane takes part)
__device__ __forceinline__ double dxi(double v) {
  double nb[4];
  xi_neighbours(v, nb);
  return central4(nb[0], nb[1], nb[2], nb[3]);
}

// 4th-order central difference from a 5-plane window
__device__ __forceinline__ double dwin(const double w[5]) {
  return central4(w[0], w[1], w[3], w[4]);
}

// The node's three viscous flux vectors E[d] = J grad xi_d . [tau; u.tau - q]
// (src/viscous_terms_kernel.cu:59-105, src/viscous_flux_kernel.cu:57-110),
// from the Cartesian gradients
//   g[a][b] = d u_a / d x_b = sum_d (d u_a / d xi_d) (d xi_d / d x_b)
// of u, v, w (a = 0..2) and T (a = 3):
//   tau = mu/Re (g + g^T - 2/3 tr(g) I),  q = -mu/(Re Pr (gamma-1) M^2) grad T.
// du[a][d]: d u_a / d xi_d; uvw: the node's velocity; T_l: its temperature;
// m: its metrics (XI_X..JAC).  T = double (plain form) or float (precision
// form: the index derivatives, metrics and their products with J are rounded
// to float, mu is formed in double).  Returns mu (unscaled).
template <class T>
__device__ __forceinline__ double visc_node_fluxes(const Consts& c, const double du[4][3],
                                                   const double uvw[3], double T_l,
                                                   const double m[10], T E[3][4]) {
#pragma clang fp contract(off)
  T g[4][3];
#pragma unroll
  for (int a = 0; a < 4; a++) {
    const T d0 = (T)du[a][0], d1 = (T)du[a][1], d2 = (T)du[a][2];
#pragma unroll
    for (int b = 0; b < 3; b++) g[a][b] = sum3(d0, (T)m[b], d1, (T)m[3 + b], d2, (T)m[6 + b]);
  }
  const double mu_d = (1.0 + c.C_T_inf) / (T_l + c.C_T_inf) * sqrt(T_l * T_l * T_l);
  const T mr = (T)(mu_d * c.Re_inv);
  const T third2 = T(2.0 / 3.0) * (g[0][0] + g[1][1] + g[2][2]);
  T tau[3][3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    tau[a][a] = mr * fma(T(2), g[a][a], -third2);
#pragma unroll
    for (int b = a + 1; b < 3; b++) tau[a][b] = tau[b][a] = mr * (g[a][b] + g[b][a]);
  }
  const T mq = mr * (T)c.qcoef;
  T e[3];  // u . tau - q
#pragma unroll
  for (int b = 0; b < 3; b++)
    e[b] = fma(-mq, g[3][b], sum3((T)uvw[0], tau[0][b], (T)uvw[1], tau[1][b], (T)uvw[2], tau[2][b]));
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const T nx = (T)(m[3 * d + 0] * m[JAC]), ny = (T)(m[3 * d + 1] * m[JAC]);
    const T nz = (T)(m[3 * d + 2] * m[JAC]);
#pragma unroll
    for (int a = 0; a < 3; a++) E[d][a] = sum3(nx, tau[0][a], ny, tau[1][a], nz, tau[2][a]);
    E[d][3] = sum3(nx, e[0], ny, e[1], nz, e[2]);
  }
  return mu_d;
}

// The workgroup's rows (64 x FROWS lanes, one row of j per wavefront) and
// the two rows on either side along j: at each plane k the lanes put their
// u,v,w,T into a plane buffer in LDS (the halo rows loaded by the first four
// wavefronts), and the eta-derivatives are differenced from it instead of
// from four loads per field.  Two buffers alternate with k, so one barrier
// per plane orders the writes of plane k+1 after the reads of plane k-1.
constexpr int VPLANE_ROWS = FROWS + 4;
static_assert(FROWS >= 4, "the halo rows are loaded by the first four wavefronts");

// Where a workgroup's lane of the flux pass sits: like tile_march_lane, but
// rows past the box along j stay (they load the values the last rows'
// stencils read and take part in the barriers).  false for the whole
// workgroup past the tile count.
__device__ inline bool visc_flux_lane(const TileMarch& t, int& i, int& j, int& k0, int& k1,
                                      bool& own) {
  const unsigned nb = (unsigned)t.ntx * t.nty * t.nkc;
  const unsigned per = (nb + N_XCD - 1) / N_XCD;
  const unsigned lb = (blockIdx.x % N_XCD) * per + blockIdx.x / N_XCD;
  if (lb >= nb) return false;
  const unsigned tx = lb % t.ntx, r = lb / t.ntx;
  const unsigned ty = r % t.nty, kc = r / t.nty;
  const int lane = (int)threadIdx.x;
  const int ti = (int)tx * (BOX_X - 2 * t.xh) - t.xh + lane, tj = ty * t.rows + threadIdx.y;
  own = tj < t.box.n[1] && lane >= t.xh && lane < BOX_X - t.xh && ti < t.box.n[0];
  i = t.box.lo[0] + ti;
  j = t.box.lo[1] + tj;
  k0 = t.box.lo[2] + (int)kc * t.chunk;
  k1 = min(k0 + t.chunk, t.box.lo[2] + t.box.n[2]);
  return true;
}

// LAM: also the spectral-radius maximum of the workgroup's nodes in
// [0, IM) x [0, JM) x [0, KM) (node_lambda, the time step's per-node term),
// written to lam_part[workgroup]; NaN if any node's is NaN.
// REF: the block has a reference axis (one-sided derivatives at its two outer
// layers); a periodic block's kernel holds no branch on the position.
// FROMQ: u, v, w, T are formed from the conservative state Q, bit for bit as the
// stage that wrote it would have, and no primitives are read: the pass has one field
// more to load (128^3 134 -> 141 us, 256^3 1026 -> 1042), the stage before it four
// fewer to store and to wrap (256^3 precision form: zeta march 1143 -> 1042, ghosts 68 ->
// 51; FP64 1459 -> 1446).  Steps: 128^3 1375 -> 1336 us, 256^3 9580 -> 9500, hybrid 9370
// -> 9040.
template <class T, bool LAM, bool REF, bool FROMQ>
__global__ void __launch_bounds__(64 * FROWS) k_visc_fluxes(Consts c, TileMarch tm,
                                                     const double* __restrict__ prim,
                                                     const double* __restrict__ Q,
                                                     const double* __restrict__ met,
                                                     T* __restrict__ vf,
                                                     double* __restrict__ lam_part) {
  __shared__ double plane[2][4][VPLANE_ROWS][BOX_X];
  int i = 0, j = 0, k0 = 0, k1 = 0;
  bool own = false;
  if (!visc_flux_lane(tm, i, j, k0, k1, own)) return;
  const int lane = threadIdx.x, ty = threadIdx.y;
  // halo row of this wavefront (the first four): j0-2, j0-1, j0+FROWS, j0+FROWS+1
  const int hr = ty < 2 ? ty : ty + FROWS;
  const int jh = j - ty - 2 + hr;
  const bool halo = FROWS == 4 || ty < 4;
  double lam = -INFINITY;
  int nan_seen = 0;
  const bool lam_line = LAM && own && i >= 0 && i < c.IM && j >= 0 && j < c.JM;
  const long S = c.S;
  const int sz = c.PXY;
  const double* f0[4] = {prim + P_U * S, prim + P_V * S, prim + P_W * S, prim + P_T * S};
  // what is loaded of a node, and its u, v, w, T
  constexpr int NL = FROMQ ? 5 : 4;
  const auto fetch = [&](int o, double v[NL]) {
#pragma unroll
    for (int f = 0; f < NL; f++) v[f] = FROMQ ? Q[f * S + o] : f0[f][o];
  };
  const auto uvwt = [&](const double v[NL], double w[4]) {
    if constexpr (FROMQ) {
      const GasT<double> g{c.gamma, c.gam1, c.gam1_inv};
      double r, p;
      q_to_prim(g, v, r, w[0], w[1], w[2], p);
      w[3] = c.gM2 * p * fast_rcp(r);
    } else {
#pragma unroll
      for (int f = 0; f < 4; f++) w[f] = v[f];
    }
  };
  // lanes and rows past the array load its last ones (their values feed no
  // node of the box)
  const int ic = min(i, c.IM + G - 1);
  const int base = idx(c, ic, min(j, c.JM + G - 1), 0);
  const int hbase = idx(c, ic, min(jh, c.JM + G - 1), 0);
  double win[4][5], hn[NL];
  {
    double v[4][NL];
#pragma unroll
    for (int s = 0; s < 4; s++) fetch(base + (k0 - 2 + s) * sz, v[s]);
    fetch(hbase + k0 * sz, hn);
#pragma unroll
    for (int s = 0; s < 4; s++) {
      double w[4];
      uvwt(v[s], w);
#pragma unroll
      for (int f = 0; f < 4; f++) win[f][s + 1] = w[f];
    }
  }
  for (int k = k0; k < k1; k++) {
    // every load of the plane up front (the halo rows of the next plane, which
    // the barrier would wait for)
    double hv[4], m[10], rp[2] = {1.0, 1.0}, pn[NL];
#pragma unroll
    for (int f = 0; f < 4; f++)
#pragma unroll
      for (int s = 0; s < 4; s++) win[f][s] = win[f][s + 1];
    uvwt(hn, hv);
    fetch(base + (k + 2) * sz, pn);
    fetch(hbase + (k + 1) * sz, hn);
#pragma unroll
    for (int q = 0; q < 10; q++) m[q] = met[q * S + base + k * sz];
    if (LAM) {
      rp[0] = prim[P_RHO * S + base + k * sz];
      rp[1] = prim[P_P * S + base + k * sz];
    }
    const int o = base + k * sz;
    const int pb = k & 1;
    double du[4][3];
#pragma unroll
    for (int f = 0; f < 4; f++) {
      plane[pb][f][ty + 2][lane] = win[f][2];
      if (halo) plane[pb][f][hr][lane] = hv[f];
    }
#pragma unroll
    for (int f = 0; f < 4; f++) du[f][0] = dxi(win[f][2]);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    // keeps the metric loads ahead of the barrier (they would sink to their use)
#pragma unroll
    for (int q = 0; q < 10; q++) asm volatile("" : "+v"(m[q]));
    {
      double w[4];
      uvwt(pn, w);
#pragma unroll
      for (int f = 0; f < 4; f++) win[f][4] = w[f];
    }
#pragma unroll
    for (int f = 0; f < 4; f++) {
      du[f][1] = central4(plane[pb][f][ty][lane], plane[pb][f][ty + 1][lane],
                          plane[pb][f][ty + 3][lane], plane[pb][f][ty + 4][lane]);
      du[f][2] = dwin(win[f]);
    }
    if (REF && own) {
      double d[4];
      if (!periodic(c, 0) && (i < 0 || i >= c.IM)) {
        dedge(f0, o, i + 2, c.IM + 4, 1, d);
#pragma unroll
        for (int f = 0; f < 4; f++) du[f][0] = d[f];
      }
      if (!periodic(c, 1) && (j < 0 || j >= c.JM)) {
        dedge(f0, o, j + 2, c.JM + 4, c.PX, d);
#pragma unroll
        for (int f = 0; f < 4; f++) du[f][1] = d[f];
      }
      if (!periodic(c, 2) && (k < 0 || k >= c.KM)) {
        dedge(f0, o, k + 2, c.KM + 4, sz, d);
#pragma unroll
        for (int f = 0; f < 4; f++) du[f][2] = d[f];
      }
    }
    const double uvw[3] = {win[0][2], win[1][2], win[2][2]};
    T E[3][4];
    visc_node_fluxes<T>(c, du, uvw, win[3][2], m, E);
    if (LAM && lam_line && k >= 0 && k < c.KM) {
      const double sl = node_lambda_v(c, rp[0], uvw[0], uvw[1], uvw[2], rp[1], win[3][2], m);
      if (isnan(sl)) nan_seen = 1;
      else lam = fmax(lam, sl);
    }
    if (own) {
#pragma unroll
      for (int d = 0; d < 3; d++)
#pragma unroll
        for (int e = 0; e < 4; e++) vf[(long)(4 * d + e) * S + o] = E[d][e];
    }
  }
  if (LAM) {
    __shared__ double lds[FROWS];
    const int tid = threadIdx.x + threadIdx.y * BOX_X;
    lam = block_max(lam, lds, tid, 64 * FROWS);
    __syncthreads();
    const int any_nan = __syncthreads_or(nan_seen);
    if (tid == 0) lam_part[blockIdx.x] = any_nan ? NAN : lam;
  }
}

// src/viscous_contribution_kernel.cu:35-67.  mode 0: dfv[e] = div; mode 1:
// out[(e+1)] -= div (the fused stage's right-hand side, momentum and energy).
// gw[e][s]: Gv component e on the zeta line of the stencil at k-2+s.
template <class T>
__device__ __forceinline__ void visc_div_node(const Consts& c, int i, int j, int k,
                                              const T gw[4][5], const T* __restrict__ vf,
                                              double* __restrict__ out, int mode) {
  const long S = c.S;
  const int sh = c.visc_centered ? 0 : -1;
  const T c0 = T(1.0 / 12.0), c1 = T(-2.0 / 3.0);
  const int ox = idx(c, i, j + sh, k + sh), oy = idx(c, i + sh, j, k + sh);
  const int sx = 1, sy = c.PX;
  const int o = idx(c, i, j, k);
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const T* Ev = vf + (long)e * S;
    const T* Fv = vf + (long)(4 + e) * S;
    T df = c0 * Ev[ox - 2 * sx] + c1 * Ev[ox - sx] - c1 * Ev[ox + sx] - c0 * Ev[ox + 2 * sx];
    df += c0 * Fv[oy - 2 * sy] + c1 * Fv[oy - sy] - c1 * Fv[oy + sy] - c0 * Fv[oy + 2 * sy];
    df += c0 * gw[e][0] + c1 * gw[e][1] - c1 * gw[e][3] - c0 * gw[e][4];
    if (mode == 0) out[e * S + o] = (double)df;
    else out[(e + 1) * S + o] -= (double)df;
  }
}

template <class T>
__global__ void __launch_bounds__(64 * VROWS) k_visc_div(Consts c, TileMarch tm,
                                                  const T* __restrict__ vf,
                                                  double* __restrict__ out, int mode) {
  int i, j, k0, k1;
  if (!tile_march_node(tm, i, j, k0, k1)) return;
  const long S = c.S;
  const int sh = c.visc_centered ? 0 : -1;
  const int sz = c.PXY;
  const int base = idx(c, i + sh, j + sh, 0);  // the zeta line of the Gv stencil
  const T* G0 = vf + 8 * S;
  T gw[4][5];
#pragma unroll
  for (int e = 0; e < 4; e++)
#pragma unroll
    for (int s = 0; s < 4; s++) gw[e][s + 1] = G0[e * S + base + (k0 - 2 + s) * sz];
  for (int k = k0; k < k1; k++) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
#pragma unroll
      for (int s = 0; s < 4; s++) gw[e][s] = gw[e][s + 1];
      gw[e][4] = G0[e * S + base + (k + 2) * sz];
    }
    visc_div_node<T>(c, i, j, k, gw, vf, out, mode);
  }
}

}  // namespace

// Workgroups of the viscous flux pass (the entries lam_part needs).
static TileMarch visc_flux_tiles(const Consts& c) {
  Box vb;
  for (int a = 0; a < 3; a++) {
    vb.lo[a] = -2;
    vb.n[a] = axis_n(c, a) + 4;
  }
  const TileMarch tm = tile_march(vb, VISC_FLUX_CHUNK, FROWS, 2);
  const bool ref = !periodic(c, 0) || !periodic(c, 1) || !periodic(c, 2);
  const long nb = (long)tm.ntx * tm.nty * tm.nkc;
  if (nb >= 448 && !(ref && nb > 512 && nb < 576)) return tm;
  return tile_march(vb, VISC_FLUX_CHUNK_SMALL, FROWS, 2);
}

long visc_flux_blocks(const Consts& c) { return (long)tile_march_blocks(visc_flux_tiles(c)); }

// vf: 12*S scratch (of T).  mode 0 writes dfv (4*S) to
// `out`, mode 1 subtracts the divergence from the right-hand side (5*S).
// lam_part (visc_flux_blocks entries) or null: the flux pass also forms the
// time step's per-workgroup spectral-radius maxima.
// q: the state to take u, v, w, T from, or null (the primitives).
template <class T>
int viscous(cbns_block* b, T* vf, double* out, int mode, double* lam_part, int parts,
            const double* q) {
  const Consts& c = b->c;
  if (parts & 1) {
    ProfScope ps(b, CBNS_K_VISC_FLUX);
    const TileMarch tm = visc_flux_tiles(c);
    const dim3 grid(tile_march_blocks(tm)), block(BOX_X, FROWS);
    const bool ref = !periodic(c, 0) || !periodic(c, 1) || !periodic(c, 2);
    if (q && (ref || lam_part)) return fail(b, CBNS_ERR_STATE, "flux pass from Q: periodic, no dt");
    const auto kern =
        q ? k_visc_fluxes<T, false, false, true>
          : (lam_part ? (ref ? k_visc_fluxes<T, true, true, false> : k_visc_fluxes<T, true, false, false>)
                      : (ref ? k_visc_fluxes<T, false, true, false>
                             : k_visc_fluxes<T, false, false, false>));
    kern<<<grid, block, 0, b->stream>>>(c, tm, b->prim, q, b->met, vf, lam_part);
    CBNS_HIP(b, hipGetLastError());
  }
  if (!(parts & 2)) return CBNS_OK;
  Box ub;
  for (int a = 0; a < 3; a++) {
    ub.lo[a] = upd_lo(c, a);
    ub.n[a] = upd_hi(c, a) - upd_lo(c, a) + 1;
  }
  ProfScope ps(b, CBNS_K_VISC_DIV);
  const TileMarch tm = tile_march(ub, VISC_CHUNK, VROWS);
  k_visc_div<T><<<tile_march_blocks(tm), dim3(BOX_X, VROWS), 0, b->stream>>>(c, tm, vf, out, mode);
  CBNS_HIP(b, hipGetLastError());
  return CBNS_OK;
}

int launch_viscous(cbns_block* b, double* vf, double* out, int mode, double* lam_part, int parts,
                   const double* q) {
  return viscous<double>(b, vf, out, mode, lam_part, parts, q);
}

// precision form: the same scratch holds 12*S floats
int launch_viscous_f32(cbns_block* b, double* scratch, double* rhs, double* lam_part, int parts,
                       const double* q) {
  return viscous<float>(b, reinterpret_cast<float*>(scratch), rhs, 1, lam_part, parts, q);
}

}  // namespace cbns
