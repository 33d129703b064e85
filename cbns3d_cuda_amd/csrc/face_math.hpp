// face_math.hpp -- per-face inviscid flux: Roe-averaged characteristic basis,
// characteristic WENO5-JS reconstruction of the conservative state on both
// sides, Lax-Friedrichs-type flux.  Method of src/rec_riemann_kernel.cu:44-89
// (calc_eigenvectors_roe, rec_weno5 x2, lf_flux), restructured for gfx950:
//   - L and R are linear and WENO5-JS is translation invariant, so the plain
//     form works on the five first differences of the stencil: they are
//     projected (five vectors for the two sides together, not ten),
//     reconstructed as deviations from the two nodes of the face and added to
//     those nodes' states;
//   - L (left eigenvectors) is applied in closed form: rows 0..2 share two
//     dot products, rows 3..4 are the tangent projections;
//   - R (right eigenvectors) is applied in closed form;
//   - each WENO5 evaluation uses one division (weights multiplied through by
//     IS1^2 IS2^2 IS3^2, the linear weights and the 1/6 of the candidate
//     stencils folded into the candidates and the normaliser) instead of
//     seven; the left and right evaluations of a field share two smoothness
//     terms and, in double, one reciprocal;
//   - the Lax-Friedrichs flux reuses 1/rho, |u|^2/2 and E of the
//     reconstructed states (the reference re-derives E from p);
//   - 1/x is formed once and multiplied where the reference divides by the
//     same x repeatedly;
//   - reciprocals and reciprocal square roots start from the hardware
//     v_rcp_f64 / v_rsq_f64 estimate (relative error <= 5.3e-8 on MI355X
//     over 2^20 arguments in [2^-30, 2^31]) and take one Newton step, which
//     leaves <= 2.3e-15 (rcp) and <= 4.2e-15 (rsq); an IEEE f64 divide or
//     sqrt costs ~11-12 VALU instructions on gfx950, this 3-4, and a second
//     step (<= 1.4e-16) would cost 2-3 more in a VALU-bound sweep.
//     Arguments are positive and finite wherever they are used.
// Every sum of products names its fused operations, so a face's bits do not depend
// on the code around it, and the marches and the tiles form it alike.  Some functions
// take which product of a sum is rounded (yz, CHAIN, SWAP; k_fused.hip's Rounding):
// in the precision and hybrid forms a last bit of a float, or a double next to one,
// shows in the step's result, and these keep the results that those forms have had.
// So the WENO lists of a hybrid round a listed face otherwise than a march would, and
// in these two forms the face at every 32nd node of an eta or zeta line is rounded
// otherwise for the node before it than for the node after it: their update conserves
// there to rounding only.
// The result equals the reference formula up to rounding (the stage parity
// bar is 1e-12 relative; tests/test_gpu_parity.py).
#pragma once

#include <hip/hip_runtime.h>

namespace cbns {

__device__ __forceinline__ double fast_rcp(double x) {
  const double r = __builtin_amdgcn_rcp(x);
  return fma(r, fma(-x, r, 1.0), r);
}
__device__ __forceinline__ float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }

// 1/sqrt(x): y <- y + y (1/2 - x y^2 / 2)
__device__ __forceinline__ double fast_rsq(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  return fma(y, fma(-0.5 * x * y, y, 0.5), y);
}
__device__ __forceinline__ float fast_rsq(float x) { return __builtin_amdgcn_rsqf(x); }

// a0 b0 + a1 b1 + a2 b2
template <class T>
__device__ __forceinline__ T sum3(T a0, T b0, T a1, T b1, T a2, T b2) {
  return fma(a2, b2, fma(a0, b0, a1 * b1));
}

template <class T>
struct GasT {
  T gamma, gam1, gam1_inv;
};

// Roe-averaged characteristic basis of a face, src/calc_eigenvectors_roe.cu:28-150.
template <class T>
struct Basis {
  T nx, ny, nz, lx, ly, lz, mx, my, mz;  // orthonormal (n normal, l,m tangents)
  T uu, vv, ww, H, c, k, qn, ql, qm;     // Roe state, k = |u|^2/2
  T K, o;                                // gam1/(2c^2), 0.5/c
};

// Characteristic basis from the face normal and the Roe-averaged state
// (u, v, w, H = X f) (src/calc_eigenvectors_roe.cu:28-150).  yz: which square of
// |l|^2 = n_y^2 + n_z^2 is rounded before the sum, n_z's or (true) n_y's.
template <class T>
__device__ __forceinline__ void basis_from_roe(const GasT<T>& g, T uu, T vv, T ww, T X, T f, T n_x,
                                               T n_y, T n_z, Basis<T>& B, bool yz = false) {
#pragma clang fp contract(off)
  T l_x = T(0), l_y = n_z, l_z = -n_y;
  T m_x, m_y, m_z;
  // |l| > 1e-8 of the reference, compared squared
  const T lm = fma(n_y, n_y, n_z * n_z);
  T l2 = yz ? fma(n_z, n_z, n_y * n_y) : lm;
  if (l2 > T(1.0e-16)) {
    m_x = -lm;
    m_y = n_x * n_y;
    m_z = n_x * n_z;
  } else {
    l2 = fma(n_x, n_x, n_z * n_z);
    l_x = -n_z; l_y = T(0); l_z = n_x;
    m_x = n_x * n_y;
    m_y = -l2;
    m_z = n_y * n_z;
  }
  const T inv_n = fast_rsq(n_z * n_z + (n_x * n_x + n_y * n_y));
  B.nx = n_x * inv_n; B.ny = n_y * inv_n; B.nz = n_z * inv_n;
  const T inv_l = fast_rsq(l2);
  B.lx = l_x * inv_l; B.ly = l_y * inv_l; B.lz = l_z * inv_l;
  // |m|^2 = |l|^2 |n|^2 for either choice of tangents
  const T inv_m = inv_l * inv_n;
  B.mx = m_x * inv_m; B.my = m_y * inv_m; B.mz = m_z * inv_m;

  B.uu = uu; B.vv = vv; B.ww = ww; B.H = X * f;
  B.k = T(0.5) * sum3(uu, uu, vv, vv, ww, ww);
  const T c2 = g.gam1 * fma(X, f, -B.k);
  const T inv_c = fast_rsq(c2);
  B.c = c2 * inv_c;
  B.qn = sum3(uu, B.nx, vv, B.ny, ww, B.nz);
  B.ql = sum3(vv, B.ly, uu, B.lx, ww, B.lz);
  B.qm = sum3(uu, B.mx, vv, B.my, ww, B.mz);
  B.o = T(0.5) * inv_c;
  B.K = T(0.5) * g.gam1 * inv_c * inv_c;
}

// From the two node states as (rho, u, v, w, H): Roe average with
// r = sqrt(rho_R / rho_L).
template <class T>
__device__ __forceinline__ void roe_basis_h(const GasT<T>& g, T rL, T uL, T vL, T wL, T HL,
                                            T rR, T uR, T vR, T wR, T HR, T n_x, T n_y, T n_z,
                                            Basis<T>& B, bool yz = false) {
  const T y = fast_rsq(rR * rL), ratio = rR * y;  // sqrt(rR / rL)
  const T inv1r = fast_rcp(fma(rR, y, T(1)));
  basis_from_roe(g, fma(ratio, uR, uL) * inv1r, fma(ratio, vR, vL) * inv1r,
                 fma(ratio, wR, wL) * inv1r, fma(ratio, HR, HL), inv1r, n_x, n_y, n_z, B, yz);
}

// From the two node states as conservative states: with a = 1/sqrt(rho),
// the Roe average sum sqrt(rho) f / sum sqrt(rho) is sum a (rho f) / sum
// sqrt(rho), and rho H = E + p.
template <class T>
__device__ __forceinline__ void roe_basis_q(const GasT<T>& g, const T qL[5], const T qR[5],
                                            T n_x, T n_y, T n_z, Basis<T>& B) {
  const T aL = fast_rsq(qL[0]), aR = fast_rsq(qR[0]);
  const T D = fast_rcp(fma(qR[0], aR, qL[0] * aL));
  const T wL = aL * D, wR = aR * D;
  // p = gam1 (E - |rho u|^2 / (2 rho)), 1/rho = a^2
  const T kL = T(0.5) * sum3(qL[1], qL[1], qL[2], qL[2], qL[3], qL[3]);
  const T kR = T(0.5) * sum3(qR[1], qR[1], qR[2], qR[2], qR[3], qR[3]);
  const T hL = fma(g.gam1, fma(-kL, aL * aL, qL[4]), qL[4]);  // rho H
  const T hR = fma(g.gam1, fma(-kR, aR * aR, qR[4]), qR[4]);
  basis_from_roe(g, fma(qR[1], wR, qL[1] * wL), fma(qR[2], wR, qL[2] * wL),
                 fma(qR[3], wR, qL[3] * wL), fma(hR, wR, hL * wL), T(1), n_x, n_y, n_z, B);
}

// From (rho, u, v, w, p): H = c^2/gam1 + |u|^2/2 with c^2 = gamma p / rho.
template <class T>
__device__ __forceinline__ void roe_basis(const GasT<T>& g, T rL, T uL, T vL, T wL, T pL,
                                          T rR, T uR, T vR, T wR, T pR, T n_x, T n_y, T n_z,
                                          Basis<T>& B) {
  const T irL = fast_rcp(rL), irR = fast_rcp(rR);
  const T HL = fma(T(0.5), sum3(uL, uL, vL, vL, wL, wL), g.gamma * pL * irL * g.gam1_inv);
  const T HR = fma(T(0.5), sum3(uR, uR, vR, vR, wR, wR), g.gamma * pR * irR * g.gam1_inv);
  roe_basis_h(g, rL, uL, vL, wL, HL, rR, uR, vR, wR, HR, n_x, n_y, n_z, B);
}

// A reconstructed face state: primitives plus 1/rho, |u|^2/2 and the
// conservative state they were derived from (momenta, total energy E;
// p = gam1 (E - rho |u|^2/2)).
template <class T>
struct Side {
  T r, u, v, w, x, p, ir, k, E, ru, rv, rw;  // x = E - rho |u|^2/2
};

// conservative -> face state (src/weno.cu:113-118 / src/primitive_bc_kernel.cu:63-67)
template <class T>
__device__ __forceinline__ Side<T> q_to_side(const GasT<T>& g, const T q[5]) {
  Side<T> s;
  s.r = q[0];
  s.ir = fast_rcp(s.r);
  s.u = q[1] * s.ir;
  s.v = q[2] * s.ir;
  s.w = q[3] * s.ir;
  s.k = T(0.5) * sum3(s.u, s.u, s.v, s.v, s.w, s.w);
  s.E = q[4];
  s.x = fma(-s.r, s.k, s.E);
  s.p = g.gam1 * s.x;
  s.ru = q[1];
  s.rv = q[2];
  s.rw = q[3];
  return s;
}

// total enthalpy of a face state, as roe_basis forms it
template <class T>
__device__ __forceinline__ T side_h(const GasT<T>& g, const Side<T>& s) {
  return fma(g.gamma * s.p * s.ir, g.gam1_inv, s.k);
}

// q0 + R W, R W in T, the sum in double, then to the face state
// (src/weno.cu:106-118): W the characteristic deviations of the side's value from
// node state q0
template <class T>
__device__ __forceinline__ Side<double> char_to_side(const GasT<double>& g, const Basis<T>& B,
                                                     const double q0[5], const T W[5]) {
  const T s = W[0] + W[2];
  const T dl = B.c * (W[2] - W[0]);
  const T r = s + W[1];
  const double q[5] = {
      q0[0] + (double)r,
      q0[1] + (double)fma(B.mx, W[4], fma(B.lx, W[3], fma(B.uu, r, B.nx * dl))),
      q0[2] + (double)fma(B.my, W[4], fma(B.ly, W[3], fma(B.vv, r, B.ny * dl))),
      q0[3] + (double)fma(B.mz, W[4], fma(B.lz, W[3], fma(B.ww, r, B.nz * dl))),
      q0[4] + (double)fma(B.qm, W[4], fma(B.ql, W[3], fma(B.qn, dl, fma(B.k, W[1], B.H * s))))};
  return q_to_side(g, q);
}

// src/lf_flux.cu:22-78 (dissipation speed |sum_d max_LR(|u_d|+c) n_d|),
//   f = (F(L).n + F(R).n - alpha (Q_R - Q_L)) / 2,  F(Q).n = (rho q_n, rho q_n u + p n, ...,
//   rho q_n H),
// on the reconstructed conservative states: the mass fluxes are (rho u).n
// and the jumps are those of rho u and E (the reference re-forms rho u and
// E from the primitives, which equals them up to rounding).
// SWAP: the sums of the two sides round the right side's product, not the left's.
template <bool SWAP = false, class T>
__device__ __forceinline__ void lf_flux(const GasT<T>& g, const Side<T>& R, const Side<T>& L,
                                        T nx, T ny, T nz, T f[5]) {
  const T aR = g.gamma * R.p * R.ir, yR = fast_rsq(aR);  // sound speed aR yR
  const T HR = fma(aR, g.gam1_inv, R.k);
  const T aL = g.gamma * L.p * L.ir, yL = fast_rsq(aL);
  const T HL = fma(aL, g.gam1_inv, L.k);
  const T s0 = fmax(fma(aR, yR, fabs(R.u)), fma(aL, yL, fabs(L.u)));
  const T s1 = fmax(fma(aR, yR, fabs(R.v)), fma(aL, yL, fabs(L.v)));
  const T s2 = fmax(fma(aR, yR, fabs(R.w)), fma(aL, yL, fabs(L.w)));
  const T ha = T(0.5) * fabs(sum3(s0, nx, s1, ny, s2, nz));
  const T hmL = T(0.5) * sum3(L.ru, nx, L.rv, ny, L.rw, nz);  // rho q_n / 2
  const T hmR = T(0.5) * sum3(R.ru, nx, R.rv, ny, R.rw, nz);
  const T hp = T(0.5) * (SWAP ? fma(g.gam1, L.x, R.p) : fma(g.gam1, R.x, L.p));
  // hmL l + hmR r
  const auto both = [&](T l, T r) { return SWAP ? fma(hmL, l, hmR * r) : fma(hmR, r, hmL * l); };
  f[0] = fma(-ha, R.r - L.r, hmL + hmR);
  f[1] = fma(-ha, R.ru - L.ru, fma(hp, nx, both(L.u, R.u)));
  f[2] = fma(-ha, R.rv - L.rv, fma(hp, ny, both(L.v, R.v)));
  f[3] = fma(-ha, R.rw - L.rw, fma(hp, nz, both(L.w, R.w)));
  f[4] = fma(-ha, R.E - L.E, both(HL, HR));
}

// conservative -> primitive (src/primitive_bc_kernel.cu:63-67)
template <class T>
__device__ __forceinline__ void q_to_prim(const GasT<T>& g, const T q[5], T& r, T& u, T& v, T& w,
                                          T& p) {
  r = q[0];
  const T ir = fast_rcp(r);
  u = q[1] * ir;
  v = q[2] * ir;
  w = q[3] * ir;
  p = g.gam1 * fma(T(-0.5) * r, sum3(u, u, v, v, w, w), q[4]);
}

// WENO5-JS on both sides of one face.  For a side's stencil a..e with differences
// E0 .. E3 = b-a .. e-d and centre c the JS weights are d_k / IS_k^2, d = (0.1,
// 0.6, 0.3), and the candidates f_k / 6; scaling numerator and normaliser by s1 s2
// s3 / 0.6, s_k = IS_k^2,
//   value - c = (p1 g1 + p2 g2 + p3 g3) / (p1 + 6 p2 + 3 p3),
//   p1 = s2 s3, p2 = s1 s3, p3 = s1 s2,
//   g1 = f1/6 - c = 5/6 E1 - 1/3 E0,  g2 = f2 - 6c = E1 + 2 E2,
//   g3 = f3/2 - 3c = 2 E2 - E3/2.
// The smoothness indicators are the polynomials of src/weno.cu:19-42 regrouped:
//   IS1 = 13/12 (E1-E0)^2 + ((E1-E0)/2 + E1)^2 + eps,
//   IS2 = 13/12 (E2-E1)^2 + ((E1+E2)/2)^2 + eps,
//   IS3 = 13/12 (E3-E2)^2 + ((E3-E2)/2 - E2)^2 + eps.
// The right side reads the differences reversed and negated; the 13/12 (.)^2 + eps
// terms of the two middle second differences serve both sides.

// p1 g1 + p2 g2 + p3 g3 and the normaliser from the indicators
template <class T>
__device__ __forceinline__ void weno5_sum(T IS1, T IS2, T IS3, T g1, T g2, T g3, T& num, T& den) {
  const T s1 = IS1 * IS1, s2 = IS2 * IS2, s3 = IS3 * IS3;
  const T p1 = s2 * s3, p2 = s1 * s3, p3 = s1 * s2;
  num = fma(p3, g3, fma(p1, g1, p2 * g2));
  den = fma(T(3), p3, fma(T(6), p2, p1));
}

// Plain form: from the differences e01 .. e45 of the six projected values w0 .. w5
// (nodes m-2 .. m+3), left = weno5(w0..w4) - w2, right = weno5(w5..w1) - w3.  The
// indicators are formed four times as large and the candidates twice (4 IS2 = 13/3
// (.)^2 + (E1+E2)^2 + 4 eps, 2 g1 = E1 + 2/3 (E1-E0), 2 g3 = 4 E2 - E3): four
// operations fewer.
__device__ __forceinline__ void weno5_pair(double e01, double e12, double e23, double e34,
                                           double e45, double& left, double& right) {
  const double k13 = 13.0 / 3.0, eps = 4.0e-6;
  const double da = e12 - e01, dc = e23 - e12, dd = e34 - e23, df = e45 - e34;
  const double tc = fma(k13 * dc, dc, eps), td = fma(k13 * dd, dd, eps);
  const double h2 = fma(2.0, e12, da), h4 = e12 + e23, h6 = fma(-2.0, e23, dd);
  const double r2 = fma(-2.0, e34, df), r4 = e23 + e34, r6 = fma(2.0, e23, dc);
  const double four = 4.0 * e23;
  double nl, dl, nr, dr;
  weno5_sum(fma(k13 * da, da, fma(h2, h2, eps)), fma(h4, h4, tc), fma(h6, h6, td),
            fma(2.0 / 3.0, da, e12), fma(2.0, e12, four), four - e34, nl, dl);
  weno5_sum(fma(k13 * df, df, fma(r2, r2, eps)), fma(r4, r4, td), fma(r6, r6, tc),
            fma(-2.0 / 3.0, df, e34), fma(2.0, e34, four), four - e12, nr, dr);
  // one reciprocal for both sides: dl, dr lie in [2e-21, 3e123] for any
  // smoothness indicator (four times as large here) below 1e30, so dl dr stays in range
  const double x = 0.5 * fast_rcp(dl * dr);
  left = nl * (dr * x);
  right = -nr * (dl * x);
}

// Precision form: from the projected deviations w0 .. w5 from node m (w2 = 0).
__device__ __forceinline__ void weno5_pair_dev(float w0, float w1, float w3, float w4, float w5,
                                               float& left, float& right) {
  const float k13 = float(13.0 / 12.0), eps = float(1.0e-6);
  const float e01 = w1 - w0, e12 = -w1, e23 = w3, e34 = w4 - w3, e45 = w5 - w4;
  const float da = e12 - e01, dc = e23 - e12, dd = e34 - e23, df = e45 - e34;
  const float tc = fma(k13 * dc, dc, eps), td = fma(k13 * dd, dd, eps);
  const float h2 = fma(0.5f, da, e12), h4 = 0.5f * (e12 + e23), h6 = fma(0.5f, dd, -e23);
  const float r2 = fma(0.5f, df, -e34), r4 = 0.5f * (e23 + e34), r6 = fma(0.5f, dc, e23);
  float nl, dl, nr, dr;
  weno5_sum(fma(k13 * da, da, fma(h2, h2, eps)), fma(h4, h4, tc), fma(h6, h6, td),
            fma(float(5.0 / 6.0), e12, -(float(1.0 / 3.0) * e01)), fma(2.0f, e23, e12),
            fma(-0.5f, e34, 2.0f * e23), nl, dl);
  weno5_sum(fma(k13 * df, df, fma(r2, r2, eps)), fma(r4, r4, td), fma(r6, r6, tc),
            fma(float(1.0 / 3.0), e45, -(float(5.0 / 6.0) * e34)), fma(-2.0f, e23, -e34),
            fma(0.5f, e12, -2.0f * e23), nr, dr);
  left = nl * fast_rcp(dl);
  right = fma(nr, fast_rcp(dr), w3);
}

// The plain form's face between nodes m and m+1 (states qm, qp): e[k] the
// differences between nodes m-2+k and m-1+k; B the face's characteristic basis;
// (nx,ny,nz) the unnormalised face vector 0.5 (J grad xi |_m + J grad xi |_{m+1}).
// Against projecting the six node states and taking each field's differences
// afterwards the face has 25 differences and a sixth of the projections fewer: the
// eta march's loop goes from 731 FP64 instructions to 696.
__device__ __forceinline__ void face_flux_basis(const GasT<double>& g, const double e[5][5],
                                                const double qm[5], const double qp[5],
                                                const Basis<double>& B, double nx, double ny,
                                                double nz, double f[5]) {
  // rows 0..2 of L e share A = K (E - u.m + |u|^2/2 rho) and Bn = o (qn rho - n.m)
  double A[5], Bn[5];
#pragma unroll
  for (int s = 0; s < 5; s++) {
    A[s] = B.K * fma(-B.ww, e[s][3],
                     fma(-B.vv, e[s][2], fma(-B.uu, e[s][1], fma(B.k, e[s][0], e[s][4]))));
    Bn[s] = B.o * fma(-B.nz, e[s][3], fma(-B.ny, e[s][2], fma(-B.nx, e[s][1], B.qn * e[s][0])));
  }
  double WL[5], WR[5], w[5];
#pragma unroll
  for (int s = 0; s < 5; s++) w[s] = A[s] + Bn[s];
  weno5_pair(w[0], w[1], w[2], w[3], w[4], WL[0], WR[0]);
#pragma unroll
  for (int s = 0; s < 5; s++) w[s] = fma(-2.0, A[s], e[s][0]);
  weno5_pair(w[0], w[1], w[2], w[3], w[4], WL[1], WR[1]);
#pragma unroll
  for (int s = 0; s < 5; s++) w[s] = A[s] - Bn[s];
  weno5_pair(w[0], w[1], w[2], w[3], w[4], WL[2], WR[2]);
#pragma unroll
  for (int s = 0; s < 5; s++)
    w[s] = fma(B.lz, e[s][3], fma(B.ly, e[s][2], fma(B.lx, e[s][1], -(B.ql * e[s][0]))));
  weno5_pair(w[0], w[1], w[2], w[3], w[4], WL[3], WR[3]);
#pragma unroll
  for (int s = 0; s < 5; s++)
    w[s] = fma(B.mz, e[s][3], fma(B.my, e[s][2], fma(B.mx, e[s][1], -(B.qm * e[s][0]))));
  weno5_pair(w[0], w[1], w[2], w[3], w[4], WL[4], WR[4]);
  lf_flux(g, char_to_side(g, B, qp, WR), char_to_side(g, B, qm, WL), nx, ny, nz, f);
}

__device__ __forceinline__ void face_flux(const GasT<double>& g, const double e[5][5],
                                          const double qm[5], const double qp[5], double nx,
                                          double ny, double nz, double f[5]) {
  Basis<double> B;
  roe_basis_q(g, qm, qp, nx, ny, nz, B);
  face_flux_basis(g, e, qm, qp, B, nx, ny, nz, f);
}

// Precision form: the Roe basis, the characteristic projection and WENO5 run in
// float on the deviations of the six stencil nodes from node m, so float's
// rounding acts on the local variation, not on the state itself.  The
// reconstructed states q_m + dq_L/R and the Lax-Friedrichs flux are formed in
// double, so face-flux differences carry no float cancellation error.

// The Roe-average inputs of a node in the precision form: rho, u, v, w and
// H of its double face state, rounded to float.
template <class T>
struct NodeT {
  T r, u, v, w, H;
};
template <class T>
__device__ __forceinline__ NodeT<T> node_t(const GasT<double>& g, const Side<double>& s) {
  return {(T)s.r, (T)s.u, (T)s.v, (T)s.w, (T)side_h(g, s)};
}

// The precision-form face from the stencil's deviations d[s] = q[s] - q[2] (d[2]
// is not read), the state of node m (qm) and the Roe inputs of nodes m and m+1;
// yz: basis_from_roe.  CHAIN: d comes from dev_from_diffs; its nodes below m, the
// negative of sums, then round another product of a sum.
template <bool CHAIN>
__device__ __forceinline__ void face_flux_dev(const GasT<double>& g, const float d[6][5],
                                              const double qm[5], const NodeT<float>& nl,
                                              const NodeT<float>& nr, double nx, double ny,
                                              double nz, bool yz, double f[5]) {
  const GasT<float> gt{(float)g.gamma, (float)g.gam1, (float)g.gam1_inv};
  Basis<float> B;
  roe_basis_h(gt, nl.r, nl.u, nl.v, nl.w, nl.H, nr.r, nr.u, nr.v, nr.w, nr.H, (float)nx, (float)ny,
              (float)nz, B, yz);
  float A[6], Bn[6], w[6];
  const auto each = [&](auto&& value) {
#pragma unroll
    for (int s = 0; s < 6; s++)
      if (s != 2) w[s] = value(s);
  };
#pragma unroll
  for (int s = 0; s < 6; s++) {
    if (s == 2) continue;
    const bool lo = CHAIN && s < 2;
    const float um = lo ? sum3(B.vv, d[s][2], B.uu, d[s][1], B.ww, d[s][3])
                        : sum3(B.uu, d[s][1], B.vv, d[s][2], B.ww, d[s][3]);
    const float nm = lo ? sum3(B.ny, d[s][2], B.nx, d[s][1], B.nz, d[s][3])
                        : sum3(B.nx, d[s][1], B.ny, d[s][2], B.nz, d[s][3]);
    A[s] = B.K * fma(B.k, d[s][0], d[s][4] - um);
    Bn[s] = fma(B.qn, d[s][0], -nm);
  }
  // t.m - qt rho for a tangent t
  const auto tangent = [&](int s, float tx, float ty, float tz, float qt) {
    const float two = CHAIN && s < 2 ? fma(-qt, d[s][0], tx * d[s][1])
                                     : fma(tx, d[s][1], -(qt * d[s][0]));
    return fma(tz, d[s][3], fma(ty, d[s][2], two));
  };
  float WL[5], WR[5];
  each([&](int s) { return fma(B.o, Bn[s], A[s]); });
  weno5_pair_dev(w[0], w[1], w[3], w[4], w[5], WL[0], WR[0]);
  each([&](int s) { return fma(-2.0f, A[s], d[s][0]); });
  weno5_pair_dev(w[0], w[1], w[3], w[4], w[5], WL[1], WR[1]);
  each([&](int s) { return fma(-B.o, Bn[s], A[s]); });
  weno5_pair_dev(w[0], w[1], w[3], w[4], w[5], WL[2], WR[2]);
  each([&](int s) { return tangent(s, B.lx, B.ly, B.lz, B.ql); });
  weno5_pair_dev(w[0], w[1], w[3], w[4], w[5], WL[3], WR[3]);
  each([&](int s) { return tangent(s, B.mx, B.my, B.mz, B.qm); });
  weno5_pair_dev(w[0], w[1], w[3], w[4], w[5], WL[4], WR[4]);
  lf_flux<!CHAIN>(g, char_to_side(g, B, qm, WR), char_to_side(g, B, qm, WL), nx, ny, nz, f);
}

// Deviations from node m of a 6-node stencil from its five consecutive
// differences e[k] = q[k+1] - q[k] (in T): a sweep carries the differences
// from face to face instead of forming five double differences per face.
template <class T>
__device__ __forceinline__ void dev_from_diffs(const T e[5][5], T d[6][5]) {
#pragma unroll
  for (int c = 0; c < 5; c++) {
    d[2][c] = T(0);
    d[1][c] = -e[1][c];
    d[0][c] = -(e[0][c] + e[1][c]);
    d[3][c] = e[2][c];
    d[4][c] = e[2][c] + e[3][c];
    d[5][c] = d[4][c] + e[4][c];
  }
}

// The differences of the six stencil nodes, in T.
template <class T>
__device__ __forceinline__ void stencil_diffs(const double q[6][5], T e[5][5]) {
#pragma unroll
  for (int s = 0; s < 5; s++)
#pragma unroll
    for (int n = 0; n < 5; n++) e[s][n] = (T)(q[s + 1][n] - q[s][n]);
}

}  // namespace cbns
