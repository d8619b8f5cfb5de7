// plate_adjoint.hpp -- reverse-mode derivative of a plate's contribution to a
// scalar L(K) (the adjoint of plate.rs:160-724 as folded in element_math.hpp).
//
// Given the local-frame gradient Gl = T (dL/dK_e) T^T of one element, lane p
// (row block of node p) produces its additive share of
//   * P[7]   dL/d(cm00, cm01, cm22, cb00, cb01, cb22, cs): the constitutive
//            constants, from which E, nu, t and k derivatives follow;
//   * gxl[6] dL/d(x1, y1, x2, y2, x4, y4): local nodal coordinates at fixed frame;
//   * hx, hy dL/d(omega_x, omega_y): an infinitesimal rotation of the element
//            frame, dR = [omega]x R.  K_e does not depend on the in-plane gauge
//            of the frame, so omega_z never contributes.
// plate_adjoint_finish turns the sums of the four lanes into parameter and
// world-frame nodal-coordinate gradients.  No K_e is stored: the forward
// integrals are recomputed.
#pragma once
#include <hip/hip_runtime.h>

#include "element_math.hpp"

namespace fem {

// plate_point (element_math.hpp) that also returns the reciprocals the
// reverse sweep of the point needs (plate_point_reverse_r)
__host__ __device__ inline void plate_point_x(const double xl[6], int ip, PlatePoint& o, double& rdet_o,
                                              double& rqr, double& rqs) {
  const double x1 = xl[0], y1 = xl[1], x2 = xl[2], y2 = xl[3], x4 = xl[4], y4 = xl[5];
  const double g = sqrt(double(ONE_THIRD_F32));
  const double r = (ip == 0 || ip == 3) ? g : -g;
  const double s = (ip < 2) ? g : -g;
  const double q4 = 0.25;
  const double pr = 1.0 + r, mr_ = 1.0 - r, ps = 1.0 + s, ms_ = 1.0 - s;
  const double usx = (x1 * ps - x2 * ps) + x4 * ms_, usy = (y1 * ps - y2 * ps) + y4 * ms_;
  const double urx = (x1 * pr + x2 * mr_) - x4 * pr, ury = (y1 * pr + y2 * mr_) - y4 * pr;
  const double j00 = usx * q4, j01 = usy * q4, j10 = urx * q4, j11 = ury * q4;
  const double det = j00 * j11 - j01 * j10;
  const double rdet = 1.0 / det;
  const double i00 = j11 * rdet, i01 = -j01 * rdet, i10 = -j10 * rdet, i11 = j00 * rdet;
  const double dr[4] = {q4 * ps, -q4 * ps, -q4 * ms_, q4 * ms_};
  const double ds[4] = {q4 * pr, q4 * mr_, -q4 * mr_, -q4 * pr};
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    o.dx[a] = i00 * dr[a] + i01 * ds[a];
    o.dy[a] = i10 * dr[a] + i11 * ds[a];
  }
  const double sqr = sqrt(urx * urx + ury * ury), sqs = sqrt(usx * usx + usy * usy);
  const double mr = sqr * 0.125 * rdet, ms = sqs * 0.125 * rdet;
  o.al[0] = ps * mr; o.al[1] = o.al[0]; o.al[2] = ms_ * mr; o.al[3] = o.al[2];
  o.be[0] = pr * ms; o.be[1] = mr_ * ms; o.be[2] = o.be[1]; o.be[3] = o.be[0];
  o.w = det;
  rdet_o = rdet;
  rqr = sqr > 0.0 ? 1.0 / sqr : 0.0;
  rqs = sqs > 0.0 ? 1.0 / sqs : 0.0;
}

// Reverse sweep of integration point ip: from the adjoints s7 = (g_det, g_i00,
// g_i01, g_i10, g_i11, g_mr, g_ms) of its forward quantities (det, the inverse
// Jacobian, the two MITC4 multipliers), summed over the element's rows, to
// gxl.  The point's reciprocals are given: rdet = 1 / det J and
// rqr, rqs = 1 / |(cx + r bx, cy + r by)|, 1 / |(ax + s bx, ay + s by)| (the
// MITC4 lengths; 0 where the length is 0), as the forward point formed them
__host__ __device__ inline void plate_point_reverse_r(const double xl[6], int ip, const double s7[7], double rdet,
                                                      double rqr, double rqs, double gxl[6]) {
  const double x1 = xl[0], y1 = xl[1], x2 = xl[2], y2 = xl[3], x4 = xl[4], y4 = xl[5];
  const double gs = sqrt(double(ONE_THIRD_F32));
  const double r = (ip == 0 || ip == 3) ? gs : -gs;
  const double s = (ip < 2) ? gs : -gs;
  const double q4 = 0.25;
  const double pr = 1.0 + r, mr_ = 1.0 - r, ps = 1.0 + s, ms_ = 1.0 - s;
  const double usx = (x1 * ps - x2 * ps) + x4 * ms_, usy = (y1 * ps - y2 * ps) + y4 * ms_;
  const double urx = (x1 * pr + x2 * mr_) - x4 * pr, ury = (y1 * pr + y2 * mr_) - y4 * pr;
  const double j00 = usx * q4, j01 = usy * q4, j10 = urx * q4, j11 = ury * q4;
  const double i00 = j11 * rdet, i01 = -j01 * rdet, i10 = -j10 * rdet, i11 = j00 * rdet;
  const double sqr = (urx * urx + ury * ury) * rqr, sqs = (usx * usx + usy * usy) * rqs;  // the lengths
  const double m_r = sqr * 0.125 * rdet, m_s = sqs * 0.125 * rdet;
  double g_det = s7[0];
  const double g_i00 = s7[1], g_i01 = s7[2], g_i10 = s7[3], g_i11 = s7[4], g_mr = s7[5], g_ms = s7[6];
  g_det -= (g_mr * m_r + g_ms * m_s) * rdet;
  const double g_sqr = g_mr * 0.125 * rdet, g_sqs = g_ms * 0.125 * rdet;
  double g_j11 = g_i00 * rdet, g_j01 = -g_i01 * rdet, g_j10 = -g_i10 * rdet, g_j00 = g_i11 * rdet;
  g_det -= (((g_i00 * i00 + g_i01 * i01) + g_i10 * i10) + g_i11 * i11) * rdet;
  g_j00 += g_det * j11;
  g_j11 += g_det * j00;
  g_j01 -= g_det * j10;
  g_j10 -= g_det * j01;
  const double kux = g_j00 * q4 + g_sqs * usx * rqs;
  const double kuy = g_j01 * q4 + g_sqs * usy * rqs;
  const double krx = g_j10 * q4 + g_sqr * urx * rqr;
  const double kry = g_j11 * q4 + g_sqr * ury * rqr;
  gxl[0] += kux * ps + krx * pr;
  gxl[1] += kuy * ps + kry * pr;
  gxl[2] += -kux * ps + krx * mr_;
  gxl[3] += -kuy * ps + kry * mr_;
  gxl[4] += kux * ms_ - krx * pr;
  gxl[5] += kuy * ms_ - kry * pr;
}

// h += antisymmetric parts (omega_x, omega_y) of K G^T + K^T G for a block's four
// pairs of 3x3 sub-blocks K, G (gl: 6x6 row-major, local frame).  K is given by
// its entries o (plate_block_entries: (u, v) x (u, v) and (w, theta_x, theta_y) x
// the same) and its drilling entry; the products with its zeros are left out.
__host__ __device__ inline void plate_frame_adjoint(const double o[13], double drilling, const double gl[36],
                                                    double& hx, double& hy) {
  // translations, then rotations: [[a, b], [c, d]] and the entry f of the axis
  const double sub[2][5] = {{o[0], o[1], o[2], o[3], o[4]}, {o[8], o[9], o[11], o[12], drilling}};
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const double* k = sub[h];
    const double* g = gl + 21 * h;
    const double g12 = g[8] + g[13], g02 = g[2] + g[12];
    hx += ((k[4] - k[3]) * g12 - k[2] * g[12]) - k[1] * g[2];
    hy += ((k[0] - k[4]) * g02 + k[1] * g[13]) + k[2] * g[8];
  }
  // (w, theta) and (theta, w)
  const double* g = gl + 3;
  hx += (o[5] * g[6] + o[6] * g[7]) - o[6] * g[14];
  hy += (o[5] * g[14] - o[5] * g[0]) - o[6] * g[1];
  g = gl + 18;
  hx += (o[7] * g[1] + o[10] * g[7]) - o[10] * g[14];
  hy += (o[7] * g[14] - o[7] * g[0]) - o[10] * g[6];
}

// dL/d(E, nu, t, k) from the constitutive partials: cm = E t/(1-nu^2),
// cb = E t^3/(12 (1-nu^2)), cs = E t k/(2 (1+nu)).  The derivatives by E, t and k are
// the products of the other factors: no parameter divides, so that a zero one
// (the modulus or thickness of a void) leaves every derivative finite.
__host__ __device__ inline void plate_adjoint_params(const double P[7], double E, double nu, double t, double k,
                                                     double grad_param[4]) {
  const double inv_n = 1.0 / ((1.0 - nu) * (1.0 + nu));  // 1 / (1 - nu^2)
  const double cm = E * t * inv_n;
  const double cb = E * (t * t * t) * (1.0 / 12.0) * inv_n;
  const double inv_1pn = (1.0 - nu) * inv_n;  // 1 / (1 + nu)
  const double cs = E * t * k * 0.5 * inv_1pn;
  const double h = (1.0 - nu) / 2.0;
  // membrane, bending and shear per unit of E t, E t^3 and E t k
  const double Lm = ((P[0] + nu * P[1]) + h * P[2]) * inv_n;
  const double Lb = ((P[3] + nu * P[4]) + h * P[5]) * ((1.0 / 12.0) * inv_n);
  const double Ls = P[6] * (0.5 * inv_1pn);
  const double tb = t * t * Lb, ks = k * Ls;
  const double dcm = cm * 2.0 * nu * inv_n, dcb = cb * 2.0 * nu * inv_n;
  grad_param[0] = t * ((Lm + tb) + ks);
  grad_param[1] = (((P[0] * dcm + P[1] * (cm + nu * dcm)) + P[2] * (h * dcm - 0.5 * cm)) +
                   ((P[3] * dcb + P[4] * (cb + nu * dcb)) + P[5] * (h * dcb - 0.5 * cb))) -
                  P[6] * cs * inv_1pn;
  grad_param[2] = E * ((Lm + 3.0 * tb) + ks);
  grad_param[3] = E * t * Ls;
}

// Element-level finish from the four lanes' sums.
//   loc[a][k]: local coordinates R (X_a - X_3) of the crate's nodes 1..4 (a = 0..3)
//   grad_param = dL/d(E, nu, t, k); gX[a][k] = dL/dX_a (world frame)
__host__ __device__ inline void plate_adjoint_finish(const double P[7], const double gxl_in[6], double hx, double hy,
                                                     const double loc[4][3], const double R[9], double E, double nu,
                                                     double t, double k, double grad_param[4], double gX[4][3]) {
  plate_adjoint_params(P, E, nu, t, k, grad_param);
  // frame rotation: local z of nodes 1, 2, 4 feed back through dxl = (omega x p)_{x,y}
  double gxl[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) gxl[i] = gxl_in[i];
  const int nidx[3] = {0, 1, 3};
  double gwx = hx, gwy = hy;
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const double z = loc[nidx[m]][2];
    gwx -= gxl[2 * m + 1] * z;
    gwy += gxl[2 * m] * z;
  }
  // omega from the normal n = (X4 - X3) x (X2 - X3): omega_x = n~_y/|n|, omega_y = -n~_x/|n|
  // with n~ = R dn = da41 x p2 + p4 x da21 (local frame)
  const double* p2 = loc[1];
  const double* p4 = loc[3];
  const double nx = p4[1] * p2[2] - p4[2] * p2[1], ny = p4[2] * p2[0] - p4[0] * p2[2], nz = p4[0] * p2[1] - p4[1] * p2[0];
  const double rn = rsqrt((nx * nx + ny * ny) + nz * nz);
  const double gnx = -gwy * rn, gny = gwx * rn;
  double ga[4][3];
  ga[0][0] = gxl[0]; ga[0][1] = gxl[1]; ga[0][2] = 0.0;
  ga[1][0] = gxl[2]; ga[1][1] = gxl[3]; ga[1][2] = 0.0;
  ga[3][0] = gxl[4]; ga[3][1] = gxl[5]; ga[3][2] = 0.0;
  // d n~_x = da41_y z2 - da41_z y2 + y4 da21_z - z4 da21_y
  // d n~_y = da41_z x2 - da41_x z2 + z4 da21_x - x4 da21_z
  const double g41[3] = {-gny * p2[2], gnx * p2[2], -gnx * p2[1] + gny * p2[0]};
  const double g21[3] = {gny * p4[2], -gnx * p4[2], gnx * p4[1] - gny * p4[0]};
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    ga[3][i] += g41[i];
    ga[1][i] += g21[i];
    ga[2][i] = -((ga[0][i] + ga[1][i]) + ga[3][i]);
  }
  // world frame: dL/dX = R^T dL/da
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int i = 0; i < 3; ++i) gX[a][i] = (R[0 * 3 + i] * ga[a][0] + R[1 * 3 + i] * ga[a][1]) + R[2 * 3 + i] * ga[a][2];
}

// plate_adjoint_finish for a plate whose frame is the identity and whose nodes
// lie in z = 0 with no frame-rotation sums (hx = hy = 0): the rotation term
// vanishes and the world gradient is the local one.
__host__ __device__ inline void plate_adjoint_finish_flat(const double P[7], const double gxl[6], double E, double nu,
                                                          double t, double k, double grad_param[4], double gX[4][3]) {
  plate_adjoint_params(P, E, nu, t, k, grad_param);
  const double g3x = -((gxl[0] + gxl[2]) + gxl[4]), g3y = -((gxl[1] + gxl[3]) + gxl[5]);
  gX[0][0] = gxl[0]; gX[0][1] = gxl[1];
  gX[1][0] = gxl[2]; gX[1][1] = gxl[3];
  gX[2][0] = g3x;    gX[2][1] = g3y;
  gX[3][0] = gxl[4]; gX[3][1] = gxl[5];
#pragma unroll
  for (int a = 0; a < 4; ++a) gX[a][2] = 0.0;
}

// Shear edge vectors of an element (plate_shear_vectors): v_a = (+-1/2, e12 or
// e43), u_a = (+-1/2, e14 or e23).
struct PlateEdges {
  double e12[2], e43[2], e14[2], e23[2];
};
__host__ __device__ inline PlateEdges plate_edges(const double xl[6]) {
  const double q = 0.25;
  PlateEdges o;
  o.e12[0] = -(xl[1] - xl[3]) * q; o.e12[1] = (xl[0] - xl[2]) * q;
  o.e43[0] = -xl[5] * q;           o.e43[1] = xl[4] * q;
  o.e14[0] = -(xl[1] - xl[5]) * q; o.e14[1] = (xl[0] - xl[4]) * q;
  o.e23[0] = -xl[3] * q;           o.e23[1] = xl[2] * q;
  return o;
}

// Compliance by strain energy: the share of the integration point (r, s) in
// L = -u_l^T k u_l, with U[a] = (u, v, w, theta_x, theta_y, theta_z) the
// local-frame displacements of node a.  Adds to P, gxl, hx, hy what
// the sixteen blocks of plate_adjoint_kernel add for G = -u_p u_q^T (but the
// drilling term: plate_compliance_drilling), without forming a block: each block
// term is a bilinear form in nodal values, so its contraction with u u^T is the
// point's quadratic form in the strains
//   membrane eps = (ux, vy, uy + vx), bending kappa = (ay, -bx, ax - by)
//   (a = theta_x, b = theta_y), shear gamma_r = mr rho, gamma_s = ms sigma
// (rho, sigma: the MITC4 tying sums of the shear vectors against U), and
// every derivative follows from the strains, the stress resultants and the
// natural-coordinate derivatives of U:
//   * P from the squared strains;
//   * the point's adjoints: det from the energy density, the inverse Jacobian from
//     resultant x natural derivative, mr and ms from the shear strains, and from
//     them the local coordinates (as plate_point_reverse_r, with the point's own
//     Jacobian, reciprocals and lengths);
//   * the shear vectors from the tying sums;
//   * hx, hy = -2 sum_a (x_a x f_a)_{x,y} over the translation and rotation
//     triples, f = k u_l the local nodal forces (their point share here).
__host__ __device__ inline void plate_compliance_point(const double xl[6], double r, double s, const PlateMat& m,
                                                       const PlateEdges& ed, const double U[4][6], double P[7],
                                                       double gxl[6], double& hx, double& hy) {
  const double x1 = xl[0], y1 = xl[1], x2 = xl[2], y2 = xl[3], x4 = xl[4], y4 = xl[5];
  const double q4 = 0.25;
  const double pr = 1.0 + r, mr_ = 1.0 - r, ps = 1.0 + s, ms_ = 1.0 - s;
  const double usx = (x1 * ps - x2 * ps) + x4 * ms_, usy = (y1 * ps - y2 * ps) + y4 * ms_;
  const double urx = (x1 * pr + x2 * mr_) - x4 * pr, ury = (y1 * pr + y2 * mr_) - y4 * pr;
  const double j00 = usx * q4, j01 = usy * q4, j10 = urx * q4, j11 = ury * q4;
  const double det = j00 * j11 - j01 * j10;
  const double rdet = 1.0 / det;
  const double i00 = j11 * rdet, i01 = -j01 * rdet, i10 = -j10 * rdet, i11 = j00 * rdet;
  // MITC4 lengths and their reciprocals (0 where the length is 0)
  const double qr = urx * urx + ury * ury, qs = usx * usx + usy * usy;
  const double rqr = qr > 0.0 ? rsqrt(qr) : 0.0, rqs = qs > 0.0 ? rsqrt(qs) : 0.0;
  const double r8 = 0.125 * rdet;
  const double mr = (qr * rqr) * r8, ms = (qs * rqs) * r8;
  const double dr[4] = {q4 * ps, -q4 * ps, -q4 * ms_, q4 * ms_};
  const double ds[4] = {q4 * pr, q4 * mr_, -q4 * mr_, -q4 * pr};
  // natural derivatives of u, v, theta_x, theta_y
  const int comp[4] = {0, 1, 3, 4};
  double fr[4], fs[4];
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    const int c = comp[f];
    fr[f] = q4 * (ps * (U[0][c] - U[1][c]) + ms_ * (U[3][c] - U[2][c]));
    fs[f] = q4 * (pr * (U[0][c] - U[3][c]) + mr_ * (U[1][c] - U[2][c]));
  }
  const double ux = i00 * fr[0] + i01 * fs[0], uy = i10 * fr[0] + i11 * fs[0];
  const double vx = i00 * fr[1] + i01 * fs[1], vy = i10 * fr[1] + i11 * fs[1];
  const double ax = i00 * fr[2] + i01 * fs[2], ay = i10 * fr[2] + i11 * fs[2];
  const double bx = i00 * fr[3] + i01 * fs[3], by = i10 * fr[3] + i11 * fs[3];
  // stress resultants: derivatives of the energy density phi with respect to
  // ux (Nux), vy (Nvy), uy and vx (Nxy), ay (May), bx (Mbx), ax (Mxy; by: -Mxy)
  const double exy = uy + vx, kxy = ax - by;
  const double Nux = 2.0 * (m.cm00 * ux + m.cm01 * vy);
  const double Nvy = 2.0 * (m.cm00 * vy + m.cm01 * ux);
  const double Nxy = 2.0 * m.cm22 * exy;
  const double May = 2.0 * (m.cb00 * ay - m.cb01 * bx);
  const double Mbx = 2.0 * (m.cb00 * bx - m.cb01 * ay);
  const double Mxy = 2.0 * m.cb22 * kxy;
  const double phi = 0.5 * (((Nux * ux + Nvy * vy) + Nxy * exy) + ((May * ay + Mbx * bx) + Mxy * kxy));
  // transverse shear: tying sums of the shear vectors against (w, theta_x, theta_y)
  const double t12 = 0.5 * (U[0][2] - U[1][2]) + (ed.e12[0] * (U[0][3] + U[1][3]) + ed.e12[1] * (U[0][4] + U[1][4]));
  const double t43 = 0.5 * (U[3][2] - U[2][2]) + (ed.e43[0] * (U[2][3] + U[3][3]) + ed.e43[1] * (U[2][4] + U[3][4]));
  const double t14 = 0.5 * (U[0][2] - U[3][2]) + (ed.e14[0] * (U[0][3] + U[3][3]) + ed.e14[1] * (U[0][4] + U[3][4]));
  const double t23 = 0.5 * (U[1][2] - U[2][2]) + (ed.e23[0] * (U[1][3] + U[2][3]) + ed.e23[1] * (U[1][4] + U[2][4]));
  const double rho = ps * t12 + ms_ * t43, sig = pr * t14 + mr_ * t23;
  const double gr = mr * rho, gz = ms * sig;
  const double w = det;
  // constitutive partials
  const double g2 = gr * gr + gz * gz;
  P[0] -= w * (ux * ux + vy * vy);
  P[1] -= w * (2.0 * ux * vy);
  P[2] -= w * (exy * exy);
  P[3] -= w * (ay * ay + bx * bx);
  P[4] += w * (2.0 * ay * bx);
  P[5] -= w * (kxy * kxy);
  P[6] -= w * g2;
  // the point's adjoints: det, inverse Jacobian, mr and ms
  const double cs2 = 2.0 * m.cs;
  const double g_i00 = -w * (((Nux * fr[0] + Nxy * fr[1]) + Mxy * fr[2]) + Mbx * fr[3]);
  const double g_i01 = -w * (((Nux * fs[0] + Nxy * fs[1]) + Mxy * fs[2]) + Mbx * fs[3]);
  const double g_i10 = -w * (((Nxy * fr[0] + Nvy * fr[1]) + May * fr[2]) - Mxy * fr[3]);
  const double g_i11 = -w * (((Nxy * fs[0] + Nvy * fs[1]) + May * fs[2]) - Mxy * fs[3]);
  const double wr = -w * cs2 * gr, wz = -w * cs2 * gz;
  const double g_mr = wr * rho, g_ms = wz * sig;
  double g_det = -(phi + m.cs * g2);
  g_det -= (g_mr * mr + g_ms * ms) * rdet;
  g_det -= (((g_i00 * i00 + g_i01 * i01) + g_i10 * i10) + g_i11 * i11) * rdet;
  const double g_sqr = g_mr * r8 * rqr, g_sqs = g_ms * r8 * rqs;
  const double kux = (g_i11 * rdet + g_det * j11) * q4 + g_sqs * usx;
  const double kuy = (-g_i01 * rdet - g_det * j10) * q4 + g_sqs * usy;
  const double krx = (-g_i10 * rdet - g_det * j01) * q4 + g_sqr * urx;
  const double kry = (g_i00 * rdet + g_det * j00) * q4 + g_sqr * ury;
  gxl[0] += kux * ps + krx * pr;
  gxl[1] += kuy * ps + kry * pr;
  gxl[2] += -kux * ps + krx * mr_;
  gxl[3] += -kuy * ps + kry * mr_;
  gxl[4] += kux * ms_ - krx * pr;
  gxl[5] += kuy * ms_ - kry * pr;
  // shear edge vectors: dL/d(tying sums) against the edges' rotation sums, a
  // quarter of the edge
  const double c12 = (wr * mr) * ps * q4, c43 = (wr * mr) * ms_ * q4, c14 = (wz * ms) * pr * q4, c23 = (wz * ms) * mr_ * q4;
  const double a12 = c12 * (U[0][3] + U[1][3]), b12 = c12 * (U[0][4] + U[1][4]);
  const double a43 = c43 * (U[2][3] + U[3][3]), b43 = c43 * (U[2][4] + U[3][4]);
  const double a14 = c14 * (U[0][3] + U[3][3]), b14 = c14 * (U[0][4] + U[3][4]);
  const double a23 = c23 * (U[1][3] + U[2][3]), b23 = c23 * (U[1][4] + U[2][4]);
  gxl[0] += b12 + b14;
  gxl[1] -= a12 + a14;
  gxl[2] += b23 - b12;
  gxl[3] += a12 - a23;
  gxl[4] += b43 - b14;
  gxl[5] += a14 - a43;
  // this point's share of the nodal forces f = k u_l
  const double hw = 0.5 * w;
  const double sr = (w * m.cs) * gr * mr, sz = (w * m.cs) * gz * ms;  // per unit tying sum
  const double fa[4] = {ps, ps, ms_, ms_}, fb[4] = {pr, mr_, mr_, pr};
  double ex = 0.0, ey = 0.0;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const double dxa = hw * (i00 * dr[a] + i01 * ds[a]), dya = hw * (i10 * dr[a] + i11 * ds[a]);
    const double cv = sr * fa[a], cu = sz * fb[a];
    const double* ev = a < 2 ? ed.e12 : ed.e43;
    const double* eu = (a == 0 || a == 3) ? ed.e14 : ed.e23;
    const double fu = Nux * dxa + Nxy * dya;
    const double fv = Nxy * dxa + Nvy * dya;
    const double fw = ((a == 0 || a == 3) ? 0.5 : -0.5) * cv + (a < 2 ? 0.5 : -0.5) * cu;
    const double fta = (Mxy * dxa + May * dya) + (cv * ev[0] + cu * eu[0]);
    const double ftb = (Mbx * dxa - Mxy * dya) + (cv * ev[1] + cu * eu[1]);
    ex += (U[a][1] * fw - U[a][2] * fv) - U[a][5] * ftb;
    ey += (U[a][2] * fu - U[a][0] * fw) + U[a][5] * fta;
  }
  hx -= 2.0 * ex;
  hy -= 2.0 * ey;
}

// the drilling forces' share (KROT6 on each node's theta_z)
__host__ __device__ inline void plate_compliance_drilling(const double U[4][6], double& hx, double& hy) {
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const double fz = KROT6 * U[a][5];
    hx -= 2.0 * (U[a][4] * fz);
    hy += 2.0 * (U[a][3] * fz);
  }
}

}  // namespace fem
