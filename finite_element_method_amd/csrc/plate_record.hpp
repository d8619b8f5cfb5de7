// plate_record.hpp -- element records of the plate kernels that sum node-pair
// blocks from point integrals (plate_lanes.hip, plate_frames.hip): the record's
// layout, and the 13 local entries of a node-pair block read from a record.
#pragma once

#include <hip/hip_runtime.h>

namespace femdev {

namespace {

typedef unsigned int pl_u32x2 __attribute__((ext_vector_type(2)));

// element record (doubles): Mxx (10, p <= q), Myy (10), Mxy (16, 4 p + q),
// A (3, alpha classes), B (3, beta classes), shear edge vectors (8), material (cm00, cm01,
// cm22, t^2/12, cs), pad
constexpr int PL_REC = 58;
constexpr int R_MYY = 10, R_MXY = 20, R_A = 36, R_B = 39, R_SH = 42, R_MAT = 50;
constexpr int PL_NINT = 42;

// index of the symmetric pair (a, b), a <= b, among the 10 pairs of 4 nodes
__device__ inline int sym_index(int a, int b) { return a * 4 - (a * (a - 1)) / 2 + (b - a); }

// both 32-bit halves of a double from the neighbouring lane (lane ^ 1), by DPP
__device__ inline double swap_pair(double v) {
  const pl_u32x2 x = __builtin_bit_cast(pl_u32x2, v);
  pl_u32x2 r;
  r.x = uint32_t(__builtin_amdgcn_mov_dpp(int(x.x), 0xB1, 0xF, 0xF, false));
  r.y = uint32_t(__builtin_amdgcn_mov_dpp(int(x.y), 0xB1, 0xF, 0xF, false));
  return __builtin_bit_cast(double, r);
}

__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// v with its sign flipped when neg is 1 (an exact sign change)
__device__ inline double with_sign(double v, int neg) {
  pl_u32x2 x = __builtin_bit_cast(pl_u32x2, v);
  x.y ^= uint32_t(neg) << 31;
  return __builtin_bit_cast(double, x);
}

// The 13 entries of the flat-plate block (p, q) (layout of plate_layout.hpp:
// (u,u) (u,v) | (v,u) (v,v) | (w,w) (w,tx) (w,ty) | (tx,.) | (ty,.)) from the
// six point integrals of the pair, plate.rs:513-672 folded over the 2x2 rule:
// membrane from cm * M, bending as t^2/12 times the matching membrane entry,
// MITC4 shear A cs v_p v_q^T + B cs u_p u_q^T with v_a = (sv_a / 2, ev_a),
// u_a = (su_a / 2, eu_a) (sv, su: sign bits).
__device__ inline void block_entries(double Mxx, double Mxy, double Myx, double Myy, double Acs, double Bcs,
                                     double cm00, double cm01, double cm22, double tb, double2 evp, double2 eup,
                                     double2 evq, double2 euq, int svp, int sup, int svq, int suq, double o[13]) {
  o[0] = __builtin_fma(cm00, Mxx, cm22 * Myy);
  o[1] = __builtin_fma(cm01, Mxy, cm22 * Myx);
  o[2] = __builtin_fma(cm01, Myx, cm22 * Mxy);
  o[3] = __builtin_fma(cm00, Myy, cm22 * Mxx);
  const double bxx = tb * o[3], bxy = -(tb * o[2]), byx = -(tb * o[1]), byy = tb * o[0];
  const double a[3] = {with_sign(0.5 * Acs, svp), Acs * evp.x, Acs * evp.y};
  const double b[3] = {with_sign(0.5 * Bcs, sup), Bcs * eup.x, Bcs * eup.y};
  const double vq[3] = {with_sign(0.5, svq), evq.x, evq.y};
  const double uq[3] = {with_sign(0.5, suq), euq.x, euq.y};
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) o[4 + 3 * i + j] = __builtin_fma(a[i], vq[j], b[i] * uq[j]);
  o[8] += bxx;
  o[9] += bxy;
  o[11] += byx;
  o[12] += byy;
}

// the 13 entries of block (p, q) from the element's record r
__device__ inline void record_block(const double* r, int p, int q, double o[13]) {
  const int si = sym_index(min(p, q), max(p, q));
  const double Mxx = r[si], Myy = r[R_MYY + si];
  const double Mxy = r[R_MXY + 4 * p + q], Myx = r[R_MXY + 4 * q + p];
  // alpha classes {0, 1} | {2, 3}; beta classes {0, 3} | {1, 2}
  const int bp = (p ^ (p >> 1)) & 1, bq = (q ^ (q >> 1)) & 1;
  const double Aa = r[R_A + (p >> 1) + (q >> 1)];
  const double Bb = r[R_B + bp + bq];
  // shear rows (plate.rs:452-508): v_a = (+-1/2, e), e = e12 for a in {0, 1},
  // e43 for {2, 3}, sign - for a in {1, 2}; u_a = (+-1/2, f), f = e14 for
  // a in {0, 3}, e23 for {1, 2}, sign - for a in {2, 3}
  const double2 evp = *reinterpret_cast<const double2*>(r + R_SH + 2 * (p >> 1));
  const double2 evq = *reinterpret_cast<const double2*>(r + R_SH + 2 * (q >> 1));
  const double2 eup = *reinterpret_cast<const double2*>(r + R_SH + 4 + 2 * bp);
  const double2 euq = *reinterpret_cast<const double2*>(r + R_SH + 4 + 2 * bq);
  const double2 m0 = *reinterpret_cast<const double2*>(r + R_MAT);
  const double2 m1 = *reinterpret_cast<const double2*>(r + R_MAT + 2);
  const double cs = r[R_MAT + 4];
  block_entries(Mxx, Mxy, Myx, Myy, Aa * cs, Bb * cs, m0.x, m0.y, m1.x, m1.y, evp, eup, evq, euq, bp, p >> 1,
                bq, q >> 1, o);
}

}  // namespace

}  // namespace femdev
