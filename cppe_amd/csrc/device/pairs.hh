// Pair field kernels shared by the direct and FMM near-field paths.
#pragma once
#include "common.hh"

namespace cppe_dev {

// v where keep has all bits set, zero where it has none (of any v, infinities included).
__device__ __forceinline__ float kept(float v, int keep) {
  return __builtin_bit_cast(float, __builtin_bit_cast(int, v) & keep);
}
__device__ __forceinline__ double kept(double v, int keep) {
  int2 b = __builtin_bit_cast(int2, v);
  b.x &= keep;
  b.y &= keep;
  return __builtin_bit_cast(double, b);
}
// that mask from bit t of skip
__device__ __forceinline__ int keep_unless(unsigned skip, int t) {
  return __builtin_amdgcn_sbfe((int)~skip, t, 1);  // (shifts the compiler turns into a compare and a select)
}

// ---------------------------------------------------------------------------------------------
// Pair kernels. d = r_target - r_source.
// ---------------------------------------------------------------------------------------------
// -T2 mu with Thole damping: fE mu / R^3 - 3 fT (d.mu) d / R^5  (P2P<1,3>, field_m1.cc:127-193),
// split into the pair's geometry (c3 = fE / R^3, cf = 3 fT / R^5) and the accumulation of one
// dipole, so that several dipole vectors can share one geometry evaluation.
// SELF0: a zero displacement (a site with itself) contributes exactly zero. keep: all bits set, or none: so does
// this pair then, whatever its displacement (1/R is masked: one and-operation for 32 bits).
template <bool DAMP, bool SELF0 = false>
__device__ __forceinline__ void geo_m1_f64(double dx, double dy, double dz, double a, double& c3, double& cf,
                                           int keep = -1) {
  const double r2   = dx * dx + dy * dy + dz * dz;
  const double rsq  = rsqrt_f64(r2);
  const double rinv = SELF0 ? (r2 > 0.0 ? rsq : 0.0) : kept(rsq, keep);
  const double ri2  = rinv * rinv;
  const double ri3  = rinv * ri2;
  double fE = 1.0, fT = 1.0;
  if (DAMP) {
    const double u = a * (r2 * rinv);
    if (u < kTholeCutoff && a > 0.0) thole_ET(u, exp(-u), fE, fT);
  }
  c3 = fE * ri3;
  cf = (3.0 * fT) * (ri3 * ri2);
}

template <bool DAMP, bool SELF0 = false>
__device__ __forceinline__ void geo_m1_f32(float dx, float dy, float dz, float a, float& c3, float& cf,
                                           int keep = -1) {
  const float r2   = dx * dx + dy * dy + dz * dz;
  const float rsq  = rsqrt_f32(r2);
  const float rinv = SELF0 ? (r2 > 0.0f ? rsq : 0.0f) : kept(rsq, keep);
  const float ri2  = rinv * rinv;
  const float ri3  = rinv * ri2;
  float fE = 1.0f, fT = 1.0f;
  if (DAMP) {
    const float u = a * (r2 * rinv);
    if (u < kTholeCutoff32 && a > 0.0f) thole_ET(u, expm_f32(u), fE, fT);
  }
  c3 = fE * ri3;
  cf = (3.0f * fT) * (ri3 * ri2);
}

// FP32 damped pair geometry for systems whose sites are all damped (alpha_iso > 0 everywhere),
// without branches. a2 = damping (s_i s_j) log2(e), so u2 = a2 R is the Thole argument v in
// base-2 units (v = u2 ln 2) and e^-v = 2^-u2 comes straight from v_exp_f32. With v = u2 ln2
//   f_E = 1 - (1 + ln2 u2 + (ln2)^2/2 u2^2) 2^-u2,   f_T = f_E - (ln2)^3/6 u2^3 2^-u2.
// SELF0: a zero displacement (the site itself) contributes exactly zero: 1/R is clamped to 2^40, so
// R = 0, u2 = 0, 2^-u2 = 1 and f_E = f_T = 0 exactly (this needs a2 finite, i.e. damped sites). keep as above.
// Large u2 (undamped in effect) gives 2^-u2 = 0 and f_E = f_T = 1.
template <bool SELF0>
__device__ __forceinline__ void geo_m1_f32_b2(float dx, float dy, float dz, float a2, float& c3, float& cf,
                                              int keep = -1) {
  constexpr float kC1 = 0.693147180559945309f;   // ln 2
  constexpr float kC2 = 0.240226506959100712f;   // (ln 2)^2 / 2
  constexpr float kC3 = 0.0555041086648215800f;  // (ln 2)^3 / 6
  const float r2   = dx * dx + dy * dy + dz * dz;
  const float rsq  = rsqrt_f32(r2);
  const float rinv = SELF0 ? __builtin_fminf(rsq, 1099511627776.0f) /* 2^40 */ : kept(rsq, keep);
  const float ri2  = rinv * rinv;
  const float ri3  = ri2 * rinv;
  const float u    = a2 * (r2 * rinv);
  const float e    = __builtin_amdgcn_exp2f(-u);
  const float u2   = u * u;
  const float p    = __builtin_fmaf(u2, kC2, __builtin_fmaf(u, kC1, 1.0f));
  const float fE   = __builtin_fmaf(-e, p, 1.0f);
  const float q    = (u2 * u) * e;
  const float fT   = __builtin_fmaf(-kC3, q, fE);
  c3 = fE * ri3;
  cf = (fT * ri3) * (3.0f * ri2);  // in this order: at R = 0, ri3 ri2 = 2^200 would overflow
}

// field += c3 mu - cf (d.mu) d
__device__ __forceinline__ void acc_m1(double c3, double cf, double dx, double dy, double dz, double mx, double my,
                                       double mz, double& fx, double& fy, double& fz) {
  const double c5 = cf * (dx * mx + dy * my + dz * mz);
  fx = __builtin_fma(c3, mx, fx);
  fx = __builtin_fma(-c5, dx, fx);
  fy = __builtin_fma(c3, my, fy);
  fy = __builtin_fma(-c5, dy, fy);
  fz = __builtin_fma(c3, mz, fz);
  fz = __builtin_fma(-c5, dz, fz);
}

__device__ __forceinline__ void acc_m1(float c3, float cf, float dx, float dy, float dz, float mx, float my,
                                       float mz, float& fx, float& fy, float& fz) {
  const float c5 = cf * (dx * mx + dy * my + dz * mz);
  fx = __builtin_fmaf(c3, mx, fx);
  fx = __builtin_fmaf(-c5, dx, fx);
  fy = __builtin_fmaf(c3, my, fy);
  fy = __builtin_fmaf(-c5, dy, fy);
  fz = __builtin_fmaf(c3, mz, fz);
  fz = __builtin_fmaf(-c5, dz, fz);
}

// FP32 undamped pair in the form field += R^-3 (mu - 3 R^-2 (d.mu) d): the same tensor as
// c3 mu - cf (d.mu) d with c3 = R^-3, cf = 3 R^-5, one multiply fewer per pair (no R^-5).
// The displacement must be nonzero.
__device__ __forceinline__ void geo_far_f32(float dx, float dy, float dz, float& ri3, float& m3) {
  const float r2   = dx * dx + dy * dy + dz * dz;
  const float rinv = rsqrt_f32(r2);
  const float ri2  = rinv * rinv;
  ri3 = ri2 * rinv;
  m3  = -3.0f * ri2;
}

__device__ __forceinline__ void acc_far_f32(float ri3, float m3, float dx, float dy, float dz, float mx, float my,
                                            float mz, float& fx, float& fy, float& fz) {
  const float q = m3 * (dx * mx + dy * my + dz * mz);
  fx = __builtin_fmaf(ri3, __builtin_fmaf(q, dx, mx), fx);
  fy = __builtin_fmaf(ri3, __builtin_fmaf(q, dy, my), fy);
  fz = __builtin_fmaf(ri3, __builtin_fmaf(q, dz, mz), fz);
}

template <bool DAMP, bool SELF0 = false>
__device__ __forceinline__ void pair_m1_f64(double dx, double dy, double dz, double mx, double my, double mz, double a,
                                            double& fx, double& fy, double& fz) {
  double c3, cf;
  geo_m1_f64<DAMP, SELF0>(dx, dy, dz, a, c3, cf);
  acc_m1(c3, cf, dx, dy, dz, mx, my, mz, fx, fy, fz);
}

template <bool DAMP, bool SELF0 = false>
__device__ __forceinline__ void pair_m1_f32(float dx, float dy, float dz, float mx, float my, float mz, float a,
                                            float& fx, float& fy, float& fz) {
  float c3, cf;
  geo_m1_f32<DAMP, SELF0>(dx, dy, dz, a, c3, cf);
  acc_m1(c3, cf, dx, dy, dz, mx, my, mz, fx, fy, fz);
}

// A static source site as the field kernels read it (device order): position, Thole scale, charge,
// dipole, the quadrupole matrix of the half-diagonal packing S (2 S0, S1, S2, 2 S3, S4, 2 S5) and its
// half trace tr = S0 + S3 + S5.
struct StaticRec {
  double x, y, z, s;
  double q, mx, my, mz;
  double xx, xy, xz, yy;
  double yz, zz, tr, pad;
};

// Static field of charge + dipole + quadrupole, combined as F(m0) - F(m1) + F(m2)
// (electric_fields.cc:163,174,186), with Thole factors from f_V/R:
//   m0: +q fE d/R^3
//   -m1: 3 fT (d.mu) d/R^5 - fE mu/R^3
//   m2: 15 fD P d/R^7 - 3 fT (tr d + Q d)/R^5, Q the source's matrix, 2 P = d.Q d
// gathered by powers of 1/R: with c5 = 3/R^5,
//   F = (fE q/R^3 + c5 (fT (d.mu - tr) + 5/2 fD (2 P)/R^2)) d - fE/R^3 mu - fT c5 Q d.
// KIND: 3 all three, 0 the charge only, 1 the dipole only (its sign as above), 2 the quadrupole only.
// About 46 FP64 instructions for an undamped pair of kind 3 (76 with the terms evaluated one by one).
template <int KIND, bool DAMP>
__device__ __forceinline__ void pair_static(double xi, double yi, double zi, double di, const StaticRec& r, double& fx,
                                            double& fy, double& fz) {
  const double dx = xi - r.x, dy = yi - r.y, dz = zi - r.z;
  const double r2   = dx * dx + dy * dy + dz * dz;
  const double rinv = rsqrt_f64(r2);
  const double ri2  = rinv * rinv;
  const double ri3  = rinv * ri2;
  double fE = 1.0, fT = 1.0, fD = 1.0;
  if (DAMP) {
    const double a = di * r.s;
    const double u = a * (r2 * rinv);
    if (u < kTholeCutoff && a > 0.0) {
      const double e = exp(-u);
      thole_ET(u, e, fE, fT);
      const double u2 = u * u;
      fD = fT - (u2 * u2 * (1.0 / 30.0)) * e;
    }
  }
  const double e3 = fE * ri3;
  if (KIND == 0) {
    const double cd = r.q * e3;
    fx += cd * dx;
    fy += cd * dy;
    fz += cd * dz;
    return;
  }
  const double c5 = 3.0 * ri3 * ri2;
  double g = 0.0, qx = 0.0, qy = 0.0, qz = 0.0;
  if (KIND == 1 || KIND == 3) g = dx * r.mx + dy * r.my + dz * r.mz;
  if (KIND == 2 || KIND == 3) {
    qx = r.xx * dx + r.xy * dy + r.xz * dz;
    qy = r.xy * dx + r.yy * dy + r.yz * dz;
    qz = r.xz * dx + r.yz * dy + r.zz * dz;
    g -= r.tr;
  }
  g *= fT;
  if (KIND == 2 || KIND == 3) g += (2.5 * fD * ri2) * (dx * qx + dy * qy + dz * qz);
  double cd = c5 * g;
  if (KIND == 3) cd += r.q * e3;
  fx += cd * dx;
  fy += cd * dy;
  fz += cd * dz;
  if (KIND == 1 || KIND == 3) {
    fx -= e3 * r.mx;
    fy -= e3 * r.my;
    fz -= e3 * r.mz;
  }
  if (KIND == 2 || KIND == 3) {
    const double t5 = fT * c5;
    fx -= t5 * qx;
    fy -= t5 * qy;
    fz -= t5 * qz;
  }
}

// i == j or j listed in the CSR exclusions of i (device order).
__device__ __forceinline__ bool excluded(int i, int j, const int* __restrict__ eoff,
                                         const int* __restrict__ eidx) {
  if (i == j) return true;
  if (eoff) {
    const int e0 = eoff[i], e1 = eoff[i + 1];
    for (int k = e0; k < e1; ++k)
      if (eidx[k] == j) return true;
  }
  return false;
}

// The exclusions of one site in registers: its first four partners, and the range of any others
// (searched in the list only inside that range).
struct SiteExclusions {
  int i, p[4], lo, hi;
  __device__ __forceinline__ SiteExclusions() {}
  __device__ __forceinline__ SiteExclusions(int i_, const int* __restrict__ eoff, const int* __restrict__ eidx)
      : i(i_), lo(0x7fffffff), hi(-1) {
    const int k0 = eoff ? eoff[i] : 0, k1 = eoff ? eoff[i + 1] : 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) p[k] = k0 + k < k1 ? eidx[k0 + k] : -1;
    for (int k = k0 + 4; k < k1; ++k) {
      const int e = eidx[k];
      if (e >= 0) {
        lo = min(lo, e);
        hi = max(hi, e);
      }
    }
  }
  // whether a source in [j0, j1) may be excluded (the site itself is)
  __device__ __forceinline__ bool meets(int j0, int j1) const {
    bool h = (i >= j0 && i < j1) || (lo < j1 && hi >= j0);
#pragma unroll
    for (int k = 0; k < 4; ++k) h = h || (p[k] >= j0 && p[k] < j1);
    return h;
  }
  __device__ __forceinline__ bool excludes(int j, const int* __restrict__ eoff, const int* __restrict__ eidx) const {
    if (j == i || j == p[0] || j == p[1] || j == p[2] || j == p[3]) return true;
    return j >= lo && j <= hi && excluded(i, j, eoff, eidx);
  }
};

}  // namespace cppe_dev
