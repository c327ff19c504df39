// Device helpers shared by the HIP translation units.
#pragma once

#include <hip/hip_runtime.h>

namespace aster {

// One coordinate of a body's kick/drift (update_leapfrog,
// src/physics/tool_chain_impl.cpp:169-185): the previous stage's second
// half-kick (dt_prev, when not 0), the drift and this stage's first
// half-kick, all with the same acceleration, in the reference's operation
// order and without contraction.
__device__ __forceinline__ void kick_drift_1(double& x, double& v, double a, double dt_prev, double dt) {
#pragma clang fp contract(off)
  double vc = v;
  if (dt_prev != 0.0) vc = vc + 0.5 * a * dt_prev;
  x = x + (vc * dt + 0.5 * a * dt * dt);
  v = vc + 0.5 * a * dt;
}

// The closing half-kick alone.
__device__ __forceinline__ double kick_1(double v, double a, double dt) {
#pragma clang fp contract(off)
  return v + 0.5 * a * dt;
}

// One coordinate of a SABA stage (src/integrators/SABA.cpp:19-553): v += (a d)
// dt, then x += (v c) dt with the kicked v; after a step's last stage also the
// next step's opening drift (cd_next, when not 0), as an addition of its own.
__device__ __forceinline__ void saba_1(double& x, double& v, double a, double d, double cd, double cd_next,
                                       double dt) {
#pragma clang fp contract(off)
  v = v + a * d * dt;
  x = x + v * cd * dt;
  if (cd_next != 0.0) x = x + v * cd_next * dt;
}

// ---- correctly rounded FP64 reciprocal square root and division ----------
//
// The reference's 1.0 / sqrt(r2) and f / m1 round twice and once; the results
// here are those doubles, at 14 + v_rsq_f64 and 4 instructions instead of
// about 30 and 10. Newton-Raphson with fused multiply-adds and an exact
// residual at the end (Markstein, IBM J. Res. Dev. 34, 111 (1990)): a quotient
// or root within one unit in the last place, corrected by its exact residual
// times a reciprocal that is good to half a unit, is the correctly rounded
// one. Ranges are the caller's business: no scaling is done.

__device__ __forceinline__ uint32_t hi32(double x) {
  return (uint32_t)((unsigned long long)__double_as_longlong(x) >> 32);
}
__device__ __forceinline__ uint32_t lo32(double x) { return (uint32_t)(unsigned long long)__double_as_longlong(x); }

// 1 / sqrt(x), both rounded, for N values x in [2^-700, 2^700], step by step
// together (their chains overlap; left alone the compiler runs one after the
// other). A root whose mantissa is all ones is the reciprocal's exception (the
// residual step would see a tie): returns whether a root ends in 32 ones; such
// results must not be used.
template <int N>
__device__ __forceinline__ bool inv_sqrt64_fast(const double* x, double* r) {
#pragma clang fp contract(off)
  double g[N], h[N], e[N], s[N];
#define ASTER_EACH(expr)                      \
  _Pragma("unroll") for (int q = 0; q < N; ++q) { expr; } \
  if (N > 1) __builtin_amdgcn_sched_barrier(0);
  ASTER_EACH(e[q] = __builtin_amdgcn_rsq(x[q]))  // to 2^-24
  ASTER_EACH(g[q] = x[q] * e[q])                 // sqrt(x)
  ASTER_EACH(h[q] = 0.5 * e[q])                  // 1 / (2 sqrt(x))
  ASTER_EACH(e[q] = fma(-h[q], g[q], 0.5))
  ASTER_EACH(g[q] = fma(g[q], e[q], g[q]))
  ASTER_EACH(h[q] = fma(h[q], e[q], h[q]))  // both to 2^-47
  ASTER_EACH(e[q] = fma(-g[q], g[q], x[q]))
  ASTER_EACH(g[q] = fma(e[q], h[q], g[q]))  // to one unit
  ASTER_EACH(e[q] = fma(-h[q], g[q], 0.5))
  ASTER_EACH(s[q] = fma(-g[q], g[q], x[q]))
  ASTER_EACH(h[q] = fma(h[q], e[q], h[q]))  // to half a unit
  ASTER_EACH(s[q] = fma(s[q], h[q], g[q]))  // the root
  ASTER_EACH(r[q] = h[q] + h[q])
  ASTER_EACH(e[q] = fma(-s[q], r[q], 1.0))
  ASTER_EACH(r[q] = fma(e[q], r[q], r[q]))
#undef ASTER_EACH
  bool odd = false;
#pragma unroll
  for (int q = 0; q < N; ++q) odd = odd || lo32(s[q]) == 0xffffffffu;
  return odd;
}

__device__ __forceinline__ double inv_sqrt64(double x) {
#pragma clang fp contract(off)
  double r;
  const bool odd = inv_sqrt64_fast<1>(&x, &r);
  // [2^-700, 2^700] by the exponent; also 0, negative numbers, infinity, NaN
  if (__builtin_expect(odd || hi32(x) - 0x14300000u >= 0x6bb00000u - 0x14300000u, 0)) r = 1.0 / sqrt(x);
  return r;
}

// A divisor with its reciprocal in two parts: y = 1 / b rounded, yl = 1 / b - y.
struct Divisor64 {
  double b, y, yl;
};
__device__ __forceinline__ Divisor64 divisor64(double b) {
#pragma clang fp contract(off)
  const double y = 1.0 / b;
  return {b, y, fma(-b, y, 1.0) * y};
}

// a / b in place for N values a, step by step together; a = 0 or |a| in
// [2^-960, 2^960], the quotient normal or 0. (A zero quotient may lose its
// sign.) The quotient of the first two steps is off by at most one unit.
template <int N>
__device__ __forceinline__ void div64_fast(double* a, const Divisor64& d) {
#pragma clang fp contract(off)
  double u[N], e[N];
#define ASTER_EACH(expr)                      \
  _Pragma("unroll") for (int q = 0; q < N; ++q) { expr; } \
  if (N > 1) __builtin_amdgcn_sched_barrier(0);
  ASTER_EACH(u[q] = a[q] * d.y)
  ASTER_EACH(u[q] = fma(a[q], d.yl, u[q]))
  ASTER_EACH(e[q] = fma(-u[q], d.b, a[q]))
  ASTER_EACH(a[q] = fma(e[q], d.y, u[q]))
#undef ASTER_EACH
}

// |x| = 0 or in [2^(lo - 1023), 2^(hi - 1023)): by the exponent field.
__device__ __forceinline__ bool zero_or_within64(double x, uint32_t lo, uint32_t hi) {
  return x == 0.0 || (hi32(x) & 0x7fffffffu) - (lo << 20) < ((hi - lo) << 20);
}

// Inputs for which the Newtonian pair force and its division by m1 stay inside
// the ranges above: coordinates 0 or 2^-100..2^100, masses 2^-150..2^150, |G|
// 2^-100..2^100 or 0, softening 0 or 2^-300..2^200. Then a separation is 0 or
// 2^-152..2^102, r^2 2^-304..2^205 (or 0: the result is NaN either way), the
// force 0 or 2^-860..2^705 and the quotient 0 or 2^-1010..2^855.
__device__ __forceinline__ bool coord_in_range64(double x) { return zero_or_within64(x, 1023 - 100, 1023 + 100); }
__device__ __forceinline__ bool mass_in_range64(double m) { return m > 0.0 && zero_or_within64(m, 1023 - 150, 1023 + 150); }
__device__ __forceinline__ bool law_in_range64(double G, double soft) {
  return zero_or_within64(G, 1023 - 100, 1023 + 100) && zero_or_within64(soft, 1023 - 300, 1023 + 200);
}

// get_pn1 (src/physics/tool_chain_impl.cpp:110-118) evaluated in the
// reference's operation order; `n` is the caller's -norm (:133).
__device__ __forceinline__ void pn1_term64(double m1, double m2, double v1x, double v1y, double v1z, double v2x,
                                           double v2y, double v2z, double inv_r, double nx, double ny, double nz,
                                           double G, double& ax, double& ay, double& az) {
#pragma clang fp contract(off)
  const double v2_sq = v2x * v2x + v2y * v2y + v2z * v2z;
  const double v1_sq = v1x * v1x + v1y * v1y + v1z * v1z;
  const double dot4 = (4.0 * v1x) * v2x + (4.0 * v1y) * v2y + (4.0 * v1z) * v2z;
  const double nv2 = nx * v2x + ny * v2y + nz * v2z;
  double s = -v1_sq - 2.0 * v2_sq;
  s = s + dot4;
  s = s + 1.5 * (nv2 * nv2);
  s = s + 5.0 * G * m1 * inv_r;
  s = s + 4.0 * G * m2 * inv_r;
  ax = nx * s;
  ay = ny * s;
  az = nz * s;
  const double n4v1 = (nx * 4.0) * v1x + (ny * 4.0) * v1y + (nz * 4.0) * v1z;
  const double n3v2 = (nx * 3.0) * v2x + (ny * 3.0) * v2y + (nz * 3.0) * v2z;
  const double t = n4v1 - n3v2;
  ax = ax + (v1x - v2x) * t;
  ay = ay + (v1y - v2y) * t;
  az = az + (v1z - v2z) * t;
  ax = ax * G * m2 * inv_r * inv_r;
  ay = ay * G * m2 * inv_r * inv_r;
  az = az * G * m2 * inv_r * inv_r;
}

// get_pn2 (tool_chain_impl.cpp:87-107), the two-body 2PN acceleration of
// body 1, in the reference's operation order: every product left to right,
// every sum left to right, the fraction constants folded as written (3.0/2.0,
// 52.0/3.0, ...). `n` is the caller's -norm.
__device__ __forceinline__ void pn2_term64(double m1, double m2, double v1x, double v1y, double v1z, double v2x,
                                           double v2y, double v2z, double inv_r, double nx, double ny, double nz,
                                           double G, double& ax, double& ay, double& az) {
#pragma clang fp contract(off)
  const double v2_sq = v2x * v2x + v2y * v2y + v2z * v2z;
  const double v1_sq = v1x * v1x + v1y * v1y + v1z * v1z;
  const double v_prod = v1x * v2x + v1y * v2y + v1z * v2z;
  const double nv1 = nx * v1x + ny * v1y + nz * v1z;
  const double nv2 = nx * v2x + ny * v2y + nz * v2z;
  const double nv22 = nv2 * nv2;
  const double pn_1 = G * m1 * inv_r;
  const double pn_2 = G * m2 * inv_r;
  const double nv12 = nv1 * nv1;
  double A = -2.0 * v2_sq * v2_sq + 4.0 * v2_sq * v_prod;
  A = A - 2.0 * v_prod * v_prod;
  A = A + 3.0 / 2.0 * v1_sq * nv22;
  A = A + 9.0 / 2.0 * v2_sq * nv22;
  A = A - 6.0 * v_prod * nv22;
  A = A - 15.0 / 8.0 * nv22 * nv22;
  double g1 = -15.0 / 4.0 * v1_sq + 5.0 / 4.0 * v2_sq;
  g1 = g1 - 5.0 / 2.0 * v_prod;
  g1 = g1 + 39.0 / 2.0 * nv12;
  g1 = g1 - 39.0 * nv1 * nv2;
  g1 = g1 + 17.0 / 2.0 * nv22;
  A = A + pn_1 * g1;
  double g2 = 4.0 * v2_sq - 8.0 * v_prod;
  g2 = g2 + 2.0 * nv12;
  g2 = g2 - 4.0 * nv1 * nv2;
  g2 = g2 - 6.0 * nv22;
  A = A + pn_2 * g2;
  double B = v1_sq * nv2 + 4.0 * v2_sq * nv1;
  B = B - 5.0 * v2_sq * nv2;
  B = B - 4.0 * v_prod * nv1;
  B = B + 4.0 * v_prod * nv2;
  B = B - 6.0 * nv1 * nv22;
  B = B + 9.0 / 2.0 * nv22 * nv2;
  B = B + pn_1 * (-63.0 / 4.0 * nv1 + 55.0 / 4.0 * nv2);
  B = B + pn_2 * (-2.0 * nv1 - 2.0 * nv2);
  const double s1 = G * m2 * inv_r * inv_r;
  const double s2 = G * G * G * m2 * inv_r * inv_r * inv_r * inv_r;
  double C = -57.0 / 4.0 * m1 * m1 - 9.0 * m2 * m2;
  C = C - 69.0 / 2.0 * m1 * m2;
  ax = (nx * A + (v1x - v2x) * B) * s1 + (nx * s2) * C;
  ay = (ny * A + (v1y - v2y) * B) * s1 + (ny * s2) * C;
  az = (nz * A + (v1z - v2z) * B) * s1 + (nz * s2) * C;
}

// get_pn25 (tool_chain_impl.cpp:73-84), the two-body 2.5PN radiation-reaction
// acceleration of body 1, in the reference's operation order. `n` is the
// caller's -norm.
__device__ __forceinline__ void pn25_term64(double m1, double m2, double v1x, double v1y, double v1z, double v2x,
                                            double v2y, double v2z, double inv_r, double nx, double ny, double nz,
                                            double G, double& ax, double& ay, double& az) {
#pragma clang fp contract(off)
  const double pn_1 = G * m1 * inv_r;
  const double pn_2 = G * m2 * inv_r;
  const double dvx = v1x - v2x, dvy = v1y - v2y, dvz = v1z - v2z;
  const double sq = dvx * dvx + dvy * dvy + dvz * dvz;
  const double k1 = -sq + 2.0 * pn_1 - 8.0 * pn_2;
  const double ndv = (nx * v1x + ny * v1y + nz * v1z) - (nx * v2x + ny * v2y + nz * v2z);
  const double k2 = 3.0 * sq - 6.0 * pn_1 + 52.0 / 3.0 * pn_2;
  double w[3] = {dvx * k1 + (nx * ndv) * k2, dvy * k1 + (ny * ndv) * k2, dvz * k1 + (nz * ndv) * k2};
#pragma unroll
  for (int c = 0; c < 3; ++c) w[c] = w[c] * 4.0 / 5.0 * G * G * m1 * m2 * inv_r * inv_r * inv_r;
  ax = w[0];
  ay = w[1];
  az = w[2];
}

// The post-Newtonian terms of compute_gravitational (tool_chain_impl.cpp:
// 129-136) that `pnf` selects (ASTER_PN1 0x10, ASTER_PN2 0x100, ASTER_PN25
// 0x1000), each scaled by 1/c^k (products of ic = 1/c taken left to right)
// and by m1, added to the force f in the reference's order.
__device__ __forceinline__ void pn_add64(int pnf, double m1, double m2, double v1x, double v1y, double v1z,
                                         double v2x, double v2y, double v2z, double inv_r, double nx, double ny,
                                         double nz, double G, double ic, double& fx, double& fy, double& fz) {
#pragma clang fp contract(off)
  double px, py, pz;
  if (pnf & 0x10) {
    const double ic2 = ic * ic;
    pn1_term64(m1, m2, v1x, v1y, v1z, v2x, v2y, v2z, inv_r, nx, ny, nz, G, px, py, pz);
    fx = fx + (px * ic2) * m1;
    fy = fy + (py * ic2) * m1;
    fz = fz + (pz * ic2) * m1;
  }
  if (pnf & 0x100) {
    const double ic4 = ic * ic * ic * ic;
    pn2_term64(m1, m2, v1x, v1y, v1z, v2x, v2y, v2z, inv_r, nx, ny, nz, G, px, py, pz);
    fx = fx + (px * ic4) * m1;
    fy = fy + (py * ic4) * m1;
    fz = fz + (pz * ic4) * m1;
  }
  if (pnf & 0x1000) {
    const double ic5 = ic * ic * ic * ic * ic;
    pn25_term64(m1, m2, v1x, v1y, v1z, v2x, v2y, v2z, inv_r, nx, ny, nz, G, px, py, pz);
    fx = fx + (px * ic5) * m1;
    fy = fy + (py * ic5) * m1;
    fz = fz + (pz * ic5) * m1;
  }
}

// compute_gravitational (tool_chain_impl.cpp:120-137): force on body 1 from
// body 2 in the reference's operation order (IEEE division and square root,
// no contraction), with the post-Newtonian terms `pnf` selects. ic = 1/c.
// The caller divides by m1 (builder_endpoint.cpp:747-752) or multiplies by
// 1/m1 (barnes_hut.cpp:238-239).
__device__ __forceinline__ void grav64(double m1, double m2, double v1x, double v1y, double v1z, double v2x,
                                       double v2y, double v2z, double p1x, double p1y, double p1z, double p2x,
                                       double p2y, double p2z, double G, double ic, double soft, int pnf,
                                       double& fx, double& fy, double& fz) {
#pragma clang fp contract(off)
  const double dx = p2x - p1x, dy = p2y - p1y, dz = p2z - p1z;
  const double r2 = dx * dx + dy * dy + dz * dz + soft;
  const double inv_r = inv_sqrt64(r2);
  const double inv_r2 = inv_r * inv_r;
  const double nx = dx * inv_r, ny = dy * inv_r, nz = dz * inv_r;
  const double scal = G * m2 * m1 * inv_r2;
  fx = nx * scal;
  fy = ny * scal;
  fz = nz * scal;
  if (pnf) pn_add64(pnf, m1, m2, v1x, v1y, v1z, v2x, v2y, v2z, inv_r, -nx, -ny, -nz, G, ic, fx, fy, fz);
}

// 1/sqrt(x) in FP64: hardware estimate (v_rsq_f64, relative error up to
// 5.2e-8) plus Newton steps y += y/2 (1 - x y^2). Measured over log-uniform x
// in [1e-30, 1e30] against a long double reference: one step 4.1e-15, two
// steps 1.4e-16 (under one ulp). Not bit-identical to 1.0/sqrt(x).
template <int STEPS>
__device__ __forceinline__ double rsqrt64_n(double x) {
  double y = __builtin_amdgcn_rsq(x);
#pragma unroll
  for (int it = 0; it < STEPS; ++it) {
    const double p = x * y;
    const double e = fma(-p, y, 1.0);
    y = fma(0.5 * y, e, y);
  }
  return y;
}
__device__ __forceinline__ double rsqrt64(double x) { return rsqrt64_n<2>(x); }

// The unused high word of a mass slot that was read counts as used here, so that
// its register is not taken for another value while the read is in flight (the
// wait on it would end the read-ahead of tile_sums). No instruction.
__device__ __forceinline__ void hold_pad(const float4&) {}
__device__ __forceinline__ void hold_pad(const double4& q) {
  asm volatile("" ::"v"((unsigned)((unsigned long long)__double_as_longlong(q.w) >> 32)));
}

// Kahan-compensated FP32 accumulation: s + (-c) carries the running sum.
__device__ __forceinline__ void kahan_add32(float& s, float& c, float t) {
  const float y = t - c;
  const float u = s + y;
  c = (u - s) - y;
  s = u;
}

// Stumpff functions c0..c3 of z: quarter z until |z| <= 0.1, 8-term nested
// series (multiplying by reciprocal constants folded at compile time, no
// division), then c3 = (c2 + c0 c3)/4, c2 = c1^2/2, c1 = c0 c1,
// c0 = 2 c0^2 - 1 once per quartering. Only +, -, *, / in a fixed order, so the result is
// the same bits on any IEEE machine (contraction off).
__device__ __forceinline__ void stumpff64(double z, double& c0, double& c1, double& c2, double& c3) {
#pragma clang fp contract(off)
  int nq = 0;
  while (fabs(z) > 0.1) {
    z = z * 0.25;
    ++nq;
  }
  c2 = 0.5 * (1.0 - z * (1.0 / 12.0) * (1.0 - z * (1.0 / 30.0) * (1.0 - z * (1.0 / 56.0) *
       (1.0 - z * (1.0 / 90.0) * (1.0 - z * (1.0 / 132.0) * (1.0 - z * (1.0 / 182.0) *
       (1.0 - z * (1.0 / 240.0) * (1.0 - z * (1.0 / 306.0)))))))));
  c3 = (1.0 / 6.0) * (1.0 - z * (1.0 / 20.0) * (1.0 - z * (1.0 / 42.0) * (1.0 - z * (1.0 / 72.0) *
       (1.0 - z * (1.0 / 110.0) * (1.0 - z * (1.0 / 156.0) * (1.0 - z * (1.0 / 210.0) *
       (1.0 - z * (1.0 / 272.0) * (1.0 - z * (1.0 / 342.0)))))))));
  c1 = 1.0 - z * c3;
  c0 = 1.0 - z * c2;
  for (int k = 0; k < nq; ++k) {
    c3 = (c2 + c0 * c3) * 0.25;
    c2 = c1 * c1 * 0.5;
    c1 = c0 * c1;
    c0 = 2.0 * c0 * c0 - 1.0;
  }
}

// Universal Kepler equation F(s) = r0 G1 + eta0 G2 + mu G3 - dt with its
// first two derivatives (G_k = s^k c_k(beta s^2)).
__device__ __forceinline__ void kepler_eval64(double r0, double eta0, double zeta0, double beta, double mu, double s,
                                              double dt, double& F, double& Fp, double& Fpp) {
#pragma clang fp contract(off)
  double c0, c1, c2, c3;
  stumpff64(beta * s * s, c0, c1, c2, c3);
  const double g1 = s * c1, g2 = s * s * c2, g3 = s * s * s * c3;
  F = r0 * g1 + eta0 * g2 + mu * g3 - dt;
  Fp = r0 * c0 + eta0 * g1 + mu * g2;
  Fpp = eta0 * c0 + zeta0 * g1;
}

// Kepler drift of relative position q and velocity u about mu for dt
// (universal variables). F is increasing (F' = r > 0): on a bound orbit dt is
// reduced modulo the period (fmod is exact) and the root lies within one
// revolution, s in [0, 2 pi / sqrt(beta)]; otherwise the bracket is grown by
// doubling. Halley steps from s = dt / r0, replaced by bisection whenever they
// leave the bracket, at most 100, until |ds| <= 1e-15 |s|; then the f and g
// functions. Every lane runs its own iteration count.
__device__ inline void kepler_drift64(double* q, double* u, double mu, double dt) {
#pragma clang fp contract(off)
  const double r0 = sqrt(q[0] * q[0] + q[1] * q[1] + q[2] * q[2]);
  const double v2 = u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
  const double eta0 = q[0] * u[0] + q[1] * u[1] + q[2] * u[2];
  const double beta = 2.0 * mu / r0 - v2;
  const double zeta0 = mu - beta * r0;
  const double sgn = dt < 0.0 ? -1.0 : 1.0;
  double F, Fp, Fpp;
  double lo = 0.0, hi;
  if (beta > 0.0) {
    const double sq = sqrt(beta);
    const double period = 6.283185307179586 * mu / (beta * sq);
    if (!(fabs(dt) < period)) dt = fmod(dt, period);
    hi = sgn * (6.283185307179586 / sq);
  } else {
    hi = dt / r0;
    for (int k = 0; k < 200; ++k) {
      kepler_eval64(r0, eta0, zeta0, beta, mu, hi, dt, F, Fp, Fpp);
      if (sgn * F >= 0.0) break;
      lo = hi;
      hi = 2.0 * hi;
    }
  }
  double s = dt / r0;
  if (!(sgn * (s - lo) > 0.0 && sgn * (hi - s) > 0.0)) s = 0.5 * (lo + hi);
  for (int it = 0; it < 100; ++it) {
    kepler_eval64(r0, eta0, zeta0, beta, mu, s, dt, F, Fp, Fpp);
    if (sgn * F < 0.0)
      lo = s;
    else
      hi = s;
    double sn = s - F / (Fp - 0.5 * F * Fpp / Fp);
    if (!(sgn * (sn - lo) > 0.0 && sgn * (hi - sn) > 0.0)) sn = 0.5 * (lo + hi);
    const double ds = sn - s;
    s = sn;
    if (fabs(ds) <= 1e-15 * fabs(s)) break;
  }
  double c0, c1, c2, c3;
  stumpff64(beta * s * s, c0, c1, c2, c3);
  const double g1 = s * c1, g2 = s * s * c2;
  const double r = r0 * c0 + eta0 * g1 + mu * g2;
  const double f = 1.0 - mu * g2 / r0;
  const double g = r0 * g1 + eta0 * g2;
  const double fd = -mu * g1 / (r * r0);
  const double gd = 1.0 - mu * g2 / r;
  double qn[3], un[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    qn[k] = f * q[k] + g * u[k];
    un[k] = fd * q[k] + gd * u[k];
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    q[k] = qn[k];
    u[k] = un[k];
  }
}

// A value known to be equal in every active lane, moved to a scalar register.
__device__ __forceinline__ float uniform_f32(float x) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}

// Compiler and memory ordering point for LDS traffic between the lanes of one
// wavefront (no cross-wave synchronisation).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The Morton box's half-extents b in every thread of a workgroup of T, and with
// `store` in box[0..2], |box| in box[3]. fmax is exact and order-independent, so
// every workgroup finds the same.
template <int T>
__device__ __forceinline__ void box_final(const BoxSource& bs, double* __restrict__ box, double* b, bool store) {
#pragma clang fp contract(off)
  __shared__ double wm[3][T / 64];
  const int t = threadIdx.x;
  if (bs.nparts == 0) {
    for (int c = 0; c < 3; ++c) b[c] = bs.part[c];
  } else {
    double r[3] = {0.0, 0.0, 0.0};
    // 8 partials per thread and round, all loaded before the first is used
    // (clamped indices), so a round costs one memory round trip
    for (int i0 = t; i0 < bs.nparts; i0 += 8 * T) {
      double q[8][3];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int i = min(i0 + u * T, bs.nparts - 1);
#pragma unroll
        for (int c = 0; c < 3; ++c) q[u][c] = bs.part[3 * i + c];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int c = 0; c < 3; ++c) r[c] = fmax(r[c], q[u][c]);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      for (int off = 32; off > 0; off >>= 1) r[c] = fmax(r[c], __shfl_xor(r[c], off, 64));
      if ((t & 63) == 0) wm[c][t >> 6] = r[c];
    }
  }
  __syncthreads();
  if (bs.nparts != 0)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      b[c] = 0.0;
      for (int q = 0; q < T / 64; ++q) b[c] = fmax(b[c], wm[c][q]);
    }
  if (store && t == 0 && bs.part != box) {
    box[0] = b[0];
    box[1] = b[1];
    box[2] = b[2];
    // bd_size = |bounding_box| (barnes_hut.cpp:405; vec3::magnitude, vectors.h:93-99)
    box[3] = sqrt(b[0] * b[0] + b[1] * b[1] + b[2] * b[2]);
  }
}

}  // namespace aster
