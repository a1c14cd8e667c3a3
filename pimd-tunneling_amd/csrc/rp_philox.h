// rp_philox.h -- counter-based Philox4x32-10 normals and Poisson draws.
//
// Written from the published description (Salmon, Moraes, Dror, Shaw, "Parallel
// random numbers: as easy as 1, 2, 3", SC11).  A trajectory owns one stream id; its
// k-th N(0,1) draw is a pure function of (seed, stream, k), so any kernel can make
// the draw the reference's sequential VSL stream would make at that position
// (verletmodule.f90:55,106,215,641) without carrying generator state.
//   block b = k >> 1 -> Philox(ctr = {b_lo, b_hi, stream_lo, stream_hi},
//                              key = {seed_lo, seed_hi}) -> two 53-bit uniforms
//   Box-Muller: draw 2b uses r cos(2 pi u1), draw 2b+1 uses r sin(2 pi u1).
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

namespace rp {

__host__ __device__ __forceinline__ void philox4x32_10(uint32_t c[4], uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    if (r) {
      k0 += 0x9E3779B9u;
      k1 += 0xBB67AE85u;
    }
    uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
    uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
    uint32_t n0 = (uint32_t)(p1 >> 32) ^ c[1] ^ k0;
    uint32_t n2 = (uint32_t)(p0 >> 32) ^ c[3] ^ k1;
    c[1] = (uint32_t)p1;
    c[3] = (uint32_t)p0;
    c[0] = n0;
    c[2] = n2;
  }
}

__host__ __device__ __forceinline__ void philox_uniform2(uint64_t seed, uint64_t stream,
                                                         uint64_t block, double& u0, double& u1) {
  uint32_t c[4] = {(uint32_t)block, (uint32_t)(block >> 32), (uint32_t)stream,
                   (uint32_t)(stream >> 32)};
  philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
  uint64_t a = ((uint64_t)c[1] << 32) | c[0], b = ((uint64_t)c[3] << 32) | c[2];
  u0 = ((double)(a >> 11) + 0.5) * 0x1.0p-53;
  u1 = ((double)(b >> 11) + 0.5) * 0x1.0p-53;
}

// Box-Muller of two uniforms in (0, 1]: z0 = r cos(2 pi u1), z1 = r sin(2 pi u1),
// r = sqrt(-2 ln u0), for exactly the arguments that occur, so without the general functions'
// range reductions and special cases.  Both the identities and the coefficients are worked
// out here: the polynomials are minimax fits (Remez exchange in 70-digit decimals) of
//   log:  ln((1+s)/(1-s)) = 2 s + s z P(z), z = s^2, |s| <= (sqrt(2)-1)/(sqrt(2)+1),
//         relative error 1.2e-18; with s = f/(2+f), ln(1+f) = f - s (f - z P), whose leading
//         term is exact;
//   sin:  sin(pi d/2) = d (pi/2 + z S(z)), z = d^2 <= 1/4, relative error 3.4e-18;
//   cos:  cos(pi d/2) = 1 + z C(z), error 3.3e-20.
__device__ __forceinline__ void box_muller(double u0, double u1, double& z0, double& z1) {
  // ln u0 = e ln 2 + ln(1 + f), 1 + f in [sqrt(1/2), sqrt(2))
  double m = __builtin_amdgcn_frexp_mant(u0);
  int e = __builtin_amdgcn_frexp_exp(u0);
  const bool low = m < 0.70710678118654752;
  m = low ? 2.0 * m : m;
  e -= low;
  const double f = m - 1.0, den = 2.0 + f;
  double q = __builtin_amdgcn_rcp(den);
  q = fma(fma(-den, q, 1.0), q, q);
  double s = f * q;
  s = fma(fma(-s, den, f), q, s);
  const double z = s * s;
  double P = 0x1.2f05637aae895p-3;
  P = fma(P, z, 0x1.39a1bab5d416ep-3);
  P = fma(P, z, 0x1.74663ee89cd65p-3);
  P = fma(P, z, 0x1.c71c52095b67cp-3);
  P = fma(P, z, 0x1.24924941f1286p-2);
  P = fma(P, z, 0x1.999999997fdb7p-2);
  P = fma(P, z, 0x1.5555555555592p-1);
  const double ed = (double)e;
  // ln 2 in two parts: e times the first (32 bits) is exact
  const double lo = fma(s, f - z * P, -ed * 1.9082149292705877e-10);
  // hi + err = e ln2_hi + f exactly: one rounding of the sum
  const double hi = fma(ed, 0x1.62e42feep-1, f), err = fma(ed, 0x1.62e42feep-1, -hi) + f;
  const double x = -2.0 * (hi - (lo - err));
  // r = sqrt(x) by the reciprocal square root estimate, one Newton step on both x^1/2 and its
  // reciprocal, and the residual; u0 = 1 gives x = 0, kept off the estimate's pole
  const double xx = fmax(x, 1e-300);
  double y = __builtin_amdgcn_rsq(xx);
  double g = xx * y, h = 0.5 * y;
  const double t = fma(-h, g, 0.5);
  g = fma(g, t, g);
  h = fma(h, t, h);
  g = fma(fma(-g, g, xx), h, g);
  // quadrant and offset of the angle (pi/2) v, v = 4 u1: adding 1.5 2^52 rounds v to the
  // integer k held in the sum's low bits
  const double v = 4.0 * u1, kk = v + 6755399441055744.0, d = v - (kk - 6755399441055744.0);
  const uint32_t k = (uint32_t)__double2loint(kk);
  const double w = d * d;
  double S = 0x1.e403d09a8a991p-25;
  S = fma(S, w, -0x1.e300a65a6ec0cp-19);
  S = fma(S, w, 0x1.5078301b629e7p-13);
  S = fma(S, w, -0x1.32d2cce3332e2p-8);
  S = fma(S, w, 0x1.466bc67758d85p-4);
  S = fma(S, w, -0x1.4abbce625be47p-1);
  S = fma(S, w, 6.123233995736766e-17);
  const double sn = fma(d, 0x1.921fb54442d18p+0, d * S);
  double C = -0x1.b26fe81e8021cp-28;
  C = fma(C, w, 0x1.f9cc6acee7764p-22);
  C = fma(C, w, -0x1.a6d1ecb73ed3fp-16);
  C = fma(C, w, 0x1.e1f50683b42adp-11);
  C = fma(C, w, -0x1.55d3c7e3c95bcp-6);
  C = fma(C, w, 0x1.03c1f081b5ab0p-2);
  C = fma(C, w, -0x1.3bd3cc9be45dep+0);
  const double cs = fma(w, C, 1.0);
  const double a = (k & 1) ? sn : cs, b = (k & 1) ? cs : sn;
  // cos is negative in quadrants 1 and 2, sin in 2 and 3
  const uint32_t sa = ((k + 1) << 30) & 0x80000000u, sb = (k << 30) & 0x80000000u;
  z0 = g * __hiloint2double(__double2hiint(a) ^ (int)sa, __double2loint(a));
  z1 = g * __hiloint2double(__double2hiint(b) ^ (int)sb, __double2loint(b));
}

// Both normals of one block (draws 2*block and 2*block+1).
__device__ __forceinline__ void philox_normal2(uint64_t seed, uint64_t stream, uint64_t block,
                                               double& z0, double& z1) {
  uint32_t c[4] = {(uint32_t)block, (uint32_t)(block >> 32), (uint32_t)stream,
                   (uint32_t)(stream >> 32)};
  philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
  // philox_uniform2's uniforms: the fma adds the exact parts and rounds once, as there
  const double u0 = fma((double)c[1], 0x1p-32, ((double)(c[0] >> 11) + 0.5) * 0x1.0p-53);
  const double u1 = fma((double)c[3], 0x1p-32, ((double)(c[2] >> 11) + 0.5) * 0x1.0p-53);
  box_muller(u0, u1, z0, z1);
}

__device__ __forceinline__ double philox_normal(uint64_t seed, uint64_t stream, int64_t index) {
  double z0, z1;
  philox_normal2(seed, stream, (uint64_t)index >> 1, z0, z1);
  return (index & 1) ? z1 : z0;
}

// Poisson(mean) on the stream's disjoint high half: inversion below mean 16, a rounded
// normal approximation above (VSL's POISNORM, which the reference selects at
// verletmodule.f90:362, is likewise a normal approximation for large means).
__host__ __device__ __forceinline__ int32_t philox_poisson(uint64_t seed, uint64_t stream,
                                                           int64_t index, double mean) {
  double u0, u1;
  philox_uniform2(seed, stream ^ 0x8000000000000000ull, (uint64_t)index, u0, u1);
  if (mean < 16.0) {
    double pk = exp(-mean), cdf = pk;
    int32_t k = 0;
    while (u0 > cdf && k < 1000) {
      ++k;
      pk *= mean / k;
      cdf += pk;
    }
    return k;
  }
  double z = sqrt(-2.0 * log(u0)) * cos(6.283185307179586 * u1);
  double k = floor(mean + sqrt(mean) * z + 0.5);
  return k < 0.0 ? 0 : (int32_t)k;
}

}  // namespace rp
