// generated by mace_onegpu/codegen.py -- harmonics of an edge direction with their tangential
// derivatives, and the split of fp32 operands for fp16 matrix instructions
#pragma once

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));

// a b = h0 + h1 + error, fp16 values rounded to nearest even, h1 from the exact residual of the product (one rounding):
// |error| <= 2^-23 |a b| where |a b| >= 2^-2, and <= 2^-25 below.  Two products at a time.
__device__ __forceinline__ void mm_split2_f16(float2v a, float2v b, unsigned& h0, unsigned& h1) {
  const half2v h = __builtin_convertvector(a * b, half2v);
  const float2v f = __builtin_convertvector(h, float2v);
  h0 = __builtin_bit_cast(unsigned, h);
  const float2v r = {fmaf(a.x, b.x, -f.x), fmaf(a.y, b.y, -f.y)};
  h1 = __builtin_bit_cast(unsigned, __builtin_convertvector(r, half2v));
}

// Polar frame of a unit vector (x, y, z): s = sin(theta), (cp, sp) = (cos, sin)(phi).  At the poles phi = 0.
__device__ __forceinline__ void mm_polar(float x, float y, float& s, float& cp, float& sp) {
  const float s2 = fmaf(x, x, y * y);
  const bool pole = s2 < 1e-30f;
  const float r0 = __builtin_amdgcn_rsqf(pole ? 1.f : s2);
  const float r = r0 * fmaf(-0.5f * s2 * r0, r0, 1.5f);   // one Newton step
  s = pole ? 0.f : s2 * r;
  cp = pole ? 1.f : x * r;
  sp = pole ? 0.f : y * r;
}

// A-operand values of one edge: F[m] A[m], m = 1..15, of the basis B_lm = F_l|m|(z) s^|m| {cos, sin}(|m| phi)
// (Y_m = c_m B_m, the c_m folded into the other operand): type 0 the value, type 1 d/dtheta, type 2 (1 / s) d/dphi, all
// times MM_POLAR_SCALE.  They stay below 4.2, so the scaled ones fill the upper end of the fp16 range: two pieces hold
// a product to 2^-23 of its value down to 2^-15, and to 2^-38 below.  The types differ in one factor per (l, |m|) and
// in where the azimuthal pairs begin, so a lane evaluates its own type only.  The pairs are turned on by x + i y, which
// is exact: rms errors of 4e-8 to 7e-8 with the split, half those of products of s, cos(m phi) and sin(m phi).
#define MM_POLAR_SCALE 8192.f
__device__ __forceinline__ void mm_polar_operands(float x, float y, float z, float s, float cp, float sp, int type,
                                                  float (&F)[16], float (&A)[16]) {
  const bool t0 = type == 0, t1 = type == 1, t2 = type == 2;
  const float z2 = z * z, s2 = fmaf(x, x, y * y), zk = MM_POLAR_SCALE * z, sk = MM_POLAR_SCALE * s, zz = z + z;
  const float f5 = fmaf(zz, zz, fmaf(z, z, -1.f));   // 5 z^2 - 1 from exact products
  // s^|m| {cos, sin}(|m| phi) (type 0), s^(|m| - 1) {cos, sin} (type 1), s^(|m| - 1) {-sin, cos} (type 2)
  const float c1 = MM_POLAR_SCALE * (t0 ? x : cp), d1 = MM_POLAR_SCALE * (t0 ? y : sp);
  const float c2 = fmaf(c1, x, -(d1 * y)), d2 = fmaf(c1, y, d1 * x);
  const float c3 = fmaf(c2, x, -(d2 * y)), d3 = fmaf(c2, y, d2 * x);
  A[1] = A[5] = A[11] = t2 ? c1 : d1;
  A[3] = A[7] = A[13] = t2 ? -d1 : c1;
  A[4] = A[10] = t2 ? c2 : d2;
  A[8] = A[14] = t2 ? -d2 : c2;
  A[9] = t2 ? c3 : d3;
  A[15] = t2 ? -d3 : c3;
  A[0] = A[2] = A[6] = A[12] = 1.f;
  // F_lm | |m| z F_lm - s^2 F'_lm (m = 0: -s F'_l0) | |m| F_lm
  F[0] = t0 ? MM_POLAR_SCALE : 0.f;
  F[2] = t0 ? zk : t1 ? -sk : 0.f;
  F[1] = F[3] = t1 ? z : 1.f;
  F[6] = t0 ? fmaf(zk, zz, fmaf(zk, z, -MM_POLAR_SCALE)) : t1 ? -6.f * z * sk : 0.f;
  F[5] = F[7] = t1 ? z2 - s2 : z;
  F[4] = F[8] = t0 ? 1.f : t1 ? zz : 2.f;
  F[12] = t0 ? zk * (f5 - 2.f) : t1 ? -3.f * sk * f5 : 0.f;
  F[11] = F[13] = t1 ? z * fmaf(-10.f, s2, f5) : f5;
  F[10] = F[14] = t0 ? z : t1 ? fmaf(2.f, z2, -s2) : zz;
  F[9] = F[15] = t0 ? 1.f : t1 ? 3.f * z : 3.f;
}
