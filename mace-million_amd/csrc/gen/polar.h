// generated by mace_onegpu/codegen.py -- harmonics of an edge direction and their tangential derivatives
#pragma once

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

// A-operand values of one edge: P[m], m = 1..15, of the basis B_lm = F_lm(z, s) {cos, sin}(|m| phi) (Y_m = c_m B_m, the
// c_m folded into the other operand): type 0 the value, type 1 d/dtheta, type 2 (1 / sin(theta)) d/dphi.  The three
// types differ in one scalar factor per (l, |m|) and in the azimuthal pair, so a lane evaluates its own type only.
__device__ __forceinline__ void mm_polar_operands(float z, float s, float cp, float sp, int type, float (&P)[16]) {
  const bool t0 = type == 0, t1 = type == 1;
  const float z2 = z * z, s2 = s * s, zs = z * s;
  const float f5 = fmaf(5.f, z2, -1.f);
  // F_lm | dF_lm/dtheta | |m| F_lm / s
  const float f10 = t0 ? z : t1 ? -s : 0.f;
  const float f11 = t0 ? s : t1 ? z : 1.f;
  const float f20 = t0 ? fmaf(3.f, z2, -1.f) : t1 ? -6.f * zs : 0.f;
  const float f21 = t0 ? zs : t1 ? z2 - s2 : z;
  const float f22 = t0 ? s2 : t1 ? 2.f * zs : 2.f * s;
  const float f30 = t0 ? z * fmaf(5.f, z2, -3.f) : t1 ? -s * fmaf(15.f, z2, -3.f) : 0.f;
  const float f31 = t0 ? s * f5 : t1 ? z * fmaf(-10.f, s2, f5) : f5;
  const float f32 = t0 ? z * s2 : t1 ? s * fmaf(2.f, z2, -s2) : 2.f * zs;
  const float f33 = t0 ? s * s2 : t1 ? 3.f * z * s2 : 3.f * s2;
  const float c2 = fmaf(cp, cp, -sp * sp), q2 = 2.f * cp * sp;
  const float c3 = fmaf(cp, c2, -sp * q2), q3 = fmaf(sp, c2, cp * q2);
  const bool t2 = type == 2;
  // azimuthal pair (cos, sin)(m phi), or its derivative / m: (-sin, cos)
  const float a1 = t2 ? -sp : cp, b1 = t2 ? cp : sp;
  const float a2 = t2 ? -q2 : c2, b2 = t2 ? c2 : q2;
  const float a3 = t2 ? -q3 : c3, b3 = t2 ? c3 : q3;
  P[0] = t0 ? 1.f : 0.f;
  P[1] = f11 * b1; P[2] = f10; P[3] = f11 * a1;
  P[4] = f22 * b2; P[5] = f21 * b1; P[6] = f20; P[7] = f21 * a1; P[8] = f22 * a2;
  P[9] = f33 * b3; P[10] = f32 * b2; P[11] = f31 * b1; P[12] = f30; P[13] = f31 * a1; P[14] = f32 * a2;
  P[15] = f33 * a3;
}
