// Minimum image of a coordinate difference, bit for bit v - L * rint(v / L) with every operation rounded separately
// (receiver_chunk_mace.py:110-111).
#pragma once

// For |v| <= L the quotient rounds to 0 or +-1, and the comparison with h = L / 2 (exact) decides which without the
// division: fl(v / L) = fl(v / h) / 2, and for v > h the ratio v / h exceeds 1 by more than 2^-53, so fl(v / h) > 1
// and rint gives 1; for |v| <= h it gives 0 (a half rounds to even).  L * n is then exact and the subtraction is the
// same.  Anything else (a coordinate outside the box, a NaN) takes the general expression.
__device__ __forceinline__ double mm_mic(double v, double L, double h) {
#pragma clang fp contract(off)
  if (__builtin_expect(!(fabs(v) <= L), 0)) return v - L * rint(v / L);
  return fabs(v) > h ? v - copysign(L, v) : v;
}

// The same for a difference known to be within [-L, L] (both coordinates in [0, L]).
__device__ __forceinline__ double mm_mic_in_box(double v, double L, double h) {
#pragma clang fp contract(off)
  return fabs(v) > h ? v - copysign(L, v) : v;
}
