"""Generates the HIP sources of the architecture-specific kernels (build step; run by mace-million_amd/build.py).

The reference generates one Triton kernel per path table at run time (conv_spline.gen_fwd/gen_bwd,
conv_spline.py:38-181).  Here the same information -- the channelwise TP terms (w, k, m, o, coef), the coupling
paths of the symmetric contraction and the spherical-harmonic polynomials -- is turned into straight-line CDNA4
HIP code once, at build time, with every coupling coefficient a compile-time constant:

  gen/sh.h          Y_lm(u) l<=3 (16 values) and the gradient of sum_m g_m Y_m(u) w.r.t. u (sympy-derived)
  gen/conv_l{1,2}.hip  fused edge convolution: spline-table radial weights x channelwise TP x receiver sum
                    (forward) and its backward (d r, d Y per edge, optional d X scattered to senders)
  gen/symc_l{1,2}.hip  per-species correlation-3 symmetric contraction, forward and backward
  gen/conv_l0123.hip   the same fused convolution for the literal 0e+1o+2e+3o node features (23 paths)
  gen/conv_l2v.hip  the layer-2 backward on the matrix cores; gen/polar.h its harmonics
  gen/tpw_*.hip     channelwise TP with explicit per-edge weights (FusedConvTP), forward and backward

Kernel/launch design is documented in the generated files' headers.
"""
import os
from collections import OrderedDict

import numpy as np
import sympy as sp

from . import o3

C = 128
NCB = 8
CB = C // NCB


def _f(x):
    """float literal with full precision."""
    r = repr(float(x))
    if "e" not in r and "." not in r:
        r += ".0"
    return r + "f"


# ----------------------------------------------------------------------------- spherical harmonics
def sh_header():
    x, y, z = sp.symbols("x y z", real=True)
    s = sp.sqrt
    Y = [sp.Integer(1),
         s(3) * y, s(3) * z, s(3) * x,
         s(15) * x * y, s(15) * y * z, s(5) / 2 * (2 * z**2 - x**2 - y**2), s(15) * x * z, s(15) / 2 * (x**2 - y**2),
         s(70) / 4 * y * (3 * x**2 - y**2), s(105) * x * y * z, s(42) / 4 * y * (4 * z**2 - x**2 - y**2),
         s(7) / 2 * z * (2 * z**2 - 3 * x**2 - 3 * y**2), s(42) / 4 * x * (4 * z**2 - x**2 - y**2),
         s(105) / 2 * z * (x**2 - y**2), s(70) / 4 * x * (x**2 - 3 * y**2)]
    L = ["// generated by mace_onegpu/codegen.py -- real spherical harmonics l<=3, component normalisation,",
         "// z-polar basis, m = -l..l (same polynomials as mace_onegpu/o3.sh_cartesian)",
         "#pragma once", ""]

    def cexpr(e):
        e = sp.expand(e)
        code = sp.ccode(sp.N(e, 17))
        return code.replace("pow(x, 2)", "(x*x)").replace("pow(y, 2)", "(y*y)").replace("pow(z, 2)", "(z*z)") \
                   .replace("pow(x, 3)", "(x*x*x)").replace("pow(y, 3)", "(y*y*y)").replace("pow(z, 3)", "(z*z*z)")

    def fl(code):
        # float literals
        import re
        return re.sub(r"(?<![\w.])(\d+\.\d+(?:e[-+]?\d+)?)(?![\w])", r"\1f", code)
    L.append("__device__ __forceinline__ void mm_sh16(float x, float y, float z, float* __restrict__ Y) {")
    for m, e in enumerate(Y):
        L.append(f"  Y[{m}] = {fl(cexpr(e)) if m else '1.0f'};")
    L.append("}")
    L.append("")
    L.append("// P_m(u) with Y_m = c_m P_m on the unit sphere (x^2 + y^2 + z^2 = 1 used to shorten l = 2, 3); the")
    L.append("// kernels that fold c_m into other constants evaluate these instead of Y (21 operations)")
    L.append("__device__ __forceinline__ void mm_shp16(float x, float y, float z, float* __restrict__ P) {")
    L.append("  const float x2 = x * x, y2 = y * y, z2 = z * z;")
    L.append("  const float d = x2 - y2, f = fmaf(5.f, z2, -1.f);")
    L.append("  P[0] = 1.f; P[1] = y; P[2] = z; P[3] = x;")
    L.append("  P[4] = x * y; P[5] = y * z; P[6] = fmaf(3.f, z2, -1.f); P[7] = x * z; P[8] = d;")
    L.append("  P[9] = y * fmaf(3.f, x2, -y2); P[10] = P[4] * z; P[11] = y * f; P[12] = z * fmaf(5.f, z2, -3.f);")
    L.append("  P[13] = x * f; P[14] = z * d; P[15] = x * fmaf(-3.f, y2, x2);")
    L.append("}")
    L.append("")
    L.append("// 1 / c_m")
    L.append("__device__ __forceinline__ float mm_sh_inv_norm(int m) {")
    L.append("  float r = 1.f;")
    for m in range(1, 16):
        L.append(f"  r = m == {m} ? {float(1.0 / SH_NORM[m])!r}f : r;")
    L.append("  return r;")
    L.append("}")
    L.append("")
    L.append("// G = grad_u sum_m g[m] Y_m(u) (Cartesian gradient of the polynomials)")
    L.append("__device__ __forceinline__ void mm_sh16_grad(float x, float y, float z, const float* __restrict__ g,"
             " float* __restrict__ G) {")
    for a, var in enumerate((x, y, z)):
        terms = []
        for m, e in enumerate(Y):
            d = sp.diff(e, var)
            if d != 0:
                terms.append(f"g[{m}] * ({fl(cexpr(d))})")
        L.append(f"  G[{a}] = " + " + ".join(terms) + ";")
    L.append("}")
    return "\n".join(L) + "\n"


def _sh_poly(x, y, z):
    """The polynomials of mm_shp16 (sympy or numpy arguments)."""
    x2, y2, z2 = x * x, y * y, z * z
    return [1 + 0 * x, y, z, x, x * y, y * z, 3 * z2 - 1, x * z, x2 - y2, y * (3 * x2 - y2), x * y * z,
            y * (5 * z2 - 1), z * (5 * z2 - 3), x * (5 * z2 - 1), z * (x2 - y2), x * (x2 - 3 * y2)]


def _sh_norms():
    """c_m with Y_m = c_m P_m on the unit sphere, from o3's harmonics, checked at random unit vectors."""
    rng = np.random.default_rng(0)
    u = rng.normal(size=(64, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    Y = np.stack(o3.sh_cartesian(u[:, 0], u[:, 1], u[:, 2]), 1)
    P = np.stack(_sh_poly(u[:, 0], u[:, 1], u[:, 2]), 1)
    c = np.array([Y[np.argmax(np.abs(P[:, m])), m] / P[np.argmax(np.abs(P[:, m])), m] for m in range(16)])
    if np.abs(P * c - Y).max() > 1e-12:
        raise AssertionError("mm_shp16 polynomials are not proportional to the harmonics")
    return c


SH_NORM = _sh_norms()


def _loop_head(A):
    """Edge loop of one 16-lane row (edge slot); the next packed record is loaded one iteration ahead."""
    A("  int e = e0 + slot;")
    A("  floatx4 pk_next = e < e1 ? e_pk[e] : floatx4{0.f, 0.f, 0.f, 0.f};")
    A("  for (; e < e1; e += 4) {")
    A("    const floatx4 pk = pk_next;   // (t, table interval row, X row, density)")
    A("    if (e + 4 < e1) pk_next = e_pk[e + 4];")


def _load_y(A, used_m, poly=False):
    """Spherical harmonics of the edge direction, evaluated from the stored unit vector (16 B per edge instead of
    64 B of harmonics: every channel block re-reads the edge records); poly: the unnormalised P_m of mm_shp16."""
    A("    const floatx4 u = e_u[e];   // (unit vector, r)")
    A("    float Yv[16];")
    A(f"    {'mm_shp16' if poly else 'mm_sh16'}(u.x, u.y, u.z, Yv);")
    for m in used_m:
        A(f"    const float Y{m} = Yv[{m}];")


# sender-feature gradient of the layer-2 backward summed per group of 4 receivers in LDS: 176 slots of 64 floats
# (51.9 KB of LDS with the hash: 3 workgroups of 4 waves per CU, the occupancy the kernel's registers allow)
GX_LDS_DEFAULT = {"r": 4, "smax": 176, "hs": 512, "maxe": 512}


def _gx_lds_prologue(A, p, nX):
    """Group of R receivers per workgroup (one per wave): the distinct senders of the group's edges get LDS slots
    (open-addressing hash of the sender row), and the sender-feature gradient of this channel block is summed in
    LDS per slot, then added to gX once per distinct sender.  Senders beyond the slot capacity, and edges beyond the
    per-group edge cap, add to gX directly."""
    R, smax, hs, maxe = p["r"], p["smax"], p["hs"], p["maxe"]
    nt = 64 * R
    lg = hs.bit_length() - 1
    assert 1 << lg == hs
    A(f"  __shared__ int hkey[{hs}];")
    A(f"  __shared__ int hslot[{hs}];")
    A(f"  __shared__ int eslot[{maxe}];")
    A(f"  __shared__ int ssend[{smax}];")
    A(f"  __shared__ float gxs[{smax * nX * 16}];   // [slot][component][16 channels]")
    A("  __shared__ int nslot;")
    A(f"  const int i0 = (blockIdx.x >> 3) * {R};")
    A("  const int i = i0 + (threadIdx.x >> 6);")
    A("  const int tid = threadIdx.x;")
    A("  const int E0g = rowptr[i0];")
    A(f"  const int nEg = min(rowptr[min(i0 + {R}, nC)] - E0g, {maxe});")
    A("  const int* __restrict__ pk_i = (const int*)e_pk;   // .z of the packed record = sender row")
    A(f"  for (int h = tid; h < {hs}; h += {nt}) hkey[h] = -1;")
    A("  if (tid == 0) nslot = 0;")
    A("  __syncthreads();")
    A(f"  for (int j = tid; j < nEg; j += {nt}) {{")
    A("    const int sj = pk_i[4 * (E0g + j) + 2];")
    A(f"    unsigned h = ((unsigned)sj * 2654435761u) >> {32 - lg};")
    A("    while (true) {")
    A("      const int prev = atomicCAS(&hkey[h], -1, sj);")
    A("      if (prev == -1 || prev == sj) break;")
    A(f"      h = (h + 1) & {hs - 1};")
    A("    }")
    A("  }")
    A("  __syncthreads();")
    A(f"  for (int h = tid; h < {hs}; h += {nt}) {{")
    A("    const int sj = hkey[h];")
    A("    if (sj >= 0) {")
    A("      const int sl = atomicAdd(&nslot, 1);")
    A("      hslot[h] = sl;")
    A(f"      if (sl < {smax}) ssend[sl] = sj;")
    A("    }")
    A("  }")
    A("  __syncthreads();")
    A(f"  const int ns = min(nslot, {smax});")
    A(f"  for (int j = tid; j < nEg; j += {nt}) {{")
    A("    const int sj = pk_i[4 * (E0g + j) + 2];")
    A(f"    unsigned h = ((unsigned)sj * 2654435761u) >> {32 - lg};")
    A(f"    while (hkey[h] != sj) h = (h + 1) & {hs - 1};")
    A("    const int sl = hslot[h];")
    A(f"    eslot[j] = sl < {smax} ? sl : -1;")
    A("  }")
    A(f"  for (int j = tid; j < ns * {nX * 16}; j += {nt}) gxs[j] = 0.f;")
    A("  __syncthreads();")


def _gx_lds_flush(A, p, nX):
    nt = 64 * p["r"]
    A("  __syncthreads();")
    A(f"  for (int j = tid; j < ns * {nX * 16}; j += {nt}) {{")
    A(f"    const int sl = j / {nX * 16}, r = j % {nX * 16};")
    A(f"    atomicAdd(gX + (size_t)ssend[sl] * {nX * C} + cb * {16 * nX} + r, gxs[j]);   // a slot: {64 * nX} contiguous bytes")
    A("  }")


# ----------------------------------------------------------------------------- edge convolution
def conv_source(tab, layer, need_gx, opts=None):
    """opts: cpl -- channels per lane of the forward kernel (default 2 for layer 2, 1 for layer 1); ybatch -- edges
    per batch of the forward's per-edge harmonic stage, a power of two from 4 to 64 (0: every lane evaluates the
    harmonics of its edge each iteration; default 64); gx_lds -- the group/slot sizes of the backward's LDS accumulation of dL/dX
    (default GX_LDS_DEFAULT)."""
    opts = opts or {}
    nX, nW, nO, terms = tab["nX"], tab["nW"], tab["nO"], tab["terms"]
    used_m = sorted({t[2] for t in terms})
    used_o = sorted({t[3] for t in terms})
    groups = OrderedDict()
    for (w, k, m, o, c) in terms:
        groups.setdefault((w, k), []).append((m, o, c))
    used_k = sorted({k for (w, k) in groups})
    # distinct |coef| * Y_m products (|coef| != 1)
    cy = OrderedDict()
    for (w, k, m, o, c) in terms:
        a = abs(c)
        if abs(a - 1.0) > 1e-12:
            key = (round(a, 14), m)
            if key not in cy:
                cy[key] = (a, m, len(cy))

    def cy_ref(m, c):
        a = abs(c)
        neg = c < 0
        if abs(a - 1.0) <= 1e-12:
            return f"Y{m}", neg
        return f"cy{cy[(round(a, 14), m)][2]}", neg

    name = f"conv{layer}"
    L = []
    A = L.append
    A(f"// generated by mace_onegpu/codegen.py -- fused edge convolution of interaction layer {layer}")
    A(f"// TP paths nW={nW}, node-feature components nX={nX}, message components nO={nO}, terms={len(terms)}")
    A("//")
    A("// out[i, o, c] = sum_{e: recv(e) = i} sum_terms coef * W(r_e; tab_e)[w, c] * X[send_e, k, c] * Y_e[m]")
    A("// W is a cubic interpolant of the fp64-sampled radial weights, stored per interval as the polynomial")
    A("// coefficients (a0, a1, a2, a3) in t in [0, 1) (same interpolant as the reference's Hermite tables).")
    # channels per lane in the forward kernel: 2 for layer 2 (per-edge work -- harmonics, coefficient products,
    # addressing -- is shared by two channels; 4 channel blocks of 32, XCDs x and x + 4 serve the same block)
    cpl = int(opts.get("cpl", 2 if layer == 2 else 1))
    if cpl not in (1, 2):
        raise ValueError(f"cpl (channels per lane of the forward) is 1 or 2, not {cpl}")
    A("// Launch: grid = 8 * ceil(nC / 4) workgroups of 256 threads; blockIdx.x % 8 = channel block cb (one per")
    A("// XCD: the XCD's L2 holds the table slice of its 16 channels); each wave handles one receiver, lanes =")
    A("// 4 edge slots x 16 channels; the 4 slot partial sums are combined with cross-lane shuffles.")
    if cpl > 1:
        A(f"// The forward kernel takes {cpl} channels per lane: {NCB // cpl} channel blocks of {16 * cpl} channels,")
        A(f"// grid = {NCB // cpl} * ceil(nC / 4), block = blockIdx.x % {NCB // cpl} (XCD x serves block x % {NCB // cpl}).")
    A('#include "../common.h"')
    A('#include "sh.h"')
    A("")
    ncb = NCB // cpl
    sub = [""] if cpl == 1 else ["a", "b"]
    A("extern \"C\" __global__ void __launch_bounds__(256)")
    A(f"mm_{name}_fwd_kernel(const int* __restrict__ rowptr, int nC, const floatx4* __restrict__ e_pk,")
    A("    const floatx4* __restrict__ e_u, const float* __restrict__ X, int x_stride,")
    A("    const floatx4* __restrict__ tab, int tab_cb_stride, float* __restrict__ out, float* __restrict__ rho) {")
    if cpl == 1:
        A("  const int cb = mm_xcd_channel_block();")
        A("  const int i = (blockIdx.x >> 3) * 4 + (threadIdx.x >> 6);")
    else:
        A(f"  const int cb = blockIdx.x & {ncb - 1};   // XCD x (= blockIdx.x % 8) always serves block x % {ncb}")
        A(f"  const int i = (blockIdx.x / {ncb}) * 4 + (threadIdx.x >> 6);")
    A("  if (i >= nC) return;")
    A("  const int lane = threadIdx.x & 63, cl = lane & 15, slot = lane >> 4;")
    A(f"  const int c = cb * {16 * cpl} + cl;")
    A("  const int e0 = rowptr[i], e1 = rowptr[i + 1];")
    for j, sfx in enumerate(sub):
        A(f"  const floatx4* __restrict__ tcb{sfx} = tab + (size_t)({cpl} * cb + {j}) * tab_cb_stride + cl;")
    for o in used_o:
        for sfx in sub:
            A(f"  float acc{o}{sfx} = 0.f;")
    A("  float dsum = 0.f;")
    yb = int(opts.get("ybatch", 64))
    if yb:
        # the edge-only factors of the terms: Y_m used with |coef| = 1 and the products cy_j = |coef| Y_m
        yvals = [f"Y{m}" for m in used_m if any(abs(abs(c) - 1.0) <= 1e-12 and mm == m for (_, _, mm, _, c) in terms)]
        yvals += [f"cy{j}" for (_, _, j) in cy.values()]
        nv4 = (len(yvals) + 3) // 4
        pk_lds = bool(opts.get("fwd_pk_lds", True))
        nv = nv4 + (1 if pk_lds else 0)
        # a batch is yb / 4 iterations of the 4 edge slots, found with masks: a power of two from 4 to 64
        if not (4 <= yb <= 64 and yb & (yb - 1) == 0):
            raise ValueError(f"ybatch must be a power of two from 4 to 64 (or 0), not {yb}")
        A(f"  // per-edge factors (harmonics, |coef| x harmonic) of a batch of {yb} edges: lane j of the wave evaluates")
        A(f"  // edge eb + j once and stores its {len(yvals)} factors in the wave's LDS rows; the 4 edge slots read them")
        A(f"  // back ({nv4} x 16 B per edge; rows of consecutive edges fall in different banks)")
        if pk_lds:
            A("  // The edge's packed record is staged with them (one coalesced load per edge, not one per channel lane).")
        A(f"  __shared__ floatx4 yf_all[4 * {yb * nv}];")
        A(f"  floatx4* __restrict__ yf = yf_all + (threadIdx.x >> 6) * {yb * nv};")
        A("  int e = e0 + slot;")
        if not pk_lds:
            A("  floatx4 pk_next = e < e1 ? e_pk[e] : floatx4{0.f, 0.f, 0.f, 0.f};")
        A(f"  // the edge vector a lane evaluates in the next batch is loaded one batch ahead")
        A(f"  floatx4 u_next = lane < {yb} && e0 + lane < e1 ? e_u[e0 + lane] : floatx4{{0.f, 0.f, 0.f, 0.f}};")
        if pk_lds:
            A(f"  floatx4 pkb_next = lane < {yb} && e0 + lane < e1 ? e_pk[e0 + lane] : floatx4{{0.f, 0.f, 0.f, 0.f}};")
        A("  for (int k = 0; e < e1; e += 4, ++k) {")
        if not pk_lds:
            A("    const floatx4 pk = pk_next;   // (t, table interval row, X row, density)")
            A("    if (e + 4 < e1) pk_next = e_pk[e + 4];")
        A(f"    if ((k & {yb // 4 - 1}) == 0) {{   // first iteration of a batch (uniform over the active lanes)")
        A("      mm_wave_lds_sync();   // the previous batch has been read")
        A(f"      const int eb = e - slot, ej = eb + lane;")
        A(f"      if (lane < {yb} && ej < e1) {{")
        A("        const floatx4 u = u_next;   // (unit vector, r) of edge ej")
        A(f"        if (ej + {yb} < e1) u_next = e_u[ej + {yb}];")
        if pk_lds:
            A(f"        yf[lane * {nv} + {nv4}] = pkb_next;")
            A(f"        if (ej + {yb} < e1) pkb_next = e_pk[ej + {yb}];")
        A("        float Yv[16];")
        A("        mm_sh16(u.x, u.y, u.z, Yv);")
        for m in used_m:
            A(f"        const float Y{m} = Yv[{m}];")
        for (a, m, j) in cy.values():
            A(f"        const float cy{j} = {_f(a)} * Y{m};")
        A(f"        floatx4* __restrict__ d = yf + lane * {nv};")
        for q in range(nv4):
            v = [yvals[4 * q + r] if 4 * q + r < len(yvals) else "0.f" for r in range(4)]
            A(f"        d[{q}] = floatx4{{{', '.join(v)}}};")
        A("      }")
        A("      mm_wave_lds_sync();")
        A("    }")
        if pk_lds:
            A(f"    const floatx4 pk = yf[((e - e0) & {yb - 1}) * {nv} + {nv4}];   // (t, table interval row, X row, density)")
    else:
        _loop_head(A)
    A("    const float t = pk.x;")
    A("    const size_t trow = (size_t)__float_as_int(pk.y) * " + str(nW * 16) + ";")
    A("    floatx4 q;")
    for w in range(nW):
        for sfx in sub:
            A(f"    q = tcb{sfx}[trow + {w * 16}];")
            A(f"    const float W{w}{sfx} = fmaf(fmaf(fmaf(q.w, t, q.z), t, q.y), t, q.x);")
    A("    const float* __restrict__ xp = X + (size_t)__float_as_int(pk.z) * x_stride + c;")
    for k in used_k:
        for j, sfx in enumerate(sub):
            A(f"    const float X{k}{sfx} = xp[{k * C + 16 * j}];")
    if yb:
        A(f"    const floatx4* __restrict__ ys = yf + ((e - e0) & {yb - 1}) * {nv};")
        for q in range(nv4):
            A(f"    const floatx4 yq{q} = ys[{q}];")
            for r in range(4):
                if 4 * q + r < len(yvals):
                    A(f"    const float {yvals[4 * q + r]} = yq{q}.{'xyzw'[r]};")
    else:
        _load_y(A, used_m)
        for (a, m, j) in cy.values():
            A(f"    const float cy{j} = {_f(a)} * Y{m};")
    for (w, k), lst in groups.items():
        for sfx in sub:
            A(f"    {{ const float p = W{w}{sfx} * X{k}{sfx};")
            for (m, o, c) in lst:
                ref, neg = cy_ref(m, c)
                A(f"      acc{o}{sfx} = fmaf({'-' if neg else ''}p, {ref}, acc{o}{sfx});")
            A("    }")
    A("    dsum += pk.w;")
    A("  }")
    for o in used_o:
        for sfx in sub:
            A(f"  acc{o}{sfx} += __shfl_xor(acc{o}{sfx}, 16); acc{o}{sfx} += __shfl_xor(acc{o}{sfx}, 32);")
    A("  dsum += __shfl_xor(dsum, 16); dsum += __shfl_xor(dsum, 32);")
    A(f"  float* __restrict__ op = out + (size_t)i * {nO * C} + c;")
    for o in range(nO):
        for j, sfx in enumerate(sub):
            v = f"acc{o}{sfx}" if o in used_o else "0.f"
            A(f"  if (slot == {o % 4}) op[{o * C + 16 * j}] = {v};")
    A("  if (cb == 0 && lane == 0) rho[i] = dsum;")
    A("}")
    A("")
    # ------------------------------------------------------------------ backward
    gx_lds_default = opts.get("gx_lds", GX_LDS_DEFAULT) if need_gx else None

    def emit_bwd(kname, gx_mode):
        """gx_mode: 'pool' (dL/dX summed per receiver group in LDS, then float atomics), 'edge' (dL/dX of every
        edge stored in its own row of gX [E, nX * 128]: no atomics, summed per sender in a fixed order by
        mm_gather_rows_csr), or None (no dL/dX).  gX rows are 16-channel-block-major ([8][nX][16])."""
        A("// Backward: given gA = dL/dout [nC, nO, 128] produce, per edge, the partial sums over this block's 16")
        A("// channels of dL/dr (already multiplied by inv_h) and dL/dY[16] in part[cb][e][17]; the 8 channel blocks")
        A("// are summed by mm_edge_grad.  With gX != nullptr also dL/dX (atomic adds: several receivers of a chunk")
        A("// share a sender), in rows of 16-channel-block-major order: gX[send][cb][k][16] holds dL/dX[send, k,")
        A("// 16 cb + channel], so that a channel block's components of a sender are contiguous (one flush of an LDS")
        A(f"// slot adds {64 * nX} contiguous bytes).")
        gx_lds = gx_lds_default if gx_mode == "pool" else None
        if gx_lds:
            A(f"// dL/dX: a workgroup serves {gx_lds['r']} consecutive receivers (one per wave; spatially close in the Morton")
            A("// order, so they share most senders).  The group's distinct senders get LDS slots (open-addressing hash of")
            A(f"// the sender row, at most {gx_lds['smax']} slots, edges of the group beyond {gx_lds['maxe']} take no slot); the")
            A("// contributions of the group's edges are summed in LDS per slot and added to gX once per distinct sender")
            A("// (about 2.1x fewer global float atomics for water).  Senders without a slot add to gX directly.")
            A(f"// Launch: grid = 8 * ceil(nC / {gx_lds['r']}) workgroups of {64 * gx_lds['r']} threads.")
        nthr = 64 * gx_lds["r"] if gx_lds else 256
        A(f"extern \"C\" __global__ void __launch_bounds__({nthr})")
        A(f"{kname}(const int* __restrict__ rowptr, int nC, const floatx4* __restrict__ e_pk,")
        A("    const floatx4* __restrict__ e_u, const float* __restrict__ X, int x_stride,")
        A("    const floatx4* __restrict__ tab, int tab_cb_stride, float inv_h,")
        A("    const float* __restrict__ gA, float* __restrict__ part, long part_stride, float* __restrict__ gX) {")
        A("  const int cb = mm_xcd_channel_block();")
        if gx_lds:
            _gx_lds_prologue(A, gx_lds, nX)
            A("  if (i < nC) {")
        else:
            A("  const int i = (blockIdx.x >> 3) * 4 + (threadIdx.x >> 6);")
            A("  if (i >= nC) return;")
        A("  const int lane = threadIdx.x & 63, cl = lane & 15, slot = lane >> 4;")
        A("  const int c = cb * 16 + cl;")
        A("  const int e0 = rowptr[i], e1 = rowptr[i + 1];")
        A("  const floatx4* __restrict__ tcb = tab + (size_t)cb * tab_cb_stride + cl;")
        A(f"  const float* __restrict__ gp = gA + (size_t)i * {nO * C} + c;")
        for o in used_o:
            A(f"  const float g{o} = gp[{o * C}];")
        # per-(w, k, m) constants G_j = sum over the terms with that (w, k, m) of coef c_m g_o: terms that differ only
        # in the output component o share one constant (86 terms -> 76 constants for layer 2), so the loop's two FMAs
        # per constant run once per distinct (w, k, m).
        # The harmonic normalisation is folded in: the loop evaluates P_m (Y_m = c_m P_m), G_j holds coef c_m g_o, and
        # the dL/dY partial is rescaled by 1 / c_m after the channel reduction.
        wkm = OrderedDict()
        for (w, k, m, o, cf) in terms:
            wkm.setdefault((w, k, m), []).append((o, cf * SH_NORM[m]))
        wkm_id = {key: j for j, key in enumerate(wkm)}
        for j, lst in enumerate(wkm.values()):
            expr = None
            for (o, cc) in lst:
                if expr is None:
                    if abs(abs(cc) - 1.0) <= 1e-12:
                        expr = f"{'-' if cc < 0 else ''}g{o}"
                    else:
                        expr = f"{_f(cc)} * g{o}"
                else:
                    expr = f"fmaf({_f(cc)}, g{o}, {expr})"
            A(f"  const float G{j} = {expr};")
        A("  const float inv_c = mm_sh_inv_norm(cl);   // 1 / c_m of the harmonic this lane reduces")
        _loop_head(A)
        A("    const float t = pk.x;")
        A("    const int s = __float_as_int(pk.z);")
        A(f"    const floatx4* __restrict__ tp = tcb + (size_t)__float_as_int(pk.y) * {nW * 16};")
        A("    floatx4 q;")
        for w in range(nW):
            A(f"    q = tp[{w * 16}];")
            # W = ((a3 t + a2) t + a1) t + a0 and dW/dt = (a3 t + (a3 t + a2)) t + ((a3 t + a2) t + a1): 5 FMAs
            A(f"    const float s{w} = fmaf(q.w, t, q.z);")
            A(f"    const float r{w} = fmaf(s{w}, t, q.y);")
            A(f"    const float W{w} = fmaf(r{w}, t, q.x);")
            A(f"    const float D{w} = fmaf(fmaf(q.w, t, s{w}), t, r{w});")
        A("    const float* __restrict__ xp = X + (size_t)s * x_stride + c;")
        for k in used_k:
            A(f"    const float X{k} = xp[{k * C}];")
        _load_y(A, used_m, poly=True)
        for m in range(16):
            A(f"    float gy{m} = 0.f;")
        A("    float gr = 0.f;")
        if need_gx:
            for k in used_k:
                A(f"    float gx{k} = 0.f;")
        wk_ms = OrderedDict()
        for (w, k, m) in wkm:
            wk_ms.setdefault((w, k), []).append(m)
        for w in range(nW):
            ks = [k for (ww, k) in groups if ww == w]
            if not ks:
                continue
            A(f"    {{ float gw = 0.f;   // dL/dW_{w} for this channel")
            for k in ks:
                A(f"      {{ const float p = W{w} * X{k}; float u = 0.f;")
                for m in wk_ms[(w, k)]:
                    j = wkm_id[(w, k, m)]
                    A(f"        u = fmaf(Y{m}, G{j}, u); gy{m} = fmaf(p, G{j}, gy{m});")
                A(f"        gw = fmaf(X{k}, u, gw);")
                if need_gx:
                    A(f"        gx{k} = fmaf(W{w}, u, gx{k});")
                A("      }")
            A(f"      gr = fmaf(gw, D{w}, gr);")
            A("    }")
        # transpose-reduction of gy over the 16 channel lanes of the slot: recursive halving with DPP partner lanes
        # (row_mirror, row_half_mirror, quad_perm [3,2,1,0], [1,0,3,2]); afterwards lane cl holds the sum of gy_cl.
        # 15 exchanges instead of 16 full row sums.
        A("    const bool b3 = cl & 8, b2 = cl & 4, b1 = cl & 2, b0 = cl & 1;")
        for j in range(8):
            A(f"    const float s8_{j} = (b3 ? gy{8 + j} : gy{j}) + mm_dpp<0x140>(b3 ? gy{j} : gy{8 + j});")
        for j in range(4):
            A(f"    const float s4_{j} = (b2 ? s8_{4 + j} : s8_{j}) + mm_dpp<0x141>(b2 ? s8_{j} : s8_{4 + j});")
        for j in range(2):
            A(f"    const float s2_{j} = (b1 ? s4_{2 + j} : s4_{j}) + mm_dpp<0x1B>(b1 ? s4_{j} : s4_{2 + j});")
        A("    const float gyl = (b0 ? s2_1 : s2_0) + mm_dpp<0xB1>(b0 ? s2_0 : s2_1);")
        A("    gr = mm_row_sum16(gr);")
        A("    float* __restrict__ pp = part + (size_t)cb * part_stride + (size_t)e * 17;")
        A("    pp[1 + cl] = gyl * inv_c;")
        A("    if (cl == 0) pp[0] = gr * mm_spline_dxdr(t, inv_h);   // zero below the table start")
        if need_gx and gx_lds:
            A(f"    const int jg = e - E0g, sl = jg < {gx_lds['maxe']} ? eslot[jg] : -1;")
            A("    if (sl >= 0) {   // the group's LDS accumulator of this sender")
            assert nX == 4 and used_k == [0, 1, 2, 3]
            A(f"      mm_lds_add4_f32(gxs + sl * {nX * 16} + cl, gx0, gx1, gx2, gx3);")
            A("    } else {")
            A(f"      float* __restrict__ gxp = gX + (size_t)s * {nX * C} + cb * {16 * nX} + cl;")
            for k in used_k:
                A(f"      atomicAdd(gxp + {k * 16}, gx{k});")
            A("    }")
        elif gx_mode == "edge":
            A(f"    float* __restrict__ gxp = gX + (size_t)e * {nX * C} + cb * {16 * nX} + cl;   // this edge's row")
            for k in used_k:
                A(f"    gxp[{k * 16}] = gx{k};")
        elif need_gx:
            A(f"    float* __restrict__ gxp = gX + (size_t)s * {nX * C} + cb * {16 * nX} + cl;")
            for k in used_k:
                A(f"    atomicAdd(gxp + {k * 16}, gx{k});")
        A("  }")
        if gx_lds:
            A("  }   // i < nC")
            _gx_lds_flush(A, gx_lds, nX)
        A("}")
        A("")

    emit_bwd(f"mm_{name}_bwd_kernel", "pool" if need_gx else None)
    if need_gx:
        A("// Deterministic variant: dL/dX of every edge in its own row (no atomics); mm_gather_rows_csr sums the rows")
        A("// per sender in ascending edge order, so repeated runs give bitwise-identical results.")
        emit_bwd(f"mm_{name}_bwd_det_kernel", "edge")
    gx_lds = gx_lds_default
    # ------------------------------------------------------------------ launchers
    A(f"extern \"C\" int mm_{name}_fwd(const int* rowptr, int nC, const float* e_pk, const float* e_u,")
    A("    const float* X, int x_stride, const float* tab, int n_tab, int M, float* out, float* rho,")
    A("    hipStream_t stream) {")
    A("  MM_CHECK_ARG(nC >= 0 && M >= 2 && n_tab >= 1, \"bad sizes\");")
    A("  if (nC == 0) return MM_OK;")
    A(f"  dim3 grid({ncb} * ((nC + 3) / 4)), block(256);")
    A(f"  hipLaunchKernelGGL(mm_{name}_fwd_kernel, grid, block, 0, stream, rowptr, nC, (const floatx4*)e_pk,")
    A(f"                     (const floatx4*)e_u, X, x_stride, (const floatx4*)tab, n_tab * (M - 1) * {nW * 16}, out,")
    A("                     rho);")
    A(f"  return mm::launch_status(\"mm_{name}_fwd\");")
    A("}")
    A("")
    A(f"extern \"C\" int mm_{name}_bwd(const int* rowptr, int nC, const float* e_pk, const float* e_u,")
    A("    const float* X, int x_stride, const float* tab, int n_tab, int M, float inv_h, const float* gA,")
    A("    float* part, long part_stride, float* gX, hipStream_t stream) {")
    A("  MM_CHECK_ARG(nC >= 0 && M >= 2 && n_tab >= 1, \"bad sizes\");")
    if not need_gx:
        A("  MM_CHECK_ARG(gX == nullptr, \"this layer has no sender-feature gradient\");")
    else:
        A("  MM_CHECK_ARG(gX != nullptr, \"gX is required\");")
    A("  if (nC == 0) return MM_OK;")
    if gx_lds:
        R = gx_lds["r"]
        A(f"  dim3 grid(8 * ((nC + {R - 1}) / {R})), block({64 * R});")
    else:
        A("  dim3 grid(8 * ((nC + 3) / 4)), block(256);")
    A(f"  hipLaunchKernelGGL(mm_{name}_bwd_kernel, grid, block, 0, stream, rowptr, nC, (const floatx4*)e_pk,")
    A(f"                     (const floatx4*)e_u, X, x_stride, (const floatx4*)tab, n_tab * (M - 1) * {nW * 16}, inv_h,")
    A("                     gA, part, part_stride, gX);")
    A(f"  return mm::launch_status(\"mm_{name}_bwd\");")
    A("}")
    if need_gx:
        A("")
        A("// gXe: [E, nX * 128] rows, one per edge of the chunk (written for every edge of a receiver's CSR range)")
        A(f"extern \"C\" int mm_{name}_bwd_det(const int* rowptr, int nC, const float* e_pk, const float* e_u,")
        A("    const float* X, int x_stride, const float* tab, int n_tab, int M, float inv_h, const float* gA,")
        A("    float* part, long part_stride, float* gXe, hipStream_t stream) {")
        A("  MM_CHECK_ARG(nC >= 0 && M >= 2 && n_tab >= 1, \"bad sizes\");")
        A("  MM_CHECK_ARG(gXe != nullptr, \"gXe is required\");")
        A("  if (nC == 0) return MM_OK;")
        A("  dim3 grid(8 * ((nC + 3) / 4)), block(256);")
        A(f"  hipLaunchKernelGGL(mm_{name}_bwd_det_kernel, grid, block, 0, stream, rowptr, nC, (const floatx4*)e_pk,")
        A(f"                     (const floatx4*)e_u, X, x_stride, (const floatx4*)tab, n_tab * (M - 1) * {nW * 16}, inv_h,")
        A("                     gA, part, part_stride, gXe);")
        A(f"  return mm::launch_status(\"mm_{name}_bwd_det\");")
        A("}")
    return "\n".join(L) + "\n"


# ----------------------------------------------------------------------------- layer-2 backward on the matrix cores
# The layer-2 edge-convolution backward on the matrix cores.
#
# The backward of the fused edge convolution (conv_source) evaluates, per edge, channel c and (path w, input
# component k), the sum u_wk = sum_m Y_m G[w, k, m, c] and contracts it with the sender features and the radial weights.
# G is a constant of the receiver, Y of the edge, so over the edges of one receiver u is a matrix product: rows = 16
# edges, columns = 16 channels, inner index = the harmonics m of the path's degree l2.  The same product with the
# harmonics' polar and azimuthal derivatives in place of Y gives du/dtheta and du/dphi, from which the angular force
# follows: the kernel returns three numbers per edge (dL/dr and two tangential derivatives) where the per-harmonic form
# returns 17.
#
# Products from fp16 matrix instructions: each operand is the sum of two fp16 values, the second from the exact residual
# (mm_split2_f16), and all four piece products are taken, side by side along the inner index: k-group 3 - 2 a - b of the
# instruction holds piece a of Y and piece b of G.  (The instruction adds its k-groups in order: the small ones first
# give a rounding error of 3.4e-8 of the sum's rms, the other way round 5.2e-8; one rounding is 2.5e-8.)  Two pieces
# hold 23 bits, an error of up to 2^-23 of the operand where fp32 has 2^-24, as long as the operand is in the upper part
# of the fp16 range; both are scaled there by powers of two.  G, per channel, to below 2^15: 23 bits down to 2^-17 of
# the channel's largest, 2^-40 of it below.  The harmonics: see mm_polar_operands.
# What that costs is won back where the harmonics are evaluated and the products rounded.  Errors of the kernel alone
# against 64 bits, same fp32 inputs, per-harmonic form -> here, water and four-species alloy: forces 1.50e-7 -> 1.42e-7
# and 1.49e-7 -> 1.43e-7, dL/dX 1.24e-7 -> 1.25e-7 and 1.20e-7 -> 1.23e-7.  Of the whole layer-2 pass (24 chunks of 785
# to 16,857 receivers): pair forces 5.93e-7 -> 5.92e-7, dL/dh1 4.02e-7 -> 4.02e-7.
#
# Measured (16,384 receivers x 90 edges, 1.47 M edges): 2.42 -> 2.17 ms, the edge gradient that reads its partials
# 0.149 -> 0.028 ms, mm_sender_slots 9 us; the layer-2 pass of that chunk 4.39 -> 3.97 ms.
# Bound by VALU issue (the spline evaluation, the two products with X and W, the operand split) at 2 waves per SIMD:
# 0.65 of the cycles issue a VALU instruction.  Left out in timing probes: the matrix instructions 0.23 ms, the LDS adds
# 0.17 ms, evaluating and splitting each receiver's operand B 0.07 ms.
# Why this form: fp32 matrix instructions (16x16x1) hold the SIMD's vector ALU while they run (2.64 ms), the fp16 ones
# run beside it; a tile of 16 edges x 16 channels is one instruction's rows and columns, so lane (edge group, channel)
# holds four edges of its channel and reads X, W and G rows of 64 contiguous bytes; a third wave per SIMD does not fit
# (252 registers, of which 64 hold B), deeper prefetch spills.
def _polar_basis(u):
    """[n, 16] B_m of unit vectors: z-polynomial x sin^|m| theta x {cos, sin}(|m| phi), the functions that
    mm_polar_operands evaluates (value type)."""
    x, y, z = u.T
    s = np.hypot(x, y)
    ph = np.arctan2(y, x)
    f = {(1, 0): z, (1, 1): s, (2, 0): 3 * z * z - 1, (2, 1): z * s, (2, 2): s * s,
         (3, 0): z * (5 * z * z - 3), (3, 1): s * (5 * z * z - 1), (3, 2): z * s * s, (3, 3): s ** 3}
    out = np.ones((len(u), 16))
    for (l, m), v in f.items():
        out[:, l * l + l + m] = v * np.cos(m * ph)
        if m:
            out[:, l * l + l - m] = v * np.sin(m * ph)
    return out


def polar_norms():
    """c_m with Y_m = c_m B_m, checked at random directions."""
    rng = np.random.default_rng(0)
    u = rng.normal(size=(64, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    Y = np.stack(o3.sh_cartesian(u[:, 0], u[:, 1], u[:, 2]), 1)
    B = _polar_basis(u)
    j = np.argmax(np.abs(B), 0)
    c = np.array([Y[j[m], m] / B[j[m], m] for m in range(16)])
    if np.abs(B * c - Y).max() > 1e-12:
        raise AssertionError("the polar basis is not proportional to the harmonics")
    return c


BWD_VEC_HEADER = """// generated by mace_onegpu/codegen.py -- layer-2 edge convolution, backward, on the matrix cores
#include "../common.h"
#include "polar.h"

typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
typedef unsigned uint2v __attribute__((ext_vector_type(2)));
typedef unsigned uint4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned mm_load_u32(const unsigned char* p) {
  unsigned v;
  __builtin_memcpy(&v, p, 4);
  return v;
}

// Slots of the distinct senders of each group of GROUP consecutive receivers (spatially close in the Morton order, so
// they share most senders): e_slot[e] = the slot of edge e's sender in its group (255: none, the sender found no slot
// or the edge lies beyond the group's first SLOT_EDGES), g_send[group][slot] = the sender, g_n[group] = slots in use.
// Once per chunk, for the 8 channel blocks of the backward (which hashed the senders 8 times before).
#define MM_SLOT_HASH 2048
extern "C" __global__ void __launch_bounds__(256)
mm_sender_slots_kernel(const int* __restrict__ rowptr, int nC, const int* __restrict__ send,
    unsigned char* __restrict__ e_slot, int* __restrict__ g_send, int* __restrict__ g_n) {
  __shared__ int hkey[MM_SLOT_HASH];
  __shared__ unsigned char hslot[MM_SLOT_HASH];
  __shared__ int nslot;
  const int i0 = blockIdx.x * GROUP, tid = threadIdx.x;
  const int E0 = rowptr[i0], nE = rowptr[min(i0 + GROUP, nC)] - E0, nH = min(nE, SLOT_EDGES);
  for (int h = tid; h < MM_SLOT_HASH; h += 256) hkey[h] = -1;
  if (tid == 0) nslot = 0;
  __syncthreads();
  for (int j = tid; j < nH; j += 256) {   // at most SLOT_EDGES keys: the probing ends at a free entry
    const int s = send[E0 + j];
    unsigned h = ((unsigned)s * 2654435761u) >> 21;
    while (true) {
      const int prev = atomicCAS(&hkey[h], -1, s);
      if (prev == -1) {
        const int sl = atomicAdd(&nslot, 1);
        hslot[h] = sl < SLOTS ? (unsigned char)sl : 255;
        if (sl < SLOTS) g_send[(size_t)blockIdx.x * SLOTS + sl] = s;
      }
      if (prev == -1 || prev == s) break;
      h = (h + 1) & (MM_SLOT_HASH - 1);
    }
  }
  __syncthreads();
  for (int j = tid; j < nE; j += 256) {
    unsigned char sl = 255;
    if (j < nH) {
      const int s = send[E0 + j];
      unsigned h = ((unsigned)s * 2654435761u) >> 21;
      while (hkey[h] != s) h = (h + 1) & (MM_SLOT_HASH - 1);
      sl = hslot[h];
    }
    e_slot[E0 + j] = sl;
  }
  if (tid == 0) g_n[blockIdx.x] = min(nslot, SLOTS);
}

extern "C" int mm_sender_slots(const int* rowptr, int nC, const int* send, unsigned char* e_slot, int* g_send, int* g_n,
    hipStream_t stream) {
  MM_CHECK_ARG(nC >= 0, "bad sizes");
  if (nC == 0) return MM_OK;
  hipLaunchKernelGGL(mm_sender_slots_kernel, dim3((nC + GROUP - 1) / GROUP), dim3(256), 0, stream, rowptr, nC, send,
                     e_slot, g_send, g_n);
  return mm::launch_status("mm_sender_slots");
}
"""

POLAR_HEADER = """// generated by mace_onegpu/codegen.py -- harmonics of an edge direction with their tangential
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
"""

GROUP = 4        # receivers per workgroup, one per wave
SLOTS = 208      # LDS accumulators (64 floats) of a workgroup's distinct senders (at most a workgroup's threads)
SLOT_EDGES = 1024   # edges of a group that take part in the slots


def conv2_bwd_vec_source(tab, depth=2):
    """Backward kernels mm_conv2_bwd_vec (dL/dX pooled per receiver group in LDS) and mm_conv2_bwd_vec_det (a row of
    dL/dX per edge)."""
    nX, nW, nO, terms = tab["nX"], tab["nW"], tab["nO"], tab["terms"]
    norm = polar_norms()
    G = OrderedDict()
    for (w, k, m, o, cf) in terms:
        G.setdefault((w, k, m), []).append((o, cf * norm[m]))
    gmax = max(sum(abs(c) for _, c in lst) for lst in G.values())
    # |G| <= gmax max|g|; the operand is scaled to at most 2^15
    b_exp = 14 - int(np.ceil(np.log2(gmax)))
    xoff = o3.Irreps(tab["in_ls"]).offsets
    paths = []                                  # (w, l2, [k])
    for w, (i1, l1, l2, l3) in enumerate(tab["paths"]):
        paths.append((w, l2, [xoff[i1] + a for a in range(2 * l1 + 1)]))
    steps = sorted([p for p in paths if p[1]], key=lambda p: (-p[1], p[0])) + [p for p in paths if not p[1]]
    n = len(steps)
    degrees = sorted({p[1] for p in paths if p[1]}, reverse=True)
    L = [BWD_VEC_HEADER.replace("SLOT_EDGES", str(SLOT_EDGES)).replace("MM_SLOT_HASH", "@H@").replace("SLOTS", str(SLOTS))
         .replace("GROUP", str(GROUP)).replace("@H@", "MM_SLOT_HASH")]
    A = L.append

    def gexpr(w, k, m):
        e = None
        for (o, cc) in G.get((w, k, m), []):
            if e is None:
                e = f"g{o}" if abs(cc - 1) < 1e-12 else f"{_f(cc)} * g{o}"
            else:
                e = f"fmaf({_f(cc)}, g{o}, {e})"
        return e or "0.f"

    def gfactors(w, k, m):
        """The two factors of an entry (a sum of several terms: the sum and 1)."""
        lst = G.get((w, k, m), [])
        return (_f(lst[0][1]), f"g{lst[0][0]}") if len(lst) == 1 else (gexpr(w, k, m), "1.f")

    def kernel(name, mode):
        pool = mode == "pool"
        A(f"extern \"C\" __global__ void __launch_bounds__({64 * GROUP}, 2)")
        A(f"{name}(const int* __restrict__ rowptr, int nC, const floatx4* __restrict__ e_pk,")
        A("    const floatx4* __restrict__ e_u, const float* __restrict__ X, int x_stride,")
        A("    const floatx4* __restrict__ tab, int tab_cb_stride, float inv_h,")
        A("    const float* __restrict__ gA, float* __restrict__ part, long part_stride, float* __restrict__ gX" +
          (",\n    const unsigned char* __restrict__ e_slot, const int* __restrict__ g_send,\n"
           "    const int* __restrict__ g_n) {" if pool else ") {"))
        A("  const int cb = mm_xcd_channel_block();")
        A(f"  __shared__ uint4v ya_all[{GROUP * 3 * len(degrees) * 32}];   // per wave: [type][degree][edge][piece] operand rows")
        A(f"  const int grp = blockIdx.x >> 3, i = grp * {GROUP} + (threadIdx.x >> 6);")
        if pool:
            A(f"  __shared__ floatx4 gxs4[{SLOTS * 4 * nX}];   // [slot][component][16 channels]")
            A(f"  __shared__ int ssend[{SLOTS}];")
            A("  float* __restrict__ gxs = (float*)gxs4;")
            A("  const int ns = g_n[grp];")
            A("  const int ir = min(i, nC - 1);   // waves past the last receiver prepare for it and take no edges")
        else:
            A("  if (i >= nC) return;")
            A("  const int ir = i;")
        A("  const int lane = threadIdx.x & 63, cl = lane & 15, eg = lane >> 4;")
        A(f"  uint4v* __restrict__ ya = ya_all + (threadIdx.x >> 6) * {3 * len(degrees) * 32};")
        A("  const int c = cb * 16 + cl;")
        A("  const int e0 = rowptr[ir], e1 = i < nC ? rowptr[ir + 1] : e0;")
        A("  const char* __restrict__ tcb = (const char*)(tab + (size_t)cb * tab_cb_stride);")
        A(f"  const float* __restrict__ gp = gA + (size_t)ir * {nO * C} + c;")
        for o in range(nO):
            A(f"  float g{o} = gp[{o * C}];")
        A("  // power-of-two scale of this channel's constants into the fp16 range")
        mx = "0.f"
        for o in range(0, nO, 2):
            mx = f"fmaxf(fmaxf(fabsf(g{o}), fabsf(g{o + 1})), {mx})" if o + 1 < nO else f"fmaxf(fabsf(g{o}), {mx})"
            if o % 8 == 6 or o + 2 >= nO:
                A(f"  {'const float mx0' if o == 6 else f'const float mx{o // 8}'} = {mx};")
                mx = f"mx{o // 8}"
        A(f"  const int gex = max(__float_as_int({mx}) >> 23, 40);")
        A(f"  const float gsc = __int_as_float(({127 + 127 + b_exp} - gex) << 23);")
        A(f"  const float gun = __int_as_float((gex - {b_exp + 13}) << 23);   // 1 / (gsc MM_POLAR_SCALE)")
        for w, l2, ks in paths:
            if l2 == 0:
                for k in ks:
                    A(f"  const float U{w}_{k} = {gexpr(w, k, 0)} * gsc * MM_POLAR_SCALE;   // l2 = 0: the same u for every edge")
        for o in range(nO):
            A(f"  g{o} *= gsc;")
        A("  // B operands: lane (channel cl, k-group eg) holds fp16 piece 1 - (eg & 1) of its channel's constants")
        A("  const bool pb = !(eg & 1);")
        for w, l2, ks in steps:
            if not l2:
                continue
            for k in ks:
                nm = 2 * l2 + 1
                nr = 2 if l2 == 1 else 4
                A(f"  uint{nr}v B{w}_{k};")
                for j in range(nr):
                    ms = [l2 * l2 + 2 * j + q for q in (0, 1)]
                    ex = [gfactors(w, k, m) if m < l2 * l2 + nm else ("0.f", "1.f") for m in ms]
                    if all(e[0] == "0.f" for e in ex):
                        A(f"  B{w}_{k}[{j}] = 0;")
                    else:
                        A(f"  {{ unsigned h0, h1; mm_split2_f16(float2v{{{ex[0][0]}, {ex[1][0]}}}, float2v{{{ex[0][1]}, {ex[1][1]}}}, h0, h1); "
                          f"B{w}_{k}[{j}] = pb ? h1 : h0; }}")

        def rec_load(eb):
            """Records of this lane's four edges of the tile at eb (clamped to the receiver's last edge)."""
            for v in range(4):
                A(f"    pkn{v} = e_pk[min({eb} + 4 * eg + {v}, e1 - 1)];")
            A(f"    un = e_u[min({eb} + cl, e1 - 1)];")

        def rec_rows():
            for v in range(4):
                A(f"    on{v} = (unsigned)__float_as_int(pkn{v}.y) * {nW * 256}u + cl * 16u;")

        def qload(j, suffix, decl):
            for v in range(4):
                A(f"    {'floatx4 ' if decl else ''}q{j}_{v} = *(const floatx4*)(tcb + o{suffix}{v} + {steps[j][0] * 256});")

        if pool:
            A(f"  if ((int)threadIdx.x < ns) ssend[threadIdx.x] = g_send[(size_t)grp * {SLOTS} + threadIdx.x];")
            A(f"  for (int j = threadIdx.x; j < ns * {4 * nX}; j += {64 * GROUP}) gxs4[j] = floatx4{{0.f, 0.f, 0.f, 0.f}};")
            A("  __syncthreads();")
        A("  if (e0 < e1) {")
        A("  floatx4 pkn0, pkn1, pkn2, pkn3, un;   // records and edge vector of the next tile")
        A("  unsigned on0, on1, on2, on3;           // its table rows")
        rec_load("e0")
        rec_rows()
        for j in range(depth):
            qload(j, "n", True)
        A("  for (int eb = e0; eb < e1; eb += 16) {")
        for v in range(4):
            A(f"    const float t{v} = pkn{v}.x;")
            A(f"    const unsigned o{v} = on{v};")
            A(f"    const float* __restrict__ xp{v} = X + (size_t)__float_as_int(pkn{v}.z) * x_stride + c;")
            for k in range(nX):
                A(f"    const float X{k}_{v} = xp{v}[{k * C}];")
        A("    const floatx4 ua = un;")
        A("    // the next tile's records and edge vector are loaded one tile ahead (the last tile reloads its own end)")
        rec_load("eb + 16")
        if pool:
            A("    const unsigned sl4 = mm_load_u32(e_slot + eb + 4 * eg);   // slots of four edges (the array is padded)")
        A("    // A operands of edge eb + cl: lane group 0 the harmonics, 1 and 2 their two derivatives")
        A("    {")
        A("      float F[16], A[16], s, cp, sp;")
        A("      mm_polar(ua.x, ua.y, s, cp, sp);")
        A("      mm_polar_operands(ua.x, ua.y, ua.z, s, cp, sp, eg, F, A);")
        A("      mm_wave_lds_sync();   // the previous tile's operands have been read")
        A("      if (eg < 3) {")
        for d, l2 in enumerate(degrees):
            nm = 2 * l2 + 1
            A(f"        {{ uint4v a = {{}}, b = {{}};")
            for j in range((nm + 1) // 2):
                m = [l2 * l2 + 2 * j + q for q in (0, 1)]
                v = [", ".join(f"{nm}[{q}]" if q < l2 * l2 + nm2 else "0.f" for q in m) for nm, nm2 in (("F", nm), ("A", nm))]
                A(f"          {{ unsigned h0, h1; mm_split2_f16(float2v{{{v[0]}}}, float2v{{{v[1]}}}, h0, h1); a[{j}] = h0; b[{j}] = h1; }}")
            A(f"          uint4v* __restrict__ d = ya + ((eg * {len(degrees)} + {d}) * 16 + cl) * 2;")
            A("          d[0] = a; d[1] = b; }")
        A("      }")
        A("      mm_wave_lds_sync();")
        A("    }")
        for v in range(4):
            A(f"    float gr{v} = 0.f, gt{v} = 0.f, gp{v} = 0.f;")
            for k in range(nX):
                A(f"    float gx{k}_{v} = 0.f;")

        def path(j, ks, src):
            """Contributions of a path; src(k, v) -> (u, dtheta, dphi) expressions for edge v (None: zero)."""
            for v in range(4):
                A("    {")
                A(f"      const floatx4 q = q{j}_{v};")
                A(f"      const float a = fmaf(q.w, t{v}, q.z);")
                A(f"      const float b = fmaf(a, t{v}, q.y);")
                A(f"      const float W = fmaf(b, t{v}, q.x);")
                A(f"      const float D = fmaf(fmaf(q.w, t{v}, a), t{v}, b);")
                for k in ks:
                    A(f"      gx{k}_{v} = fmaf(W, {src(k, v)[0]}, gx{k}_{v});")
                for ty, (g, f) in enumerate((("gr", "D"), ("gt", "W"), ("gp", "W"))):
                    if src(ks[0], v)[ty] is None:
                        continue
                    e = None
                    for k in ks:
                        u = src(k, v)[ty]
                        e = f"X{k}_{v} * {u}" if e is None else f"fmaf(X{k}_{v}, {u}, {e})"
                    A(f"      {g}{v} = fmaf({e}, {f}, {g}{v});")
                A("    }")
        last = None
        for j, (w, l2, ks) in enumerate(steps):
            if l2:
                ht = "half4v" if l2 == 1 else "half8v"
                mf = "__builtin_amdgcn_mfma_f32_16x16x16f16" if l2 == 1 else "__builtin_amdgcn_mfma_f32_16x16x32_f16"
                if l2 != last:
                    d = degrees.index(l2)
                    for ty in range(3):
                        row = f"ya[(({ty * len(degrees) + d}) * 16 + cl) * 2 + 1 - (eg >> 1)]"
                        if l2 == 1:
                            A(f"    const half4v A{l2}_{ty} = __builtin_bit_cast(half4v, *(const uint2v*)&{row});")
                        else:
                            A(f"    const half8v A{l2}_{ty} = __builtin_bit_cast(half8v, {row});")
                    last = l2
                for k in ks:
                    for ty in range(3):
                        A(f"    const floatx4 D{ty}_{w}_{k} = {mf}(A{l2}_{ty}, __builtin_bit_cast({ht}, B{w}_{k}), floatx4{{0.f, 0.f, 0.f, 0.f}}, 0, 0, 0);")
                path(j, ks, lambda k, v: tuple(f"D{ty}_{w}_{k}[{v}]" for ty in range(3)))
            else:
                path(j, ks, lambda k, v: (f"U{w}_{k}", None, None))
            # keep the accumulation here (the compiler would sink the sums below the loop body's branches and hold
            # every path's W and u until then)
            ops = ", ".join(f'"+v"(gx{k}_{v})' for k in ks for v in range(4))
            A(f"    asm volatile(\"\" : {ops});")
            if j + depth == n:
                rec_rows()
            if j + depth < n:
                qload(j + depth, "", True)
            else:
                qload(j + depth - n, "n", False)
        A("    const int n_own = min(e1 - (eb + 4 * eg), 4);   // this lane's edges inside the receiver's range (may be <= 0)")
        A("    // sums over the 16 channels of the row: transpose-reduction, lane cl = 3 v + j ends with value j of edge v")
        vals = [f"{nm}{v}" for v in range(4) for nm in ("gr", "gt", "gp")]
        for x in vals:
            A(f"    {x} *= gun;")
        A("    const bool b3 = cl & 8, b2 = cl & 4, b1 = cl & 2, b0 = cl & 1;")
        for j in range(8):
            hi = vals[8 + j] if 8 + j < 12 else "0.f"
            A(f"    const float s8_{j} = (b3 ? {hi} : {vals[j]}) + mm_dpp<0x140>(b3 ? {vals[j]} : {hi});")
        for j in range(4):
            A(f"    const float s4_{j} = (b2 ? s8_{4 + j} : s8_{j}) + mm_dpp<0x141>(b2 ? s8_{j} : s8_{4 + j});")
        for j in range(2):
            A(f"    const float s2_{j} = (b1 ? s4_{2 + j} : s4_{j}) + mm_dpp<0x1B>(b1 ? s4_{j} : s4_{2 + j});")
        A("    float sum = (b0 ? s2_1 : s2_0) + mm_dpp<0xB1>(b0 ? s2_0 : s2_1);")
        A("    const float tc = cl < 3 ? t0 : cl < 6 ? t1 : cl < 9 ? t2 : t3;")
        A("    if (cl == 0 || cl == 3 || cl == 6 || cl == 9) sum *= mm_spline_dxdr(tc, inv_h);   // zero below the table start")
        A("    if (cl < 12 && cl < 3 * n_own)")
        A("      part[(size_t)cb * part_stride + (size_t)(eb + 4 * eg) * 3 + cl] = sum;")
        if pool:
            for v in range(4):
                A(f"    const unsigned sl{v} = (sl4 >> {8 * v}) & 255u;")
            A("    // the group's LDS accumulators of the senders by 32-bit compare-and-swap, all issued together and repeated only")
            A("    // where another wave came between; edges without a slot add to gX directly")
            A("    if (__all(n_own == 4 && !(sl0 == 255 || sl1 == 255 || sl2 == 255 || sl3 == 255))) {")
            vk = [(v, k) for v in range(4) for k in range(nX)]
            for v in range(4):
                A(f"      unsigned* __restrict__ l{v} = (unsigned*)gxs + sl{v} * {16 * nX} + cl;")
            for v, k in vk:
                A(f"      unsigned a{k}_{v} = l{v}[{16 * k}];")
            for v, k in vk:
                A(f"      unsigned r{k}_{v} = atomicCAS(l{v} + {16 * k}, a{k}_{v}, "
                  f"__float_as_uint(fmaf(gx{k}_{v}, gun, __uint_as_float(a{k}_{v}))));")
            A("      if (" + " | ".join(f"(r{k}_{v} != a{k}_{v})" for v, k in vk) + ") {")
            for v, k in vk:
                A(f"        while (r{k}_{v} != a{k}_{v}) {{ a{k}_{v} = r{k}_{v}; r{k}_{v} = atomicCAS(l{v} + {16 * k}, "
                  f"a{k}_{v}, __float_as_uint(fmaf(gx{k}_{v}, gun, __uint_as_float(a{k}_{v})))); }}")
            A("      }")
            A("    } else {")
            for v in range(4):
                A(f"      if ({v} < n_own) {{")
                A(f"        if (sl{v} != 255) {{")
                A(f"          mm_lds_add4_f32(gxs + sl{v} * {16 * nX} + cl, gx0_{v} * gun, gx1_{v} * gun, gx2_{v} * gun, gx3_{v} * gun);")
                A("        } else {")
                A(f"          float* __restrict__ gxp = gX + (size_t)__float_as_int(e_pk[eb + 4 * eg + {v}].z) * {nX * C} + cb * {16 * nX} + cl;")
                for k in range(nX):
                    A(f"          atomicAdd(gxp + {16 * k}, gx{k}_{v} * gun);")
                A("        }")
                A("      }")
            A("    }")
        else:
            for v in range(4):
                A(f"    if ({v} < n_own) {{")
                A(f"      float* __restrict__ gxp = gX + (size_t)(eb + 4 * eg + {v}) * {nX * C} + cb * {16 * nX} + cl;")
                for k in range(nX):
                    A(f"      gxp[{16 * k}] = gx{k}_{v} * gun;")
                A("    }")
        A("  }")
        A("  }   // edges")
        if pool:
            A("  __syncthreads();")
            A(f"  for (int j = threadIdx.x; j < ns * 64; j += {64 * GROUP}) {{")
            A("    const int sl = j >> 6, r = j & 63;   // a slot: 256 contiguous bytes [component][channel] of its sender's row")
            A(f"    atomicAdd(gX + (size_t)ssend[sl] * {nX * C} + cb * {16 * nX} + r, gxs[j]);")
            A("  }")
        A("}")
        A("")
        A(f"extern \"C\" int {name[:-7]}(const int* rowptr, int nC, const float* e_pk, const float* e_u,")
        A("    const float* X, int x_stride, const float* tab, int n_tab, int M, float inv_h, const float* gA,")
        A("    float* part, long part_stride, float* gX," + (" const unsigned char* e_slot, const int* g_send, const int* g_n,"
                                                           if pool else "") + " hipStream_t stream) {")
        A("  MM_CHECK_ARG(nC >= 0 && M >= 2 && n_tab >= 1, \"bad sizes\");")
        if pool:
            A("  MM_CHECK_ARG(e_slot && g_send && g_n, \"the groups' sender slots (mm_sender_slots) are required\");")
        A("  MM_CHECK_ARG(gX != nullptr, \"the sender-feature gradient buffer is required\");")
        A(f"  MM_CHECK_ARG((long)n_tab * (M - 1) * {nW * 256} < (1L << 32), \"a channel block's tables exceed 4 GiB\");")
        A("  if (nC == 0) return MM_OK;")
        A(f"  hipLaunchKernelGGL({name}, dim3(8 * ((nC + 3) / 4)), dim3(256), 0, stream, rowptr, nC,")
        A(f"                     (const floatx4*)e_pk, (const floatx4*)e_u, X, x_stride, (const floatx4*)tab,")
        A(f"                     n_tab * (M - 1) * {nW * 16}, inv_h, gA, part, part_stride, gX" +
          (", e_slot, g_send, g_n);" if pool else ");"))
        A(f"  return mm::launch_status(\"{name[:-7]}\");")
        A("}")
        A("")
    kernel("mm_conv2_bwd_vec_kernel", "pool")
    kernel("mm_conv2_bwd_vec_det_kernel", "edge")
    return "\n".join(L) + "\n"


# ----------------------------------------------------------------------------- explicit-weight convolution
TPW_TABLES = o3.COMPILED_TP_TABLES


# When the four waves of a workgroup of the explicit-weight kernels share one receiver's edges instead of taking a
# receiver each.  With few receivers it is the parallelism that pays (501 receivers of 37 edges, shared against not:
# forward l1 34 -> 14 us, l2 68 -> 26; backward l1 83 -> 27, l2 106 -> 62); with many, a wave streams contiguous rows of
# W next to its neighbours' (16,384 receivers of 90 edges: forward l2 1,651 -> 1,559 us, backward 4,121 -> 4,015), but
# each pays for its part of the reduction or its own receiver constants, so short receivers stay whole. Mean edges per
# receiver from which they are shared, by the accumulators (forward) or constants (backward) per lane: at 16,384
# receivers forward l1 (32) 3 edges 39 -> 39 us, 7 83 -> 72; l2 (80) 7 199 -> 198, 13 306 -> 287; l0123 (99) 13 718 ->
# 732, 20 1,037 -> 1,019; backward l1 (32) 3 85 -> 83, l2 (76) 7 407 -> 417, 13 689 -> 680.  A backward in path groups
# (l0123) has several waves per receiver already: shared up to SHARE_WAVES of them (37 edges: 1,500 waves 139 -> 94 us,
# 9,000 633 -> 619, 12,000 799 -> 817).
SHARE_WAVES = 8192


def _share_edges(state):
    return 4 if state <= 40 else 10 if state <= 88 else 18


def tpw_layout(tab):
    """Lane layout of the explicit-weight kernels of one path table.  A wave serves one receiver and a row of 64
    or 128 channels: cpl channels per lane (c = 64 h + lane + 64 j, j < cpl), nh = 2 / cpl waves per receiver
    (channel halves h).  Two channels per lane while the per-lane state fits (forward: 2 nO accumulators;
    backward: 2 x terms constants coef g_o), else one; unroll = edges whose loads are issued together (2, or 1
    when the doubled W / X registers would cost occupancy).  parts = dL/dY partial rows per edge (one per
    channel half of the backward)."""
    nO, nT, nW, nX = tab["nO"], len(tab["terms"]), tab["nW"], tab["nX"]
    cpl_f = 2 if 2 * nO <= 96 else 1
    # the backward keeps one constant per (path, X component, harmonic) and channel across the edge loop (at most
    # one per term); a table with more terms than fit is split into path groups (one wave each, _path_groups)
    cpl_b = 2 if 2 * nT <= 64 else 1
    pgs = _path_groups(tab)
    npg = len(pgs)
    unroll_f = 2 if cpl_f * (nO + 2 * (nW + nX)) <= 160 else 1
    g_terms = max(sum(1 for t in tab["terms"] if t[0] in g) for g in pgs)
    state_b = cpl_b * g_terms + 16 + cpl_b * nX
    unroll_b = 2 if state_b + 2 * cpl_b * (nW // npg + nX) <= 180 else 1
    unroll_b = 1 if npg > 1 else unroll_b
    return dict(cpl_fwd=cpl_f, nh_fwd=2 // cpl_f, unroll_fwd=unroll_f, cpl_bwd=cpl_b, nh_bwd=2 // cpl_b,
                unroll_bwd=unroll_b, npg=npg, parts=(2 // cpl_b) * npg)


def _tpw_groups(tab):
    """(w, k) term groups of a table, in (w, k) order."""
    groups = OrderedDict()
    for (w, k, m, o, c) in sorted(tab["terms"], key=lambda t: (t[0], t[1])):
        groups.setdefault((w, k), []).append((m, o, c))
    return groups


def _path_groups(tab, max_terms=140):
    """The backward's path groups of at most about max_terms terms: paths with the same input components k (one
    input irrep) are grouped together, so that a group adds the dL/dX of few components (one atomic add per
    component, channel and group); a larger irrep's paths are split into balanced parts, and the smallest groups
    are merged while the merge stays within max_terms.  One group when the whole table has at most max_terms
    terms."""
    groups = _tpw_groups(tab)
    used_w = sorted({w for (w, k) in groups})
    if len(tab["terms"]) <= max_terms:
        return [used_w]
    ks = {w: frozenset(k for (ww, k) in groups if ww == w) for w in used_w}
    cnt = {w: sum(len(lst) for (ww, k), lst in groups.items() if ww == w) for w in used_w}
    bins = {}
    for w in used_w:
        bins.setdefault(ks[w], []).append(w)
    out = []
    for b in bins.values():          # a bin above max_terms: split into balanced parts (largest paths first)
        n = -(-sum(cnt[w] for w in b) // max_terms)
        parts, load = [[] for _ in range(n)], [0] * n
        for w in sorted(b, key=lambda w: (-cnt[w], w)):
            j = min(range(n), key=lambda q: (load[q], q))
            parts[j].append(w)
            load[j] += cnt[w]
        out += parts
    out = sorted(out, key=lambda g: sum(cnt[w] for w in g))
    while len(out) > 1 and sum(cnt[w] for w in out[0] + out[1]) <= max_terms:
        out = sorted([out[0] + out[1]] + out[2:], key=lambda g: sum(cnt[w] for w in g))
    return [sorted(g) for g in sorted(out, key=min)]


def _bwd_constants(gsel):
    """The backward's receiver constants: one per (path w, X component k, harmonic m),
    G[w, k, m] = sum over the table's terms (w, k, m, o) of coef g_o (the terms of one (w, k, m) differ only in o).
    Returns (index of each (w, k, m), the distinct m of each (w, k) in term order, [(o, coef), ...] per index)."""
    tid, gm, sums = {}, OrderedDict(), []
    for (w, k), lst in gsel:
        ms = OrderedDict()
        for (m, o, cf) in lst:
            ms.setdefault(m, []).append((o, cf))
        gm[(w, k)] = list(ms)
        for m, ocs in ms.items():
            tid[(w, k, m)] = len(tid)
            sums.append(ocs)
    return tid, gm, sums


def _const_expr(ocs, g):
    """sum of coef g(o) over ocs = [(o, coef), ...], as one product and a chain of FMAs."""
    e = (("-" if ocs[0][1] < 0 else "") + g(ocs[0][0]) if abs(abs(ocs[0][1]) - 1.0) <= 1e-12
         else f"{_f(ocs[0][1])} * {g(ocs[0][0])}")
    for (o, cf) in ocs[1:]:
        e = f"fmaf({_f(cf)}, {g(o)}, {e})"
    return e


def tpw_source(tab, name):
    """gather(sender) x channelwise TP with per-edge weights W [E, nW, 128] x receiver-CSR sum, and its backward
    (dW, dY, dX): the kernels behind FusedConvTP (fused_conv.py:33-37 of the reference).  These kernels read
    explicit weights, not a table, so nothing gains from keeping channel blocks on XCDs: a wave takes whole rows
    of channels (tpw_layout), every W / X / gW access is a 256-byte run per instruction, the harmonics of an
    edge are read once (a wave-uniform address) and dL/dY is reduced over the wave's channels in the kernel."""
    nX, nW, nO, terms = tab["nX"], tab["nW"], tab["nO"], tab["terms"]
    lay = tpw_layout(tab)
    used_m = sorted({t[2] for t in terms})
    used_o = sorted({t[3] for t in terms})
    groups = OrderedDict()
    for (w, k, m, o, c) in sorted(terms, key=lambda t: (t[0], t[1])):
        groups.setdefault((w, k), []).append((m, o, c))
    used_k = sorted({k for (w, k) in groups})
    used_w = sorted({w for (w, k) in groups})

    def coef_mul(c, v):
        if abs(abs(c) - 1.0) <= 1e-12:
            return ("-" if c < 0 else "") + v
        return f"{_f(c)} * {v}"

    kn = f"tpw_{name}"
    L = []
    A = L.append

    def head(kind, nh, npg=1, shared=False):
        """Wave -> (receiver i, sub-wave h): h = channel half * npg + path group; c = first channel of the lane
        (channel half * 64 + lane), always < 128.  shared: one (i, h) per workgroup, a quarter of the receiver's edges
        per wave."""
        if shared:
            A("  const int wave = threadIdx.x >> 6;")
            A("  const int gw = blockIdx.x;   // receiver i, sub-wave h")
        else:
            A(f"  const int gw = blockIdx.x * 4 + (threadIdx.x >> 6);   // global wave: receiver i, sub-wave h")
        A(f"  const int i = gw / {nh}, h = gw % {nh};" if nh > 1 else "  const int i = gw, h = 0;")
        A("  if (i >= nR) return;")
        A("  const int lane = threadIdx.x & 63;")
        A(f"  const int c = (h / {npg}) * 64 + lane;" if npg > 1 else "  const int c = h * 64 + lane;")
        if shared:
            A("  const int r0 = rowptr[i], nr = rowptr[i + 1] - r0;")
            A("  const int p0 = r0 + (int)((long)nr * wave / 4), p1 = r0 + (int)((long)nr * (wave + 1) / 4);")
        else:
            A("  const int p0 = rowptr[i], p1 = rowptr[i + 1];")

    def edge_loads(t, cpl, pidx, guard=None, ws=None, ks=None):
        ws = used_w if ws is None else ws
        ks = used_k if ks is None else ks
        e = f"e{t}"
        # the edge and its sender are the same for the whole wave: readfirstlane makes that visible to the
        # compiler, so the harmonics and the indices come through scalar loads
        if guard is None:
            A(f"    const int {e} = __builtin_amdgcn_readfirstlane(eid ? eid[{pidx}] : {pidx});")
        else:
            A(f"    const int {e} = {guard} ? __builtin_amdgcn_readfirstlane(eid ? eid[{pidx}] : {pidx}) : ea;")
        A(f"    const int s{t} = __builtin_amdgcn_readfirstlane(send[{e}]);")
        A(f"    const float* __restrict__ wp{t} = W + (size_t){e} * w_stride + c;")
        for w in ws:
            for j in range(cpl):
                A(f"    const float W{w}_{j}_{t} = wp{t}[{w * C + 64 * j}];")
        A(f"    const float* __restrict__ xp{t} = X + (size_t)s{t} * x_stride + c;")
        for k in ks:
            for j in range(cpl):
                A(f"    const float X{k}_{j}_{t} = xp{t}[{k * C + 64 * j}];")
        A(f"    const float* __restrict__ yp{t} = Y + (size_t){e} * y_stride;")
        for m in used_m:
            A(f"    const float Y{m}_{t} = yp{t}[{m}];")

    # ------------------------------------------------------------------ header comment
    A(f"// generated by mace_onegpu/codegen.py -- explicit-weight channelwise TP '{name}'")
    A(f"// nX={nX}, nW={nW}, nO={nO}, terms={len(terms)}")
    A("//")
    A("// out[i, o, c] = sum_{p in [rowptr[i], rowptr[i+1])} sum_terms coef * W[e, w, c] * X[send[e], k, c] * Y[e, m],")
    A("// e = eid[p] (or p when eid is null): receiver-CSR over a permutation, so edges need not be stored sorted.")
    A(f"// Forward: one wave per receiver and channel half, {lay['cpl_fwd']} channel(s) per lane (c = 64 h + lane + 64 j),")
    A(f"// {lay['nh_fwd']} wave(s) per receiver, {lay['unroll_fwd']} edge(s) loaded together.  Backward: "
      f"{lay['cpl_bwd']} channel(s) per lane, {lay['nh_bwd']} wave(s)")
    A(f"// per receiver, {lay['unroll_bwd']} edge(s) loaded together; dL/dY partials: {lay['parts']} per edge "
      "(one per channel half).")
    A('#include "../common.h"')
    A("")
    # ------------------------------------------------------------------ forward
    def forward(shared):
        cpl, nh, un = lay["cpl_fwd"], lay["nh_fwd"], lay["unroll_fwd"]
        A("extern \"C\" __global__ void __launch_bounds__(256)")
        A(f"mm_{kn}_fwd{'_shared' if shared else ''}_kernel(const int* __restrict__ rowptr, int nR, const int* __restrict__ eid,")
        A("    const int* __restrict__ send, const float* __restrict__ Y, long y_stride, const float* __restrict__ W,")
        A("    long w_stride, const float* __restrict__ X, long x_stride, float* __restrict__ out, long out_stride) {")
        accs = [f"acc{o}_{j}" for o in used_o for j in range(cpl)]
        if shared:
            A(f"  __shared__ float red[{len(accs)} * 64];   // one wave's sums [accumulator][lane]")
        head("fwd", nh, shared=shared)
        for o in used_o:
            for j in range(cpl):
                A(f"  float acc{o}_{j} = 0.f;")

        def fwd_body(t):
            # per (w, k) group: q = W X, one product q |coef| per distinct |coef| of the group, then one FMA per term
            # with the edge's (wave-uniform) harmonic
            for (w, k), lst in groups.items():
                mags = OrderedDict()
                for (m, o, c) in lst:
                    if abs(abs(c) - 1.0) > 1e-12:
                        mags.setdefault(round(abs(c), 12), (len(mags), abs(c)))
                for j in range(cpl):
                    A(f"    {{ const float q = W{w}_{j}_{t} * X{k}_{j}_{t};")
                    for key, (idx, ac) in mags.items():
                        A(f"      const float q{idx} = {_f(ac)} * q;")
                    for (m, o, c) in lst:
                        key = round(abs(c), 12)
                        qv = f"q{mags[key][0]}" if key in mags else "q"
                        A(f"      acc{o}_{j} = fmaf({'-' if c < 0 else ''}{qv}, Y{m}_{t}, acc{o}_{j});")
                    A("    }")

        if un == 2:
            A("  for (int p = p0; p < p1; p += 2) {")
            A("    const bool two = p + 1 < p1;   // wave-uniform")
            edge_loads("a", cpl, "p")
            edge_loads("b", cpl, "p + 1", guard="two")
            fwd_body("a")
            A("    if (two) {")
            fwd_body("b")
            A("    }")
            A("  }")
        else:
            A("  for (int p = p0; p < p1; ++p) {")
            edge_loads("a", cpl, "p")
            fwd_body("a")
            A("  }")
        if shared:
            A("  for (int s = 1; s < 4; ++s) {   // the waves' sums in wave order")
            A("    if (wave == s) {")
            for q, v in enumerate(accs):
                A(f"      red[{64 * q} + lane] = {v};")
            A("    }")
            A("    __syncthreads();")
            A("    if (wave == 0) {")
            for q, v in enumerate(accs):
                A(f"      {v} += red[{64 * q} + lane];")
            A("    }")
            A("    __syncthreads();")
            A("  }")
            A("  if (wave) return;")
        A("  float* __restrict__ op = out + (size_t)i * out_stride + c;")
        for o in range(nO):
            for j in range(cpl):
                v = f"acc{o}_{j}" if o in used_o else "0.f"
                A(f"  op[{o * C + 64 * j}] = {v};")
        A("}")
        A("")

    forward(False)
    forward(True)
    # ------------------------------------------------------------------ backward
    def backward(shared):
        cpl, nh, un, npg = lay["cpl_bwd"], lay["nh_bwd"], lay["unroll_bwd"], lay["npg"]
        pgroups = _path_groups(tab)
        A("// Backward from gO = dL/dout: gW[e, w, c] (written), gYp[part][e][m] = partial sums of dL/dY[e, m] over")
        A(f"// the channels and paths of one wave ({lay['parts']} partial(s): channel half h x path group g, part")
        A(f"// h * {npg} + g; summed by the caller), gX[send, k, c] (atomic adds).  Null outputs are skipped.")
        if npg > 1:
            A(f"// Path groups (one wave each): {pgroups}.")
        A("extern \"C\" __global__ void __launch_bounds__(256)")
        A(f"mm_{kn}_bwd{'_shared' if shared else ''}_kernel(const int* __restrict__ rowptr, int nR, const int* __restrict__ eid,")
        A("    const int* __restrict__ send, const float* __restrict__ Y, long y_stride, const float* __restrict__ W,")
        A("    long w_stride, const float* __restrict__ X, long x_stride, const float* __restrict__ gO, long g_stride,")
        A("    float* __restrict__ gW, long gw_stride, float* __restrict__ gYp, long gy_cb_stride,")
        A("    float* __restrict__ gX, long gx_stride) {")
        head("bwd", nh * npg, npg, shared)
        if npg > 1:
            A(f"  const int pg = h % {npg};   // path group; channel half h / {npg}")
        A("  const int part = h;")
        A("  const int cl = lane & 15;")
        A("  const bool b3 = cl & 8, b2 = cl & 4, b1 = cl & 2, b0 = cl & 1;")

        def bwd_group(gi, wsel):
            gsel = [(wk, lst) for wk, lst in groups.items() if wk[0] in wsel]
            ksel = sorted({k for (w, k), _ in gsel})
            osel = sorted({o for _, lst in gsel for (m, o, cf) in lst})
            A("  const float* __restrict__ gp = gO + (size_t)i * g_stride + c;")
            for o in osel:
                for j in range(cpl):
                    A(f"  const float g{o}_{j} = gp[{o * C + 64 * j}];")
            tid, gm, sums = _bwd_constants(gsel)
            for n, ocs in enumerate(sums):
                for j in range(cpl):
                    A(f"  const float G{n}_{j} = {_const_expr(ocs, lambda o: f'g{o}_{j}')};")

            def bwd_body(t):
                for m in range(16):
                    A(f"    float gy{m} = 0.f;")
                for k in ksel:
                    for j in range(cpl):
                        A(f"    float gx{k}_{j} = 0.f;")
                A(f"    float* __restrict__ gwp = gW ? gW + (size_t)e{t} * gw_stride + c : nullptr;")
                for w in wsel:
                    A("    {")
                    for j in range(cpl):
                        A(f"      float gw{j} = 0.f;")
                    for (ww, k), lst in gsel:
                        if ww != w:
                            continue
                        for j in range(cpl):
                            A(f"      {{ const float q = W{w}_{j}_{t} * X{k}_{j}_{t}; float u = 0.f;")
                            for m in gm[(w, k)]:
                                G = f"G{tid[(w, k, m)]}_{j}"
                                A(f"        u = fmaf(Y{m}_{t}, {G}, u); gy{m} = fmaf(q, {G}, gy{m});")
                            A(f"        gw{j} = fmaf(X{k}_{j}_{t}, u, gw{j}); gx{k}_{j} = fmaf(W{w}_{j}_{t}, u, gx{k}_{j});")
                            A("      }")
                    for j in range(cpl):
                        A(f"      if (gwp) gwp[{w * C + 64 * j}] = gw{j};")
                    A("    }")
                if gi == 0:
                    for w in range(nW):
                        if w not in used_w:
                            for j in range(cpl):
                                A(f"    if (gwp) gwp[{w * C + 64 * j}] = 0.f;")
                A("    if (gYp) {")
                A("      // transpose-reduction over each 16-lane row (lane cl ends with the row's sum of gy_cl), then the"
                  " 4 rows")
                for j in range(8):
                    A(f"      const float s8_{j} = (b3 ? gy{8 + j} : gy{j}) + mm_dpp<0x140>(b3 ? gy{j} : gy{8 + j});")
                for j in range(4):
                    A(f"      const float s4_{j} = (b2 ? s8_{4 + j} : s8_{j}) + mm_dpp<0x141>(b2 ? s8_{j} : s8_{4 + j});")
                for j in range(2):
                    A(f"      const float s2_{j} = (b1 ? s4_{2 + j} : s4_{j}) + mm_dpp<0x1B>(b1 ? s4_{j} : s4_{2 + j});")
                A("      float gyl = (b0 ? s2_1 : s2_0) + mm_dpp<0xB1>(b0 ? s2_0 : s2_1);")
                A("      gyl += __shfl_xor(gyl, 16);")
                A("      gyl += __shfl_xor(gyl, 32);")
                A(f"      if (lane < 16) gYp[(size_t)part * gy_cb_stride + (size_t)e{t} * 16 + lane] = gyl;")
                A("    }")
                A("    if (gX) {")
                A(f"      float* __restrict__ gxp = gX + (size_t)s{t} * gx_stride + c;")
                for k in ksel:
                    for j in range(cpl):
                        A(f"      atomicAdd(gxp + {k * C + 64 * j}, gx{k}_{j});")
                A("    }")

            if un == 2:
                A("  for (int p = p0; p < p1; p += 2) {")
                A("    const bool two = p + 1 < p1;   // wave-uniform")
                edge_loads("a", cpl, "p", ws=wsel, ks=ksel)
                edge_loads("b", cpl, "p + 1", guard="two", ws=wsel, ks=ksel)
                bwd_body("a")
                A("    if (two) {")
                bwd_body("b")
                A("    }")
                A("  }")
            else:
                A("  for (int p = p0; p < p1; ++p) {")
                edge_loads("a", cpl, "p", ws=wsel, ks=ksel)
                bwd_body("a")
                A("  }")

        if npg == 1:
            bwd_group(0, pgroups[0])
        else:
            for gi, wsel in enumerate(pgroups):
                A(f"  {'if' if gi == 0 else 'else if'} (pg == {gi}) {{")
                bwd_group(gi, wsel)
                A("  }")
        A("}")
        A("")

    backward(False)
    backward(True)
    # ------------------------------------------------------------------ entry points
    for kind, nh_k in (("fwd", lay["nh_fwd"]), ("bwd", lay["nh_bwd"] * lay["npg"])):
        state = (lay["cpl_fwd"] * len(used_o) if kind == "fwd" else
                 lay["cpl_bwd"] * len(_bwd_constants(list(groups.items()))[2]))
        few = f"waves <= {SHARE_WAVES}" if kind == "bwd" and lay["npg"] > 1 else "true"
        if kind == "fwd":
            A(f"extern \"C\" int mm_{kn}_fwd_n(long E, const int* rowptr, int nR, const int* eid, const int* send, const float* Y,")
            A("    long y_stride, const float* W, long w_stride, const float* X, long x_stride, float* out, long out_stride,")
            A("    hipStream_t stream) {")
            A("  MM_CHECK_ARG(nR >= 0, \"bad sizes\");")
            A(f"  MM_CHECK_ARG(y_stride >= 16 && w_stride >= {nW * C} && x_stride >= {nX * C} && out_stride >= {nO * C},")
            A("               \"row strides smaller than the path table's widths\");")
        else:
            A(f"extern \"C\" int mm_{kn}_bwd_n(long E, const int* rowptr, int nR, const int* eid, const int* send, const float* Y,")
            A("    long y_stride, const float* W, long w_stride, const float* X, long x_stride, const float* gO, long g_stride,")
            A("    float* gW, long gw_stride, float* gYp, long gy_cb_stride, float* gX, long gx_stride, hipStream_t stream) {")
            A("  MM_CHECK_ARG(nR >= 0, \"bad sizes\");")
            A(f"  MM_CHECK_ARG(y_stride >= 16 && w_stride >= {nW * C} && x_stride >= {nX * C} && g_stride >= {nO * C},")
            A("               \"row strides smaller than the path table's widths\");")
            A(f"  MM_CHECK_ARG(!gW || gw_stride >= {nW * C}, \"gW row stride\");")
            A(f"  MM_CHECK_ARG(!gX || gx_stride >= {nX * C}, \"gX row stride\");")
        A("  if (nR == 0) return MM_OK;")
        A(f"  const long waves = (long)nR * {nh_k};")
        A("  // E < 0: unknown, shared where the receivers alone leave most of the chip idle")
        A("  // (a launch takes fewer than 2^32 threads)")
        A(f"  const bool shared = E < 0 ? waves <= 2048 : {few} && waves < (1L << 24) && E >= {_share_edges(state)}L * nR;")
        A("  dim3 grid((unsigned)(shared ? waves : (waves + 3) / 4)), block(256);")
        if kind == "fwd":
            A(f"  hipLaunchKernelGGL(shared ? mm_{kn}_fwd_shared_kernel : mm_{kn}_fwd_kernel, grid, block, 0, stream, rowptr, nR, eid, send, Y, y_stride, W,")
            A("                     w_stride, X, x_stride, out, out_stride);")
        else:
            A(f"  hipLaunchKernelGGL(shared ? mm_{kn}_bwd_shared_kernel : mm_{kn}_bwd_kernel, grid, block, 0, stream, rowptr, nR, eid, send, Y, y_stride, W,")
            A("                     w_stride, X, x_stride, gO, g_stride, gW, gw_stride, gYp, gy_cb_stride, gX, gx_stride);")
        A(f"  return mm::launch_status(\"mm_{kn}_{kind}\");")
        A("}")
        A("")
        args = ("rowptr, nR, eid, send, Y, y_stride, W, w_stride, X, x_stride, " +
                ("out, out_stride" if kind == "fwd" else "gO, g_stride, gW, gw_stride, gYp, gy_cb_stride, gX, gx_stride"))
        A(f"extern \"C\" int mm_{kn}_{kind}(const int* rowptr, int nR, const int* eid, const int* send, const float* Y,")
        A("    long y_stride, const float* W, long w_stride, const float* X, long x_stride,")
        A("    float* out, long out_stride, hipStream_t stream) {" if kind == "fwd" else
          "    const float* gO, long g_stride, float* gW, long gw_stride, float* gYp, long gy_cb_stride, float* gX,\n"
          "    long gx_stride, hipStream_t stream) {")
        A(f"  return mm_{kn}_{kind}_n(-1, {args}, stream);")
        A("}")
        A("")
    return "\n".join(L)


def conv_wide_source(tab, name):
    """Fused spline-table radial weights x channelwise TP x receiver sum for a wide path table (the benchmark's
    literal node features 0e+1o+2e+3o: 16 components, 23 paths, 353 terms), forward and backward: the
    reference's generated ConvSpline kernels for any path table (conv_spline.py:38-94, 97-181).  Layout as the
    explicit-weight kernels (tpw_layout: whole channel rows per wave, path groups in the backward), with W and
    dW/dt evaluated per edge from the interval coefficients (the layer-2 table layout, any nW) and the harmonics
    from the edge's unit vector; the backward writes per-edge partial rows (inv_h dL/dr, dL/dY[16]) for
    mm_edge_grad, one per wave of a receiver, and adds dL/dX to the senders."""
    nX, nW, nO, terms = tab["nX"], tab["nW"], tab["nO"], tab["terms"]
    lay = tpw_layout(tab)
    groups = _tpw_groups(tab)
    used_m = sorted({t[2] for t in terms})
    used_o = sorted({t[3] for t in terms})
    used_w = sorted({w for (w, k) in groups})

    def coef_mul(c, v):
        if abs(abs(c) - 1.0) <= 1e-12:
            return ("-" if c < 0 else "") + v
        return f"{_f(c)} * {v}"

    kn = f"conv{name}"
    L = []
    A = L.append

    def head(nh, npg=1):
        A("  const int gw = blockIdx.x * 4 + (threadIdx.x >> 6);   // global wave: receiver i, sub-wave h")
        A(f"  const int i = gw / {nh}, h = gw % {nh};" if nh > 1 else "  const int i = gw, h = 0;")
        A("  if (i >= nC) return;")
        A("  const int lane = threadIdx.x & 63;")
        A(f"  const int c = (h / {npg}) * 64 + lane;   // channel of the lane, < 128" if npg > 1 else
          "  const int c = h * 64 + lane;   // channel of the lane, < 128")
        A("  const floatx4* __restrict__ tcl = tab + (size_t)(c >> 4) * tab_cb_stride + (c & 15);")
        A("  const int e0 = rowptr[i], e1 = rowptr[i + 1];")

    def edge_in(ws, ks, deriv):
        A("    const floatx4 pk = e_pk[e];   // (t, interval row, sender row, density); the same for the wave")
        A("    const floatx4 u = e_u[e];     // (unit vector, r)")
        A("    const float t = pk.x;")
        A("    const int s = __float_as_int(pk.z);")
        A(f"    const floatx4* __restrict__ tp = tcl + (size_t)__float_as_int(pk.y) * {nW * 16};")
        for w in ws:
            A(f"    const floatx4 q{w} = tp[{w * 16}];")
        A("    const float* __restrict__ xp = X + (size_t)s * x_stride + c;")
        for k in ks:
            A(f"    const float X{k} = xp[{k * C}];")
        for w in ws:
            A(f"    const float s{w} = fmaf(q{w}.w, t, q{w}.z), r{w} = fmaf(s{w}, t, q{w}.y);")
            A(f"    const float W{w} = fmaf(r{w}, t, q{w}.x);")
            if deriv:
                A(f"    const float D{w} = fmaf(fmaf(q{w}.w, t, s{w}), t, r{w});   // dW/dt")
        A("    float Yv[16];")
        A("    mm_sh16(u.x, u.y, u.z, Yv);")

    A(f"// generated by mace_onegpu/codegen.py -- fused spline-table channelwise TP '{name}' (spline W x TP x sum)")
    A(f"// nX={nX}, nW={nW}, nO={nO}, terms={len(terms)}")
    A("//")
    A("// out[i, o, c] = sum_{e in [rowptr[i], rowptr[i+1])} sum_terms coef * W(t_e; row_e)[w, c] * X[s_e, k, c] * Y_m(u_e),")
    A("// rho[i] = sum of the edges' densities; W from the interval coefficients tab (float4 [cb][row][w][16],")
    A("// row = table * (M - 1) + interval, as built by mm_spline_coeffs).  Edge records as the layer-2 kernels:")
    A("// e_pk = (t, row, sender row, density), e_u = (unit vector, r).")
    A("// Forward: per channel block of 16 (one per XCD, blockIdx.x % 8) and path group one wave per receiver, lanes =")
    A("// 4 edge slots x 16 channels.  Backward: one channel per lane, " + str(lay['nh_bwd'] * lay['npg']) +
      " waves per receiver (channel half x path group);")
    A(f"// backward partial rows part[h][e][17] = (inv_h dL/dr, dL/dY), h < {lay['parts']}.")
    A('#include "../common.h"')
    A('#include "sh.h"')
    A("")
    assert lay["cpl_fwd"] == 1 and lay["cpl_bwd"] == 1, "the wide kernels take one channel per lane"
    # ------------------------------------------------------------------ forward
    # the outputs o of different paths are disjoint, so the backward's path groups split the forward as well:
    # each wave accumulates only its group's outputs and loads only its group's table rows and X components.
    # Layout of the layer-2 kernels: blockIdx.x % 8 = the channel block of 16 channels, served by one XCD, whose
    # table slice (M - 1 rows x nW x 16 x 16 B) stays in that XCD's L2; a wave takes 4 edges of its receiver at a
    # time (lanes = 4 edge slots x 16 channels) and sums the slots at the end.
    pgroups = _path_groups(tab)
    npf = len(pgroups)
    A("extern \"C\" __global__ void __launch_bounds__(256)")
    A(f"mm_{kn}_fwd_kernel(const int* __restrict__ rowptr, int nC, const floatx4* __restrict__ e_pk,")
    A("    const floatx4* __restrict__ e_u, const float* __restrict__ X, int x_stride, const floatx4* __restrict__ tab,")
    A("    long tab_cb_stride, float* __restrict__ out, float* __restrict__ rho) {")
    A("  const int cb = mm_xcd_channel_block();")
    A("  const int gw = (blockIdx.x >> 3) * 4 + (threadIdx.x >> 6);   // receiver i, path group pg")
    A(f"  const int i = gw / {npf}, pg = gw % {npf};" if npf > 1 else "  const int i = gw, pg = 0;")
    A("  if (i >= nC) return;")
    A("  const int lane = threadIdx.x & 63, cl = lane & 15, slot = lane >> 4;")
    A("  const int c = cb * 16 + cl;")
    A("  const floatx4* __restrict__ tcl = tab + (size_t)cb * tab_cb_stride + cl;")
    A("  const int e0 = rowptr[i], e1 = rowptr[i + 1];")
    A(f"  float* __restrict__ op = out + (size_t)i * {nO * C} + c;")
    for o in range(nO):
        if o not in used_o:
            A(f"  if (pg == 0 && slot == {o % 4}) op[{o * C}] = 0.f;")
    for gi, wsel in enumerate(pgroups):
        gsel = [(wk, lst) for wk, lst in groups.items() if wk[0] in wsel]
        ksel = sorted({k for (w, k), _ in gsel})
        osel = sorted({o for _, lst in gsel for (m, o, cf) in lst})
        A(f"  {'if' if gi == 0 else 'else if'} (pg == {gi}) {{")
        for o in osel:
            A(f"    float acc{o} = 0.f;")
        if gi == 0:
            A("    float dsum = 0.f;")
        A("    for (int e = e0 + slot; e < e1; e += 4) {")
        edge_in(wsel, ksel, False)
        if gi == 0:
            A("      dsum += pk.w;")
        for (w, k), lst in gsel:
            mags = OrderedDict()
            for (m, o, cf) in lst:
                if abs(abs(cf) - 1.0) > 1e-12:
                    mags.setdefault(round(abs(cf), 12), (len(mags), abs(cf)))
            A(f"      {{ const float q = W{w} * X{k};")
            for key, (idx, ac) in mags.items():
                A(f"        const float q{idx} = {_f(ac)} * q;")
            for (m, o, cf) in lst:
                key = round(abs(cf), 12)
                qv = f"q{mags[key][0]}" if key in mags else "q"
                A(f"        acc{o} = fmaf({'-' if cf < 0 else ''}{qv}, Yv[{m}], acc{o});")
            A("      }")
        A("    }")
        for o in osel:
            A(f"    acc{o} += __shfl_xor(acc{o}, 16); acc{o} += __shfl_xor(acc{o}, 32);")
            A(f"    if (slot == {o % 4}) op[{o * C}] = acc{o};")
        if gi == 0:
            A("    dsum += __shfl_xor(dsum, 16); dsum += __shfl_xor(dsum, 32);")
            A("    if (cb == 0 && lane == 0) rho[i] = dsum;")
        A("  }")
    A("}")
    A("")
    # ------------------------------------------------------------------ backward
    nh, npg = lay["nh_bwd"], lay["npg"]
    pgroups = _path_groups(tab)
    A("// Backward from gA = dL/dout [nC, nO, 128]: part[h][e] = (inv_h dL/dr, dL/dY[16]) summed over the channels")
    A("// and paths of sub-wave h (mm_edge_grad sums the partial rows); gX[s, k, c] += dL/dX (atomic adds, when gX is")
    A("// not null).")
    A(f"// Path groups (one wave each): {pgroups}.")
    A("extern \"C\" __global__ void __launch_bounds__(256)")
    A(f"mm_{kn}_bwd_kernel(const int* __restrict__ rowptr, int nC, const floatx4* __restrict__ e_pk,")
    A("    const floatx4* __restrict__ e_u, const float* __restrict__ X, int x_stride, const floatx4* __restrict__ tab,")
    A("    long tab_cb_stride, float inv_h, const float* __restrict__ gA, float* __restrict__ part, long part_stride,")
    A("    float* __restrict__ gX) {")
    head(nh * npg, npg)
    if npg > 1:
        A(f"  const int pg = h % {npg};")
    A("  const int cl = lane & 15;")
    A("  const bool b3 = cl & 8, b2 = cl & 4, b1 = cl & 2, b0 = cl & 1;")
    A(f"  const float* __restrict__ gp = gA + (size_t)i * {nO * C} + c;")
    A("  float* __restrict__ pb = part + (size_t)h * part_stride;")

    def group(wsel):
        gsel = [(wk, lst) for wk, lst in groups.items() if wk[0] in wsel]
        ksel = sorted({k for (w, k), _ in gsel})
        osel = sorted({o for _, lst in gsel for (m, o, cf) in lst})
        for o in osel:
            A(f"    const float g{o} = gp[{o * C}];")
        tid, gm, sums = _bwd_constants(gsel)
        for n, ocs in enumerate(sums):
            A(f"    const float G{n} = {_const_expr(ocs, lambda o: f'g{o}')};")
        A("    for (int e = e0; e < e1; ++e) {")
        edge_in(wsel, ksel, True)
        for m in range(16):
            A(f"      float gy{m} = 0.f;")
        for k in ksel:
            A(f"      float gx{k} = 0.f;")
        A("      float gr = 0.f;")
        for w in wsel:
            A("      { float gw = 0.f;")
            for (ww, k), lst in gsel:
                if ww != w:
                    continue
                A(f"        {{ const float q = W{w} * X{k}; float uu = 0.f;")
                for m in gm[(w, k)]:
                    G = f"G{tid[(w, k, m)]}"
                    A(f"          uu = fmaf(Yv[{m}], {G}, uu); gy{m} = fmaf(q, {G}, gy{m});")
                A(f"          gw = fmaf(X{k}, uu, gw); gx{k} = fmaf(W{w}, uu, gx{k});")
                A("        }")
            A(f"        gr = fmaf(gw, D{w}, gr);")
            A("      }")
        A("      // transpose-reduction over each 16-lane row (lane cl ends with the row's sum of gy_cl), then the 4 rows")
        for j in range(8):
            A(f"      const float s8_{j} = (b3 ? gy{8 + j} : gy{j}) + mm_dpp<0x140>(b3 ? gy{j} : gy{8 + j});")
        for j in range(4):
            A(f"      const float s4_{j} = (b2 ? s8_{4 + j} : s8_{j}) + mm_dpp<0x141>(b2 ? s8_{j} : s8_{4 + j});")
        for j in range(2):
            A(f"      const float s2_{j} = (b1 ? s4_{2 + j} : s4_{j}) + mm_dpp<0x1B>(b1 ? s4_{j} : s4_{2 + j});")
        A("      float gyl = (b0 ? s2_1 : s2_0) + mm_dpp<0xB1>(b0 ? s2_0 : s2_1);")
        A("      gyl += __shfl_xor(gyl, 16);")
        A("      gyl += __shfl_xor(gyl, 32);")
        A("      gr = mm_row_sum16(gr);")
        A("      gr += __shfl_xor(gr, 16);")
        A("      gr += __shfl_xor(gr, 32);")
        A("      float* __restrict__ pp = pb + (size_t)e * 17;")
        A("      if (lane < 16) pp[1 + lane] = gyl;")
        A("      if (lane == 0) pp[0] = gr * mm_spline_dxdr(t, inv_h);   // zero below the table start")
        A("      if (gX) {")
        A("        float* __restrict__ gxp = gX + (size_t)s * x_stride + c;")
        for k in ksel:
            A(f"        atomicAdd(gxp + {k * C}, gx{k});")
        A("      }")
        A("    }")

    for gi, wsel in enumerate(pgroups):
        A(f"  {'if' if gi == 0 else 'else if'} ({'pg' if npg > 1 else '0'} == {gi}) {{")
        group(wsel)
        A("  }")
    A("}")
    A("")
    tab_stride = f"(long)n_tab * (M - 1) * {nW * 16}"
    A(f"extern \"C\" int mm_{kn}_fwd(const int* rowptr, int nC, const float* e_pk, const float* e_u, const float* X,")
    A("    int x_stride, const float* tab, int n_tab, int M, float* out, float* rho, hipStream_t stream) {")
    A(f"  MM_CHECK_ARG(nC >= 0 && M >= 2 && n_tab >= 1 && x_stride >= {nX * C}, \"bad sizes\");")
    A("  if (nC == 0) return MM_OK;")
    A(f"  dim3 grid((unsigned)(8 * (((long)nC * {len(_path_groups(tab))} + 3) / 4))), block(256);")
    A(f"  hipLaunchKernelGGL(mm_{kn}_fwd_kernel, grid, block, 0, stream, rowptr, nC, (const floatx4*)e_pk,")
    A(f"                     (const floatx4*)e_u, X, x_stride, (const floatx4*)tab, {tab_stride}, out, rho);")
    A(f"  return mm::launch_status(\"mm_{kn}_fwd\");")
    A("}")
    A("")
    A(f"extern \"C\" int mm_{kn}_bwd(const int* rowptr, int nC, const float* e_pk, const float* e_u, const float* X,")
    A("    int x_stride, const float* tab, int n_tab, int M, float inv_h, const float* gA, float* part,")
    A("    long part_stride, float* gX, hipStream_t stream) {")
    A(f"  MM_CHECK_ARG(nC >= 0 && M >= 2 && n_tab >= 1 && x_stride >= {nX * C}, \"bad sizes\");")
    A("  if (nC == 0) return MM_OK;")
    A(f"  dim3 grid((unsigned)(((long)nC * {nh * npg} + 3) / 4)), block(256);")
    A(f"  hipLaunchKernelGGL(mm_{kn}_bwd_kernel, grid, block, 0, stream, rowptr, nC, (const floatx4*)e_pk,")
    A(f"                     (const floatx4*)e_u, X, x_stride, (const floatx4*)tab, {tab_stride}, inv_h, gA, part,")
    A("                     part_stride, gX);")
    A(f"  return mm::launch_status(\"mm_{kn}_bwd\");")
    A("}")
    A("")
    return "\n".join(L)


def tpw_tables():
    """{name: path table} of the explicit-weight kernels that the build compiles."""
    return OrderedDict((n, o3.tp_table(list(a), b, c)) for n, (a, b, c) in TPW_TABLES.items())


# ----------------------------------------------------------------------------- symmetric contraction
def symc_model_flops(paths, out_ls, C=128):
    """Forward FLOPs per node of one symmetric contraction by the dense-coefficient convention: every non-zero of
    every path's coupling tensor U_p[M, i1..i_nu] costs nu + 1 multiplications-with-accumulate (the weight and the
    nu features) per channel, at 2 flops each -- the count of the reference's flop budget
    (scripts/flop_budget.py:11-35, 52-56).  The generated kernels evaluate the same sums factorised (shared
    intermediates, nu = 3 paths grouped before the last coupling) and execute fewer operations."""
    import numpy as np
    tot = 0
    for L in out_ls:
        for nu in sorted(paths[L]):
            for pth in paths[L][nu]:
                if pth[0] == "1":
                    nnz = 2 * L + 1
                elif pth[0] == "2":
                    _, l1, l2 = pth
                    nnz = int((np.abs(o3.coupling(l1, l2, L)) > 1e-12).sum())
                else:
                    _, l1, l2, J, l3 = pth
                    U = np.einsum("abj,jcm->mabc", o3.coupling(l1, l2, J), o3.coupling(J, l3, L))
                    nnz = int((np.abs(U) > 1e-12).sum())
                tot += 2 * (int(pth[0]) + 1) * nnz
    return tot * C


def kernel_body(src, kernel):
    """Text of the __global__ function `kernel` in generated source `src` (up to the next extern "C")."""
    i = src.index(kernel + "(")
    j = src.find('extern "C"', i)
    return src[i:j if j >= 0 else len(src)]


def written_flops(body):
    """Floating-point operations written in a generated kernel body, per thread: every arithmetic statement
    (`const float v = e;`, `v = e;`, `v += e;`) whose expression reads no memory, with fmaf counted as 2, every other
    binary * and + (or -) as 1, a += as 1, and multiplications by the literal 1.0f not counted (the compiler folds
    them).  Address arithmetic and loads / stores (expressions with [ ]) and the cross-lane reductions are not
    counted."""
    import re
    total = 0
    for stmt in body.split(";"):
        st = stmt.strip()
        m = re.match(r"^(?:const\s+float\s+)?([A-Za-z_][A-Za-z0-9_]*)\s*(\+?=)\s*(.+)$", st, re.S)
        if not m or "[" in st or "__shfl" in st or "(size_t)" in st:
            continue
        if m.group(1) in ("node", "c", "h", "o") or not re.search(r"[A-Za-z_]", m.group(3)):
            continue
        e = re.sub(r"\b1\.0f\s*\*\s*", "", m.group(3))
        n_fma = e.count("fmaf(")
        total += 2 * n_fma + e.count("*") + len(re.findall(r"\s[+-]\s", e)) + (1 if m.group(2) == "+=" else 0)
    return total


def asm_valu_flops(asm, kernel):
    """fp32 VALU arithmetic of `kernel` in gfx950 assembly text, per thread: every v_fma / v_fmac / v_fmamk /
    v_fmaak _f32 counts 2 flops, every v_mul / v_add / v_sub / v_subrev _f32 1 (exact executed work for
    straight-line code; packed-FP32 instructions are disabled in this build and counted 4 if present)."""
    import re
    start = asm.index(f"\n{kernel}:")
    end = asm.index("s_endpgm", start)
    body = asm[start:end]
    fma = len(re.findall(r"^\s+v_(?:fma|fmac|fmamk|fmaak)_f32", body, re.M))
    one = len(re.findall(r"^\s+v_(?:mul|add|sub|subrev)_f32", body, re.M))
    pk = len(re.findall(r"^\s+v_pk_(?:fma|mul|add)_f32", body, re.M))
    return dict(flops=2 * fma + one + 4 * pk, fma=fma, mul_add=one, packed=pk)


def symc_executed_flops(gen_dir, layer, C=128, ops_json=None):
    """{'fwd': F, 'bwd': F}: floating-point operations per node that the generated contraction kernels of `layer`
    execute: from the kernels' gfx950 assembly when the build's ops_json holds them (asm_valu_flops), otherwise
    the source-level count (written_flops), per channel thread times C channels."""
    import json
    import os
    if ops_json and os.path.exists(ops_json):
        with open(ops_json) as fh:
            ops = json.load(fh)
        return {d: C * ops[f"mm_symc{layer}_{d}_kernel"]["flops"] for d in ("fwd", "bwd")}
    src = open(os.path.join(gen_dir, f"symc_l{layer}.hip")).read()
    return {d: C * written_flops(kernel_body(src, f"mm_symc{layer}_{d}_kernel")) for d in ("fwd", "bwd")}


def symc_source(paths, out_ls, in_ls, layer):
    """paths: {L: {nu: [path]}}.  Weight layout: Wsc[species][p][128] with p enumerating, for L in out_ls, for
    nu = 1..3, the paths in order."""
    xin = o3.Irreps(in_ls)
    off = {l: xin.offsets[i] for i, l in enumerate(in_ls)}
    outI = o3.Irreps(out_ls)
    nOut = outI.dim
    plist = []
    for L in out_ls:
        for nu in sorted(paths[L]):
            for pth in paths[L][nu]:
                plist.append((L, pth))
    P = len(plist)
    # distinct nu=3 intermediates (l1, l2, J) and nu=3 groups (L, J, l3)
    inter = OrderedDict()
    groups = OrderedDict()
    for pi_, (L, pth) in enumerate(plist):
        if pth[0] == "3":
            _, l1, l2, J, l3 = pth
            inter.setdefault((l1, l2, J), len(inter))
            groups.setdefault((L, J, l3), []).append((pi_, (l1, l2, J)))

    def cg(a, b, c):
        return o3.coupling(a, b, c)

    def nz(T, tol=1e-12):
        import numpy as np
        return [(idx, float(T[idx])) for idx in zip(*np.nonzero(np.abs(T) > tol))]

    def xv(l, a):
        return f"x{off[l] + a}"

    L_ = []
    A = L_.append
    A(f"// generated by mace_onegpu/codegen.py -- symmetric contraction (correlation 3) of product block {layer}")
    A(f"// inputs {xin} per channel, outputs {outI}, {P} coupling paths (weights Wsc[species][path][128]).")
    A("// out_L[M] = sum_nu sum_paths W[s, p, c] * P_p(x)[M] with P built from real coupling coefficients along")
    A("// ((l1 l2) J l3) -> L; the nu=3 paths sharing (L, J, l3) are summed before the last coupling.")
    A("// One thread per (node, channel); block = 256 threads = 2 nodes x 128 channels.")
    A('#include "../common.h"')
    A("")
    # ------------------------------------------------------------------ forward body helper
    def emit_Z(A, ind):
        for (l1, l2, J), zi in inter.items():
            T = cg(l1, l2, J)
            for j in range(2 * J + 1):
                terms = [(a, b, v) for (a, b, jj), v in nz(T) if jj == j]
                expr = " + ".join(f"{_f(v)} * {xv(l1, a)} * {xv(l2, b)}" for a, b, v in terms) or "0.f"
                A(f"{ind}const float z{zi}_{j} = {expr};")

    A(f"extern \"C\" __global__ void __launch_bounds__(256)")
    A(f"mm_symc{layer}_fwd_kernel(int n, const float* __restrict__ x, long x_stride, const int* __restrict__ spec,")
    A("    const float* __restrict__ Wsc, float* __restrict__ out, long out_stride) {")
    A("  const int node = blockIdx.x * 2 + (threadIdx.x >> 7);")
    A("  if (node >= n) return;")
    A("  const int c = threadIdx.x & 127;")
    A("  const float* __restrict__ xp = x + (size_t)node * x_stride + c;")
    for j in range(xin.dim):
        A(f"  const float x{j} = xp[{j * C}];")
    A(f"  const float* __restrict__ wp = Wsc + (size_t)spec[node] * {P * C} + c;")
    for p in range(P):
        A(f"  const float w{p} = wp[{p * C}];")
    emit_Z(A, "  ")
    for L in out_ls:
        for M in range(2 * L + 1):
            A(f"  float o{L}_{M} = 0.f;")
    for pi_, (L, pth) in enumerate(plist):
        if pth[0] == "1":
            for M in range(2 * L + 1):
                A(f"  o{L}_{M} = fmaf(w{pi_}, {xv(pth[1], M)}, o{L}_{M});")
        elif pth[0] == "2":
            _, l1, l2 = pth
            T = cg(l1, l2, L)
            for M in range(2 * L + 1):
                terms = [(a, b, v) for (a, b, mm), v in nz(T) if mm == M]
                expr = " + ".join(f"{_f(v)} * {xv(l1, a)} * {xv(l2, b)}" for a, b, v in terms)
                A(f"  o{L}_{M} = fmaf(w{pi_}, {expr}, o{L}_{M});")
    for gi, ((L, J, l3), mem) in enumerate(groups.items()):
        for j in range(2 * J + 1):
            expr = " + ".join(f"w{pi_} * z{inter[key]}_{j}" for pi_, key in mem)
            A(f"  const float zs{gi}_{j} = {expr};")
        T = cg(J, l3, L)
        for M in range(2 * L + 1):
            terms = [(j, d, v) for (j, d, mm), v in nz(T) if mm == M]
            if terms:
                expr = " + ".join(f"{_f(v)} * zs{gi}_{j} * {xv(l3, d)}" for j, d, v in terms)
                A(f"  o{L}_{M} += {expr};")
    A("  float* __restrict__ op = out + (size_t)node * out_stride + c;")
    for L in out_ls:
        for M in range(2 * L + 1):
            A(f"  op[{(outI.offsets[out_ls.index(L)] + M) * C}] = o{L}_{M};")
    A("}")
    A("")
    # ------------------------------------------------------------------ backward
    A("// Backward: g_x = (d out / d x)^T g_out; also g_rho[node] = -inv(node) * sum_{comp, c} x * g_x with")
    A("// inv = 1 / (rho + 1) (x is the density-normalised message, so this is dL/drho).")
    A(f"extern \"C\" __global__ void __launch_bounds__(256)")
    A(f"mm_symc{layer}_bwd_kernel(int n, const float* __restrict__ x, long x_stride, const int* __restrict__ spec,")
    A("    const float* __restrict__ Wsc, const float* __restrict__ gout, long gout_stride, float* __restrict__ gx,")
    A("    long gx_stride, const float* __restrict__ rho, float* __restrict__ g_rho) {")
    A("  __shared__ float red[4];")
    A("  const int node = blockIdx.x * 2 + (threadIdx.x >> 7);")
    A("  const int c = threadIdx.x & 127;")
    A("  const bool active = node < n;")
    A("  float dot = 0.f;")
    A("  if (active) {")
    A("  const float* __restrict__ xp = x + (size_t)node * x_stride + c;")
    for j in range(xin.dim):
        A(f"  const float x{j} = xp[{j * C}];")
        A(f"  float gx{j} = 0.f;")
    A(f"  const float* __restrict__ wp = Wsc + (size_t)spec[node] * {P * C} + c;")
    for p in range(P):
        A(f"  const float w{p} = wp[{p * C}];")
    A("  const float* __restrict__ gp = gout + (size_t)node * gout_stride + c;")
    for L in out_ls:
        for M in range(2 * L + 1):
            A(f"  const float g{L}_{M} = gp[{(outI.offsets[out_ls.index(L)] + M) * C}];")
    emit_Z(A, "  ")

    def gxv(l, a):
        return f"gx{off[l] + a}"
    for pi_, (L, pth) in enumerate(plist):
        if pth[0] == "1":
            for M in range(2 * L + 1):
                A(f"  {gxv(pth[1], M)} = fmaf(w{pi_}, g{L}_{M}, {gxv(pth[1], M)});")
        elif pth[0] == "2":
            _, l1, l2 = pth
            T = cg(l1, l2, L)
            A("  {")
            for M in range(2 * L + 1):
                A(f"    const float q{M} = w{pi_} * g{L}_{M};")
            for (a, b, M), v in nz(T):
                A(f"    {gxv(l1, a)} = fmaf({_f(v)} * q{M}, {xv(l2, b)}, {gxv(l1, a)});")
                A(f"    {gxv(l2, b)} = fmaf({_f(v)} * q{M}, {xv(l1, a)}, {gxv(l2, b)});")
            A("  }")
    # nu=3: gz for intermediates
    for (l1, l2, J), zi in inter.items():
        for j in range(2 * J + 1):
            A(f"  float gz{zi}_{j} = 0.f;")
    for gi, ((L, J, l3), mem) in enumerate(groups.items()):
        for j in range(2 * J + 1):
            expr = " + ".join(f"w{pi_} * z{inter[key]}_{j}" for pi_, key in mem)
            A(f"  const float zs{gi}_{j} = {expr};")
        T = cg(J, l3, L)
        for j in range(2 * J + 1):
            A(f"  float gzs{gi}_{j} = 0.f;")
        for (j, d, M), v in nz(T):
            A(f"  gzs{gi}_{j} = fmaf({_f(v)} * g{L}_{M}, {xv(l3, d)}, gzs{gi}_{j});")
            A(f"  {gxv(l3, d)} = fmaf({_f(v)} * g{L}_{M}, zs{gi}_{j}, {gxv(l3, d)});")
        for pi_, key in mem:
            zi = inter[key]
            for j in range(2 * J + 1):
                A(f"  gz{zi}_{j} = fmaf(w{pi_}, gzs{gi}_{j}, gz{zi}_{j});")
    for (l1, l2, J), zi in inter.items():
        T = cg(l1, l2, J)
        for (a, b, j), v in nz(T):
            A(f"  {gxv(l1, a)} = fmaf({_f(v)} * gz{zi}_{j}, {xv(l2, b)}, {gxv(l1, a)});")
            A(f"  {gxv(l2, b)} = fmaf({_f(v)} * gz{zi}_{j}, {xv(l1, a)}, {gxv(l2, b)});")
    A("  float* __restrict__ gxp = gx + (size_t)node * gx_stride + c;")
    for j in range(xin.dim):
        A(f"  gxp[{j * C}] = gx{j};")
        A(f"  dot = fmaf(x{j}, gx{j}, dot);")
    A("  }")
    A("  // sum dot over the 128 channel threads of the node (2 waves)")
    A("  for (int o = 32; o >= 1; o >>= 1) dot += __shfl_xor(dot, o);")
    A("  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = dot;")
    A("  __syncthreads();")
    A("  if (active && c == 0) {")
    A("    const int h = (threadIdx.x >> 7) * 2;")
    A("    g_rho[node] = -(red[h] + red[h + 1]) / (rho[node] + 1.f);")
    A("  }")
    A("}")
    A("")
    A(f"extern \"C\" int mm_symc{layer}_fwd(int n, const float* x, long x_stride, const int* spec, const float* Wsc,")
    A("    float* out, long out_stride, hipStream_t stream) {")
    A("  MM_CHECK_ARG(n >= 0, \"bad sizes\");")
    A("  if (n == 0) return MM_OK;")
    A(f"  hipLaunchKernelGGL(mm_symc{layer}_fwd_kernel, dim3((n + 1) / 2), dim3(256), 0, stream, n, x, x_stride,")
    A("                     spec, Wsc, out, out_stride);")
    A(f"  return mm::launch_status(\"mm_symc{layer}_fwd\");")
    A("}")
    A("")
    A(f"extern \"C\" int mm_symc{layer}_bwd(int n, const float* x, long x_stride, const int* spec, const float* Wsc,")
    A("    const float* gout, long gout_stride, float* gx, long gx_stride, const float* rho, float* g_rho,")
    A("    hipStream_t stream) {")
    A("  MM_CHECK_ARG(n >= 0, \"bad sizes\");")
    A("  if (n == 0) return MM_OK;")
    A(f"  hipLaunchKernelGGL(mm_symc{layer}_bwd_kernel, dim3((n + 1) / 2), dim3(256), 0, stream, n, x, x_stride,")
    A("                     spec, Wsc, gout, gout_stride, gx, gx_stride, rho, g_rho);")
    A(f"  return mm::launch_status(\"mm_symc{layer}_bwd\");")
    A("}")
    return "\n".join(L_) + "\n", P, plist


def generate(out_dir, tables):
    """Writes the generated sources into out_dir; returns {name: metadata}."""
    os.makedirs(out_dir, exist_ok=True)
    files = {"sh.h": sh_header(),
             "conv_l1.hip": conv_source(tables.tp1, 1, need_gx=False),
             "conv_l2.hip": conv_source(tables.tp2, 2, need_gx=True)}
    s1, P1, pl1 = symc_source(tables.sc1, [0, 1], [0, 1, 2, 3], 1)
    s2, P2, pl2 = symc_source(tables.sc2, [0], [0, 1, 2, 3], 2)
    files["symc_l1.hip"] = s1
    files["symc_l2.hip"] = s2
    for n, tab in tpw_tables().items():
        files[f"tpw_{n}.hip"] = tpw_source(tab, n)
    files["conv_l0123.hip"] = conv_wide_source(tpw_tables()["l0123"], "0123")
    files.update({"polar.h": POLAR_HEADER, "conv_l2v.hip": conv2_bwd_vec_source(tables.tp2)})
    for name, src in files.items():
        path = os.path.join(out_dir, name)
        if not os.path.exists(path) or open(path).read() != src:
            with open(path, "w") as fh:
                fh.write(src)
    return dict(symc1_paths=pl1, symc2_paths=pl2)


def symc_path_order(paths, out_ls):
    """Path enumeration order of the generated symmetric-contraction kernels (weight rows of Wsc)."""
    out = []
    for L in out_ls:
        for nu in sorted(paths[L]):
            for pth in paths[L][nu]:
                out.append((L, nu, pth))
    return out
