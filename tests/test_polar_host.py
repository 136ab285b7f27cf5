"""The operands of the layer-2 backward's matrix instructions (csrc/gen/polar.h, compiled for the host): two fp16 pieces
hold what their comments say, also for small operands, and the harmonics and tangential derivatives made of them agree
with 64-bit ones."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from mace_onegpu import codegen

GEN = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mace-million_amd", "csrc", "gen")
CLANG = "/opt/rocm/llvm/bin/clang++"
SCALE = 8192.0

SOURCE = f"""
#include <cmath>
using std::fmaf;
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_rsqf(x) (1.0f / std::sqrt(x))
#include "{GEN}/polar.h"
static void pieces(unsigned h0, unsigned h1, float* o) {{
  const half2v a = __builtin_bit_cast(half2v, h0), b = __builtin_bit_cast(half2v, h1);
  o[0] = (float)a.x; o[1] = (float)b.x; o[2] = (float)a.y; o[3] = (float)b.y;
}}
extern "C" void split(const float* a, const float* b, float* o, long n) {{   // n even; o [n][2]
  for (long i = 0; i < n; i += 2) {{
    unsigned h0, h1;
    mm_split2_f16(float2v{{a[i], a[i + 1]}}, float2v{{b[i], b[i + 1]}}, h0, h1);
    pieces(h0, h1, o + 2 * i);
  }}
}}
extern "C" void operands(const float* u, int type, float* o, long n) {{      // o [n][16][2]
  for (long i = 0; i < n; ++i) {{
    float s, cp, sp, F[16], A[16];
    mm_polar(u[3 * i], u[3 * i + 1], s, cp, sp);
    mm_polar_operands(u[3 * i], u[3 * i + 1], u[3 * i + 2], s, cp, sp, type, F, A);
    for (int m = 0; m < 16; m += 2) {{
      unsigned h0, h1;
      mm_split2_f16(float2v{{F[m], F[m + 1]}}, float2v{{A[m], A[m + 1]}}, h0, h1);
      pieces(h0, h1, o + 32 * i + 2 * m);
    }}
  }}
}}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if not os.path.exists(CLANG):
        pytest.skip("no clang with _Float16")
    d = tmp_path_factory.mktemp("polar")
    (d / "polar.cpp").write_text(SOURCE)
    so = d / "polar.so"
    subprocess.run([CLANG, "-O1", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared", "-w", str(d / "polar.cpp"),
                    "-o", str(so)], check=True)
    return ctypes.CDLL(str(so))


def _p(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def test_two_pieces_of_a_product(lib):
    """|a b - h0 - h1| <= 2^-23 |a b| down to 1/4, 2^-25 below (half a subnormal fp16 step)."""
    rng = np.random.default_rng(0)
    n = 200000
    mag = 2.0 ** rng.uniform(-30, 15, n)
    f = 2.0 ** rng.uniform(-8, 0, n)
    a = (np.sign(rng.normal(size=n)) * mag / f).astype(np.float32)
    b = f.astype(np.float32)
    b[::4] = 1.0
    a[::4] = np.minimum(np.abs(a[::4]), 32768)
    a[:8], b[:8] = [1 + 2.0 ** -12 + 2.0 ** -23, 0, -0.0, 2.0 ** -24, 32768, 2.0 ** -25, 4095.75, 3 * 2.0 ** -26], 1.0
    out = np.empty((n, 2), np.float32)
    lib.split(_p(a), _p(b), _p(out), ctypes.c_long(n))
    x = a.astype(np.float64) * b
    err = np.abs(out.astype(np.float64).sum(1) - x)
    assert (err <= np.where(np.abs(x) >= 0.25, 2.0 ** -23 * np.abs(x), 2.0 ** -25)).all()
    assert err[0] == 2.0 ** -23                # a value that two fp16 pieces do not hold


def _reference(u):
    """[3, n, 16]: the basis, d/dtheta and (1 / sin theta) d/dphi at the directions u, in 64 bits."""
    import torch
    th = torch.from_numpy(np.arctan2(np.hypot(u[:, 0], u[:, 1]), u[:, 2])).requires_grad_(True)
    ph = torch.from_numpy(np.arctan2(u[:, 1], u[:, 0])).requires_grad_(True)
    z, s = torch.cos(th), torch.sin(th)
    f = {(0, 0): torch.ones_like(z), (1, 0): z, (1, 1): s, (2, 0): 3 * z * z - 1, (2, 1): z * s, (2, 2): s * s,
         (3, 0): z * (5 * z * z - 3), (3, 1): s * (5 * z * z - 1), (3, 2): z * s * s, (3, 3): s ** 3}
    out = np.zeros((3, len(u), 16))
    for (l, m), v in f.items():
        for sign in (1, -1) if m else (1,):
            B = v * (torch.cos(m * ph) if sign > 0 else torch.sin(m * ph))
            j = l * l + l + sign * m
            out[0, :, j] = B.detach().numpy()
            if l:
                gt, gp = torch.autograd.grad(B.sum(), [th, ph], retain_graph=True, allow_unused=True)
                out[1, :, j] = gt.numpy()
                out[2, :, j] = 0 if gp is None or not m else (gp / s.detach()).numpy()
    assert np.allclose(out[0], codegen._polar_basis(u), atol=1e-12)
    return out


@pytest.mark.parametrize("kind", ["anywhere", "near the z axis", "near the planes"])
def test_harmonics_and_derivatives(lib, kind):
    """Products without a cancelling sum are right to 2^-21 of their own value down to 2^-15 (the split's 2^-23, and up
    to six fp32 roundings of 2^-24 in the direction and the factors), everything to 2.5e-6 absolute (the rounding of
    the direction, 2^-23 along it, times the steepest polynomial's 15, and six roundings of values up to 4)."""
    rng = np.random.default_rng(1)
    v = rng.normal(size=(20000, 3))
    if kind == "near the z axis":
        v[:, :2] *= 2.0 ** rng.uniform(-14, 0, (20000, 1))
    if kind == "near the planes":
        v *= 2.0 ** rng.uniform(-9, 0, v.shape)
    u = (v / np.linalg.norm(v, axis=1)[:, None]).astype(np.float32)
    w = u.astype(np.float64) / np.linalg.norm(u.astype(np.float64), axis=1)[:, None]
    ref = _reference(w)
    for t in range(3):
        out = np.empty((len(u), 16, 2), np.float32)
        lib.operands(_p(u), ctypes.c_int(t), _p(out), ctypes.c_long(len(u)))
        got = out.astype(np.float64).sum(2) / SCALE
        err = np.abs(got - ref[t])
        assert err.max() <= 2.5e-6
        # y, z, x, x y, y z, x z, x y z and their like: m of single products per type
        mono = {0: [1, 2, 3, 4, 5, 7, 10], 1: [1, 2, 3, 6], 2: [1, 3, 5, 7]}[t]
        small = np.abs(ref[t][:, mono]) >= 2.0 ** -15
        assert (err[:, mono][small] <= 2.0 ** -21 * np.abs(ref[t][:, mono][small])).all()
