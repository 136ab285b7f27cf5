"""The division-free minimum image of the kernels (csrc/mic.h, compiled for the host) equals v - L * rint(v / L) bit
for bit: random differences, values around 0, L / 2, L and 3 L / 2, and what falls to the general expression."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mace-million_amd", "csrc", "mic.h")


@pytest.fixture(scope="module")
def mic(tmp_path_factory):
    d = tmp_path_factory.mktemp("mic")
    (d / "mic.cpp").write_text('#include <cmath>\nusing std::fabs; using std::rint;\n#define __device__\n'
                               f'#define __forceinline__ inline\n#include "{HEADER}"\n'
                               'extern "C" void mic(const double* v, double L, double* o, long n) {\n'
                               '  for (long i = 0; i < n; ++i) o[i] = mm_mic(v[i], L, 0.5 * L);\n}\n')
    so = d / "mic.so"
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-fPIC", "-shared", "-w", str(d / "mic.cpp"), "-o", str(so)],
                   check=True)
    lib = ctypes.CDLL(str(so))

    def call(v, L):
        v = np.ascontiguousarray(v, dtype=np.float64)
        out = np.empty_like(v)
        p = ctypes.POINTER(ctypes.c_double)
        lib.mic(v.ctypes.data_as(p), ctypes.c_double(L), out.ctypes.data_as(p), ctypes.c_long(v.size))
        return out
    return call


@pytest.mark.parametrize("L", [12.417, 16.0, 24.833999999999996, 180.0, np.nextafter(16.0, 0), 1.0 + 2.0 ** -52])
def test_equals_the_rounded_quotient_form(mic, L):
    rng = np.random.default_rng(0)
    v = [rng.uniform(-L, L, 200000), rng.uniform(-4 * L, 4 * L, 20000)]
    for c in (0.0, L / 2, L, 1.5 * L, 2.5 * L):
        for s in (-1.0, 1.0):
            x = s * c
            near = [x]
            for _ in range(6):
                near += [np.nextafter(near[-1], np.inf)]
            near += [x]
            for _ in range(6):
                near += [np.nextafter(near[-1], -np.inf)]
            v.append(np.array(near))
    v.append(np.array([-0.0, 0.0, np.inf, -np.inf, np.nan, 1e300, 5e-324]))
    v = np.concatenate(v)
    with np.errstate(invalid="ignore"):
        ref = v - L * np.round(v / L)
    assert np.array_equal(mic(v, L), ref, equal_nan=True)
