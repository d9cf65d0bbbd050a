"""The slopes of the stencil weights that the particle backward takes (SlopePair in
csrc/stencil.h), compiled for the host, against FP64: rounded once to FP32, that is within half
an ulp of a value below 2 (6e-8), where a correctly rounded FP32 cosine minus 1 would be within
9e-8."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from ckmpm_amd import build

SRC = """
#include "stencil.h"
extern "C" void slopes(const float* t0, const float* t1, int n, float* d0, float* d1) {
    for (int i = 0; i < n; ++i) ckmpm::SlopePair(t0[i], t1[i], d0[i], d1[i]);
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("slopes")
    src, out = d / "slopes.hip", d / "libslopes.so"
    src.write_text(SRC)
    subprocess.run([build.HIPCC, "--offload-host-only", "-O2", "-std=c++17", "-fPIC", "-shared", "-I", build.CSRC, str(src),
                    "-o", str(out)], check=True, env={**os.environ, "TMPDIR": str(d)})
    return ctypes.CDLL(str(out))


def test_slopes_are_rounded_once(lib):
    # t as MakeStencilPair gives it: a multiple of 2^-22 (positions of 2 to 8 cells) in [0, 1],
    # or just outside, and the other grid's t half a cell away
    k = np.concatenate([np.arange(-400, 2 ** 22 + 400, 7), np.arange(-400, 400), 2 ** 20 + np.arange(-400, 400),
                        2 ** 21 + np.arange(-400, 400), 3 * 2 ** 20 + np.arange(-400, 400), 2 ** 22 + np.arange(-400, 400)])
    t0 = (k / 2.0 ** 22).astype(np.float32)
    t1 = np.where(t0 >= 0.5, t0 - np.float32(0.5), t0 + np.float32(0.5)).astype(np.float32)
    d = [np.empty_like(t0) for _ in range(2)]
    p = [a.ctypes.data_as(ctypes.POINTER(ctypes.c_float)) for a in (t0, t1, *d)]
    lib.slopes(p[0], p[1], t0.shape[0], p[2], p[3])
    for t, got in ((t0, d[0]), (t1, d[1])):
        want = -2.0 * np.sin(np.pi * t.astype(np.float64)) ** 2  # = -1 + cos(2 pi t)
        worst = np.abs(got - want).max()
        print("largest error", worst)
        assert worst <= 2.0 ** -24 * 1.01
