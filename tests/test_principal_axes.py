"""The principal axes of csrc/svd3.h on the CPU (the header compiled for the host):
gradients whose smaller singular values lie anywhere between the largest and far
below its rounding noise, of lower rank, graded, and at the ends of FP32's range.
U and V have to be orthonormal and right-handed, and U S V^T the matrix again."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import PKG

RUNTIME = r"""
#pragma once
#include <cmath>
#include <cstdlib>
#include <cstring>
using std::fabs; using std::fma; using std::fmax; using std::fmin; using std::sqrt; using std::copysign;
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_rsq(d) (1.0 / std::sqrt(d))
inline int __double2hiint(double d) { long long b; std::memcpy(&b, &d, 8); return (int)(b >> 32); }
"""
SOURCE = r"""
#include "svd3.h"
extern "C" int axes(const float* in, double* U, double* S, double* V) {
    float F[3][3]; double u[3][3], v[3][3] = {}, s[3], r[3];
    std::memcpy(F, in, sizeof F);
    const bool regular = mpmx::principal_axes(F, u, s, r);
    if (!regular) mpmx::principal_axes_singular(F, r, u, v);
    std::memcpy(U, u, sizeof u); std::memcpy(S, s, sizeof s); std::memcpy(V, v, sizeof v);
    return regular;
}
"""


@pytest.fixture(scope="module")
def axes(tmp_path_factory):
    d = tmp_path_factory.mktemp("axes")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (d / "axes.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-I", str(d),
                    "-I", os.path.join(PKG, "csrc"), "-o", str(d / "axes.so"), str(d / "axes.cpp")], check=True)
    lib = ctypes.CDLL(str(d / "axes.so"))
    out = ctypes.POINTER(ctypes.c_double)

    def run(F):
        F = np.ascontiguousarray(F, np.float32)
        U, S, V = np.zeros((3, 3)), np.zeros(3), np.zeros((3, 3))
        ok = lib.axes(F.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), *[a.ctypes.data_as(out) for a in (U, S, V)])
        return bool(ok), U, S, V

    return run


def rotations(rng, n):
    q, r = np.linalg.qr(rng.standard_normal((n, 3, 3)))
    q[:, :, 0] *= np.linalg.det(q)[:, None]
    return q


def matrices(kind, n, rng):
    if kind.startswith("rank"):
        r = int(kind[4])
        a = rng.integers(1, 9, (n, 3, r)) * rng.choice([-1, 1], (n, 3, r))
        b = rng.integers(1, 9, (n, 3, r)) * rng.choice([-1, 1], (n, 3, r))
        return (a @ b.transpose(0, 2, 1)) / 4.0 * 10.0 ** rng.choice([-30, 0, 30], (n, 1, 1))
    S = np.zeros((n, 3, 3))
    S[:, 0, 0] = 1.0
    S[:, 1, 1] = 10.0 ** rng.uniform(-30, 0, n)
    S[:, 2, 2] = 10.0 ** rng.uniform(-30, 0, n) * rng.choice([-1, 1], n)
    if kind in ("rotated", "left"):
        S = rotations(rng, n) @ S
    if kind in ("rotated", "right"):
        S = S @ rotations(rng, n)
    return S


@pytest.mark.parametrize("kind", ["rank0", "rank1", "rank2", "rotated", "left", "right", "diagonal"])
def test_orthonormal_axes(axes, kind):
    """1e-10: a thousandth of what shows in FP32 outputs of the largest entry; the
    rotations stop at 2^-50 of a pair's lengths."""
    some = 0
    for F in matrices(kind, 1000, np.random.default_rng(3)):
        ok, U, S, V = axes(F)
        F = F.astype(np.float32).astype(np.float64)
        assert np.abs(U.T @ U - np.eye(3)).max() < 1e-10, F
        if ok:
            continue
        some += 1
        assert np.abs(V.T @ V - np.eye(3)).max() < 1e-10, F
        assert np.linalg.det(U) > 0 and np.linalg.det(V) > 0, F
        assert np.abs(U @ np.diag(S) @ V.T - F).max() <= 1e-10 * np.abs(F).max(), F
    assert some > 300
