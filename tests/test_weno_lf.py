"""FP64 Lax-Friedrichs face flux (two reconstructions over one reciprocal, split
fluxes scaled by 2^-20) against the oracle's WENO5-JS formula, on the host."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from oracle.flux import _weno_core

HERE = os.path.dirname(os.path.abspath(__file__))
D = ctypes.POINTER(ctypes.c_double)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("weno") / "shim_weno.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-x", "c++",
                    os.path.join(HERE, "host", "shim_weno.cpp"), "-o", so], check=True)
    lib = ctypes.CDLL(so)
    lib.host_weno_lf.restype = ctypes.c_double
    return lib


def _stencils(rng, kind, scale):
    if kind == "random":
        return rng.standard_normal(6) * scale
    if kind == "jump":
        return np.where(np.arange(6) < rng.integers(0, 7), 1.0, rng.uniform(0, 1)) * scale
    if kind == "smooth":
        return scale * np.sin(0.05 * np.arange(6) + rng.uniform(0, 6))
    return np.full(6, scale * rng.uniform(-1, 1))          # constant


@pytest.mark.parametrize("kind", ["random", "jump", "smooth", "constant"])
def test_lf_face_flux(lib, kind):
    """Each e_k carries a few roundings on a quadratic form of condition 18
    (about 40 eps relative), the candidates' offsets are at most 4 times the
    stencil's scale and the two values add: 2e-14 of the two scales."""
    rng = np.random.default_rng(1)
    for scale in 10.0 ** np.arange(-9, 16, 1.0):
        for _ in range(60):
            f, g = _stencils(rng, kind, scale), _stencils(rng, kind, scale * 10 **
                                                          rng.uniform(-3, 3))
            p, m = np.ascontiguousarray(f[:5]), np.ascontiguousarray(g[1:])
            got = lib.host_weno_lf(p.ctypes.data_as(D), m.ctypes.data_as(D))
            ref = _weno_core(*p) + _weno_core(*m[::-1])
            assert abs(got - ref) <= 2e-14 * (np.abs(p).max() + np.abs(m).max())


@pytest.mark.parametrize("kind", ["random", "jump", "smooth", "constant"])
def test_face_values(lib, kind):
    """Left and right values over one reciprocal: as the flux above, each value
    within 2e-14 of its stencil's scale."""
    rng = np.random.default_rng(3)
    out = np.zeros(2)
    for scale in 10.0 ** np.arange(-9, 16, 1.0):
        for _ in range(60):
            v = np.ascontiguousarray(_stencils(rng, kind, scale))
            lib.host_weno_LR(v.ctypes.data_as(D), out.ctypes.data_as(D))
            tol = 2e-14 * np.abs(v).max()
            assert abs(out[0] - _weno_core(*v[:5])) <= tol
            assert abs(out[1] - _weno_core(*v[:0:-1])) <= tol
