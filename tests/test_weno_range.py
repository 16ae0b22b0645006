"""Range of the FP64 face values that share a reciprocal, on the host: finite
and accurate up to the largest stencils stated beside them, far past where the
product of the two denominators leaves FP64."""
import ctypes

import numpy as np
import pytest

from oracle.flux import _weno_core
from test_weno_lf import D, _stencils, lib  # noqa: F401  (the module's host build)

KINDS = ["random", "jump", "smooth", "constant", "alternating"]


def _stencil(rng, kind, scale):
    if kind == "alternating":
        return scale * (-1.0) ** np.arange(6)
    return _stencils(rng, kind, scale)


@pytest.mark.parametrize("kind", KINDS)
def test_face_values_range(lib, kind):  # noqa: F811
    """As at ordinary scales: each value within 2e-14 of its stencil's scale."""
    rng = np.random.default_rng(7)
    out = np.zeros(2)
    for scale in 10.0 ** np.arange(10, 33, 0.5):
        for _ in range(20):
            v = np.ascontiguousarray(_stencil(rng, kind, scale))
            lib.host_weno_LR(v.ctypes.data_as(D), out.ctypes.data_as(D))
            tol = 2e-14 * np.abs(v).max()
            assert abs(out[0] - _weno_core(*v[:5])) <= tol
            assert abs(out[1] - _weno_core(*v[:0:-1])) <= tol


@pytest.mark.parametrize("kind", KINDS)
def test_lf_face_flux_range(lib, kind):  # noqa: F811
    rng = np.random.default_rng(8)
    for k in np.arange(10, 22.6, 0.5):
        for _ in range(20):
            f = _stencil(rng, kind, 10.0 ** k)
            g = _stencil(rng, kind, 10.0 ** rng.uniform(k - 3, min(k + 3, 22.5)))
            p, m = np.ascontiguousarray(f[:5]), np.ascontiguousarray(g[1:])
            got = lib.host_weno_lf(p.ctypes.data_as(D), m.ctypes.data_as(D))
            ref = _weno_core(*p) + _weno_core(*m[::-1])
            assert abs(got - ref) <= 2e-14 * (np.abs(p).max() + np.abs(m).max())


def test_trace_increments_keep_their_precision(lib):  # noqa: F811
    """Stencils of trace mass fluxes (numerical diffusion leaves 1e-80 and less
    ahead of a front): every e_k is eps, so the value is the linear scheme's, and eps^8 under the shared
    reciprocal must not underflow."""
    rng = np.random.default_rng(9)
    w = np.array([2.0, -13.0, 47.0, 27.0, -3.0]) / 60.0
    for scale in 10.0 ** np.arange(-120, -9, 2.0):
        for _ in range(20):
            p, m = scale * rng.uniform(0.5, 1, 5), scale * rng.uniform(0.5, 1, 5)
            got = lib.host_weno_lf(p.ctypes.data_as(D), m.ctypes.data_as(D))
            assert abs(got - (w @ p + w[::-1] @ m)) <= 1e-14 * scale
