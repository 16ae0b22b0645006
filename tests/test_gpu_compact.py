"""The compact stage kernel (small grids) against the wide one.

A single context runs the compact kernel up to 200000 cells; the batch API
runs the wide 64-column kernel for every case, so a batch of one case is the
same step by the other kernel.  The arithmetic per cell and per face is the
same, so states and time steps are equal bit for bit.  Sizes: both sides of
every line of the rule, thin and square grids, prime sides, the smallest
grid; source-cell halos (tube, periodic channel) and strips (inlet, outlet)."""
import pytest

from janc_amd import cases
from janc_amd.mechanism import Mechanism

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]

SIZES = [("tube", 4, 4), ("tube", 4, 3001), ("tube", 2999, 5), ("box", 61, 67),
         ("tube", 128, 112), ("box", 128, 113), ("annulus", 150, 101), ("tube", 250, 200),
         ("annulus", 251, 200), ("tube", 400, 500), ("tube", 401, 500)]


def _case(mech, kind, nx, ny):
    if kind == "tube":
        return cases.detonation_tube(mech, nx=nx, ny=ny, driver=max(1, nx // 8)) + (None,)
    if kind == "box":
        return cases.periodic_box(mech, nx=nx, ny=ny) + (None,)
    return cases.rdc_annulus(mech, nx=nx, ny=ny, seed_cols=nx // 5)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kind,nx,ny", SIZES)
def test_compact_equals_wide(kind, nx, ny, precision):
    from janc_amd.batch import BatchSimulator
    from janc_amd.solver import Simulator
    U, aux, g, theta = _case(Mechanism(), kind, nx, ny)
    cfg = cases.simulation_config(g, cfl=0.3, precision=precision, theta=theta)
    dt = torch.float64 if precision == "fp64" else torch.float32
    U = torch.as_tensor(U).to(dtype=dt).cuda()
    aux = torch.as_tensor(aux).to(dtype=dt).cuda()
    Us, As = U.clone(), aux.clone()
    _, _, hist = Simulator(cfg).advance(Us, As, 3)
    b = BatchSimulator([cfg], [U], [aux])
    hb = b.advance(3, graph=False, dt_hist=True)
    torch.cuda.synchronize()
    assert torch.isfinite(Us).all()
    assert torch.equal(U, Us) and torch.equal(aux, As) and torch.equal(hb[0], hist)
