"""The compact stage kernel (small grids, AMR levels) against the wide one.

A single context runs the compact kernel up to 200000 cells; the batch API
runs the wide 64-column kernel for every case, so a batch of one case is the
same step by the other kernel.  The arithmetic per cell and per face is the
same, so states and time steps are equal bit for bit.  Sizes: both sides of
every line of the rule, thin and square grids, prime sides, the smallest
grid; source-cell halos (tube, periodic channel) and strips (inlet, outlet).
The level step of a uniform block grid is compared with the padded path."""
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


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nbx,nby,bnx,bny", [(3, 2, 21, 37), (4, 4, 20, 20), (2, 3, 40, 50),
                                             (2, 2, 7, 130), (5, 3, 4, 4), (1, 1, 33, 70)])
def test_level_step_equals_padded_path(nbx, nby, bnx, bny, precision):
    from janc_amd.amr import BlockSolver, UniformBlockGrid

    class Padded(UniformBlockGrid):      # another hierarchy object: the general path
        pass

    nx, ny = nbx * bnx, nby * bny
    U, aux, g, _ = _case(Mechanism(), "tube", nx, ny)
    sol = BlockSolver(cases.simulation_config(g, dt=1e-9, precision=precision))
    dt = torch.float64 if precision == "fp64" else torch.float32
    out = []
    for cls in (UniformBlockGrid, Padded):
        grid = cls(g["boundary_config"], nbx, nby, bnx, bny)
        blk = grid.split(torch.as_tensor(U).to(dtype=dt).cuda(),
                         torch.as_tensor(aux).to(dtype=dt).cuda())
        if cls is UniformBlockGrid and bnx == 21:    # interiors read through strides
            pad = torch.full((blk.shape[0], 14, bnx + 2, bny + 4), float("nan"),
                             dtype=dt, device="cuda")
            pad[:, :, 1:-1, 2:-2] = blk
            blk = pad[:, :, 1:-1, 2:-2]
        for _ in range(2):
            blk = sol.advance_one_step(1, None, g["dx"], g["dy"], 1e-9, blk, None, amr=grid)
        out.append(blk)
    assert torch.isfinite(out[0]).all() and torch.equal(out[0], out[1])
    assert sol.health() == 0
