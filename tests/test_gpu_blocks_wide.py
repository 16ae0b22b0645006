"""Padded AMR blocks by the wide and by the compact stage body, bit for bit.

Many blocks whose rows fill 64 columns run the wide body, few of them the
compact one, so the same blocks handed in together and a few at a time are the
same stage by both kernels; sizes with ragged rows and columns of the 8 x 64
tile, and one that is compact either way."""
import pytest

from janc_amd import cases
from janc_amd.mechanism import Mechanism

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,bnx,bny", [(64, 64, 64), (512, 8, 60), (128, 16, 125), (86, 23, 128),
                                       (64, 62, 61), (64, 20, 20)])
def test_wide_equals_compact(n, bnx, bny, precision):
    from janc_amd.amr import BlockSolver, UniformBlockGrid
    U, aux, g = cases.detonation_tube(Mechanism(), nx=n * bnx, ny=bny, driver=n * bnx // 3)
    dt = torch.float64 if precision == "fp64" else torch.float32
    gen = torch.Generator().manual_seed(3)
    U = torch.as_tensor(U).clone()
    U[1:3] += 30.0 * U[0] * torch.randn((2,) + tuple(U.shape[1:]), generator=gen,
                                        dtype=torch.float64)
    grid = UniformBlockGrid(g["boundary_config"], n, 1, bnx, bny)
    pad = grid.get_ghost_block_data(grid.split(U.to(dtype=dt).cuda(),
                                               torch.as_tensor(aux).to(dtype=dt).cuda()))
    mid = pad.clone()
    mid[:, 3] *= 1.01                               # another state than U^n
    sol = BlockSolver(cases.simulation_config(g, dt=1e-9, precision=precision))
    args = (g["dx"], g["dy"], 1e-9)
    few = range(0, n, 7)
    for s in range(3):
        out = sol.stage(s, mid, pad, *args)
        assert torch.isfinite(out).all()
        for i in few:
            assert torch.equal(sol.stage(s, mid[i:i + 3], pad[i:i + 3], *args), out[i:i + 3])
    rhs = sol.flux_func(mid, *args)
    for i in few:
        assert torch.equal(sol.flux_func(mid[i:i + 3], *args), rhs[i:i + 3])
    assert sol.health() == 0
