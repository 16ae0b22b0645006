"""The step of a uniform block level on its own grid (blocks read in place)
against the padded path, bit for bit."""
import pytest

from janc_amd import cases
from janc_amd.mechanism import Mechanism

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]

DTYPE = {"fp64": torch.float64, "mixed": torch.float32}


@pytest.mark.parametrize("precision,stride", [("mixed", 195225787), ("fp64", 195225787),
                                              ("mixed", 2 ** 31 + 6)])
def test_plane_stride_of_any_size(precision, stride):
    """A level that is a view into a plane-major buffer: 11 planes are 2^31
    elements apart from the first stride on, one plane from the last."""
    from janc_amd.amr import BlockSolver, UniformBlockGrid
    U, aux, g = cases.detonation_tube(Mechanism(), nx=12, ny=14, driver=3)
    sol = BlockSolver(cases.simulation_config(g, dt=1e-9, precision=precision))
    grid = UniformBlockGrid(g["boundary_config"], 2, 2, 6, 7)
    blk = grid.split(torch.as_tensor(U).to(dtype=DTYPE[precision]).cuda(),
                     torch.as_tensor(aux).to(dtype=DTYPE[precision]).cuda())
    count = 13 * stride + 4 * 42
    if torch.cuda.mem_get_info()[0] < count * blk.element_size() + 2 ** 31:
        pytest.skip("needs %d GB" % (count * blk.element_size() >> 30))
    buf = torch.empty((count,), dtype=blk.dtype, device="cuda")
    far = buf.as_strided(tuple(blk.shape), (42, stride, 7, 1))
    for v in range(14):
        far[:, v].copy_(blk[:, v])
    torch.cuda.synchronize()
    print("level in place", precision, stride, flush=True)
    args = (1, None, g["dx"], g["dy"], 1e-9)
    got = sol.advance_one_step(*args, far, None, amr=grid)
    ref = sol.advance_one_step(*args, blk, None, amr=grid)
    assert torch.isfinite(ref).all() and torch.equal(got, ref)
    del far, buf
    torch.cuda.empty_cache()


@pytest.mark.parametrize("name,where", [("get_ghost_block_data", "object"),
                                        ("update_external_boundary", "object"),
                                        ("get_ghost_block_data", "class"),
                                        ("update_external_boundary", "class")])
def test_replaced_ghost_functions_are_asked(name, where, monkeypatch):
    """A caller's own ghost function, put on a UniformBlockGrid or on the
    class, is called for every stage and its result used."""
    from janc_amd.amr import BlockSolver, UniformBlockGrid
    U, aux, g = cases.detonation_tube(Mechanism(), nx=12, ny=14, driver=3)
    sol = BlockSolver(cases.simulation_config(g, dt=1e-9))
    grid = UniformBlockGrid(g["boundary_config"], 2, 2, 6, 7)
    blk = grid.split(torch.as_tensor(U).cuda(), torch.as_tensor(aux).cuda())
    own, calls = getattr(grid, name), []

    def replaced(*args):
        calls.append(name)
        out = own(*args[1:] if where == "class" else args).clone()
        out[:, 2] += 1.0                       # the caller's change of rho v
        return out

    args = (1, None, g["dx"], g["dy"], 1e-9, blk, None)
    plain = sol.advance_one_step(*args, amr=grid)
    monkeypatch.setattr(grid if where == "object" else UniformBlockGrid, name, replaced)
    out = sol.advance_one_step(*args, amr=grid)
    assert calls == [name] * 3
    assert not torch.equal(out, plain)


# left, right, bottom, top: both momenta flipped on one ghost, copies across the
# domain with the off-by-one pre-pad, each alone and against a wall
KINDS = [("no_slip_wall", "no_slip_wall", "no_slip_wall", "no_slip_wall"),
         ("periodic", "periodic", "periodic", "periodic"),
         ("periodic", "periodic", "no_slip_wall", "slip_wall"),
         ("slip_wall", "no_slip_wall", "periodic", "periodic"),
         ("slip_wall", "slip_wall", "slip_wall", "zero_gradient")]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kinds", KINDS)
def test_boundary_kinds(kinds, precision):
    """Every copied ghost kind, with momenta at the edges that a wrong or
    missing flip or source cell would show in; the two steps of the level read
    in place equal the padded path's."""
    from janc_amd.amr import BlockSolver, UniformBlockGrid

    class Padded(UniformBlockGrid):
        pass

    nbx, nby, bnx, bny = 3, 2, 11, 19
    U, aux, g = cases.detonation_tube(Mechanism(), nx=nbx * bnx, ny=nby * bny, driver=8)
    gen = torch.Generator().manual_seed(5)
    U, aux = torch.as_tensor(U).clone(), torch.as_tensor(aux)
    noise = 200.0 * (torch.rand((2,) + tuple(U.shape[1:]), generator=gen,
                                dtype=torch.float64) - 0.4)
    kin = 0.5 * (U[1] ** 2 + U[2] ** 2) / U[0]
    U[1:3] += U[0] * noise
    U[3] += 0.5 * (U[1] ** 2 + U[2] ** 2) / U[0] - kin
    bc = dict(zip(("left_boundary", "right_boundary", "bottom_boundary", "top_boundary"), kinds))
    sol = BlockSolver(cases.simulation_config(dict(g, boundary_config=bc), dt=2e-9,
                                              precision=precision))
    out = []
    for cls in (UniformBlockGrid, Padded):
        grid = cls(bc, nbx, nby, bnx, bny)
        blk = grid.split(U.to(DTYPE[precision]).cuda(), aux.to(DTYPE[precision]).cuda())
        for _ in range(2):
            blk = sol.advance_one_step(1, None, g["dx"], g["dy"], 2e-9, blk, None, amr=grid)
        out.append(blk)
    assert torch.isfinite(out[0]).all() and torch.equal(out[0], out[1])
