"""Which stage kernel a context runs: the compact one on small grids by
default, the chosen variant of the wide one after set_tile.  Every variant
gives the default kernel's states and time steps bit for bit, on a small grid
and on one past the compact kernel's range, with strips (inlet, outlet) and
with source-cell halos (wall kinds, periodic)."""
import pytest

from janc_amd import cases
from janc_amd.autotune import variants
from janc_amd.mechanism import Mechanism
from janc_amd.solver import Simulator

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]

SIDES = ("left_boundary", "right_boundary", "bottom_boundary", "top_boundary")
CHANNEL = dict(zip(SIDES, ("periodic", "periodic", "no_slip_wall", "slip_wall")))


def _case(kind, nx, ny):
    mech = Mechanism()
    if kind == "annulus":
        return cases.rdc_annulus(mech, nx=nx, ny=ny, seed_cols=nx // 5)
    U, aux, g = cases.detonation_tube(mech, nx=nx, ny=ny, driver=nx // 8)
    return U, aux, dict(g, boundary_config=CHANNEL), None


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kind,nx,ny,small", [("annulus", 131, 77, True), ("channel", 131, 77, True),
                                              ("annulus", 459, 467, False),
                                              ("channel", 459, 467, False)])
def test_set_tile_runs_the_variant(kind, nx, ny, small, precision):
    U0, aux0, g, theta = _case(kind, nx, ny)
    dt = torch.float64 if precision == "fp64" else torch.float32
    U0, aux0 = (torch.as_tensor(v).to(dtype=dt).cuda() for v in (U0, aux0))
    sim = Simulator(cases.simulation_config(g, cfl=0.3, precision=precision, theta=theta))
    assert sim.compact(U0, theta) == small
    ref = [U0.clone(), aux0.clone()]
    ref.append(sim.advance(ref[0], ref[1], 3, theta)[2])
    for v in variants():
        sim.set_tile(U0, v["variant"], theta)
        assert not sim.compact(U0, theta) and sim.get_tile(U0, theta) == v["variant"]
        U, aux = U0.clone(), aux0.clone()
        hist = sim.advance(U, aux, 3, theta)[2]
        torch.cuda.synchronize()
        print(kind, nx, ny, precision, "variant", v, flush=True)
        assert torch.isfinite(U).all()
        assert torch.equal(U, ref[0]) and torch.equal(aux, ref[1]) and torch.equal(hist, ref[2])


@pytest.mark.parametrize("nx,ny,small", [(131, 77, True), (459, 467, False)])
def test_autotune_times_variants_where_they_run(nx, ny, small, tmp_path, monkeypatch):
    """A small grid has no variants to time: nothing is stored, in memory or in
    the cache file, and the compact kernel stays."""
    import janc_amd.autotune as at
    path = tmp_path / "tune.json"
    monkeypatch.setenv("JANC_AMD_TUNE_CACHE", str(path))
    monkeypatch.setattr(at, "_MEM", {})
    U, aux, g, _ = _case("channel", nx, ny)
    U, aux = torch.as_tensor(U).cuda(), torch.as_tensor(aux).cuda()
    sim = Simulator(cases.simulation_config(g, cfl=0.3))
    t = sim.autotune(U, aux, steps=1)
    assert at.tunable(sim) and at.tunable(sim, U) != small
    assert sim.compact(U) == small
    assert path.exists() != small and bool(at._MEM) != small
    if small:
        assert t["tuned"] is False and t["variant"] == sim.get_tile(U)
    else:
        assert sorted(int(k) for k in t["ms_per_step"]) == [v["variant"] for v in variants()]


@pytest.mark.parametrize("nx,ny,groups", [(4, 4, 12), (128, 112, 12), (120, 120, 6), (200, 140, 6),
                                          (2000, 14, 6), (280, 100, 2), (200, 150, 2),
                                          (250, 200, 2), (3000, 60, 2), (720, 250, 2),
                                          (740, 250, 0), (400, 500, 0)])
def test_compact_rule_goes_by_tiles(nx, ny, groups):
    """12 and 6 groups only while their tiles are at most one for each of the
    256 CUs, 2 groups up to three; each form equals the wide kernel."""
    mech = Mechanism()
    U0, aux0, g = cases.detonation_tube(mech, nx=nx, ny=ny, driver=max(1, nx // 8))
    for precision, dt in (("fp64", torch.float64), ("mixed", torch.float32)):
        Ui, ai = (torch.as_tensor(v).to(dtype=dt).cuda() for v in (U0, aux0))
        sim = Simulator(cases.simulation_config(g, cfl=0.3, precision=precision))
        ctx = sim._context(Ui, None)
        assert ctx.lib.jh_ctx_compact(ctx.h) == groups
        out = []
        for _ in range(2):
            U, aux = Ui.clone(), ai.clone()
            out.append((U, aux, sim.advance(U, aux, 2)[2]))
            sim.set_tile(Ui, sim.get_tile(Ui))
        assert torch.isfinite(out[0][0]).all()
        assert all(torch.equal(a, b) for a, b in zip(*out))
