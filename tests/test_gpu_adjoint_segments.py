"""Row segments of the adjoint's x pass: 8, 16 or 32 rows by the number of waves
the grid gives (24 per 64 columns and segment, 1024 wanted).  The other adjoint
tests' grids take 8 rows; these take 16 and 32, with a ragged last segment, under
the same bar against the differentiable twin of the oracle."""
import pytest

from janc_amd import cases
from janc_amd.mechanism import Mechanism

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]

from oracle.torch_step import TorchOracle  # noqa: E402
from test_gpu_adjoint import DT, TWIN_TOL, _cotangents, rel_err  # noqa: E402
from test_oracle_adjoint import tie_free_state  # noqa: E402


@pytest.mark.parametrize("nx", [200, 330])
def test_longer_segments_match_twin(mech_path, nx):
    from janc_amd.adjoint import step
    from janc_amd.solver import Simulator
    mech = Mechanism(mech_path)
    U, aux, g = tie_free_state(mech_path, mech, "tube", nx, 200)
    W, Wa = _cotangents(U, aux)
    sim = Simulator(cases.simulation_config(g, mech_path, cfl=0.3, dt=DT))
    x = [torch.tensor(v, device="cuda", requires_grad=True) for v in (U, aux)]
    got = torch.autograd.grad(list(step(sim, x[0], x[1], DT)), x,
                              [torch.tensor(v, device="cuda") for v in (W, Wa)])
    print("device gradient done", nx, flush=True)
    to = TorchOracle(mech_path, g["boundary_config"], g["dx"], g["dy"])
    y = [torch.tensor(v, requires_grad=True) for v in (U, aux)]
    U4, a4 = to.advance_one_step(y[0], y[1], DT)
    ((U4 * torch.tensor(W)).sum() + (a4 * torch.tensor(Wa)).sum()).backward()
    assert rel_err(got[0], y[0].grad).max() <= TWIN_TOL
    assert rel_err(got[1], y[1].grad).max() <= TWIN_TOL
