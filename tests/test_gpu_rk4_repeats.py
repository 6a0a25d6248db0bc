"""FP64 time integration on "auto": equal calls give equal bits whatever ran on
the operator before, and every call that is answered eagerly is answered under
graph capture too."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _operator(cuda, n=30, order=None):
    from openfpm_numerics_amd import Laplacian, ParticleSet

    rng = np.random.default_rng(n)
    g = (np.arange(n) + 0.5) / n
    pos = np.stack(np.meshgrid(g, g, indexing="ij"), -1).reshape(-1, 2)
    pos = np.mod(pos + rng.uniform(-0.1 / n, 0.1 / n, pos.shape), 1.0)
    if order is not None:
        pos = pos[order]
    ps = ParticleSet(pos, [0.0] * 2, [1.0] * 2, bc=[1, 1], device=cuda)
    return Laplacian(ps, ps.getVerlet(3.1 / n), 2, 3.1 / n), torch.as_tensor(rng.standard_normal(n * n), device=cuda)


@pytest.fixture
def small(monkeypatch):
    """The thresholds of lists of millions brought down to this test's."""
    from openfpm_numerics_amd import ode

    monkeypatch.setitem(ode.CSR_MAX, torch.float64, 0)
    return ode


def test_equal_calls_equal_bits(cuda, small):
    lap, f = _operator(cuda)
    first = {steps: small.rk4(lap, f.clone(), 1e-6, steps) for steps in (1, 9, 10, 20)}
    one = torch.empty_like(f)
    small.stage(lap, f, 1.0, f, 0.5, one, None, 0.0, None)
    for use in (lambda: None, lambda: lap(f), lambda: small.rk4(lap, f.clone(), 1e-6, 100)):
        use()
        for steps, want in first.items():
            assert torch.equal(small.rk4(lap, f.clone(), 1e-6, steps), want), steps
        again = torch.empty_like(f)
        small.stage(lap, f, 1.0, f, 0.5, again, None, 0.0, None)
        assert torch.equal(again, one)


def test_single_stages_of_large_lists(cuda, small, monkeypatch):
    """On the copy from the first stage on, unless copies are deferred."""
    from openfpm_numerics_amd import dcpse

    monkeypatch.setattr(small, "SELL64_LARGE", 0)
    lap, f = _operator(cuda)
    outs = [torch.empty_like(f) for _ in range(3)]
    small.stage(lap, f, 1.0, f, 0.5, outs[0], None, 0.0, None)
    assert lap.dcpse._W.get("bundle16_64") is not None
    small.stage(lap, f, 1.0, f, 0.5, outs[1], None, 0.0, None)
    small.stage(lap, f, 1.0, f, 0.5, outs[2], None, 0.0, None, layout="bundle16")
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    monkeypatch.setattr(dcpse, "SELL_AFTER", 1000)
    lap, f = _operator(cuda)
    small.stage(lap, f, 1.0, f, 0.5, outs[0], None, 0.0, None)
    assert lap.dcpse._W.get("bundle16_64") is None


def test_deferred_copies(cuda, small, monkeypatch):
    from openfpm_numerics_amd import dcpse

    monkeypatch.setattr(dcpse, "SELL_AFTER", 1000)
    lap, f = _operator(cuda)
    small.rk4(lap, f.clone(), 1e-6, 20)
    assert lap.dcpse._W.get("bundle16_64") is None


@pytest.mark.parametrize("layout", ["auto", "bundle16", "sell"])
@pytest.mark.parametrize("warm", [0, 1, 20])
def test_captured_calls(cuda, small, layout, warm):
    """Steps before the capture as given; 20 captured, more than build the copy."""
    lap, f0 = _operator(cuda)
    if warm:
        small.rk4(lap, f0.clone(), 1e-6, warm)
    f, work = f0.clone(), torch.empty(3 * f0.numel(), dtype=torch.float64, device=cuda)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        small.rk4(lap, f, 1e-6, 20, layout=layout, work=work)
    want = small.rk4(lap, f0.clone(), 1e-6, 20)
    # 80 stages, each rounding sums of 60 products of any order in FP64
    tol = 80 * 64 * 2.0 ** -53 * float(want.abs().max())
    for _ in range(3):
        f.copy_(f0)
        graph.replay()
        torch.cuda.synchronize()
        assert float((f - want).abs().max()) <= tol
