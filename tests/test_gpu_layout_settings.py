"""The choice between 16-bit and 32-bit columns of a list follows the limits in
force at the call, whatever was chosen before."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _operators(cuda, n=260):
    """A set half of whose particles lie shuffled in memory: many far neighbours."""
    from openfpm_numerics_amd import Derivative_x, Laplacian, ParticleSet

    rng = np.random.default_rng(1)
    g = (np.arange(n) + 0.5) / n
    pos = np.stack(np.meshgrid(g, g, indexing="ij"), -1).reshape(-1, 2)
    pos = np.mod(pos + rng.uniform(-0.1 / n, 0.1 / n, pos.shape), 1.0)
    some = rng.permutation(n * n)[: n * n // 2]
    pos[np.sort(some)] = pos[some]
    ps = ParticleSet(pos, [0.0] * 2, [1.0] * 2, bc=[1, 1], device=cuda)
    vl = ps.getVerlet(3.1 / n)
    return vl, [K(ps, vl, 2, 3.1 / n) for K in (Laplacian, Derivative_x)], n * n, rng


def test_the_share_of_far_neighbours_is_asked_each_time(cuda):
    vl, _, _, _ = _operators(cuda)
    assert vl.col16(0.0) is None  # counted, refused
    far = vl.col16(1.0)[-1]
    assert far > 0
    assert vl.col16(0.5 * far / vl.nnz) is None
    assert vl.col16(1.0) is not None


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_settings_in_force(cuda, dtype, monkeypatch):
    from openfpm_numerics_amd import dcpse, fused

    vl, ops, n, rng = _operators(cuda)
    f = torch.as_tensor(rng.standard_normal(n), dtype=dtype, device=cuda)
    runs = []
    for least, share in ((10 ** 9, 1.0), (0, 1.0), (0, 0.0), (0, 1.0), (10 ** 9, 1.0)):
        monkeypatch.setattr(dcpse, "COL16_MIN", least)
        monkeypatch.setattr(dcpse, "BUNDLE16_MAX_EXC", share)
        used = [fused(*ops, f=f), fused(*ops, f=f)]
        key = (f.dtype, ops[1].dcpse._gen)
        name = ops[0].dcpse._plans[key].name
        assert ("col16" in name) == (least == 0 and share == 1.0)
        # a list that has seen no other setting
        fresh = _operators(cuda)[1]
        for got in used:
            for a, b in zip(got, fused(*fresh, f=f)):
                assert torch.equal(a, b)
        runs.append(used[0])
    for a, b in zip(runs[0], runs[4]):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_small_lists_do_not_depend_on_earlier_calls(cuda, dtype):
    """Several operators of a list below COL16_MIN, before and after another call
    has built the list's 16-bit columns."""
    from openfpm_numerics_amd import fused

    vl, ops, n, rng = _operators(cuda)
    f = torch.as_tensor(rng.standard_normal(n), dtype=dtype, device=cuda)
    want = fused(*ops, f=f)
    vl2, ops2, _, _ = _operators(cuda)
    assert vl2.col16(1.0)[-1] > 0
    for a, b in zip(fused(*ops2, f=f), want):
        assert torch.equal(a, b)
