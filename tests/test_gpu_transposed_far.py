"""The FP32 transposed apply on the 16-bit bundle with neighbours beyond 16-bit
offsets: equal to the transposed CSR kernel up to the order of summation."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_transposed_bundle16_with_far_neighbours(cuda, monkeypatch):
    from openfpm_numerics_amd import Laplacian, ParticleSet, dcpse, workloads as W

    w = W.jittered_2d(300, seed=4)
    n = w["pos"].shape[0]
    order = np.concatenate([np.arange(n // 2), n // 2 + np.random.default_rng(6).permutation(n - n // 2)])
    ps = ParticleSet(w["pos"][order], w["box_lo"], w["box_hi"], bc=[1, 1], device=cuda)
    vl = ps.getVerlet(w["rcut"])
    d = Laplacian(ps, vl, 2, w["rcut"]).dcpse
    assert vl.far16()[1] > 0
    monkeypatch.setattr(dcpse, "BUNDLE16_MAX_EXC", 1.0)
    g = torch.as_tensor(np.random.default_rng(1).standard_normal(n), dtype=torch.float32, device=cuda)
    got = d.applyTranspose(g)
    assert d._T.get("bundle16") is not None
    want = d.applyTranspose(g.double())
    # FP32 weights and one rounding of the result, the sums in FP64
    scale = torch.zeros(n, dtype=torch.float64, device=cuda)
    rows = torch.repeat_interleave(torch.arange(n, device=cuda), vl.row_lengths())
    Wabs = d.weights(torch.float64).abs()
    scale.index_add_(0, vl.col.long(), Wabs * g.double().abs()[rows]).index_add_(0, rows, Wabs * g.double().abs()[rows])
    assert bool(((got.double() - want).abs() <= 4 * 2.0 ** -24 * scale).all())
