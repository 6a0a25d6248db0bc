"""Prepared applies of several operators: the weights of the others are not held
by the first one's plans."""
import weakref

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_other_operators_weights_are_released(cuda, dtype):
    from openfpm_numerics_amd import Derivative_x, Laplacian, ParticleSet, fused

    n = 40
    rng = np.random.default_rng(0)
    g = (np.arange(n) + 0.5) / n
    pos = np.stack(np.meshgrid(g, g, indexing="ij"), -1).reshape(-1, 2)
    pos = np.mod(pos + rng.uniform(-0.1 / n, 0.1 / n, pos.shape), 1.0)
    ps = ParticleSet(pos, [0.0] * 2, [1.0] * 2, bc=[1, 1], device=cuda)
    vl = ps.getVerlet(3.1 / n)
    lap, dx = (K(ps, vl, 2, 3.1 / n) for K in (Laplacian, Derivative_x))
    f = torch.as_tensor(rng.standard_normal(n * n), dtype=dtype, device=cuda)
    key = "sell" if dtype == torch.float32 else "sell64"
    want = fused(lap, dx, f=f)
    for again in range(3):  # assembled again: new weights, the old ones go
        weights = weakref.ref(dx.dcpse._W[key])
        assert weights() is not None
        dx.update(ps)
        assert weights() is None
        for _ in range(2):
            for a, b in zip(fused(lap, dx, f=f), want):
                assert torch.equal(a, b)
    weights = weakref.ref(dx.dcpse._W[key])
    del dx
    assert weights() is None
    # copies taken out of an operator: the plan that used them is made anew
    dx = Derivative_x(ps, vl, 2, 3.1 / n)
    fused(lap, dx, f=f)
    del dx.dcpse._W[key]
    for a, b in zip(fused(lap, dx, f=f), want):
        assert torch.equal(a, b)
