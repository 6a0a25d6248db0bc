"""Neighbour lists of few particles in large boxes, a cut-off per particle:
against brute force."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _brute(pos, rc, lo, hi, bc):
    d = pos[:, None] - pos[None]
    for k in range(pos.shape[1]):
        if bc[k]:
            d[..., k] -= (hi[k] - lo[k]) * np.round(d[..., k] / (hi[k] - lo[k]))
    near = (d ** 2).sum(2) < (rc ** 2)[:, None]
    np.fill_diagonal(near, False)
    return np.concatenate([[0], np.cumsum(near.sum(1))]), np.nonzero(near)[1]


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("across", [2.5, 2.96, 2.999, 3.0, 3.4])
def test_narrow_periodic_strip(cuda, dim, across):
    """Periodic across, 2.5 and more of the largest cut-off; long and nearly
    empty along the rest, so that the cells are coarsened to one per cut-off."""
    from openfpm_numerics_amd import ParticleSet

    rng = np.random.default_rng(int(across * 1000) + dim)
    n, hi = 300, [1.0] + ([30.0] if dim == 3 else []) + [3000.0]
    pos = rng.random((n, dim)) * hi
    pos[n // 2:] = pos[:n - n // 2] + rng.uniform(-0.2, 0.2, (n - n // 2, dim))  # pairs within reach
    pos[:, 1:] = np.clip(pos[:, 1:], 0.0, hi[1:])
    pos[:, 0] %= 1.0
    bc = [1] + [0] * (dim - 1)
    rc = rng.uniform(0.5, 1.0, n) / across
    rc[0] = 1.0 / across
    ps = ParticleSet(pos, [0.0] * dim, hi, bc=bc, device=cuda)
    vl = ps.getVerlet(torch.as_tensor(rc, device=cuda))
    rp, col = _brute(pos, rc, [0.0] * dim, hi, bc)
    assert len(col) > n // 4
    assert np.array_equal(vl.row_ptr.cpu().numpy(), rp) and np.array_equal(vl.col.cpu().numpy(), col)
