"""Cell lists where neighbours in memory share a cell (one atomic per run of
lanes): counts around a wavefront, all particles in one cell, runs of every
length, and no runs, against all pairs in FP64.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_particle", [False, True])
@pytest.mark.parametrize("order", ["runs", "shuffled", "one_cell"])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 129, 1000, 4097])
def test_lists_of_runs(cuda, n, order, per_particle):
    from openfpm_numerics_amd import ParticleSet

    rng = np.random.default_rng(n)
    r = 0.09
    pos = rng.random((n, 2))
    if order == "one_cell":
        pos = 0.5 + 0.02 * (pos - 0.5)
        pos = pos[: min(n, 700)]  # a row holds at most as many neighbours as the library takes
    elif order == "runs":
        q = np.floor(pos / r).astype(int)
        pos = pos[np.lexsort((q[:, 1], q[:, 0]))]
    m = len(pos)
    rc = rng.uniform(0.5 * r, r, m) if per_particle else np.full(m, r)
    ps = ParticleSet(pos, [0.0, 0.0], [1.0, 1.0], bc=[1, 1], device=cuda)
    vl = ps.getVerlet(torch.as_tensor(rc, device=cuda) if per_particle and m > 1 else float(rc[0]))
    d = pos[:, None] - pos[None]
    d -= np.rint(d)
    near = (d ** 2).sum(-1) < (rc ** 2)[:, None]
    np.fill_diagonal(near, False)
    assert np.array_equal(vl.row_ptr.cpu().numpy(), np.concatenate([[0], np.cumsum(near.sum(1))]))
    assert np.array_equal(vl.col.cpu().numpy(), np.nonzero(near)[1])
