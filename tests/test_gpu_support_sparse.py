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


def test_memory_of_a_nearly_empty_box(cuda):
    """500 cut-offs a side: no more memory than the cells of a search without
    groups (6.7e7 of 12 bytes, and as much again for a workspace that doubled)."""
    from openfpm_numerics_amd import _lib

    n, side = 2000, 500.0
    rng = np.random.default_rng(0)
    pos = rng.uniform(240.0, 246.0, (n, 3))
    rc = rng.uniform(0.9, 1.0, n)
    rc[0] = 1.0
    soa = torch.as_tensor(pos.T.copy(), device=cuda)
    rcd = torch.as_tensor(rc, device=cuda)
    lo, hi = np.zeros(3), np.full(3, side)
    rp = torch.empty(n + 1, dtype=torch.int64, device=cuda)
    nnz = np.zeros(1, np.int64)
    ctx, p = _lib.Context(cuda.index or 0), _lib.ptr
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    args = (3, p(soa), n, None)
    ctx.call("dcpse_support_count", *args, n, p(rcd), 1, p(lo), p(hi), 0, p(rp), p(nnz))
    assert free - torch.cuda.mem_get_info()[0] < 2 * 12 * 6.7e7 + 64e6
    col = torch.empty(int(nnz[0]), dtype=torch.int32, device=cuda)
    ctx.call("dcpse_support_fill_counted", *args, None, n, p(rcd), 1, p(lo), p(hi), 0, p(rp), p(col))
    want = _brute(pos, rc, lo, hi, [0, 0, 0])
    assert np.array_equal(rp.cpu().numpy(), want[0]) and np.array_equal(col.cpu().numpy(), want[1])


def test_large_lists_are_given_back(cuda):
    """The candidate lists of 30M particles with a cut-off each (650 bytes per
    particle, more than a sixteenth of the memory) go with the fill; those of a
    small set stay for the next count, and both searches repeat."""
    from openfpm_numerics_amd import _lib

    ctx, p = _lib.Context(cuda.index or 0), _lib.ptr
    lo, hi = np.zeros(3), np.ones(3)
    kept = []
    for n in (30_000_000, 100_000):
        gen = torch.Generator("cuda").manual_seed(n)
        soa = torch.rand((3, n), generator=gen, dtype=torch.float64, device=cuda)
        h = (1.0 / n) ** (1 / 3)
        rc = h * (1.0 + 0.2 * torch.rand(n, generator=gen, dtype=torch.float64, device=cuda))
        rp = torch.empty(n + 1, dtype=torch.int64, device=cuda)
        nnz = np.zeros(1, np.int64)
        args = (3, p(soa), n, None)
        box = (p(lo), p(hi), 7, p(rp))
        ctx.call("dcpse_support_count", *args, n, p(rc), 1, *box, p(nnz))
        cols = [torch.full((int(nnz[0]),), -1, dtype=torch.int32, device=cuda) for _ in range(2)]
        torch.cuda.synchronize()
        held = torch.cuda.mem_get_info()[0]
        ctx.call("dcpse_support_fill_counted", *args, None, n, p(rc), 1, *box, p(cols[0]))
        kept.append(torch.cuda.mem_get_info()[0] - held)
        ctx.call("dcpse_support_fill", *args, n, p(rc), 1, *box, p(cols[1]))
        assert torch.equal(*cols)
        del soa, rc, rp, cols
    assert kept[0] > torch.cuda.get_device_properties(cuda).total_memory // 16
    assert kept[1] == 0
