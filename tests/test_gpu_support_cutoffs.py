"""Fills with a cut-off per particle after a count of other cut-offs with the
same extremes, and after cut-offs that changed in place."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


class Lists:
    """Count and fill of one 3D set through the C entry points."""

    def __init__(self, cuda, n=2500):
        from openfpm_numerics_amd import ParticleSet, _lib

        rng = np.random.default_rng(4)
        self.ps = ParticleSet(rng.random((n, 3)), [0.0] * 3, [1.0] * 3, bc=[1] * 3, device=cuda)
        self.ctx, self.p, self.n = _lib.context(cuda.index or 0), _lib.ptr, n
        r = rng.uniform(0.08, 0.16, n)
        # the same values at other particles
        self.rc = [torch.as_tensor(v, device=cuda) for v in (r, rng.permutation(r))]
        self.box = (self.ps.box_lo.ctypes.data, self.ps.box_hi.ctypes.data, self.ps.periodic_mask)

    def count(self, rc):
        rp, nnz = torch.empty(self.n + 1, dtype=torch.int64, device=rc.device), np.zeros(1, np.int64)
        self.ctx.call("dcpse_support_count", 3, self.p(self.ps.pos_soa), self.n, None, self.n, self.p(rc), 1, *self.box,
                      self.p(rp), nnz.ctypes.data)
        return rp, torch.empty(int(nnz[0]), dtype=torch.int32, device=rc.device)

    def fill(self, rc, rp, col, counted):
        name, ids = ("dcpse_support_fill_counted", (None,)) if counted else ("dcpse_support_fill", ())
        self.ctx.call(name, 3, self.p(self.ps.pos_soa), self.n, None, *ids, self.n, self.p(rc), 1, *self.box, self.p(rp),
                      self.p(col))


@pytest.mark.parametrize("counted", [False, True])
def test_two_counts_then_the_first_fill(cuda, counted):
    lists = Lists(cuda)
    want = [lists.ps.getVerlet(rc) for rc in lists.rc]
    assert not torch.equal(want[0].row_ptr, want[1].row_ptr)
    made = [lists.count(rc) for rc in lists.rc]
    for rc, (rp, col), vl in zip(lists.rc, made, want):
        lists.fill(rc, rp, col, counted)
        assert torch.equal(rp, vl.row_ptr) and torch.equal(col, vl.col)


def test_changed_in_place_is_refused(cuda):
    from openfpm_numerics_amd import _lib

    lists = Lists(cuda)
    rp, col = lists.count(lists.rc[0])
    lists.rc[0].copy_(lists.rc[1])
    with pytest.raises(_lib.DcpseError, match="changed since count"):
        lists.fill(lists.rc[0], rp, col, False)
