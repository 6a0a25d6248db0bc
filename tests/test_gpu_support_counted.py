"""Neighbour lists by the counted entry points (cut-off known to the host, the
fill continuing the count) against count and fill called apart, entry for
entry: one set, a subset, two sets, one cut-off and one per particle, and a
fill whose count was of other arguments.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _apart(ps, rc, domain=None):
    """The lists by dcpse_support_count / _fill, the fill after another count."""
    from openfpm_numerics_amd import _lib, ParticleSubset

    ctx, p = _lib.context(ps.device.index or 0), _lib.ptr
    dom = ps if domain is None else domain
    n_dom, per = dom.size_local(), int(rc.numel() > 1)
    sub = isinstance(domain, ParticleSubset)
    sets = (ps.dims, p(ps.pos_soa), ps.size_local(), None if domain is None else p(dom.pos_soa),
            *((p(dom.ids),) if sub else ()), n_dom, p(rc), per, ps.box_lo.ctypes.data, ps.box_hi.ctypes.data,
            ps.periodic_mask)
    rp, nnz = torch.empty(n_dom + 1, dtype=torch.int64, device=ps.device), np.zeros(1, np.int64)
    ctx.call("dcpse_support_count" + "_subset" * sub, *sets, p(rp), nnz.ctypes.data)
    ps.getVerlet(0.3)
    col = torch.empty(max(int(nnz[0]), 1), dtype=torch.int32, device=ps.device)
    ctx.call("dcpse_support_fill" + "_subset" * sub, *sets, p(rp), p(col))
    return rp, col[: int(nnz[0])]


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("kind", ["scalar", "numpy", "tensor", "per_particle"])
@pytest.mark.parametrize("domain", ["same", "subset", "two_sets"])
def test_counted_lists(cuda, dim, kind, domain):
    from openfpm_numerics_amd import ParticleSet, ParticleSubset, VerletList

    rng = np.random.default_rng(dim)
    n = 1500
    ps = ParticleSet(rng.random((n, dim)), [0.0] * dim, [1.0] * dim, bc=[1] * dim, device=cuda)
    dom = {"same": None, "subset": ParticleSubset(ps, np.arange(3, n, 7)),
           "two_sets": ParticleSet(rng.random((333, dim)), [0.0] * dim, [1.0] * dim, bc=[1] * dim, device=cuda)}[domain]
    n_dom = n if dom is None else dom.size_local()
    r = 0.08 if dim == 2 else 0.15
    rcut = {"scalar": r, "numpy": np.float64(r), "tensor": torch.tensor([r], dtype=torch.float64, device=cuda),
            "per_particle": torch.as_tensor(rng.uniform(0.5 * r, r, n_dom), device=cuda)}[kind]
    rc = torch.as_tensor(rcut, dtype=torch.float64, device=cuda).reshape(-1)
    rp, col = _apart(ps, rc, dom)
    vl = VerletList.build(ps, rcut, domain=dom)
    assert vl.nnz > 0 and torch.equal(vl.row_ptr, rp) and torch.equal(vl.col, col)
    assert torch.equal(vl.rcut, rc)


def test_fill_of_another_count(cuda):
    """A counted fill whose last count had another cut-off reads its own."""
    from openfpm_numerics_amd import ParticleSet, _lib

    rng = np.random.default_rng(9)
    n, p = 900, _lib.ptr
    ps = ParticleSet(rng.random((n, 2)), [0.0, 0.0], [1.0, 1.0], bc=[1, 1], device=cuda)
    ctx = _lib.context(cuda.index or 0)
    rc = [torch.tensor([r], dtype=torch.float64, device=cuda) for r in (0.05, 0.2)]
    rp = [torch.empty(n + 1, dtype=torch.int64, device=cuda) for _ in rc]
    nnz = np.zeros(2, np.int64)
    box = (ps.box_lo.ctypes.data, ps.box_hi.ctypes.data, ps.periodic_mask)
    for i, r in enumerate((0.05, 0.2)):
        ctx.call("dcpse_support_count_one", 2, p(ps.pos_soa), n, None, None, n, p(rc[i]), r, *box, p(rp[i]),
                 nnz[i:].ctypes.data)
    col = torch.empty(int(nnz[0]), dtype=torch.int32, device=cuda)
    ctx.call("dcpse_support_fill_counted", 2, p(ps.pos_soa), n, None, None, n, p(rc[0]), 0, *box, p(rp[0]), p(col))
    want = ps.getVerlet(0.05)
    assert torch.equal(want.row_ptr, rp[0]) and torch.equal(want.col, col)
