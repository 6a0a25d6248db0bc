"""Batches on a domain that is the leading part of its support set: f_self is f
itself, and columns reach past the domain's rows. Bit for bit the single-field
applies, which are checked against FP64 numpy."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("nb", [2, 3, 4, 13, 16])
def test_leading_domain(cuda, nb, dtype):
    from openfpm_numerics_amd import _lib

    rng = np.random.default_rng(nb)
    n, n_sup = 700, 5000
    lens = rng.integers(0, 70, n)
    rows = np.repeat(np.arange(n), lens)
    rp = np.concatenate([[0], np.cumsum(lens)])
    nnz = int(rp[-1])
    c = rng.integers(0, n_sup, nnz)
    w, x = rng.standard_normal(nnz), rng.standard_normal((nb, n_sup))
    if dtype == torch.float32:
        w, x = w.astype(np.float32).astype(np.float64), x.astype(np.float32).astype(np.float64)
    rpd, cd = torch.as_tensor(rp, device=cuda), torch.as_tensor(c, dtype=torch.int32, device=cuda)
    W, f = torch.as_tensor(w, dtype=dtype, device=cuda), torch.as_tensor(x, dtype=dtype, device=cuda)
    ctx, p = _lib.context(cuda.index or 0), _lib.ptr
    name = "dcpse_apply_f32" if dtype == torch.float32 else "dcpse_apply_f64"

    def run(k, src, dst):
        ctx.call(name, n, p(rpd), p(cd), 1, _lib.ptr_array([W]), p(src), n_sup, k, p(src), n_sup,
                 _lib.ptr_array([dst]), n, 1.0, 0.0)

    want, got = (torch.zeros((nb, n), dtype=dtype, device=cuda) for _ in range(2))
    for b in range(nb):
        run(1, f[b], want[b])
    run(nb, f, got)
    assert torch.equal(got, want)
    # each sum: at most 70 products rounded in FP64, and once to the result type
    tiny = 72 * 2.0 ** -53 + (2.0 ** -24 if dtype == torch.float32 else 0.0)
    for b in range(nb):
        terms = w * (x[b, c] - x[b, rows])
        ref = np.bincount(rows, terms, minlength=n)
        size = np.bincount(rows, np.abs(w) * (np.abs(x[b, c]) + np.abs(x[b, rows])), minlength=n)
        assert (np.abs(got[b].double().cpu().numpy() - ref) <= tiny * size).all()
