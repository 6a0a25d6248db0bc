"""The launch shape of an apply follows from its list, not from a list that lay
at the same address before: same bits as in a context that has seen no other."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_lists_at_one_address(cuda, dtype):
    from openfpm_numerics_amd import _lib

    p, n, most = _lib.ptr, 4000, 120
    t = "f32" if dtype == torch.float32 else "f64"
    rng = np.random.default_rng(2)
    rp = torch.zeros(n + 1, dtype=torch.int64, device=cuda)
    col = torch.as_tensor(rng.integers(0, n, n * most), dtype=torch.int32, device=cuda)
    W, f = (torch.as_tensor(rng.standard_normal(s), dtype=dtype, device=cuda) for s in (n * most, (5, n)))
    used = _lib.Context(cuda.index or 0)

    def run(ctx, nb, nnz):
        out = torch.zeros_like(f)
        scratch = torch.empty(8 * n, dtype=dtype, device=cuda)
        ctx.call(f"dcpse_apply_nnz_{t}", n, nnz, p(rp), p(col), 1, _lib.ptr_array([W]), p(f), n, nb, None, n,
                 _lib.ptr_array([out]), n, 1.0, 0.0, p(scratch), scratch.numel() * scratch.element_size())
        return out

    for mean in (20, 50, 100, 20):  # 4, 8 and 12 nonzeros per lane
        lens = rng.integers(mean - 15, mean + 16, n)
        rp.copy_(torch.as_tensor(np.concatenate([[0], np.cumsum(lens)])))
        for nb in (1, 5):
            assert torch.equal(run(used, nb, int(lens.sum())), run(_lib.Context(cuda.index or 0), nb, int(lens.sum())))
