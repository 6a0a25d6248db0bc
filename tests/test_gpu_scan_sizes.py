"""The exclusive scan behind row pointers, through the transposed row pointer,
at the edges of its forms: one block, tiles whose blocks add up the sums before
them, and tile sums scanned by a kernel of their own.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 2047, 8191, 8192, 8193, 10_241, 524_289, 2048 * 4096, 2048 * 4096 + 1])
def test_row_pointer_scan(cuda, n):
    from openfpm_numerics_amd import _lib

    gen = torch.Generator(cuda).manual_seed(n)
    nnz = 3 * n + 5
    col = torch.randint(0, n, (nnz,), generator=gen, dtype=torch.int32, device=cuda)
    col[:5] = n - 1
    rp = torch.tensor([0, nnz], dtype=torch.int64, device=cuda)
    got = torch.full((n + 1,), -1, dtype=torch.int64, device=cuda)
    _lib.context(cuda.index or 0).call("dcpse_transpose_count", 1, n, _lib.ptr(rp), _lib.ptr(col), _lib.ptr(got))
    want = torch.zeros(n + 1, dtype=torch.int64, device=cuda)
    want[1:] = torch.cumsum(torch.bincount(col, minlength=n), 0)
    assert torch.equal(got, want)
