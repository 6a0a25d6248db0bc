"""Batched FP32 applies on rows of every length: the particle-major kernels
against one single-field pass per field, bit for bit (they sum in its order).
The patterns are made here: empty rows, rows of one to a few hundred
nonzeros (whole chunks, remainders, the strided tail), sets smaller than a
wavefront's rows and arrays shorter than one vector load.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = {
    "one_nonzero": [1],
    "three_nonzeros": [1, 0, 2],
    "all_empty_but_last": [0] * 20 + [3],
    "every_length": list(range(0, 75)),
    "around_chunks": [3, 4, 5, 31, 32, 33, 63, 64, 65, 127, 128, 129] * 3,
    "long_rows": [300, 1, 0, 200, 64, 1000, 7],
    "alike_2d": [28, 29, 30, 29, 28, 27, 32, 29] * 40 + [5],
    "last_row_empty": [17] * 33 + [0],
}


@pytest.mark.parametrize("nb", [4, 8, 16, 21])
@pytest.mark.parametrize("name", list(ROWS))
def test_batch_equals_single_fields(cuda, name, nb):
    from openfpm_numerics_amd import _lib

    rng = np.random.default_rng(nb)
    lens = np.array(ROWS[name])
    n = len(lens)
    rp = torch.as_tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int64, device=cuda)
    nnz = int(lens.sum())
    col = torch.as_tensor(rng.integers(0, n, nnz), dtype=torch.int32, device=cuda)
    W = torch.as_tensor(rng.standard_normal(nnz), dtype=torch.float32, device=cuda)
    diag = torch.as_tensor(rng.standard_normal(n), dtype=torch.float32, device=cuda)
    f = torch.as_tensor(rng.standard_normal((nb, n)), dtype=torch.float32, device=cuda)
    ctx = _lib.context(cuda.index or 0)
    p = _lib.ptr

    def forward(x, k, out):
        ctx.call("dcpse_apply_f32", n, p(rp), p(col), 1, _lib.ptr_array([W]), p(x), n, k, None, n,
                 _lib.ptr_array([out]), n, 1.5, 0.25)

    def transposed(x, k, out):
        ctx.call("dcpse_apply_transpose_f32", n, p(rp), p(col), p(W), p(diag), p(x), n, k, p(out), n, 1.5, 0.25)

    for apply in (forward, transposed):
        got = torch.ones((nb, n), dtype=torch.float32, device=cuda)
        apply(f, nb, got)
        for b in range(nb):
            want = torch.ones(n, dtype=torch.float32, device=cuda)
            apply(f[b].contiguous(), 1, want)
            assert torch.equal(got[b], want), (name, apply.__name__, b)
