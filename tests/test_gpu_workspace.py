"""A workspace that cannot be had is an error of that call alone."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_refused_workspace(cuda):
    from openfpm_numerics_amd import _lib

    ctx, p = _lib.Context(cuda.index or 0), _lib.ptr
    n, nb = 3000, 16
    rng = np.random.default_rng(0)
    lens = rng.integers(0, 40, n)
    rp = torch.as_tensor(np.concatenate([[0], np.cumsum(lens)]), device=cuda)
    col = torch.as_tensor(rng.integers(0, n, int(lens.sum())), dtype=torch.int32, device=cuda)
    W = torch.as_tensor(rng.standard_normal(int(lens.sum())), device=cuda)
    f = torch.as_tensor(rng.standard_normal((nb, n)), device=cuda)
    slice_ptr = torch.zeros(n // 64 + 2, dtype=torch.int64, device=cuda)
    sell_row = torch.zeros(n + 64, dtype=torch.int32, device=cuda)
    slots = C.c_int64()

    def batch():
        out = torch.zeros_like(f)
        ctx.call("dcpse_apply_f64", n, p(rp), p(col), 1, _lib.ptr_array([W]), p(f), n, nb, None, n,
                 _lib.ptr_array([out]), n, 1.0, 0.0)
        return out

    want = batch()
    ctx.call("dcpse_sell_count", n, p(rp), p(slice_ptr), p(sell_row), C.addressof(slots))
    first = slots.value
    # 2^48 bytes of workspace: refused by the allocator before any launch
    with pytest.raises(_lib.DcpseError, match="workspace"):
        ctx.call("dcpse_sell_count", 1 << 52, p(rp), p(slice_ptr), p(sell_row), C.addressof(slots))
    ctx.call("dcpse_sell_count", n, p(rp), p(slice_ptr), p(sell_row), C.addressof(slots))
    assert slots.value == first
    assert torch.equal(batch(), want)
