"""The sliced-ELL layout builds against the same layouts formed by torch from
the CSR arrays: rows of every length up to several tiles of 32 slots, empty
rows, a last slice that is not full, with and without row scales. Equal bit for
bit (the scaled weights are one product each)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = {
    "one": [3],
    "tile_edges": [0, 1, 3, 4, 5, 31, 32, 33, 63, 64, 65, 95, 96, 97, 200] * 5,
    "a_slice": list(range(64)),
    "uneven": list(np.random.default_rng(0).integers(0, 150, 1000)),
    "empty": [0] * 70 + [2],
}


@pytest.mark.parametrize("name", list(ROWS))
def test_fills_match_torch(cuda, name):
    from openfpm_numerics_amd import _lib
    from openfpm_numerics_amd.dcpse import bundle16
    from openfpm_numerics_amd.particles import VerletList, sell_cols, sell_slices, sell_weights

    lens = np.array(ROWS[name])
    n, nnz = len(lens), int(lens.sum())
    rng = np.random.default_rng(1)
    rp = torch.as_tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int64, device=cuda)
    col = torch.as_tensor(rng.integers(0, n, nnz), dtype=torch.int32, device=cuda)
    K = torch.as_tensor(rng.standard_normal(nnz), device=cuda)
    scale = torch.as_tensor(rng.uniform(0.5, 2.0, n), device=cuda)
    slice_ptr, sell_row, n_slots = sell_slices(rp, n)
    # slot of every neighbour
    lane_of = torch.zeros(n, dtype=torch.int64, device=cuda)
    lanes = torch.nonzero(sell_row[: 64 * ((n + 63) // 64)] >= 0).ravel()
    lane_of[sell_row[lanes].long()] = lanes
    row = torch.repeat_interleave(torch.arange(n, device=cuda), rp[1:] - rp[:-1])
    j = torch.arange(nnz, device=cuda) - rp[row]
    lane = lane_of[row]
    slot = slice_ptr[lane // 64] + (j // 4) * 256 + 4 * (lane % 64) + j % 4

    def placed(v):
        out = torch.zeros(max(n_slots, 4), dtype=v.dtype, device=cuda)
        out[slot] = v
        return out

    assert torch.equal(sell_cols(rp, col, n, slice_ptr, sell_row, n_slots)[:n_slots], placed(col)[:n_slots])
    W32 = K.float()
    assert torch.equal(sell_weights(rp, W32, (slice_ptr, sell_row, n_slots), n)[:n_slots], placed(W32)[:n_slots])
    p = _lib.ptr
    ctx = _lib.context(cuda.index or 0)
    got = torch.full((max(n_slots, 4),), 7.0, dtype=torch.float64, device=cuda)
    ctx.call("dcpse_sell_fill_weights_f64", n, p(rp), p(K), p(slice_ptr), p(sell_row), p(got))
    assert torch.equal(got[:n_slots], placed(K)[:n_slots])
    W64 = scale[row] * K
    got.fill_(7.0)
    ctx.call("dcpse_sell_fill_weights_scaled_f64", n, p(rp), p(K), p(scale), p(slice_ptr), p(sell_row), p(got))
    assert torch.equal(got[:n_slots], placed(W64)[:n_slots])
    vl = VerletList(rp, col, n, 1.0)
    plain, scaled = bundle16(vl, [W64, K]), bundle16(vl, [K, K], [scale, torch.ones_like(scale)])
    for a, b in zip(plain[:2], scaled[:2]):  # the bundle and its lanes (no far neighbours: the lists are empty)
        assert torch.equal(a.flatten()[: 2 * n_slots], b.flatten()[: 2 * n_slots])
    # far neighbours per lane, plain offsets (a small set: none)
    exc_ptr, n_exc = vl.far16()
    assert n_exc == 0 and int(exc_ptr.abs().max()) == 0
