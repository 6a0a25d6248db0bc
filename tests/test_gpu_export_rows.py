"""Sparse export on rows of every length: every number of lanes per row, with
weights given and formed on the way, against numpy.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = {
    "empty_rows": [0, 0, 3],
    "one": [1],
    "short": list(range(0, 18)),  # mean below 32: 16 lanes
    "mean_32": [32, 31, 33, 16, 48, 15, 49, 32],
    "middle": [33, 63, 64, 65, 31, 96, 1, 90],  # 32 lanes
    "mean_80": [80] * 5,
    "long": [81, 127, 128, 129, 255, 300, 0, 64],  # 64 lanes
}


@pytest.mark.parametrize("name", list(ROWS))
def test_export_rows(cuda, name):
    from openfpm_numerics_amd import _lib

    rng = np.random.default_rng(4)
    lens = np.array(ROWS[name])
    n_rows = len(lens)
    n = max(n_rows, 400)  # the listed lengths over and over, which keeps their mean
    lens = np.concatenate([lens] * (n // n_rows + 1))[:n]
    rows = [np.sort(rng.choice(np.delete(np.arange(n), i), k, replace=False)) for i, k in enumerate(lens)]
    rp = np.concatenate([[0], np.cumsum(lens)])
    col = np.concatenate(rows).astype(np.int32)
    nnz = len(col)
    K, s = rng.standard_normal(max(nnz, 1)), rng.uniform(0.5, 2.0, n)
    row_of = np.repeat(np.arange(n), lens)
    W = np.zeros(max(nnz, 1))
    W[:nnz] = K[:nnz] * s[row_of]
    d = {k: torch.as_tensor(v, device=cuda) for k, v in
         dict(rp=rp.astype(np.int64), col=np.concatenate([col, [0]]).astype(np.int32), K=K, s=s, W=W,
              W32=W.astype(np.float32)).items()}
    ctx = _lib.context(cuda.index or 0)
    p = _lib.ptr

    def outs(dt):
        return (torch.full((n + 1,), -1, dtype=torch.int64, device=cuda),
                torch.full((nnz + n,), -1, dtype=torch.int32, device=cuda),
                torch.full((nnz + n,), float("nan"), dtype=dt, device=cuda))

    got = {}
    for key, fn, args, dt in (
            ("W", "dcpse_export_csr_nnz_f64", (n, nnz, p(d["rp"]), p(d["col"]), p(d["W"]), None), torch.float64),
            ("K", "dcpse_export_csr_nnz_f64", (n, nnz, p(d["rp"]), p(d["col"]), p(d["K"]), p(d["s"])), torch.float64),
            ("plain", "dcpse_export_csr_f64", (n, p(d["rp"]), p(d["col"]), p(d["W"])), torch.float64),
            ("f32", "dcpse_export_csr_nnz_f32", (n, nnz, p(d["rp"]), p(d["col"]), p(d["W32"])), torch.float32)):
        o = outs(dt)
        ctx.call(fn, *args, -1.0, *map(p, o))
        got[key] = [t.cpu().numpy() for t in o]
    for key, (grp, gcol, gval) in got.items():
        w = W.astype(np.float32) if key == "f32" else W
        eps = 2.0 ** -23 if key == "f32" else 2.0 ** -52
        assert np.array_equal(grp, rp + np.arange(n + 1)), key
        for i in range(n):
            r, k = rows[i], int((rows[i] < i).sum())
            a = w[rp[i]:rp[i + 1]]
            assert np.array_equal(gcol[grp[i]:grp[i + 1]], np.insert(r, k, i)), (key, i)
            v = gval[grp[i]:grp[i + 1]]
            assert np.array_equal(np.delete(v, k), a), (key, i)
            # FP64 sums of len(a) terms in any order, one rounding to the value type
            bound = len(a) * 2.0 ** -52 * np.abs(a.astype(np.float64)).sum() + eps * abs(a.astype(np.float64).sum())
            assert abs(v[k] + a.astype(np.float64).sum()) <= bound, (key, i)
    assert np.array_equal(got["K"][2], got["W"][2])
