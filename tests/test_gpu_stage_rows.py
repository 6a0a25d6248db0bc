"""Fused time-integration stages on the CSR kernel: rows of every length around
its steps (16 lanes by 4 up to 8,192 rows, 8 lanes by 4 beyond), with the outputs
aliasing their inputs, against FP64 numpy; and the layout "auto" picks.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n", [1, 5, 400, 8192, 8193, 20_011])
def test_stage_rows(cuda, n, dtype):
    from openfpm_numerics_amd import _lib

    rng = np.random.default_rng(n)
    lens = np.resize([0, 1, 3, 4, 7, 8, 9, 31, 32, 33, 63, 64, 65, 127, 130, 28, 56], n)
    rp = np.concatenate([[0], np.cumsum(lens)])
    nnz = int(rp[-1])
    np_t = np.float32 if dtype == torch.float32 else np.float64
    col = rng.integers(0, n, max(nnz, 1)).astype(np.int32)
    W, u, y, acc = (rng.standard_normal(k).astype(np_t) for k in (max(nnz, 1), n, n, n))
    d = [torch.as_tensor(v, device=cuda) for v in (rp.astype(np.int64), col, W, u, y, acc)]
    out = torch.full((n,), float("nan"), dtype=dtype, device=cuda)
    ctx, p = _lib.context(cuda.index or 0), _lib.ptr
    name = "dcpse_stage_f32" if dtype == torch.float32 else "dcpse_stage_f64"
    ctx.call(name, n, p(d[0]), p(d[1]), p(d[2]), p(d[3]), 0.75, p(d[4]), 0.25, p(out), p(d[5]), -1.5, p(d[5]))
    w, u64 = W.astype(np.float64), u.astype(np.float64)
    row = np.repeat(np.arange(n), lens)
    terms = w[:nnz] * (u64[col[:nnz]] - u64[row])
    k = 0.75 * np.bincount(row, terms, n)
    mag = 0.75 * np.bincount(row, np.abs(terms), n)
    for got, c, base in ((out, 0.25, y), (d[5], -1.5, acc)):
        want = base.astype(np.float64) + c * k
        # FP64 sums of at most 130 terms in any order, one rounding to the state's type
        bound = 140 * 2.0 ** -52 * (abs(c) * mag + np.abs(base)) + np.finfo(np_t).eps * np.abs(want)
        assert bool((np.abs(got.cpu().numpy().astype(np.float64) - want) <= bound).all())


def test_auto_layout_by_size(cuda, monkeypatch):
    from openfpm_numerics_amd import Laplacian, ParticleSet, ode

    rng = np.random.default_rng(2)
    g = (np.arange(24) + 0.5) / 24
    pos = np.stack(np.meshgrid(g, g, indexing="ij"), -1).reshape(-1, 2) + rng.uniform(-0.004, 0.004, (576, 2))
    ps = ParticleSet(np.mod(pos, 1.0), [0.0, 0.0], [1.0, 1.0], bc=[1, 1], device=cuda)
    f0 = torch.as_tensor(rng.standard_normal(576), device=cuda)
    for dtype, key in ((torch.float32, "bundle16"), (torch.float64, "bundle16_64")):
        vl = ps.getVerlet(3.1 / 24)
        lap = Laplacian(ps, vl, 2, 3.1 / 24)
        small = ode.rk4(lap, f0.to(dtype), 1e-5, 16)
        assert lap.dcpse._W.get(key) is None
        assert torch.equal(small, ode.rk4(lap, f0.to(dtype), 1e-5, 16, layout="csr"))
        monkeypatch.setitem(ode.CSR_MAX, dtype, vl.nnz - 1)
        large = ode.rk4(lap, f0.to(dtype), 1e-5, 16)
        assert lap.dcpse._W.get(key) is not None
        assert torch.equal(large, ode.rk4(lap, f0.to(dtype), 1e-5, 16, layout="bundle16"))
