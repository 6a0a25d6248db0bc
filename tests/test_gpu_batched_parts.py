"""Batched FP32 applies whose fields do not fill a pass and whose rows are
shared by four or eight lanes: every batch size around the passes of 4, 8 and
16 fields, bit for bit against one single-field pass per field.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# mean rows below 24, below 40, 40 to 56, 56 to 72 and above 72 (the launch
# shapes), each with rows shorter and longer than a pass covers
LENGTHS = {"short": (0, 40), "middle": (0, 70), "mean_48": (30, 67), "mean_64": (1, 128), "long": (70, 131)}


@pytest.mark.parametrize("few", [True, False])
@pytest.mark.parametrize("name", list(LENGTHS))
def test_batch_parts(cuda, name, few):
    from openfpm_numerics_amd import _lib

    rng = np.random.default_rng(len(name))
    n = 999 if few else 140_001  # eight lanes per row up to 131,072 rows
    lens = rng.integers(*LENGTHS[name], n)
    rp = torch.as_tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int64, device=cuda)
    nnz = int(lens.sum())
    col = torch.as_tensor(rng.integers(0, n, nnz), dtype=torch.int32, device=cuda)
    W = torch.as_tensor(rng.standard_normal(nnz), dtype=torch.float32, device=cuda)
    diag = torch.as_tensor(rng.standard_normal(n), dtype=torch.float32, device=cuda)
    f = torch.as_tensor(rng.standard_normal((19, n)), dtype=torch.float32, device=cuda)
    ctx, p = _lib.context(cuda.index or 0), _lib.ptr

    def forward(nb, src, dst):
        ctx.call("dcpse_apply_f32", n, p(rp), p(col), 1, _lib.ptr_array([W]), p(src), n, nb, None, n,
                 _lib.ptr_array([dst]), n, 1.0, 0.5)

    def transposed(nb, src, dst):
        ctx.call("dcpse_apply_transpose_f32", n, p(rp), p(col), p(W), p(diag), p(src), n, nb, p(dst), n, 1.0, 0.5)

    for run in (forward, transposed):
        want = torch.ones_like(f)
        for b in range(len(f)):
            run(1, f[b], want[b])
        for nb in ((2, 3, 4, 5, 7, 8, 9, 12, 13, 16, 17, 18, 19) if few else (3, 6, 13, 19)):
            got = torch.ones_like(f)
            run(nb, f, got)
            assert torch.equal(got[:nb], want[:nb]), (run.__name__, nb)
            assert bool((got[nb:] == 1).all()), (run.__name__, nb)  # fields beyond the batch are not written


@pytest.mark.parametrize("few", [True, False])
@pytest.mark.parametrize("name", ["short", "mean_64", "long"])
def test_fp64_batches(cuda, name, few):
    """FP64 batches against single fields of the CSR kernel, bit for bit."""
    from openfpm_numerics_amd import _lib

    rng = np.random.default_rng(7 + few)
    n = 999 if few else 40_003
    lens = rng.integers(*LENGTHS[name], n)
    lens[[0, n // 2, n - 1]] = 0
    rp = torch.as_tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int64, device=cuda)
    nnz = int(lens.sum())
    col = torch.as_tensor(rng.integers(0, n, nnz), dtype=torch.int32, device=cuda)
    W = torch.as_tensor(rng.standard_normal(nnz), device=cuda)
    diag = torch.as_tensor(rng.standard_normal(n), device=cuda)
    f = torch.as_tensor(rng.standard_normal((19, n)), device=cuda)
    ctx, p = _lib.context(cuda.index or 0), _lib.ptr
    def forward(nb, src, dst):
        ctx.call("dcpse_apply_f64", n, p(rp), p(col), 1, _lib.ptr_array([W]), p(src), n, nb, None, n,
                 _lib.ptr_array([dst]), n, 0.75, 0.5)

    def transposed(nb, src, dst):
        ctx.call("dcpse_apply_transpose_f64", n, p(rp), p(col), p(W), p(diag), p(src), n, nb, p(dst), n, 0.75, 0.5)

    for run in (forward, transposed):
        want = torch.ones_like(f)
        for b in range(len(f)):
            run(1, f[b], want[b])
        for nb in (2, 3, 4, 5, 8, 9, 16, 17, 19):
            got = torch.ones_like(f)
            run(nb, f, got)
            assert torch.equal(got[:nb], want[:nb]), (run.__name__, nb)
            assert bool((got[nb:] == 1).all()), (run.__name__, nb)


@pytest.mark.parametrize("direction", ["forward", "transposed"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("nb", [3, 13])
def test_captured_batches(cuda, nb, dtype, direction):
    """A captured batch keeps no workspace: lists that outgrow it come between
    capture and replay."""
    from openfpm_numerics_amd import Laplacian, ParticleSet

    rng = np.random.default_rng(nb)

    def lattice(n):
        g = (np.arange(n) + 0.5) / n
        pos = np.stack(np.meshgrid(g, g, indexing="ij"), -1).reshape(-1, 2)
        return ParticleSet(np.mod(pos + rng.uniform(-0.1 / n, 0.1 / n, pos.shape), 1.0), [0.0] * 2, [1.0] * 2, bc=[1, 1],
                           device=cuda)

    ps = lattice(48)
    d = Laplacian(ps, ps.getVerlet(3.1 / 48), 2, 3.1 / 48).dcpse
    f = torch.as_tensor(rng.standard_normal((nb, ps.size_local())), dtype=dtype, device=cuda)
    run = d if direction == "forward" else d.applyTranspose
    run(f)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run(f)
    lattice(700).getVerlet(3.1 / 700)
    for k in range(3):
        f.copy_(torch.as_tensor(rng.standard_normal(f.shape), dtype=dtype))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, run(f)), k
