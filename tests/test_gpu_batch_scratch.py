"""Batches with the caller's scratch for the particle-major copies: any size of
it, eager and captured, bit for bit one single-field apply per field."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _problem(cuda, dtype, n, nb):
    rng = np.random.default_rng(n + nb)
    lens = rng.integers(0, 60, n)
    rp = torch.as_tensor(np.concatenate([[0], np.cumsum(lens)]), device=cuda)
    nnz = int(lens.sum())
    col = torch.as_tensor(rng.integers(0, n, nnz), dtype=torch.int32, device=cuda)
    W, diag, f = (torch.as_tensor(rng.standard_normal(s), dtype=dtype, device=cuda) for s in (nnz, n, (nb, n)))
    return nnz, rp, col, W, diag, f


def _runs(ctx, dtype, n, nnz, rp, col, W, diag):
    from openfpm_numerics_amd import _lib

    p, t = _lib.ptr, "f32" if dtype == torch.float32 else "f64"

    def forward(k, src, dst, scratch, size):
        ctx.call(f"dcpse_apply_nnz_{t}", n, nnz, p(rp), p(col), 1, _lib.ptr_array([W]), p(src), n, k, None, n,
                 _lib.ptr_array([dst]), n, 0.75, 0.5, p(scratch), size)

    def transposed(k, src, dst, scratch, size):
        ctx.call(f"dcpse_apply_transpose_nnz_{t}", n, nnz, p(rp), p(col), p(W), p(diag), p(src), n, k, p(dst), n, 0.75,
                 0.5, p(scratch), size)

    return forward, transposed


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("nb", [1, 2, 3, 5, 16, 19])
def test_any_scratch(cuda, nb, dtype):
    from openfpm_numerics_amd import _lib

    n = 1337
    nnz, rp, col, W, diag, f = _problem(cuda, dtype, n, nb)
    one = f.element_size()
    for run in _runs(_lib.context(cuda.index or 0), dtype, n, nnz, rp, col, W, diag):
        want = torch.ones_like(f)
        for b in range(nb):
            run(1, f[b], want[b], None, 0)
        # values of room: none, one short of a pass of 4, of 4, 8 and 16 fields, and more
        for room in (0, 4 * n - 1, 4 * n, 8 * n - 1, 8 * n, 16 * n, 17 * n):
            scratch = torch.full((room + 64,), 7.0, dtype=dtype, device=cuda)
            got = torch.ones_like(f)
            run(nb, f, got, scratch, room * one)
            assert torch.equal(got, want), (run.__name__, room)
            assert bool((scratch[room:] == 7.0).all()), (run.__name__, room)


def test_scratch_is_checked(cuda):
    from openfpm_numerics_amd import _lib

    n = 100
    nnz, rp, col, W, diag, f = _problem(cuda, torch.float64, n, 4)
    scratch = torch.empty(4 * n + 2, dtype=torch.float64, device=cuda)
    for run in _runs(_lib.context(cuda.index or 0), torch.float64, n, nnz, rp, col, W, diag):
        with pytest.raises(_lib.DcpseError, match="16-byte"):
            run(4, f, torch.ones_like(f), scratch[1:], 4 * n * 8)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("nb", [4, 16])
def test_captured_batch_is_particle_major(cuda, nb, dtype):
    """A captured batch runs the passes of an eager one: every replay leaves its
    fields particle-major in the scratch."""
    from openfpm_numerics_amd import _lib

    n = 2000
    nnz, rp, col, W, diag, f = _problem(cuda, dtype, n, nb)
    scratch = torch.zeros(nb * n, dtype=dtype, device=cuda)
    size = scratch.numel() * scratch.element_size()
    rng = np.random.default_rng(3)
    for run in _runs(_lib.context(cuda.index or 0), dtype, n, nnz, rp, col, W, diag):
        out, want = torch.zeros_like(f), torch.zeros_like(f)
        run(nb, f, out, scratch, size)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            run(nb, f, out, scratch, size)
        for k in range(3):
            f.copy_(torch.as_tensor(rng.standard_normal((nb, n)), dtype=dtype))
            scratch.zero_()
            out.zero_()
            want.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(scratch.view(n, nb), f.t()), (run.__name__, k)
            for b in range(nb):
                run(1, f[b], want[b], None, 0)
            assert torch.equal(out, want), (run.__name__, k)
