"""Batches on several streams of one context without a wait between them: the
particle-major copies of a batch stay whole until it has read them. Results
bit for bit those of the same calls one after another."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _operator(cuda, n, rcut):
    from openfpm_numerics_amd import Laplacian, ParticleSet

    rng = np.random.default_rng(n)
    g = (np.arange(n) + 0.5) / n
    pos = np.stack(np.meshgrid(g, g, indexing="ij"), -1).reshape(-1, 2)
    pos = np.mod(pos + rng.uniform(-0.1 / n, 0.1 / n, pos.shape), 1.0)
    ps = ParticleSet(pos, [0.0] * 2, [1.0] * 2, bc=[1, 1], device=cuda)
    return ps, Laplacian(ps, ps.getVerlet(rcut / n), 2, rcut / n).dcpse


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("nb", [3, 13, 20])
def test_batches_on_two_streams(cuda, nb, dtype):
    from openfpm_numerics_amd import _lib

    _, d = _operator(cuda, 300, 3.1)
    vl = d.verletList
    n = vl.n_rows
    f = torch.randn((2, nb, n), generator=torch.Generator("cuda").manual_seed(nb), dtype=dtype, device=cuda)
    W = d.weights(dtype)
    rowT, colT, WT, diag = d.transposed(dtype)
    ctx, p = _lib.context(cuda.index or 0), _lib.ptr
    t = "f32" if dtype == torch.float32 else "f64"

    def forward(src, dst):
        ctx.call(f"dcpse_apply_{t}", n, p(vl.row_ptr), p(vl.col), 1, _lib.ptr_array([W]), p(src), n, nb, None, n,
                 _lib.ptr_array([dst]), n, 1.0, 0.0)

    def transposed(src, dst):
        ctx.call(f"dcpse_apply_transpose_{t}", n, p(rowT), p(colT), p(WT), p(diag), p(src), n, nb, p(dst), n, 1.0, 0.0)

    def python(src, dst):
        d.computeDifferentialOperator(src, out=dst)

    def python_transposed(src, dst):
        d.applyTranspose(src, out=dst)

    streams = [torch.cuda.Stream(cuda) for _ in range(2)]
    for run in (forward, transposed, python, python_transposed):
        want = [torch.empty_like(x) for x in f]
        for x, o in zip(f, want):
            run(x, o)
            torch.cuda.synchronize()
        got = [[torch.zeros_like(x) for x in f] for _ in range(4)]
        torch.cuda.synchronize()
        for outs in got:
            for s, x, o in zip(streams, f, outs):
                with torch.cuda.stream(s):
                    run(x, o)
        torch.cuda.synchronize()
        for outs in got:
            for o, w in zip(outs, want):
                assert torch.equal(o, w), run.__name__


def test_batch_beside_a_search(cuda):
    """A batch on one stream, neighbour lists and an operator's transpose on
    another; the lists first outgrow the workspace."""
    ps, d = _operator(cuda, 200, 3.1)
    f = torch.randn((16, ps.size_local()), generator=torch.Generator("cuda").manual_seed(1), dtype=torch.float64,
                    device=cuda)
    want = d(f)
    other, _ = _operator(cuda, 260, 3.1)
    rc = 3.1 / 260
    ref = other.getVerlet(rc)
    torch.cuda.synchronize()
    side = torch.cuda.Stream(cuda)
    for _ in range(3):
        got = [torch.empty_like(f) for _ in range(2)]
        torch.cuda.synchronize()
        for o in got:
            d.computeDifferentialOperator(f, out=o)
        with torch.cuda.stream(side):
            vl = other.getVerlet(rc)
        torch.cuda.synchronize()
        assert torch.equal(vl.row_ptr, ref.row_ptr) and torch.equal(vl.col, ref.col)
        for o in got:
            assert torch.equal(o, want)
