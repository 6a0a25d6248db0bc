"""Operators whose first use is inside a graph capture: what the capture builds
(FP64 weights, layouts, prepared calls) has its values only at a replay, so
eager calls before and after the replays build their own."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _operators(cuda, kinds):
    import openfpm_numerics_amd as A

    n = 40
    rng = np.random.default_rng(1)
    g = (np.arange(n) + 0.5) / n
    pos = np.stack(np.meshgrid(g, g, indexing="ij"), -1).reshape(-1, 2)
    pos = np.mod(pos + rng.uniform(-0.1 / n, 0.1 / n, pos.shape), 1.0)
    ps = A.ParticleSet(pos, [0.0] * 2, [1.0] * 2, bc=[1, 1], device=cuda)
    vl = ps.getVerlet(3.1 / n)
    return [getattr(A, k)(ps, vl, 2, 3.1 / n) for k in kinds], ps.size_local()


def _runs(A, name):
    return {
        "apply": lambda lap, dx, f: [dx(f)],
        "fused": lambda lap, dx, f: A.fused(dx, lap, f=f),
        "batch": lambda lap, dx, f: [dx(torch.stack([f, 2 * f, 3 * f, 4 * f]))],
        "rk4": lambda lap, dx, f: [A.rk4(dx, f.clone(), 1e-4, 2)],
        "rk4_sell": lambda lap, dx, f: [A.rk4(dx, f.clone(), 1e-4, 2, layout="sell")],
        "rk4_bundle16": lambda lap, dx, f: [A.rk4(dx, f.clone(), 1e-4, 2, layout="bundle16")],
    }[name]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("name", ["apply", "fused", "batch", "rk4", "rk4_sell", "rk4_bundle16"])
def test_first_use_in_a_capture(cuda, name, dtype):
    import openfpm_numerics_amd as A

    run = _runs(A, name)
    kinds = ("Laplacian", "Derivative_x")
    (lap, dx), n = _operators(cuda, kinds)
    fresh, _ = _operators(cuda, kinds)
    rng = np.random.default_rng(2)
    fs = [torch.as_tensor(rng.standard_normal(n), dtype=dtype, device=cuda) for _ in range(4)]
    want = [run(*fresh, f) for f in fs]
    lap(fs[0])  # the list's own layout; dx has not been used
    f = fs[0].clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run(lap, dx, f)
    for k, x in enumerate(fs):
        for a, b in zip(run(lap, dx, x), want[k]):  # eager, first before any replay
            assert torch.equal(a, b), k
        f.copy_(x)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, want[k]):
            assert torch.equal(a, b), k
