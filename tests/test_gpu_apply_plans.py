"""The prepared path of repeated single-field applies against the first apply
of fresh operators: after reassembly, a load, a new list, on another stream, in
a captured graph, for alternating operators, copies, and inputs the plan does
not take (strided, batched, wrong length).
"""
import copy

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _set(cuda, seed=0, n=20):
    from openfpm_numerics_amd import ParticleSet

    rng = np.random.default_rng(seed)
    g = (np.arange(n) + 0.5) / n
    pos = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    pos = np.mod(pos + rng.uniform(-0.1 / n, 0.1 / n, pos.shape), 1.0)
    return ParticleSet(pos, [0.0] * 3, [1.0] * 3, bc=[1] * 3, device=cuda), 2.4 / n, rng


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_repeated_applies(cuda, dtype, tmp_path):
    from openfpm_numerics_amd import Derivative_x, Derivative_y, Laplacian, fused

    ps, rc, rng = _set(cuda)
    vl = ps.getVerlet(rc)
    kinds = (Laplacian, Derivative_x, Derivative_y)
    ops = [K(ps, vl, 2, rc) for K in kinds]
    n = ps.size_local()
    fs = [torch.as_tensor(rng.standard_normal(n), dtype=dtype, device=cuda) for _ in range(3)]

    def first(k, f):  # the first apply of new operators on a new list
        v = ps.getVerlet(rc)
        return fused(*[kinds[i](ps, v, 2, rc) for i in k], f=f)

    for k in ((0,), (0, 1), (0, 2), (0, 1), (0, 1, 2), (2, 0)):
        for f in fs:
            for got, want in zip(fused(*[ops[i] for i in k], f=f), first(k, f)):
                assert torch.equal(got, want), k
    # strided and batched inputs, outputs given, a wrong length
    wide = torch.stack(fs, 1)
    assert torch.equal(ops[0](wide[:, 1]), ops[0](fs[1]))
    assert ops[0](fs[0][None]).shape == (1, n)
    out = torch.ones_like(fs[0])
    want = 2.0 * ops[0](fs[0]).double() + 0.5
    ops[0].apply(fs[0], out=out, alpha=2.0, beta=0.5)
    assert float((out.double() - want).abs().max()) <= 4 * torch.finfo(dtype).eps * float(want.abs().max())
    with pytest.raises(ValueError):
        ops[0](fs[0][:-1])
    # another stream
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = ops[0](fs[2])
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(got, first((0,), fs[2])[0])
    # copies make their own plans
    twin = copy.deepcopy(ops[1].dcpse)
    assert torch.equal(twin(fs[0]), ops[1](fs[0])) and twin._plans is not ops[1].dcpse._plans
    # moved particles: refused until the update, then the new kernels
    ops[0].save(ps, str(tmp_path / "k"))
    old = ops[0](fs[0])
    ps.set_positions(torch.remainder(ps.positions() + 0.01 / 20 * torch.sin(6.28 * ps.positions().flip(1)), 1.0))
    with pytest.raises(RuntimeError):
        ops[0](fs[0])
    ps.updateVerlet(vl, rc)
    ops[0].update(ps)
    moved = ops[0](fs[0])
    assert torch.equal(moved, first((0,), fs[0])[0]) and not torch.equal(moved, old)
    # the list replaced under the same operators
    before = ops[0].dcpse.verletList
    ops[0].dcpse.verletList = ps.getVerlet(rc)
    assert torch.equal(ops[0](fs[1]), first((0,), fs[1])[0])
    ops[0].dcpse.verletList = before


def test_load_renews_plans(cuda, tmp_path):
    from openfpm_numerics_amd import Laplacian

    ps, rc, rng = _set(cuda, 3)
    vl = ps.getVerlet(rc)
    a, b = Laplacian(ps, vl, 2, rc), Laplacian(ps, vl, 2, rc, h_over_eps=0.8)
    f = torch.as_tensor(rng.standard_normal(ps.size_local()), device=cuda)
    want = a(f)
    assert not torch.equal(b(f), want)
    a.save(ps, str(tmp_path / "k"))
    b.load(ps, str(tmp_path / "k"))
    got = b(f)
    assert float((got - want).abs().max()) <= 1e-13 * float(want.abs().max())


def test_planned_apply_in_a_graph(cuda):
    from openfpm_numerics_amd import Laplacian

    ps, rc, rng = _set(cuda, 4)
    lap = Laplacian(ps, ps.getVerlet(rc), 2, rc)
    f = torch.as_tensor(rng.standard_normal(ps.size_local()), dtype=torch.float32, device=cuda)
    lap(f)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = lap(f)
    for k in range(3):
        f.copy_(torch.as_tensor(rng.standard_normal(ps.size_local()), dtype=torch.float32))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, lap(f)), k


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_columns_by_list_size(cuda, dtype, monkeypatch):
    from openfpm_numerics_amd import Derivative_x, Laplacian, dcpse, fused

    ps, rc, rng = _set(cuda, 5)
    f = torch.as_tensor(rng.standard_normal(ps.size_local()), dtype=dtype, device=cuda)
    got = []
    for least in (dcpse.COL16_MIN, 0):
        monkeypatch.setattr(dcpse, "COL16_MIN", least)
        vl = ps.getVerlet(rc)
        got.append(fused(Laplacian(ps, vl, 2, rc), Derivative_x(ps, vl, 2, rc), f=f))
        assert bool(vl._col16) == (least == 0) and (vl._sell is None) == (least == 0)
    for a, b in zip(*got):
        assert float((a - b).abs().max()) <= 2 * torch.finfo(dtype).eps * float(a.abs().max())
