"""The particles per wavefront that the assembly picks from the number of
particles, on both sides of each line, against 18 per wavefront, bit for bit.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 7, 16384, 16385, 131072, 131073, 524288, 524289])
def test_default_batches(cuda, n):
    from openfpm_numerics_amd import Derivative_x, Laplacian, ParticleSet, VerletList, _lib
    from openfpm_numerics_amd.dcpse import assemble_together

    # n domain particles on a support of a lattice: ring-shaped lists by index, no search
    m = 64
    g = (np.arange(m) + 0.5) / m
    rng = np.random.default_rng(1)
    pos = np.stack(np.meshgrid(g, g, indexing="ij"), -1).reshape(-1, 2) + rng.uniform(-0.1 / m, 0.1 / m, (m * m, 2))
    sup = ParticleSet(np.mod(pos, 1.0), [0.0, 0.0], [1.0, 1.0], bc=[1, 1], device=cuda)
    home = rng.integers(0, m * m, n)
    dom = ParticleSet(np.mod(pos[home] + rng.uniform(-0.2 / m, 0.2 / m, (n, 2)), 1.0), [0.0, 0.0], [1.0, 1.0], bc=[1, 1],
                      device=cuda)
    dy, dx = np.meshgrid(np.arange(-2, 3), np.arange(-2, 3))
    near = ((home // m)[:, None] + dx.ravel()) % m * m + ((home % m)[:, None] + dy.ravel()) % m
    vl = VerletList(torch.arange(0, 25 * n + 1, 25, device=cuda),
                    torch.as_tensor(np.sort(near, 1).astype(np.int32).ravel(), device=cuda), m * m, 3.0 / m, dom)
    ops = [K(sup, vl, 2, 3.0 / m, particlesDomain=dom).dcpse for K in (Laplacian, Derivative_x)]
    ctx = _lib.context(cuda.index or 0)
    got = [(d.localEps.clone(), d.calcKernels.clone(), d.info.clone()) for d in ops if not assemble_together([d])]
    pair = assemble_together(ops) or [d.calcKernels.clone() for d in ops]
    try:
        ctx.call("dcpse_set_assembly_launch", 0, 18, 64, 0)
        for d, (eps, K, info) in zip(ops, got):
            assemble_together([d])
            assert torch.equal(d.localEps, eps) and torch.equal(d.calcKernels, K) and torch.equal(d.info, info)
        assemble_together(ops)
        assert all(torch.equal(d.calcKernels, K) for d, K in zip(ops, pair))
    finally:
        ctx.call("dcpse_set_assembly_launch", 0, 0, 64, 0)
