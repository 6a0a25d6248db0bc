"""Neighbour lists of one set, with one cut-off or one per particle: the group
kernels (candidate lists sorted in registers, FP32 tests with an FP64 decision
near the cut-off) against the per-particle kernel, which a subset domain holding every particle
runs through. Both take the same distance formula, so the lists must be equal
entry for entry, ties at the cut-off included.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _uniform(n, dim, seed=0):
    return np.random.default_rng(seed).random((n, dim))


def _lattice(n, dim):
    g = (np.arange(n) + 0.5) / n
    return np.stack([a.ravel() for a in np.meshgrid(*([g] * dim), indexing="ij")], axis=1)


def _clustered(n, dim, seed=1):
    """A thin background and one dense cluster: its cells exceed the candidate lists."""
    rng = np.random.default_rng(seed)
    return np.concatenate([rng.random((n, dim)), 0.5 + 0.03 * rng.random((n // 8, dim))])


def _duplicates(n, dim, seed=2):
    p = np.random.default_rng(seed).random((n, dim))
    return np.concatenate([p, p[::3]])


# (points, dim, cut-off, box, periodicity). The mean candidate count of a cell
# runs through every register width (1 to 32 keys per lane) and past the
# per-cell kernels' limit; cells hold none to over 64 particles.
CASES = {
    "few_3d": (lambda: _uniform(300, 3), 0.21, 1),
    "sparse_3d": (lambda: _uniform(6000, 3), 0.06, 1),
    "widths_3d_160": (lambda: _uniform(6000, 3), 0.1, 1),
    "widths_3d_740": (lambda: _uniform(20000, 3), 0.11, 1),
    "beyond_3d_2500": (lambda: _uniform(20000, 3), 0.16, 1),
    "beyond_3d_5200": (lambda: _uniform(24000, 3), 0.2, 1),
    "widths_3d_200": (lambda: _uniform(8000, 3), 0.1, 1),
    "widths_3d_1600": (lambda: _uniform(7500, 3), 0.2, 1),
    "beyond_3d": (lambda: _uniform(12000, 3), 0.249, 1),
    "widths_2d_10": (lambda: _uniform(3000, 2), 0.02, 1),
    "widths_2d_90": (lambda: _uniform(9001, 2), 0.033, 1),
    "widths_2d_300": (lambda: _uniform(9000, 2), 0.06, 1),
    "widths_2d_700": (lambda: _uniform(9000, 2), 0.09, 1),
    "three_cells": (lambda: _uniform(900, 3), 0.3, 1),
    "four_cells": (lambda: _uniform(2000, 3), 0.24, 1),
    "open_3d": (lambda: _uniform(8000, 3), 0.11, 0),
    "open_two_cells": (lambda: _uniform(500, 3), 0.4, 0),
    "clustered_3d": (lambda: _clustered(8000, 3), 0.05, 1),
    "clustered_2d": (lambda: _clustered(4000, 2), 0.03, 1),
    "ties_3d": (lambda: _lattice(16, 3), 2.0 / 16, 1),
    "ties_2d": (lambda: _lattice(48, 2), 3.0 / 48, 1),
    "ties_odd_2d": (lambda: _lattice(43, 2), 5.0 / 43, 0),
    "coincident": (lambda: _duplicates(3000, 3), 0.12, 1),
    "outside_open": (lambda: np.concatenate([_uniform(3000, 3), 40.0 * _uniform(50, 3) - 20.0]), 0.12, 0),
    "unwrapped": (lambda: _uniform(4000, 3) + np.random.default_rng(3).integers(-3, 4, (4000, 3)), 0.11, 1),
    "one_particle": (lambda: _uniform(1, 3), 0.2, 1),
    "below_a_slice": (lambda: _uniform(63, 2), 0.2, 1),
}


def _graded(n, dim, ratio, seed=6):
    """Points thinning out along x and cut-offs to match (spread 1 : ratio)."""
    rng = np.random.default_rng(seed)
    p = rng.random((n, dim))
    p[:, 0] = p[:, 0] ** 2
    return p, (1.0 + (ratio - 1.0) * p[:, 0]) * rng.uniform(0.95, 1.0, n)


# a cut-off per particle: (points and cut-offs, periodicity)
OWN = {
    "spread_1": (lambda: (_uniform(4000, 3), 0.09 + 1e-9 * np.arange(4000)), 1),
    "spread_2": (lambda: (lambda p, r: (p, 0.06 * r))(*_graded(9000, 3, 2.0)), 1),
    "spread_4": (lambda: (lambda p, r: (p, 0.05 * r))(*_graded(9000, 3, 4.0)), 1),
    "spread_9_open": (lambda: (lambda p, r: (p, 0.03 * r))(*_graded(9000, 3, 9.0)), 0),
    "spread_100": (lambda: (_uniform(3000, 3), 0.003 + 0.297 * np.random.default_rng(7).random(3000) ** 8), 1),
    "shuffled_cutoffs": (lambda: (_uniform(5000, 3), np.random.default_rng(8).uniform(0.03, 0.13, 5000)), 1),
    "spread_3_2d": (lambda: (lambda p, r: (p, 0.02 * r))(*_graded(9001, 2, 3.0)), 1),
    "spread_20_2d": (lambda: (lambda p, r: (p, 0.01 * r))(*_graded(7000, 2, 20.0)), 0),
    "small_box": (lambda: (_uniform(700, 3), np.random.default_rng(9).uniform(0.2, 0.33, 700)), 1),
    "mixed_box": (lambda: (_uniform(900, 2), np.random.default_rng(9).uniform(0.05, 0.33, 900)), 1),
    "dense": (lambda: (_uniform(20000, 3), np.random.default_rng(10).uniform(0.1, 0.2, 20000)), 1),
    "ties": (lambda: (_lattice(16, 3), np.where(np.arange(4096) % 3 == 0, 2.0, 1.0) / 16), 1),
    "outside_open": (lambda: (np.concatenate([_uniform(3000, 3), 9.0 * _uniform(90, 3) - 4.0]),
                              np.random.default_rng(11).uniform(0.05, 0.3, 3090)), 0),
    "unwrapped": (lambda: (_uniform(4000, 3) + np.random.default_rng(3).integers(-3, 4, (4000, 3)),
                           np.random.default_rng(12).uniform(0.05, 0.11, 4000)), 1),
    "coincident": (lambda: (_duplicates(3000, 3), np.full(4000, 0.1) + 1e-4 * np.arange(4000) / 4000), 1),
    "sparse": (lambda: (_uniform(400, 3), np.random.default_rng(13).uniform(0.002, 0.02, 400)), 1),
    "two_particles": (lambda: (np.array([[0.1, 0.1], [0.9, 0.9]]), np.array([0.3, 0.1])), 1),
}


def _compare(pos, rcut, lo, hi, periodic, cuda):
    from openfpm_numerics_amd import ParticleSet, ParticleSubset

    ps = ParticleSet(pos, lo, hi, bc=[periodic] * pos.shape[1], device=cuda)
    got = ps.getVerlet(rcut)
    want = ParticleSubset(ps, np.arange(len(pos), dtype=np.int32)).getVerlet(rcut)
    assert torch.equal(got.row_ptr, want.row_ptr)
    assert torch.equal(got.col, want.col)
    return got


@pytest.mark.parametrize("name", list(CASES))
def test_cell_lists_equal_per_particle_lists(cuda, name):
    make, rcut, periodic = CASES[name]
    pos = make()
    dim = pos.shape[1]
    vl = _compare(pos, rcut, [0.0] * dim, [1.0] * dim, periodic, cuda)
    print(f"[support] {name}: {len(pos)} particles, mean row {vl.nnz / len(pos):.1f}", flush=True)


@pytest.mark.parametrize("name", list(OWN))
def test_own_cutoffs_equal_per_particle_lists(cuda, name):
    make, periodic = OWN[name]
    pos, rcut = make()
    dim = pos.shape[1]
    vl = _compare(pos, torch.as_tensor(rcut, device=cuda), [0.0] * dim, [1.0] * dim, periodic, cuda)
    print(f"[support] {name}: {len(pos)} particles, mean row {vl.nnz / len(pos):.1f}", flush=True)


@pytest.mark.parametrize("scale,shift", [(1e-9, 0.0), (3e7, 0.0), (1.0, 1e4), (1.0, 3e6), (1.0, -1e10)])
def test_units_and_offsets(cuda, scale, shift):
    """Other length units, boxes away from the origin (at 3e6 and 1e10 the FP64
    kernels take over) and positions of little resolution."""
    pos = _uniform(5000, 3, seed=4) * scale + shift
    _compare(pos, 0.11 * scale, [shift] * 3, [scale + shift] * 3, 1, cuda)
    own = torch.as_tensor(np.random.default_rng(14).uniform(0.05, 0.11, 5000) * scale, device=cuda)
    _compare(pos, own, [shift] * 3, [scale + shift] * 3, 1, cuda)


def test_fill_follows_new_positions(cuda):
    """Lists built again after every particle moved use no old candidate list."""
    from openfpm_numerics_amd import ParticleSet

    pos = _uniform(5000, 3, seed=5)
    ps = ParticleSet(pos, [0.0] * 3, [1.0] * 3, bc=[1] * 3, device=cuda)
    vl = ps.getVerlet(0.1)
    for k in range(3):
        pos = np.mod(pos + 0.03 * (k + 1), 1.0)[::-1].copy()
        ps.set_positions(pos)
        vl = ps.updateVerlet(vl, 0.1)
        want = _compare(pos, 0.1, [0.0] * 3, [1.0] * 3, 1, cuda)
        assert torch.equal(vl.row_ptr, want.row_ptr) and torch.equal(vl.col, want.col)
