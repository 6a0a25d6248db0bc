"""The work a user of this framework has it do, as measurable cases.

Every case goes through the Python entry points of the package: neighbour
support (``getVerlet``), operator assembly (``assemble_together``, ``update``),
applies (operators called on fields, ``fused``, ``Gradient``), gradients
through ``dcpse_apply``, explicit time integration (``rk4``) and the sparse
matrix handed to implicit solvers (``export_csr``).

The listed sizes are those of the repository's workloads, tests and benchmark:

  apply_2d_64_f64          the 64 x 64 periodic lattice: the smallest set, where one
                           call's launches and host work are all there is
  apply_2d_512_f32         one Laplacian on the 512 x 512 jittered set in FP32, the
                           plain ``op(f)`` of an explicit solver
  fused_3d_128_f32         Laplacian and d/dx of one field in one pass on the
                           benchmark's set (128^3 lattice, 10% removed)
  gradient_3d_77_f64       all first derivatives of a field in FP64 on an odd size
  adjoint_2d_1024_b16_f32  a loss and its gradient with respect to 16 fields (an
                           inverse problem): forward and transposed applies
  rk4_adaptive_1m_f32      explicit diffusion on the adaptive set of a million
                           particles (spacing 4 : 1, own cut-off per particle)
  rk4_3d_64_f64            the same integration in FP64 on an ordinary set
  support_3d_128           neighbour lists of the benchmark's set
  support_adaptive_500k    neighbour lists with one cut-off per particle
  assemble_3d_128          kernels of Laplacian and d/dx on the benchmark's set
  moving_3d_75_f64         one Lagrangian step: the particles have moved, so lists,
                           kernels and the first apply on them are all new
  export_3d_96_f64         the operator as a sparse matrix for an implicit solver

``draw`` spreads the same kinds of work over their whole ranges: dimensions,
sizes, orders of the particles in memory, operators, value types, batches.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from openfpm_numerics_amd import (Derivative_x, Derivative_xx, Derivative_xy, Derivative_y, Gradient, Laplacian,
                                  ParticleSet, dcpse_apply, fused, rk4)
from openfpm_numerics_amd.dcpse import assemble_together

_DTYPES = {"f32": torch.float32, "f64": torch.float64}
_OPS = {"lap": Laplacian, "dx": Derivative_x, "dy": Derivative_y, "dxx": Derivative_xx, "dxy": Derivative_xy}


def _case(kind, dim, n, dtype="f64", **kw):
    """A case with every option spelled out. ``set``: "jittered" (an n^dim
    lattice with jitter, a share ``drop`` of it removed) or "adaptive" (about n
    particles, spacing growing ``ratio`` times along x); ``rcut``: cut-off in
    spacings; ``order``: of the particles in memory; ``ops``: operators;
    ``batch``: fields; ``steps``: of the integration."""
    c = {"kind": kind, "set": "jittered", "dim": dim, "n": n, "dtype": dtype, "ops": "lap", "rcut": 3.1 if dim == 2 else 2.4,
         "jitter": 0.1, "drop": 0.0, "ratio": 4.0, "order": "lattice", "batch": 1, "steps": 0}
    c.update(kw)
    return c


def listed():
    named = {
        "apply_2d_64_f64": _case("apply", 2, 64, jitter=0.0),
        "apply_2d_512_f32": _case("apply", 2, 512, "f32"),
        "fused_3d_128_f32": _case("apply", 3, 128, "f32", ops="lap,dx", drop=0.1),
        "gradient_3d_77_f64": _case("gradient", 3, 77, drop=0.1, ops="grad"),
        "adjoint_2d_1024_b16_f32": _case("adjoint", 2, 1024, "f32", batch=16),
        "rk4_adaptive_1m_f32": _case("rk4", 3, 1_000_000, "f32", set="adaptive", steps=20),
        "rk4_3d_64_f64": _case("rk4", 3, 64, steps=20, drop=0.1),
        "support_3d_128": _case("support", 3, 128, drop=0.1),
        "support_adaptive_500k": _case("support", 3, 500_000, set="adaptive"),
        "assemble_3d_128": _case("assemble", 3, 128, drop=0.1, ops="lap,dx"),
        "moving_3d_75_f64": _case("moving", 3, 75, drop=0.1),
        "export_3d_96_f64": _case("export", 3, 96, drop=0.1),
    }
    return [{**c, "name": name} for name, c in named.items()]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["apply", "apply", "gradient", "adjoint", "rk4", "support", "assemble", "moving", "export"])
    dim = rng.choice([2, 3])
    big = kind in ("apply", "support")
    n = _log_int(rng, 40, 1000 if big else 700) if dim == 2 else _log_int(rng, 16, 120 if big else 90)
    c = _case(kind, dim, n, rng.choice(["f32", "f64"]), drop=rng.choice([0.0, 0.05, 0.1]),
              jitter=rng.uniform(0.02, 0.15), rcut=rng.uniform(3.1, 4.1) if dim == 2 else rng.uniform(2.4, 2.9))
    if kind == "apply":
        c["ops"] = rng.choice(["lap", "dx", "dxx", "lap,dx", "dx,dy", "lap,dx,dy"])
    elif kind == "gradient":
        c["ops"] = "grad"
    elif kind == "assemble":
        c["ops"] = rng.choice(["lap", "dx", "lap,dx", "dx,dy", "dxx,dxy"])
    elif kind == "adjoint":
        c["batch"] = rng.choice([1, 1, 2, 3, 6, 13, 16])
    elif kind == "rk4":
        c["steps"] = rng.randint(1, 20)
    if kind in ("rk4", "support", "assemble", "moving") and dim == 3 and rng.random() < 0.3:
        c.update(set="adaptive", n=_log_int(rng, 20_000, 700_000), rcut=2.4, drop=0.0, jitter=0.1,
                 ratio=rng.uniform(1.5, 4.0))
    elif rng.random() < 0.2:
        c["order"] = "morton"
    if c["ops"] == "lap" and kind in ("adjoint", "moving", "export") and rng.random() < 0.3:
        c["ops"] = "dx"
    return c


# ---- inputs --------------------------------------------------------------------


def _adaptive(n_target, ratio, rng, jitter, rcut):
    """Planes along x, the spacing growing from h0 to ratio * h0; every plane a
    square lattice of its own spacing. y and z are periodic, x is open."""

    def planes(h0):
        out, x = [], 0.5 * h0
        while x < 1.0:
            h = h0 * (1.0 + (ratio - 1.0) * x)
            out.append((x, h, max(int(round(1.0 / h)), 4)))
            x += h
        return out

    lo, hi = 1e-3, 0.1
    for _ in range(40):
        h0 = math.sqrt(lo * hi)
        if sum(m * m for _, _, m in planes(h0)) > n_target:
            lo = h0
        else:
            hi = h0
    made = np.random.default_rng(5)
    shift = rng.random(2)
    pos, hs = [], []
    for x, h, m in planes(h0):
        g = (np.arange(m) + 0.5) / m
        p = np.empty((m * m, 3))
        p[:, 0] = x
        p[:, 1] = np.repeat(g, m)
        p[:, 2] = np.tile(g, m)
        p += made.uniform(-jitter * h, jitter * h, size=p.shape)
        p[:, 1:] = np.mod(p[:, 1:] + shift, 1.0)
        at = np.minimum((p[:, 1:] * m).astype(np.int64), m - 1)
        pos.append(p[np.argsort(at[:, 0] * m + at[:, 1], kind="stable")])
        hs.append(np.full(m * m, h))
    pos, hs = np.concatenate(pos), np.concatenate(hs)
    pad = ratio * h0
    return pos, rcut * hs, [-pad, 0.0, 0.0], [1.0 + pad, 1.0, 1.0], [0, 1, 1], h0


def _morton(pos):
    """Permutation along the Z-order curve over the unit box."""
    q = (np.clip(pos, 0.0, 1.0) * 1023).astype(np.int64)
    code = np.zeros(len(pos), np.int64)
    for b in range(10):
        for d in range(pos.shape[1]):
            code |= ((q[:, d] >> b) & 1) << (b * pos.shape[1] + d)
    return np.argsort(code, kind="stable")


def _points(case, seed):
    """(positions, cut-off or cut-offs, box_lo, box_hi, periodicity, smallest spacing).

    The seed moves one irregular set through its periodic box (and the particles
    in memory with it), so that sets of other seeds have other positions and
    neighbours at every index, and as many of them in all."""
    rng = np.random.default_rng(seed)
    dim, n = case["dim"], case["n"]
    if case["set"] == "adaptive":
        return _adaptive(n, case["ratio"], rng, case["jitter"], case["rcut"])
    h = 1.0 / n
    made = np.random.default_rng(3)
    axes = tuple(range(dim))
    shift = tuple(int(v) for v in rng.integers(0, n, dim))
    g = (np.arange(n) + 0.5) * h
    pos = np.stack(np.meshgrid(*([g] * dim), indexing="ij"), axis=-1)
    if case["jitter"]:
        off = made.uniform(-case["jitter"] * h, case["jitter"] * h, size=pos.shape)
        pos = np.mod(pos + np.roll(off, shift, axes), 1.0)
    pos = pos.reshape(-1, dim)
    if case["drop"]:
        keep = made.random((n,) * dim) >= case["drop"]
        pos = pos[np.roll(keep, shift, axes).ravel()]
    if case["order"] == "morton":
        pos = pos[_morton(pos)]
    return np.ascontiguousarray(pos), case["rcut"] * h, [0.0] * dim, [1.0] * dim, [1] * dim, h


def _field(pos, seed):
    """A smooth periodic field, the phases and amplitudes drawn from the seed."""
    rng = np.random.default_rng(seed + 7)
    f = np.zeros(len(pos))
    for k in (1.0, 2.0, 3.0):
        term = np.full(len(pos), rng.uniform(0.5, 1.0) / k)
        for d in range(pos.shape[1]):
            term *= np.sin(2 * np.pi * (k * pos[:, d] + rng.random()))
        f += term
    return f


def _diffusion(h):
    """(alpha, dt) of a stable explicit step of df/dt = alpha Lap f."""
    return 0.01, 0.02 * h * h / 0.01


def _batch(case, n, seed):
    """(fields, targets) of the loss, N(0, 1)."""
    g = torch.Generator("cuda").manual_seed(seed + 11)
    shape = (case["batch"], n) if case["batch"] > 1 else (n,)
    dt = _DTYPES[case["dtype"]]
    return (torch.randn(shape, generator=g, dtype=dt, device="cuda"),
            torch.randn(shape, generator=g, dtype=dt, device="cuda"))


def prepare(case, seed):
    pos, rcut, lo, hi, bc, h = _points(case, seed)
    kind, dt = case["kind"], _DTYPES[case["dtype"]]
    s = {"kind": kind, "rcut": rcut}
    if kind == "moving":
        # the set one step earlier: the same particles, displaced by a fraction of the spacing
        before = pos + 0.02 * h * np.sin(2 * np.pi * pos[:, ::-1])
        before = np.where(np.array(bc) > 0, np.mod(before, 1.0), before)
        s["now"] = torch.as_tensor(pos, device="cuda")
        s["parts"] = ParticleSet(before, lo, hi, bc=bc)
    else:
        s["parts"] = ParticleSet(pos, lo, hi, bc=bc)
    if np.ndim(rcut):
        s["rcut"] = torch.as_tensor(rcut, device="cuda")
    if kind == "support":
        return s
    parts, rcut = s["parts"], s["rcut"]
    s["list"] = parts.getVerlet(rcut)
    if kind == "gradient":
        s["ops"] = [Gradient(parts, s["list"], 2, rcut)]
    else:
        s["ops"] = [_OPS[o](parts, s["list"], 2, rcut) for o in case["ops"].split(",")]
    if kind == "adjoint":
        s["f"], s["target"] = _batch(case, len(pos), seed)
    elif kind not in ("assemble", "export"):
        s["f"] = torch.as_tensor(_field(pos, seed), dtype=dt, device="cuda")
    if kind == "rk4":
        s["alpha"], s["dt"] = _diffusion(h)
        s["steps"] = case["steps"]
    if kind == "export":
        s["dtype"] = dt
    return s


def _kernels(op):
    d = op.dcpse
    return {"eps": d.localEps, "scale": d.localEpsInvPow, "kernels": d.calcKernels,
            "weights": d.weights(torch.float32), "info": d.info}


def run(state):
    kind = state["kind"]
    if kind == "support":
        vl = state["parts"].getVerlet(state["rcut"])
        return {"row_ptr": vl.row_ptr, "col": vl.col}
    ops = state["ops"]
    if kind == "apply":
        return {"out": [ops[0](state["f"])] if len(ops) == 1 else fused(*ops, f=state["f"])}
    if kind == "gradient":
        return {"out": ops[0](state["f"])}
    if kind == "adjoint":
        f = state["f"].detach().requires_grad_(True)
        y = dcpse_apply(ops[0], f)
        loss = ((y - state["target"]) ** 2).sum()
        return {"out": y.detach(), "grad": torch.autograd.grad(loss, f)[0]}
    if kind == "rk4":
        return {"f": rk4(ops[0], state["f"].clone(), state["dt"], state["steps"], alpha=state["alpha"])}
    if kind == "assemble":
        assemble_together([op.dcpse for op in ops])
        return {"ops": [_kernels(op) for op in ops]}
    if kind == "moving":
        parts = state["parts"]
        parts.set_positions(state["now"])
        vl = parts.updateVerlet(state["list"], state["rcut"])
        ops[0].update(parts)
        return {"row_ptr": vl.row_ptr, "col": vl.col, "kernels": ops[0].dcpse.calcKernels, "out": ops[0](state["f"])}
    if kind == "export":
        row_ptr, col, val = ops[0].export_csr(state["dtype"])
        return {"row_ptr": row_ptr, "col": col, "val": val}
    raise ValueError(kind)


# ---- work ----------------------------------------------------------------------


def _mean_row(case):
    """Mean neighbours of a particle: the lattice offsets inside the cut-off,
    each with the chance that jitter leaves it there."""
    dim, r = case["dim"], case["rcut"]
    k = int(math.ceil(r)) + 1
    off = np.stack([a.ravel() for a in np.meshgrid(*([np.arange(-k, k + 1)] * dim), indexing="ij")], axis=1)
    off = off[np.any(off != 0, axis=1)]
    rng = np.random.default_rng(0)
    j = case["jitter"] * (rng.uniform(-1, 1, (128, 1, dim)) - rng.uniform(-1, 1, (128, 1, dim)))
    inside = np.mean(np.sum((off[None] + j) ** 2, axis=2) < r * r, axis=0)
    return float(inside.sum()) * (1.0 - (case["drop"] if case["set"] == "jittered" else 0.0))


def _signatures(op, dim):
    unit = np.eye(dim, dtype=int)
    return {"dx": [unit[0]], "dy": [unit[1]], "dxx": [2 * unit[0]], "dxy": [unit[0] + unit[1]],
            "lap": [2 * u for u in unit]}[op]


def _operators(case):
    """Signatures of every operator of the case."""
    dim = case["dim"]
    if case["ops"] == "grad":
        return [[u] for u in np.eye(dim, dtype=int)]
    return [_signatures(o, dim) for o in case["ops"].split(",")]


def _basis(order_b, dim):
    """Exponents with 1 (even derivatives) or 0 <= |alpha| < |beta| + 2."""
    top = order_b + 2
    e = np.stack([a.ravel() for a in np.meshgrid(*([np.arange(top)] * dim), indexing="ij")], axis=1)
    s = e.sum(axis=1)
    return e[(s < top) & (s >= (1 if order_b % 2 == 0 else 0))]


def work(case):
    dim, kind = case["dim"], case["kind"]
    n = case["n"] if case["set"] == "adaptive" else case["n"] ** dim * (1.0 - case["drop"])
    nnz = n * _mean_row(case)
    t = 4 if case["dtype"] == "f32" else 8
    ops = _operators(case)
    rows = 8 * (n + 1)
    sup_b, sup_f = 8 * dim * n + rows + 4 * nnz, nnz * 3 * dim
    asm_b = 8 * dim * n + rows + 4 * nnz + len(ops) * (12 * nnz + 20 * n)
    asm_f = 0.0
    for sig in ops:
        m = len(_basis(int(sum(sig[0])), dim))
        # the moments, one factorisation and solve, the weighted polynomial
        moments = math.comb(2 * (int(sum(sig[0])) + 1) + dim, dim)
        asm_f += 2 * nnz * moments + n * (m ** 3 / 3 + 2 * m * m) + 2 * nnz * m
    app_b = nnz * (4 + t * len(ops)) + rows + t * n * (1 + len(ops))
    app_f = nnz * (1 + 2 * len(ops))
    if kind == "support":
        return {"bytes": sup_b, "flops": sup_f}
    if kind == "assemble":
        return {"bytes": asm_b, "flops": asm_f}
    if kind in ("apply", "gradient"):
        return {"bytes": app_b, "flops": app_f}
    if kind == "adjoint":
        b = case["batch"]
        # fields, targets and outputs once; columns and weights for either direction
        return {"bytes": 2 * (nnz * (4 + t) + rows) + 4 * b * t * n, "flops": b * (nnz * 5 + 4 * n)}
    if kind == "rk4":
        return {"bytes": case["steps"] * (4 * (nnz * (4 + t) + rows) + 13 * t * n), "flops": case["steps"] * nnz * 12}
    if kind == "moving":
        return {"bytes": sup_b + asm_b + app_b, "flops": sup_f + asm_f + app_f}
    if kind == "export":
        return {"bytes": nnz * (4 + t) * 2 + 2 * rows + (4 + t) * n, "flops": nnz}
    raise ValueError(kind)


# ---- the same results in 64 bits, in plain torch -------------------------------


def _image(d, k, lo, hi, bc):
    if not bc[k]:
        return d
    box = hi[k] - lo[k]
    return d - box * torch.round(d / box)


def _neighbours(pos, rcut, lo, hi, bc):
    """(row_ptr, col) of every q != p with |x_p - x_q| < rcut_p, ascending."""
    n, dim = pos.shape
    rc = torch.as_tensor(rcut, dtype=torch.float64, device=pos.device)
    rmax, rmin = float(rc.max()), float(rc.min())
    rc = rc.expand(n) if rc.dim() == 0 else rc
    edge = rmax / max(1, min(4, math.ceil(rmax / rmin - 1e-9)))
    nc = [max(1, int((hi[d] - lo[d]) / edge)) for d in range(dim)]
    size = [(hi[d] - lo[d]) / nc[d] for d in range(dim)]
    cell = [torch.clamp(((pos[:, d] - lo[d]) / size[d]).long(), 0, nc[d] - 1) for d in range(dim)]
    key = cell[0]
    for d in range(1, dim):
        key = key * nc[d] + cell[d]
    members = torch.argsort(key, stable=True)
    count = torch.bincount(key, minlength=math.prod(nc))
    start = torch.cumsum(count, 0) - count
    wide = int(count.max())
    reach = [min(int(math.ceil(rmax / size[d])), (nc[d] - 1) // 2 if bc[d] else nc[d]) for d in range(dim)]
    lane = torch.arange(wide, device=pos.device)
    keys = []
    for off in np.ndindex(*[2 * r + 1 for r in reach]):
        off = [o - r for o, r in zip(off, reach)]
        gap = math.sqrt(sum((max(0, abs(o) - 1) * size[d]) ** 2 for d, o in enumerate(off)))
        ok = rc > gap
        other = torch.zeros(n, dtype=torch.long, device=pos.device)
        for d in range(dim):
            c = cell[d] + off[d]
            if bc[d]:
                c = c % nc[d]
            else:
                ok = ok & (c >= 0) & (c < nc[d])
            other = other * nc[d] + torch.clamp(c, 0, nc[d] - 1)
        rows = torch.nonzero(ok).ravel()
        step = max(1, 60_000_000 // wide)
        for i in range(0, len(rows), step):
            p = rows[i:i + step]
            o = other[p]
            have = lane[None, :] < count[o][:, None]
            q = members[torch.clamp(start[o][:, None] + lane[None, :], max=n - 1)]
            d2 = torch.zeros(q.shape, dtype=torch.float64, device=pos.device)
            for d in range(dim):
                d2 += _image(pos[p, d][:, None] - pos[:, d][q], d, lo, hi, bc) ** 2
            take = have & (d2 < (rc[p] ** 2)[:, None]) & (q != p[:, None])
            keys.append((p[:, None] * n + q)[take])
    keys = torch.sort(torch.cat(keys)).values
    row = torch.div(keys, n, rounding_mode="floor")
    row_ptr = torch.zeros(n + 1, dtype=torch.long, device=pos.device)
    row_ptr[1:] = torch.cumsum(torch.bincount(row, minlength=n), 0)
    return row_ptr, keys - row * n


def _padded(row_ptr, a, b):
    """(entries, mask) of rows a .. b - 1 as a rectangle."""
    length = row_ptr[a + 1:b + 1] - row_ptr[a:b]
    lane = torch.arange(int(length.max()), device=row_ptr.device)
    mask = lane[None, :] < length[:, None]
    last = int(row_ptr[-1]) - 1
    return torch.clamp(row_ptr[a:b, None] + lane[None, :], max=last), mask


def _solve(A, b):
    """Solutions of the symmetric positive definite systems A x = b."""
    m = A.shape[-1]
    L = torch.zeros_like(A)
    for k in range(m):
        L[:, k, k] = torch.sqrt(A[:, k, k] - (L[:, k, :k] ** 2).sum(1))
        if k + 1 < m:
            s = A[:, k + 1:, k] - (L[:, k + 1:, :k] * L[:, k:k + 1, :k]).sum(2)
            L[:, k + 1:, k] = s / L[:, k, k][:, None]
    x = b.expand(len(A), m).clone()
    for k in range(m):
        x[:, k] = (x[:, k] - (L[:, k, :k] * x[:, :k]).sum(1)) / L[:, k, k]
    for k in reversed(range(m)):
        x[:, k] = (x[:, k] - (L[:, k + 1:, k] * x[:, k + 1:]).sum(1)) / L[:, k, k]
    return x


def _assembled(pos, row_ptr, col, lo, hi, bc, sigs):
    """eps, eps^-|beta| and kernels K of the operator sum over sigs."""
    n, dim = pos.shape
    border = int(sum(sigs[0]))
    e = _basis(border, dim)
    m = len(e)
    b = torch.zeros(m, dtype=torch.float64, device=pos.device)
    for s in sigs:
        i = int(np.nonzero((e == np.asarray(s)).all(1))[0][0])
        b[i] += (-1.0) ** border * math.prod(math.factorial(int(v)) for v in s)
    eps = torch.empty(n, dtype=torch.float64, device=pos.device)
    K = torch.empty(len(col), dtype=torch.float64, device=pos.device)
    for r0 in range(0, n, 50_000):
        r1 = min(n, r0 + 50_000)
        at, mask = _padded(row_ptr, r0, r1)
        q = col[at]
        z = [_image(pos[r0:r1, d][:, None] - pos[:, d][q], d, lo, hi, bc) for d in range(dim)]
        ep = torch.where(mask, sum(v.abs() for v in z), 0.0).sum(1) / mask.sum(1) / 0.9
        eps[r0:r1] = ep
        z = [v / ep[:, None] for v in z]
        w = torch.where(mask, torch.exp(-sum(v * v for v in z)), 0.0)
        powers = [[torch.ones_like(v)] for v in z]
        for d in range(dim):
            for _ in range(border + 1):
                powers[d].append(powers[d][-1] * z[d])
        V = torch.stack([math.prod(powers[d][int(a[d])] for d in range(dim)) for a in e], dim=2)
        A = torch.bmm((V * w[:, :, None]).transpose(1, 2).contiguous(), V)
        x = _solve(A, b)
        K[at[mask]] = (torch.bmm(V, x[:, :, None])[:, :, 0] * w)[mask]
    return eps, eps ** -border, K


def _difference(row_ptr, col, W, f):
    """sum_q W_pq (f_q - f_p) for fields (..., N)."""
    out = torch.empty(f.shape, dtype=torch.float64, device=f.device)
    n = f.shape[-1]
    for r0 in range(0, n, 400_000):
        r1 = min(n, r0 + 400_000)
        at, mask = _padded(row_ptr, r0, r1)
        w = torch.where(mask, W[at], 0.0)
        q = col[at]
        for g, o in zip(f.reshape(-1, n), out.reshape(-1, n)):
            o[r0:r1] = (w * (g[q] - g[r0:r1, None])).sum(1)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "support":
        return None  # whole numbers
    pos, rcut, lo, hi, bc, h = _points(case, seed)
    n = len(pos)
    dt = _DTYPES[case["dtype"]]
    p = torch.as_tensor(pos, device="cuda")
    rp, col = _neighbours(p, torch.as_tensor(rcut, dtype=torch.float64, device="cuda"), lo, hi, bc)
    asm = [_assembled(p, rp, col, lo, hi, bc, s) for s in _operators(case)]
    row = torch.repeat_interleave(torch.arange(n, device="cuda"), rp[1:] - rp[:-1])
    if kind == "assemble":
        return {"ops": [{"eps": e, "scale": s, "kernels": K, "weights": K * s[row], "info": None} for e, s, K in asm]}
    Ws = [K * s[row] for _, s, K in asm]
    W = Ws[0]
    if kind == "adjoint":
        f, target = (v.double() for v in _batch(case, n, seed))
        y = _difference(rp, col, W, f)
        g = (2.0 * (y - target)).reshape(-1, n)
        grad = torch.empty_like(g)
        for i in range(len(g)):
            back = torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, col, W * g[i][row])
            grad[i] = back - torch.zeros_like(back).index_add_(0, row, W) * g[i]
        return {"out": y, "grad": grad.reshape(f.shape)}
    if kind == "export":
        border = int(sum(_operators(case)[0][0]))
        sign = -1.0 if border % 2 == 0 else 1.0
        diag = sign * torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, row, W)
        at = torch.arange(n, device="cuda")
        order = torch.argsort(torch.cat([row * n + col, at * n + at]))
        return {"row_ptr": None, "col": None, "val": torch.cat([W, diag])[order]}
    f = torch.as_tensor(_field(pos, seed), dtype=dt, device="cuda").double()
    if kind == "apply":
        return {"out": [_difference(rp, col, w, f) for w in Ws]}
    if kind == "gradient":
        return {"out": torch.stack([_difference(rp, col, w, f) for w in Ws])}
    if kind == "moving":
        return {"row_ptr": None, "col": None, "kernels": asm[0][2], "out": _difference(rp, col, W, f)}
    if kind == "rk4":
        alpha, dt_ = _diffusion(h)
        for _ in range(case["steps"]):
            k1 = alpha * _difference(rp, col, W, f)
            k2 = alpha * _difference(rp, col, W, f + 0.5 * dt_ * k1)
            k3 = alpha * _difference(rp, col, W, f + 0.5 * dt_ * k2)
            k4 = alpha * _difference(rp, col, W, f + dt_ * k3)
            f = f + dt_ / 6.0 * (k1 + 2.0 * k2 + 2.0 * k3 + k4)
        return {"f": f}
    raise ValueError(kind)
