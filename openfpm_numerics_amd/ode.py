"""Explicit time integration on the device for DC-PSE right-hand sides.

Classic RK4 of df/dt = alpha * D f, the integration the reference runs with
boost::odeint's runge_kutta4 over its vector_dist state
(src/OdeIntegrators/OdeIntegrators.hpp:63-135,
src/OdeIntegrators/tests/OdeIntegratores_base_tests.cpp:478-577). Each stage
is one launch of the library (dcpse_stage_* / dcpse_rk4_*): the operator
gather with the stage's axpys fused into its epilogue, so the state stays in
HBM for the whole integration and a step costs four operator passes.
"""
from __future__ import annotations

import torch

from . import _lib
from . import dcpse as _dcpse_module
from .dcpse import Dcpse
from .particles import capturing

#: Neighbours up to which "auto" stays on the CSR kernel: its eight lanes per
#: row keep a small set busy where the sliced-ELL layouts' one lane does not
#: (FP32, us per stage CSR / "bundle16": 30,000 particles in 3D 4.9 / 8.8, 90,000
#: in 2D 6.6 / 8.2, 131,000 in 2D 9.1 / 8.6; FP64 30,000 5.4 / 7.7, 90,000 8.3 /
#: 8.2)
CSR_MAX = {torch.float32: 3_600_000, torch.float64: 2_600_000}
#: FP64 stages of one call from which "auto" runs on the sliced-ELL copy of a
#: list of at least SELL64_LARGE neighbours, or of a smaller one, whose weights
#: and columns (12 bytes a neighbour on CSR) the 256 MB last-level cache holds.
#: us per stage CSR / "bundle16" and for building the copy: 4M neighbours 11.4 /
#: 9.8, 80; 8.7M 21.1 / 21.7, 100; 15M 32.0 / 28.8, 115; 18M 38.5 / 35.2, 125; 28M
#: 89 / 64, 180; 45M 142 / 112, 240: paid for by some 50, -, 36, 37, 7 and 8
#: stages. A single ``stage`` counts as SELL64_AFTER: it is one of a longer
#: integration, which the caller drives
SELL64_AFTER = 8
SELL64_LARGE = 20_000_000
SELL64_AFTER_SMALL = 40


_NAMES = {"bundle16": "bundle16_", "col16": "col16_", "sell": "sell_", "csr": ""}


def _layout(d: Dcpse, dtype, layout: str, stages: int) -> str:
    """The layout a call of this many stages runs on. In FP64 it follows from
    the list and the call alone, so equal calls give equal bits; only a call
    under graph capture, which may not wait for the copy's counts, runs on CSR
    where the copy is not there."""
    nnz = d.verletList.nnz
    if dtype == torch.float32:
        if layout != "auto":
            return layout
        d._n32["fwd"] += stages - 1
        ready = d._count_apply32("fwd")
    else:
        if layout in _NAMES:
            return "csr" if capturing() and not d.verletList.counted(layout) else layout
        after = SELL64_AFTER if nnz >= SELL64_LARGE else SELL64_AFTER_SMALL
        ready = stages >= max(after, _dcpse_module.SELL_AFTER)
    if not ready or d.verletList.n_rows == 0 or nnz <= CSR_MAX[dtype]:
        return "csr"
    if dtype == torch.float64 and capturing() and not d.sell_ready64():
        return "csr"
    return "bundle16" if d.bundle16_suits() else "col16" if d.col16() is not None else "sell"


def _dcpse(op) -> Dcpse:
    d = op.dcpse if hasattr(op, "dcpse") else op
    if not d.same_set:
        raise ValueError("time integration needs an operator whose support and domain sets are the same")
    return d


def _operator(d: Dcpse, dtype, layout: str):
    """The arrays and counts that describe operator d on a layout, as the library
    takes them after n_rows; held by the caller until the call that uses them has
    been made (inside a graph capture nothing else holds what is built for it)."""
    vl = d.verletList
    if layout == "bundle16":
        bundle, row16, exc_ptr, exc_col, exc_W, ne = d.sell_bundle16(dtype)
        return [vl.row_ptr, vl.sell_slices()[0], row16, bundle, exc_ptr, exc_col, exc_W, ne]
    W = (d.sell_weights if dtype == torch.float32 else d.sell_weights64)
    if layout == "col16":
        c16 = d.col16()
        if c16 is None:
            raise ValueError("too many neighbours of this list do not fit 16-bit columns")
        return [vl.row_ptr, *c16, W()]
    if layout == "sell":
        return [vl.row_ptr, *vl.sell(), W()]
    if layout == "csr":
        return [vl.row_ptr, vl.col, d.weights(dtype)]
    raise ValueError(f"unknown layout {layout!r}")


def _args(held):
    return [x if isinstance(x, int) else _lib.ptr(x) for x in held]


def rk4(op, f: torch.Tensor, dt: float, n_steps: int, alpha: float = 1.0, layout: str = "auto",
        work: torch.Tensor | None = None) -> torch.Tensor:
    """Advances f (N,) in place by n_steps RK4 steps of df/dt = alpha * D f and returns it.

    float32 and float64 state run the kernels of their type on layout "bundle16"
    (sliced-ELL with 16-bit column offsets, the fewest bytes), "col16" (the
    list's 16-bit columns), "sell" (32-bit columns), "csr", or "auto": "csr" up
    to ``CSR_MAX`` neighbours; above, in FP32, the 4 n_steps stage applies count
    towards the operator's ``dcpse.SELL_AFTER`` and run on "bundle16" once it is
    reached (its copy is then built; "col16", then "sell", where too many
    neighbours do not fit, ``dcpse.BUNDLE16_MAX_EXC``), on "csr" before; in FP64
    a call of at least ``SELL64_AFTER`` stages (``SELL64_AFTER_SMALL`` below
    ``SELL64_LARGE`` neighbours, ``dcpse.SELL_AFTER`` if that is larger) runs on
    it, a shorter one on "csr", as does one being captured before the copy was
    built.
    ``work`` (3N of f's dtype) may be passed to avoid an allocation per call.
    """
    d = _dcpse(op)
    vl = d.verletList
    n = vl.n_rows
    if f.dim() != 1 or f.numel() != n or not f.is_contiguous():
        raise ValueError("f must be a contiguous (N,) tensor on the operator's particles")
    if f.dtype not in (torch.float32, torch.float64):
        raise TypeError("state must be float32 or float64")
    if work is None:
        work = torch.empty(3 * n, dtype=f.dtype, device=f.device)
    elif work.numel() < 3 * n or work.dtype != f.dtype or not work.is_contiguous():
        raise ValueError("work must be a contiguous tensor of 3N elements of f's dtype")
    ctx = _lib.context(f.device.index or 0)
    ctx.bind_current_stream()
    layout = _layout(d, f.dtype, layout, 4 * int(n_steps))
    p = _lib.ptr
    t = "f32" if f.dtype == torch.float32 else "f64"
    end = (float(alpha), float(dt), int(n_steps), p(f), p(work))
    held = _operator(d, f.dtype, layout)
    ctx.call(f"dcpse_rk4_{_NAMES[layout]}{t}", n, *_args(held), *end)
    return f


def stage(op, u: torch.Tensor, alpha: float, y_a: torch.Tensor | None, ca: float, out_a: torch.Tensor | None,
          y_b: torch.Tensor | None, cb: float, out_b: torch.Tensor | None, layout: str = "auto"):
    """One fused stage: k = alpha * D u; out_a = y_a + ca k; out_b = y_b + cb k (outputs may be None).

    Layouts as for rk4; "auto" counts one apply towards ``dcpse.SELL_AFTER`` in
    FP32 and runs as a call of ``SELL64_AFTER`` stages in FP64."""
    d = _dcpse(op)
    vl = d.verletList
    ctx = _lib.context(u.device.index or 0)
    ctx.bind_current_stream()
    p = _lib.ptr
    layout = _layout(d, u.dtype, layout, 1 if u.dtype == torch.float32 else SELL64_AFTER)
    t = "f32" if u.dtype == torch.float32 else "f64"
    held = _operator(d, u.dtype, layout)
    ctx.call(f"dcpse_stage_{_NAMES[layout]}{t}", vl.n_rows, *_args(held), p(u), float(alpha), p(y_a), float(ca), p(out_a),
             p(y_b), float(cb), p(out_b))
