"""Reverse-mode differentiation of the mixing path through torch.autograd.

The reference is differentiated by JAX's autodiff of its own code
(veros/core/utilities.py:51-59 and veros/core/isoneutral/diffusion.py:172-207
under ``jax.grad``); here each forward kernel has a hand-written adjoint
kernel in libvxmix.so behind a ``torch.autograd.Function``:

* ``solve_implicit_ad(a, b, c, d, kbot, b_edge=None, d_edge=None)`` — the
  kbot-masked tridiagonal solve, differentiable in a, b, c, d, b_edge and
  d_edge (vx_tdma_adjoint_f64: a transposed Thomas sweep that recomputes the
  elimination factors from a, b, c instead of storing them).
* ``isoneutral_step(state, T_tau, T_taup1, K_iso)`` — one isoneutral tracer
  step (iso=True, energy branch off) with the state's isoneutral tensor held
  fixed, differentiable in T[tau], T[taup1] and K_iso
  (vx_iso_diffusion_adjoint_f64: transposed K33 solve, then the transposed
  flux stencil scattered with float64 atomics).
* ``mixing_step(state, a, b, c, d, T_tau, K_iso, kbot)`` — the two composed
  in one autograd node: the solve's result becomes the tracer's taup1 level on
  the interior.

Forward passes run the same kernels as the non-differentiable API; the TDMA
forward may use the mixed float32 + float64-refinement solve
(``precision="mixed"``), its backward is always float64.
"""
from __future__ import annotations

import torch

from . import _native
from ._arrays import ptr, stream_handle, to_device
from .isoneutral import _check_array, grid_struct, params_struct
from .layout import LEVELS_OUTER
from .utilities import solve_implicit_kbot


def _contig(t):
    return None if t is None else t.contiguous()


def _solve_adjoint(a, b, c, b_edge, d_edge, kbot, x, gx):
    """(ga, gb, gc, gd, gb_edge, gd_edge) of the solve; gx in a's layout."""
    nx, ny, nz = a.shape
    ga, gb, gc, gd = (torch.empty_like(a) for _ in range(4))
    gbe = torch.empty_like(a) if b_edge is not None else None
    gde = torch.empty_like(a) if d_edge is not None else None
    sx, sy, _ = a.stride()
    rc = _native.lib().vx_tdma_adjoint_f64(
        stream_handle(), ptr(a), ptr(b), ptr(c), ptr(b_edge), ptr(d_edge), ptr(kbot), kbot.stride(0),
        kbot.stride(1), ptr(x), ptr(gx), ptr(ga), ptr(gb), ptr(gc), ptr(gd), ptr(gbe), ptr(gde),
        nx, ny, nz, sx, sy)
    _native.check(rc, "vx_tdma_adjoint_f64")
    return ga, gb, gc, gd, gbe, gde


class TdmaSolve(torch.autograd.Function):
    """x = solve_implicit(a, b, c, d) with gradients for a, b, c, d, b_edge, d_edge."""

    @staticmethod
    def forward(ctx, a, b, c, d, b_edge, d_edge, kbot, precision, refine_steps):
        x = solve_implicit_kbot(a, b, c, d, kbot, b_edge=b_edge, d_edge=d_edge, precision=precision,
                                refine_steps=refine_steps)
        ctx.save_for_backward(a, b, c, b_edge, d_edge, kbot, x)
        return x

    @staticmethod
    def backward(ctx, gx):
        return (*_solve_adjoint(*ctx.saved_tensors, gx.contiguous()), None, None, None)


def _solve_operands(*ts):
    for t in ts:
        if t is not None and (not isinstance(t, torch.Tensor) or t.device.type != "cuda"):
            raise TypeError("solve_implicit_ad takes torch tensors on the GPU")
    return [_contig(t) for t in ts]


def solve_implicit_ad(a, b, c, d, kbot, b_edge=None, d_edge=None, *, precision="fp64", refine_steps=1):
    """Differentiable solve_implicit on kbot-masked columns (float64 tensors on the GPU)."""
    a, b, c, d, b_edge, d_edge = _solve_operands(a, b, c, d, b_edge, d_edge)
    kb, _ = to_device(kbot, torch.int32)
    return TdmaSolve.apply(a, b, c, d, b_edge, d_edge, kb.contiguous(), precision, refine_steps)


_TENSOR = ("Ai_ez", "Ai_nz", "Ai_bx", "Ai_by", "K_11", "K_22", "K_33")
# the levels of the two-level tracer buffers below, stored one after another
_TAU, _TAUP1 = 0, 1


def _isoneutral_tensor(vs, X, Y, nz):
    return [_check_array(n, getattr(vs, n), (X, Y, nz, 2, 2) if n.startswith("Ai") else (X, Y, nz)) for n in _TENSOR]


def _step_forward(state, tr, K_iso):
    """One step in place on tr (2, X, Y, nz), levels _TAU and _TAUP1."""
    vs = state.variables
    _, X, Y, nz = tr.shape
    if int(vs.tau) == int(vs.taup1):
        raise ValueError("tau and taup1 must differ")
    keep = []
    g = grid_struct(vs, keep, LEVELS_OUTER)
    p = params_struct(state.settings)
    tensors = _isoneutral_tensor(vs, X, Y, nz)
    dtr = torch.zeros((X, Y, nz), dtype=torch.float64, device=tr.device)
    L = _native.lib()
    ws = torch.empty(L.vx_iso_workspace_bytes(g, 1), dtype=torch.uint8, device=tr.device)
    rc = L.vx_iso_diffusion_f64(stream_handle(), g, p, ptr(tr), _TAU, _TAUP1, ptr(K_iso), *(ptr(t) for t in tensors),
                                ptr(dtr), None, None, ptr(ws))
    _native.check(rc, "isoneutral_step")


def _step_adjoint(state, tr, K_iso, g_new):
    """(dL/dT_tau, dL/dT_taup1, dL/dK_iso) of _step_forward."""
    vs, st = state.variables, state.settings
    X, Y, nz = K_iso.shape
    keep = []
    g = grid_struct(vs, keep, LEVELS_OUTER)
    p = params_struct(st)
    g_new = g_new.contiguous()
    g_tau, g_taup1, g_K = (torch.empty((X, Y, nz), dtype=torch.float64, device=K_iso.device) for _ in range(3))
    L = _native.lib()
    ws = torch.empty(L.vx_iso_adjoint_workspace_bytes(g), dtype=torch.uint8, device=K_iso.device)
    rc = L.vx_iso_diffusion_adjoint_f64(stream_handle(), g, p, ptr(tr), _TAU, ptr(K_iso),
                                        *(ptr(getattr(vs, n)) for n in _TENSOR), ptr(g_new), ptr(g_tau),
                                        ptr(g_taup1), ptr(g_K), ptr(ws))
    _native.check(rc, "isoneutral_step (adjoint)")
    return g_tau, g_taup1, g_K


class _IsoStep(torch.autograd.Function):
    @staticmethod
    def forward(ctx, T_tau, T_taup1, K_iso, state):
        tr = torch.empty((2,) + tuple(K_iso.shape), dtype=torch.float64, device=K_iso.device)
        tr[_TAU].copy_(T_tau)
        tr[_TAUP1].copy_(T_taup1)
        _step_forward(state, tr, K_iso)
        ctx.state = state
        ctx.save_for_backward(tr, K_iso)
        return tr[_TAUP1].clone()

    @staticmethod
    def backward(ctx, g_new):
        tr, K_iso = ctx.saved_tensors
        return (*_step_adjoint(ctx.state, tr, K_iso, g_new), None)


class _MixingStep(torch.autograd.Function):
    """The solve and the step in one node: between them only the solution is
    copied into the tracer's taup1 level (halo from ``base``), and back."""

    @staticmethod
    def forward(ctx, a, b, c, d, b_edge, d_edge, T_tau, K_iso, base, kbot, state, precision, refine_steps):
        x = solve_implicit_kbot(a, b, c, d, kbot, b_edge=b_edge, d_edge=d_edge, precision=precision,
                                refine_steps=refine_steps)
        tr = torch.empty((2,) + tuple(K_iso.shape), dtype=torch.float64, device=K_iso.device)
        tr[_TAU].copy_(T_tau)
        tr[_TAUP1].copy_(base)
        tr[_TAUP1, 2:-2, 2:-2].copy_(x)
        _step_forward(state, tr, K_iso)
        ctx.state = state
        ctx.save_for_backward(a, b, c, b_edge, d_edge, kbot, x, tr, K_iso)
        return tr[_TAUP1].clone()

    @staticmethod
    def backward(ctx, g_new):
        a, b, c, b_edge, d_edge, kbot, x, tr, K_iso = ctx.saved_tensors
        need = ctx.needs_input_grad
        g_tau, g_taup1, g_K = _step_adjoint(ctx.state, tr, K_iso, g_new)
        gs = (None,) * 6
        if any(need[:6]):
            gs = _solve_adjoint(a, b, c, b_edge, d_edge, kbot, x, g_taup1[2:-2, 2:-2].contiguous())
        g_base = None
        if need[8]:
            g_taup1[2:-2, 2:-2] = 0.0
            g_base = g_taup1
        return (*gs, g_tau, g_K, g_base, None, None, None, None)


def _check_step_inputs(state, **tensors):
    shape = tuple(state.variables.K_iso.shape)
    for name, t in tensors.items():
        if not isinstance(t, torch.Tensor) or t.device.type != "cuda" or t.dtype != torch.float64:
            raise TypeError(f"{name} must be a float64 torch tensor on the GPU")
        if tuple(t.shape) != shape:
            raise ValueError(f"{name} must have shape {shape}, got {tuple(t.shape)}")


def isoneutral_step(state, T_tau, T_taup1, K_iso):
    """T_new = tracer[..., taup1] after one isoneutral step of the tracer whose
    levels tau / taup1 are ``T_tau`` / ``T_taup1`` (each (X, Y, nz)), with
    ``K_iso`` in place of the state's and the state's Ai_*, K_11, K_22, K_33
    held fixed (veros/core/isoneutral/diffusion.py:172-207, iso=True, energy
    branch off). Differentiable in T_tau, T_taup1 and K_iso."""
    _check_step_inputs(state, T_tau=T_tau, T_taup1=T_taup1, K_iso=K_iso)
    return _IsoStep.apply(T_tau, T_taup1, K_iso.contiguous(), state)


def mixing_step(state, a, b, c, d, T_tau, K_iso, b_edge=None, d_edge=None, *, precision="fp64",
                refine_steps=1):
    """solve_implicit of d on the interior columns (the state's kbot), whose
    result replaces the interior of the tracer's taup1 level (halo from
    ``state.variables.temp``), then one isoneutral step. Differentiable in
    a, b, c, d, b_edge, d_edge, T_tau and K_iso."""
    vs = state.variables
    a, b, c, d, b_edge, d_edge = _solve_operands(a, b, c, d, b_edge, d_edge)
    base = vs.temp[..., vs.taup1]
    if isinstance(base, torch.Tensor) and not base.is_complex():
        base = base.to(torch.float64)
    _check_step_inputs(state, T_tau=T_tau, T_taup1=base, K_iso=K_iso)
    X, Y, nz = K_iso.shape
    if tuple(a.shape) != (X - 4, Y - 4, nz):
        raise ValueError(f"the systems must have the interior's shape {(X - 4, Y - 4, nz)}, got {tuple(a.shape)}")
    kb, _ = to_device(vs.kbot, torch.int32)
    # the solve's own copy: kbot may change in place before backward
    return _MixingStep.apply(a, b, c, d, b_edge, d_edge, T_tau, K_iso.contiguous(), base, kb[2:-2, 2:-2].clone(),
                             state, precision, refine_steps)
