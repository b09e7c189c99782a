"""The adjoint kernels over their range of depths: the solve's at depths either
side of every number of levels per lane, in each storage that the entry point
takes, and the isoneutral step's, two columns of its gradients against unit
perturbations of the oracle (exact: the step is affine in each input)."""
import numpy as np
import pytest
import torch

import test_gpu_adjoint as TA
from conftest import rel_err
from oracle import adjoint as OA
from oracle import tdma as OT
from veros_amd import workloads as W

pytestmark = pytest.mark.gpu


def _strided(a, form):
    """a's values on the GPU: rows apart, columns with spare levels, or 8 bytes off 16-byte alignment."""
    nx, ny, nz = a.shape
    if form == "offset":
        w = torch.zeros(a.size + 1, dtype=torch.float64, device="cuda")[1:].view(a.shape)
    elif form == "interior":
        w = torch.zeros((nx + 4, ny + 4, nz), dtype=torch.float64, device="cuda")[2:-2, 2:-2]
    else:
        w = torch.zeros((nx, ny, nz + 3), dtype=torch.float64, device="cuda")[..., :nz]
    w.copy_(torch.from_numpy(a))
    return w


@pytest.mark.parametrize("nz", [1, 2, 9, 16, 17, 33, 47, 64, 65, 97, 112, 128])
@pytest.mark.parametrize("form", ["offset", "interior", "padded"])
def test_solve_adjoint_depths_and_strides(nz, form):
    from veros_amd import _native
    from veros_amd._arrays import ptr, stream_handle
    rng = np.random.default_rng(nz)
    p = W.diffusion_tdma(rng, 13, 11, nz, dz=W.geometric_dz(nz, 10.0, 500.0), land_frac=0.2, independent_ac=True,
                         with_b_edge=True, with_d_edge=True)
    p.kbot[0, 0], p.kbot[-1, -1] = 1, nz
    gx = rng.standard_normal(p.a.shape)
    x = OT.solve_implicit_kbot(p.a, p.b, p.c, p.d, p.kbot, b_edge=p.b_edge, d_edge=p.d_edge, solver="dense")
    ins = [_strided(v, form) for v in (p.a, p.b, p.c, p.b_edge, p.d_edge, x, gx)]
    outs = [_strided(np.full(p.a.shape, 7.0), form) for _ in range(6)]
    a, b, c, be, de, xt, g = (ptr(t) for t in ins)
    kb = torch.from_numpy(p.kbot).cuda()
    sx, sy, _ = ins[0].stride()
    _native.check(_native.lib().vx_tdma_adjoint_f64(stream_handle(), a, b, c, be, de, ptr(kb), *kb.stride(), xt, g,
                                                    *(ptr(t) for t in outs), 13, 11, nz, sx, sy), "adjoint")
    ref = OA.tdma_vjp(p.a, p.b, p.c, p.kbot, x, gx, b_edge=p.b_edge, d_edge=p.d_edge)  # a, b, c, d, b_edge, d_edge
    for name, t, r in zip(("a", "b", "c", "d", "b_edge", "d_edge"), outs, ref):
        assert rel_err(t.cpu().numpy(), r) <= 1e-12, name
    for t in outs:  # nothing beside the columns is written
        t.zero_()
        assert torch.count_nonzero(t._base) == 0


@pytest.mark.parametrize("nz", [9, 16, 17, 33, 65, 97, 128])
def test_step_adjoint_depths(nz):
    from veros_amd.autodiff import isoneutral_step
    from veros_amd.state import to_device_state
    st, rng = TA._iso_state(nz, 4, 3, nz, cyclic=False)
    vs = st.variables
    T0, K = vs.temp[..., vs.tau].copy(), vs.K_iso.copy()
    T1, g = (rng.standard_normal(K.shape) for _ in range(2))
    t0, t1, k = TA._t(T0, True), TA._t(T1, True), TA._t(K, True)
    isoneutral_step(to_device_state(st), t0, t1, k).backward(TA._t(g))
    zero = np.zeros_like(T1)
    base = float(np.sum(g * OA.iso_step(st, T0, zero, K)))
    wet = np.argwhere(vs.kbot[2:-2, 2:-2] > 0) + 2
    deep = min(wet.tolist(), key=lambda c: vs.kbot[c[0], c[1]])
    for i, j in (deep, (deep[0] - 1, deep[1])):
        ref = np.zeros((3, nz))
        for lev in range(nz):
            for q, x in enumerate((T0, zero, K)):
                h = max(float(np.max(np.abs(x))), 1.0)
                xp = x.copy()
                xp[i, j, lev] += h
                args = [T0, zero, K]
                args[q] = xp
                ref[q, lev] = (float(np.sum(g * OA.iso_step(st, *args))) - base) / h
        for name, t, r in (("T_tau", t0, ref[0]), ("T_taup1", t1, ref[1]), ("K_iso", k, ref[2])):
            scale = float(t.grad.abs().max())
            assert np.abs(t.grad[i, j].cpu().numpy() - r).max() <= 1e-10 * scale, (name, i, j)
