"""The work a user of veros_amd has it do, as measurable cases.

A case is one pass through public entry points on one grid:

* ``solve``        ``utilities.solve_implicit_kbot`` (float64 or mixed precision)
* ``solve_masks``  ``utilities.solve_implicit`` with the reference's boolean masks
* ``batch``        ``batched.TdmaBatch.run`` over many grids of different shapes
* ``iso_step``     ``isoneutral.isoneutral_pre_and_diffusion_temp_salt`` (the one call)
* ``iso_calls``    pre, temperature and salinity diffusion, and with ``skew`` the
                   skew diffusion of both and the streamfunction, call by call
* ``vertical``     ``thermodynamics.vertmix_tempsalt`` and
                   ``friction.implicit_vert_friction``
* ``turbulence``   ``turbulence.integrate_{tke,eke,idemix}_kernel``
* ``solve_grad``   ``autodiff.solve_implicit_ad``, forward and backward
* ``step_grad``    ``autodiff.mixing_step``, forward and backward

Grids run from a coarse global model (90x40x15) over 1-degree channels to the
quarter-degree grid 1440x720x80 of the benchmark; depths are even and odd;
``levels`` is the storage of the time-level arrays, ``inner`` (the
reference's) or ``outer`` (veros_amd.layout). The bottom index is uniform in
[kmin, nz] with a land fraction, the vertical spacing grows geometrically
from 10 m, tracers are an exponential thermocline with noise: the recipes of
veros_amd.workloads, made on the GPU.
"""
from __future__ import annotations

import math
import random
from types import SimpleNamespace

import torch

F64 = torch.float64
GRAV, RHO_0 = 9.81, 1024.0
DEG = 6370e3 * math.pi / 180.0
# a linear equation of state's drho/dT, drho/dS
DRHODT, DRHODS = -1.67e-4 * 1024.0, 0.78e-3 * 1024.0
TAU, TAUP1, TAUM1 = 0, 1, 2


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def listed():
    return [
        # one small solve: a regional model's tracer column solve, latency bound
        dict(name="solve_64x64x40", kind="solve", nx=64, ny=64, nz=40, land=0.3, kmin=1, precision="fp64", edges=False),
        # the drop-in call as veros makes it, masks and an edge diagonal, 1-degree grid of odd depth
        dict(name="masks_360x160x45", kind="solve_masks", nx=360, ny=160, nz=45, land=0.25, kmin=1, edges=True),
        # the benchmark's solve: quarter degree, float32 sweeps with float64 refinement
        dict(name="mixed_1440x720x80", kind="solve", nx=1440, ny=720, nz=80, land=0.35, kmin=5, precision="mixed",
             edges=False),
        # many independent sub-domains of uneven shape and depth through one kept plan
        dict(name="batch_32_grids", kind="batch", systems=32, lo=48, hi=480, zlo=15, zhi=100, shapes=1003, land=0.3,
             precision="fp64"),
        # the isoneutral step of a coarse global model in the reference's layout: launches count
        dict(name="iso_90x40x15", kind="iso_step", nx=90, ny=40, nz=15, land=0.3, kmin=1, levels="inner"),
        # a 1-degree channel, the reference's calls one after the other, with the skew (GM) branch
        dict(name="iso_calls_360x160x60", kind="iso_calls", nx=360, ny=160, nz=60, land=0.25, kmin=1, levels="inner",
             skew=True),
        # the benchmark's isoneutral step: quarter degree
        dict(name="iso_1440x720x80", kind="iso_step", nx=1440, ny=720, nz=80, land=0.35, kmin=5, levels="outer"),
        # vertical mixing and friction of the 1-degree channel in the reference's layout
        dict(name="vert_360x160x60", kind="vertical", nx=360, ny=160, nz=60, land=0.25, kmin=1, levels="inner"),
        # and of the quarter-degree grid
        dict(name="vert_1440x720x80", kind="vertical", nx=1440, ny=720, nz=80, land=0.35, kmin=5, levels="outer"),
        # the energy closures on a 1-degree grid of odd depth in the reference's layout
        dict(name="turb_360x160x45", kind="turbulence", nx=360, ny=160, nz=45, land=0.25, kmin=1, levels="inner",
             hor=True),
        # and on the quarter-degree grid
        dict(name="turb_1440x720x80", kind="turbulence", nx=1440, ny=720, nz=80, land=0.35, kmin=5, levels="outer",
             hor=True),
        # the differentiated mixing step, forward and backward, of the 2-degree grid
        dict(name="grad_180x90x40", kind="step_grad", nx=180, ny=90, nz=40, land=0.25, kmin=1, precision="fp64"),
    ]


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve_masks", "batch", "iso_step", "iso_step", "iso_calls", "vertical",
                       "vertical", "turbulence", "turbulence", "solve_grad", "step_grad"])
    if kind == "batch":
        hi = int(round(math.exp(rng.uniform(math.log(64), math.log(480)))))
        return dict(kind=kind, systems=rng.randint(4, 40), lo=max(8, hi // 8), hi=hi, zlo=rng.randint(8, 30),
                    zhi=rng.randint(40, 110), shapes=rng.randint(0, 10 ** 6), land=round(rng.uniform(0.0, 0.5), 2),
                    precision=rng.choice(["fp64", "mixed"]))
    nz = rng.randint(10, 100)
    top = {"solve_grad": 8e6, "step_grad": 3e6, "iso_calls": 2e7}.get(kind, 4e7)
    cells = math.exp(rng.uniform(math.log(4e4), math.log(top)))
    ncol = max(64.0, cells / nz)
    nx = max(8, int(math.sqrt(ncol * math.exp(rng.uniform(0.0, 1.4)))))
    ny = max(8, int(ncol / nx))
    case = dict(kind=kind, nx=nx, ny=ny, nz=nz, land=round(rng.uniform(0.0, 0.45), 2),
                kmin=rng.randint(1, max(1, nz // 2)))
    if kind in ("solve", "solve_grad", "step_grad"):
        case["precision"] = rng.choice(["fp64", "mixed"])
    if kind in ("solve", "solve_masks", "solve_grad"):
        case["edges"] = rng.random() < 0.5
    if kind in ("iso_step", "iso_calls", "vertical", "turbulence"):
        case["levels"] = rng.choice(["inner", "outer"])
    if kind == "iso_calls":
        case["skew"] = rng.random() < 0.5
    if kind == "turbulence":
        case["hor"] = rng.random() < 0.75
    return case


# ---------------------------------------------------------------------------
# inputs, made on the GPU from the seed
# ---------------------------------------------------------------------------

class _Rand:
    def __init__(self, seed):
        self.dev = _device()
        self.g = torch.Generator(device=self.dev)
        self.g.manual_seed(int(seed))

    def u(self, shape, lo=0.0, hi=1.0):
        return torch.rand(shape, generator=self.g, dtype=F64, device=self.dev).mul_(hi - lo).add_(lo)

    def n(self, shape, scale=1.0):
        return torch.randn(shape, generator=self.g, dtype=F64, device=self.dev).mul_(scale)

    def logu(self, shape, lo, hi):
        return self.u(shape, math.log(lo), math.log(hi)).exp_()

    def kbot(self, nx, ny, nz, kmin, land):
        kb = torch.randint(min(kmin, nz), nz + 1, (nx, ny), generator=self.g, device=self.dev, dtype=torch.int32)
        return torch.where(self.u((nx, ny)) < land, torch.zeros_like(kb), kb)


def _dz(nz, top=10.0, bottom=250.0):
    r = (bottom / top) ** (1.0 / max(nz - 1, 1))
    return torch.tensor([top * r ** (nz - 1 - k) for k in range(nz)], dtype=F64, device=_device())


def _solve_inputs(r, nx, ny, nz, land, kmin, edges, kbot=None):
    """Vertical-diffusion systems: a = -dt kappa / dz^2 (c alike with its own kappa), b = 1 - a - c."""
    shape, dz = (nx, ny, nz), _dz(nz)
    a = r.logu(shape, 1e-5, 1e-2).mul_(-3600.0).div_(dz ** 2)
    c = r.logu(shape, 1e-5, 1e-2).mul_(-3600.0).div_(dz ** 2)
    p = SimpleNamespace(a=a, b=1.0 - a - c, c=c, d=r.n(shape), b_edge=None, d_edge=None)
    p.kbot = r.kbot(nx, ny, nz, kmin, land) if kbot is None else kbot
    if edges:
        p.b_edge = 1.0 - c + 0.1 * r.u(shape)
    return p


def _masks(kbot, nz):
    ks = kbot.to(torch.int64)[:, :, None] - 1
    k = torch.arange(nz, device=kbot.device)
    return (ks >= 0) & (k >= ks), (ks >= 0) & (k == ks)


def _cyclic(t):
    t[-2:] = t[2:4].clone()
    t[:2] = t[-4:-2].clone()
    return t


def _levels(t):
    """Three time levels of t, levels innermost."""
    return t[..., None].expand(*t.shape, 3).contiguous()


def _grid(r, case):
    """A cyclic channel with 2-cell halos in degrees; the variables' names are veros's."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    X, Y, dev = nx + 4, ny + 4, _device()
    v = SimpleNamespace(tau=TAU, taup1=TAUP1, taum1=TAUM1)
    dx, dy = 360.0 / nx, min(150.0 / ny, 1.0)
    v.dxt = torch.full((X,), dx * DEG, dtype=F64, device=dev)
    v.dxu = v.dxt.clone()
    v.dyt = torch.full((Y,), dy * DEG, dtype=F64, device=dev)
    v.dyu = v.dyt.clone()
    lat = (torch.arange(Y, dtype=F64, device=dev) - Y / 2) * dy
    v.cost, v.cosu = torch.cos(lat * math.pi / 180.0), torch.cos((lat + dy / 2) * math.pi / 180.0)
    v.dzt = _dz(nz)
    v.dzw = torch.cat([0.5 * (v.dzt[1:] + v.dzt[:-1]), v.dzt[-1:]])
    zw = torch.flip(torch.cumsum(torch.flip(v.dzt, [0]), 0), [0])  # depth of each cell's lower face
    v.zt = -(zw - 0.5 * v.dzt)
    v.kbot = torch.zeros((X, Y), dtype=torch.int32, device=dev)
    v.kbot[2:-2, 2:-2] = r.kbot(nx, ny, nz, case["kmin"], case["land"])
    _cyclic(v.kbot)
    return v


def _settings(case):
    """veros's settings (its defaults where it has them) that the entry points read."""
    return SimpleNamespace(
        nx=case["nx"], ny=case["ny"], nz=case["nz"], dt_tracer=3600.0, dt_mom=3600.0, K_iso_steep=500.0,
        iso_slopec=1e-2, iso_dslope=5e-3, enable_conserve_energy=True, enable_cyclic_x=True, grav=GRAV, rho_0=RHO_0,
        eq_of_state_type=1, drhodT=DRHODT, drhodS=DRHODS, enable_neutral_diffusion=True, enable_skew_diffusion=True,
        alpha_tke=30.0, c_eps=0.7, K_h_tke=2000.0, enable_tke_hor_diffusion=bool(case.get("hor")),
        enable_tke_superbee_advection=False, enable_tke_upwind_advection=False, enable_store_cabbeling_heat=False,
        enable_store_bottom_friction_tke=False, enable_eke=True, enable_idemix=True, eke_c_eps=1.0, alpha_eke=1.0,
        enable_eke_superbee_advection=False, enable_eke_upwind_advection=False, tau_v=86400.0, tau_h=15.0 * 86400.0,
        enable_idemix_hor_diffusion=bool(case.get("hor")), enable_eke_diss_bottom=False,
        enable_eke_diss_surfbot=False, eke_diss_surfbot_frac=1.0, enable_idemix_superbee_advection=False,
        enable_idemix_upwind_advection=False)


def _tracers(r, v, X, Y, nz):
    v.temp = _levels(_cyclic(20.0 * torch.exp(v.zt / 800.0) + r.n((X, Y, nz), 0.1)))
    v.salt = _levels(_cyclic(35.0 + r.n((X, Y, nz), 0.3)))


def _iso_state(r, case):
    v, s = _grid(r, case), _settings(case)
    X, Y, nz = case["nx"] + 4, case["ny"] + 4, case["nz"]
    _tracers(r, v, X, Y, nz)
    v.K_iso = r.u((X, Y, nz), 500.0, 1500.0)
    v.K_gm = r.u((X, Y, nz), 500.0, 1500.0) if case.get("skew") else None
    depth = v.zt.abs().expand(X, Y, nz)
    v.int_drhodT, v.int_drhodS = _levels(depth * DRHODT), _levels(depth * DRHODS)

    def zeros(*more):
        return torch.zeros((X, Y, nz) + more, dtype=F64, device=r.dev)

    for n in ("Ai_ez", "Ai_nz", "Ai_bx", "Ai_by"):
        setattr(v, n, zeros(2, 2))
    for n in ("K_11", "K_22", "K_33", "dtemp_iso", "dsalt_iso", "P_diss_iso"):
        setattr(v, n, zeros())
    if case.get("skew"):
        v.P_diss_skew, v.B1_gm, v.B2_gm = zeros(), zeros(), zeros()
    return SimpleNamespace(variables=v, settings=s)


def _vertical_state(r, case):
    v, s = _grid(r, case), _settings(case)
    X, Y, nz = case["nx"] + 4, case["ny"] + 4, case["nz"]
    _tracers(r, v, X, Y, nz)
    v.kappaH, v.kappaM = r.logu((X, Y, nz), 1e-5, 1e-2), r.logu((X, Y, nz), 1e-5, 1e-2)
    v.forc_temp_surface, v.forc_salt_surface = r.n((X, Y), 1e-5), r.n((X, Y), 1e-6)
    v.u, v.v = r.n((X, Y, nz, 3), 0.1), r.n((X, Y, nz, 3), 0.1)
    v.area_t = v.cost * v.dyt * v.dxt[:, None]
    v.area_v = v.cosu * v.dyu * v.dxt[:, None]
    for n in ("dtemp_vmix", "dsalt_vmix", "du_mix", "dv_mix", "K_diss_v"):
        setattr(v, n, torch.zeros((X, Y, nz), dtype=F64, device=r.dev))
    return SimpleNamespace(variables=v, settings=s)


_TERMS = ("K_diss_v", "P_diss_v", "P_diss_adv", "P_diss_nonlin", "eke_diss_tke", "iw_diss", "K_diss_bot",
          "eke_diss_iw", "K_diss_gm", "K_diss_h", "P_diss_skew", "P_diss_hmix", "P_diss_iso")


def _turbulence_state(r, case):
    v, s = _grid(r, case), _settings(case)
    X, Y, nz = case["nx"] + 4, case["ny"] + 4, case["nz"]
    f3 = (X, Y, nz)
    wet = _masks(v.kbot, nz)[0]
    v.kappaM = r.logu(f3, 1e-5, 1e-2)
    v.tke = r.u(f3 + (3,), 1e-5, 1e-2)
    v.sqrttke = v.tke[..., TAU].sqrt()
    v.mxl = r.u(f3, 1.0, 100.0)
    v.forc_tke_surface = r.n((X, Y), 2e-5)
    v.eke = r.u(f3 + (3,), 1e-4, 1e-2)
    v.sqrteke = v.eke[..., TAU].sqrt()
    v.eke_len = r.u(f3, 1e3, 1e5)
    v.K_gm = r.u(f3, 150.0, 450.0)
    v.E_iw = r.u(f3 + (3,), -1e-5, 1e-3)
    v.dE_iw = torch.zeros((1,), dtype=F64, device=r.dev)  # not touched by the path
    v.c0, v.v0, v.alpha_c = r.u(f3) * wet, r.u(f3, 0.0, 0.5) * wet, r.u(f3, 0.0, 1e-3) * wet
    v.forc_iw_bottom, v.forc_iw_surface = r.u((X, Y), 0.0, 1e-6), r.u((X, Y), 0.0, 1e-6)
    for n in _TERMS:
        setattr(v, n, r.n(f3, 1e-9) * wet)
    v.tke_surf_corr = torch.zeros((X, Y), dtype=F64, device=r.dev)
    v.tke_diss = torch.zeros(f3, dtype=F64, device=r.dev)
    return SimpleNamespace(variables=v, settings=s)


_STATES = {"iso_step": _iso_state, "iso_calls": _iso_state, "vertical": _vertical_state,
           "turbulence": _turbulence_state}


def _batch_shapes(case):
    s = random.Random(case["shapes"])
    return [(s.randint(case["lo"], case["hi"]), s.randint(case["lo"], case["hi"]), s.randint(case["zlo"], case["zhi"]))
            for _ in range(case["systems"])]


def _inputs(case, seed):
    r, kind = _Rand(seed), case["kind"]
    if kind in ("solve", "solve_masks", "solve_grad"):
        p = _solve_inputs(r, case["nx"], case["ny"], case["nz"], case["land"], case["kmin"], case["edges"])
        if kind == "solve_grad":
            p.w = r.n(p.a.shape)
        return p
    if kind == "batch":
        return [_solve_inputs(r, nx, ny, nz, case["land"], 1, False) for nx, ny, nz in _batch_shapes(case)]
    if kind == "step_grad":
        st = _iso_state(r, case)
        st.settings.enable_conserve_energy = False
        kb = st.variables.kbot[2:-2, 2:-2].contiguous()
        p = _solve_inputs(r, case["nx"], case["ny"], case["nz"], 0.0, 1, True, kbot=kb)
        return st, p, r.n(st.variables.K_iso.shape)
    return _STATES[kind](r, case)


# ---------------------------------------------------------------------------
# the framework
# ---------------------------------------------------------------------------

def prepare(case, seed):
    from veros_amd import batched, isoneutral, layout

    kind, data = case["kind"], _inputs(case, seed)
    st = SimpleNamespace(case=case, kind=kind)
    if kind == "solve_masks":
        data.water, data.edge = _masks(data.kbot, case["nz"])
    if kind == "batch":
        sys = [dict(a=p.a, b=p.b, c=p.c, d=p.d, kbot=p.kbot, x=torch.empty_like(p.d)) for p in data]
        st.plan, st.x = batched.TdmaBatch(sys, precision=case["precision"]), [s["x"] for s in sys]
        return st
    if kind == "solve_grad":
        st.leaves = [t.requires_grad_(True) for t in (data.a, data.b, data.c, data.d, data.b_edge) if t is not None]
    if kind == "step_grad":
        st.state, p, st.w = data
        isoneutral.isoneutral_diffusion_pre(st.state)  # the tensor the step holds fixed
        v = st.state.variables
        T = v.temp[..., TAU].contiguous()
        st.leaves = [t.requires_grad_(True) for t in (p.a, p.b, p.c, p.d, T, v.K_iso.clone(), p.b_edge)]
        return st
    if kind in _STATES:
        if case["levels"] == "outer":
            layout.set_state_layout(data, layout.LEVELS_OUTER)
        st.state = data
        return st
    st.p = data
    return st


def run(st):
    from veros_amd import autodiff, friction, isoneutral, thermodynamics, turbulence, utilities

    kind, case = st.kind, st.case
    if kind == "solve":
        p = st.p
        return utilities.solve_implicit_kbot(p.a, p.b, p.c, p.d, p.kbot, b_edge=p.b_edge, precision=case["precision"])
    if kind == "solve_masks":
        p = st.p
        return utilities.solve_implicit(p.a, p.b, p.c, p.d, p.water, p.edge, b_edge=p.b_edge)
    if kind == "batch":
        st.plan.run()
        return st.x
    if kind == "solve_grad":
        p = st.p
        x = autodiff.solve_implicit_ad(p.a, p.b, p.c, p.d, p.kbot, p.b_edge, precision=case["precision"])
        return [x.detach(), *torch.autograd.grad(x, st.leaves, p.w)]
    if kind == "step_grad":
        a, b, c, d, T, K, be = st.leaves
        new = autodiff.mixing_step(st.state, a, b, c, d, T, K, b_edge=be, precision=case["precision"])
        return [new.detach(), *torch.autograd.grad(new, st.leaves, st.w)]
    v = st.state.variables
    if kind == "iso_step":
        isoneutral.isoneutral_pre_and_diffusion_temp_salt(st.state)
        return [v.Ai_ez, v.Ai_nz, v.Ai_bx, v.Ai_by, v.K_11, v.K_22, v.K_33, v.temp, v.salt, v.dtemp_iso, v.dsalt_iso,
                v.P_diss_iso]
    if kind == "iso_calls":
        out = [*isoneutral.isoneutral_diffusion_pre(st.state)]
        isoneutral.isoneutral_diffusion(st.state, v.temp, True)
        isoneutral.isoneutral_diffusion(st.state, v.salt, False)
        out += [v.temp, v.salt, v.dtemp_iso, v.dsalt_iso, v.P_diss_iso]
        if case["skew"]:
            isoneutral.isoneutral_skew_diffusion(st.state, v.temp, True)
            isoneutral.isoneutral_skew_diffusion(st.state, v.salt, False)
            isoneutral.isoneutral_diag_streamfunction(st.state)
            out += [v.P_diss_skew, v.B1_gm, v.B2_gm]
        return out
    if kind == "vertical":
        return [*thermodynamics.vertmix_tempsalt(st.state), *friction.implicit_vert_friction(st.state)]
    t = turbulence.integrate_tke_kernel(st.state)
    e = turbulence.integrate_eke_kernel(st.state)
    # IDEMIX takes the dissipation EKE just formed, as one model step does
    i = turbulence.integrate_idemix_kernel(st.state)
    return [t.tke, t.tke_surf_corr, t.tke_diss, e.eke, e.eke_diss_iw, e.eke_diss_tke, i.E_iw, i.iw_diss]


def work(case):
    """Bytes each input is read and each output written once, wet cells where only they are needed."""
    kind = case["kind"]
    if kind == "batch":
        b = 0.0
        for nx, ny, nz in _batch_shapes(case):
            wet = nx * ny * (1 - case["land"]) * (nz + 1) / 2
            b += 32 * wet + 8.0 * nx * ny * nz + 4.0 * nx * ny
        return {"bytes": b, "flops": b / 3}
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    cells, cols = float(nx) * ny * nz, float(nx) * ny
    wet = cols * (1 - case["land"]) * (nz - (min(case["kmin"], nz) + nz) / 2.0 + 1)
    edge = 8 * cols if case.get("edges") else 0.0  # one diagonal per column
    if kind == "solve":
        return {"bytes": 32 * wet + 8 * cells + 4 * cols + edge, "flops": 12 * wet}
    if kind == "solve_masks":
        return {"bytes": 32 * wet + 8 * cells + cells + edge, "flops": 12 * wet}
    if kind == "solve_grad":  # forward; backward reads a, b, c, x, g and writes the gradients
        grads = 5 if case["edges"] else 4
        return {"bytes": 32 * wet + 8 * cells + 40 * wet + 8 * grads * cells + edge, "flops": 30 * wet}
    # per wet cell: K_iso, T and S at tau, both at taup1 and their tendencies read and written, two
    # int_drhodX, P_diss read and written; per cell: the tensor written
    if kind == "iso_step":
        return {"bytes": 120 * wet + 152 * cells + 4 * cols, "flops": 900 * wet}
    if kind == "iso_calls":  # each tracer reads the tensor again
        b = (24 * wet + 152 * cells) + 2 * (152 + 64) * wet
        if case["skew"]:
            b += 2 * (144 + 64) * wet + 72 * wet + 16 * cells
        return {"bytes": b, "flops": (1400 if case["skew"] else 1100) * wet}
    if kind == "vertical":  # kappaH, T, S in; T, S, tendencies out; kappaM, u, v, tendencies, dissipation
        return {"bytes": 40 * wet + 16 * cells + 40 * wet + 32 * cells + 16 * cells, "flops": 120 * wet}
    if kind == "turbulence":
        # TKE: kappaM, sqrttke, mxl, 7 terms, tau in; EKE: kappaM, sqrteke, eke_len, K_gm, 5 terms, tau;
        # IDEMIX: c0, v0, alpha_c, 2 terms, tau; the energy on wet cells and the diagnostics out
        return {"bytes": (88 + 80 + 48 + 24) * wet + 32 * cells, "flops": 300 * wet}
    # step_grad: solve and its adjoint (5 gradients), the step and its adjoint (tensor read twice)
    return {"bytes": 72 * wet + 48 * cells + 2 * 152 * wet + 10 * 8 * cells, "flops": 400 * wet}


# ---------------------------------------------------------------------------
# the same results from plain torch in float64
# ---------------------------------------------------------------------------

def _shift(t, di, dj, dk):
    """t at (i + di, j + dj, k + dk); the wrapped edges are never used."""
    return torch.roll(t, (-di, -dj, -dk), (0, 1, 2))


def _thomas(a, b, c, d, kbot, b_edge=None, d_edge=None):
    """The masked systems' solution, 0 off the wet levels, by sweeps along z."""
    nz = a.shape[2]
    water, edge = _masks(kbot, nz)
    zero, one = torch.zeros((), dtype=F64, device=a.device), torch.ones((), dtype=F64, device=a.device)
    b = b if b_edge is None else torch.where(edge, b_edge, b)
    d = d if d_edge is None else torch.where(edge, d_edge, d)
    a, b = torch.where(water & ~edge, a, zero), torch.where(water, b, one)
    c, d = torch.where(water, c, zero), torch.where(water, d, zero)
    cp, dp = [], []
    for k in range(nz):
        up = c[..., k] if k < nz - 1 else torch.zeros_like(c[..., k])
        den = b[..., k] - (a[..., k] * cp[-1] if k else 0.0)
        cp.append(up / den)
        dp.append((d[..., k] - (a[..., k] * dp[-1] if k else 0.0)) / den)
    x = [dp[-1]]
    for k in range(nz - 2, -1, -1):
        x.append(dp[k] - cp[k] * x[-1])
    return torch.where(water, torch.stack(x[::-1], -1), zero)


def _wet(v, nz):
    return _masks(v.kbot, nz)[0].to(F64)


def _set_top(t, value):
    t = t.clone()
    t[..., -1] = value
    return t


def _iso_tensor(v, s):
    """Ai_ez, Ai_nz, Ai_bx, Ai_by, K_11, K_22, K_33 from T, S at tau and K_iso."""
    X, Y, nz = v.K_iso.shape
    T, S, K, m = v.temp[..., TAU], v.salt[..., TAU], v.K_iso, _wet(v, v.K_iso.shape[2])
    rho = s.drhodT * T + s.drhodS * S  # linear: density gradients are gradients of this
    mU, mV = m * _shift(m, 1, 0, 0), m * _shift(m, 0, 1, 0)
    mW = _set_top(m * _shift(m, 0, 0, 1), 0.0)
    rx = mU * (_shift(rho, 1, 0, 0) - rho) / (v.dxu[:, None, None] * v.cost[None, :, None])
    ry = mV * (_shift(rho, 0, 1, 0) - rho) / v.dyu[None, :, None]
    rz = mW * (_shift(rho, 0, 0, 1) - rho) / v.dzw

    def slope(num, den):
        sl = -num / (torch.clamp(den, max=0.0) - 1e-20)
        return sl, 0.5 * (1.0 + torch.tanh((s.iso_slopec - sl.abs()) / s.iso_dslope))

    outs = []
    for di, dj, mask, r, cols in ((1, 0, mU, rx, (slice(1, X - 2), slice(2, Y - 2))),
                                  (0, 1, mV, ry, (slice(2, X - 2), slice(1, Y - 2)))):
        dl = K + _shift(K, di, dj, 0)
        lower = dl[..., :1]
        dl = torch.cat([0.5 * lower, 0.25 * (dl[..., 1:] + dl[..., :-1])], -1)
        A, acc = torch.zeros((X, Y, nz, 2, 2), dtype=F64, device=K.device), torch.zeros_like(K)
        for kr in (0, 1):
            lo = 1 - kr
            dz = v.dzw if kr else torch.roll(v.dzw, 1)
            for ip in (0, 1):
                mp = _shift(m, ip * di, ip * dj, 0)
                sl, t = slope(mp * r, mp * _shift(rz, ip * di, ip * dj, kr - 1))
                acc[..., lo:] += (dz * mask * torch.clamp(dl * t, min=s.K_iso_steep))[..., lo:]
                A[cols[0], cols[1], lo:, ip, kr] = (t * sl * mask)[cols[0], cols[1], lo:]
        Kd = torch.zeros_like(K)
        Kd[cols] = (acc / (4.0 * v.dzt))[cols]
        outs.append((A, Kd))
    inner = (slice(2, X - 2), slice(2, Y - 2), slice(0, nz - 1))
    K33, tops = torch.zeros_like(K), []
    for di, dj, r, w, den in ((1, 0, rx, v.dxu[:, None, None].expand(X, Y, 1), 4 * v.dxt[:, None, None]),
                              (0, 1, ry, (v.cosu * v.dyu)[None, :, None].expand(X, Y, 1),
                               (4 * v.dyt * v.cost)[None, :, None])):
        B, acc = torch.zeros((X, Y, nz, 2, 2), dtype=F64, device=K.device), torch.zeros_like(K)
        for kr in (0, 1):
            mk = _shift(m, 0, 0, kr)
            for ip in (0, 1):
                g = _shift(r, (ip - 1) * di, (ip - 1) * dj, kr)
                sl, t = slope(mk * g, mk * rz)
                acc += _shift(w, (ip - 1) * di, (ip - 1) * dj, 0) * K * t * sl ** 2 * mW
                B[inner + (ip, kr)] = (t * sl * mW)[inner]
        K33[inner] += (acc / den)[inner]
        tops.append(B)
    (ez, k11), (nz_, k22) = outs
    return ez, nz_, tops[0], tops[1], k11, k22, K33


def _fluxes(v, tensor, T, K1, K2):
    """East, north and top fluxes of T; K1 for the lateral faces, K2 for the top ones."""
    ez, nz_, bx, by, k11, k22, _ = tensor
    X, Y, nz = T.shape

    def kshift(t, n):  # clamped along z
        if n == 0:
            return t
        return torch.cat([t[..., 1:], t[..., -1:]], -1) if n > 0 else torch.cat([t[..., :1], t[..., :-1]], -1)

    out = []
    for di, dj, A, Kd, met, scale, cols in (
            (1, 0, ez, k11, v.dxu[:, None, None] * v.cost[None, :, None], 1.0, (slice(1, X - 2), slice(2, Y - 2))),
            (0, 1, nz_, k22, v.dyu[None, :, None], v.cosu[None, :, None], (slice(2, X - 2), slice(1, Y - 2)))):
        dl = K1 + _shift(K1, di, dj, 0)
        dl = torch.cat([0.5 * dl[..., :1], 0.25 * (dl[..., 1:] + dl[..., :-1])], -1)
        acc = 0.0
        for kr in (0, 1):
            for ip in (0, 1):
                t = _shift(T, ip * di, ip * dj, 0)
                acc = acc + dl * A[..., ip, kr] * (kshift(t, kr) - kshift(t, kr - 1))
        full = scale * (acc / (4.0 * v.dzt) + (_shift(T, di, dj, 0) - T) / met * Kd)
        keep = torch.zeros((X, Y, 1), dtype=F64, device=T.device)
        keep[cols] = 1.0
        out.append(full * keep)
    ft = 0.0
    for di, dj, B, w, den in ((1, 0, bx, (1.0 / v.cost)[None, :, None].expand(X, Y, 1), 4 * v.dxt[:, None, None]),
                              (0, 1, by, v.cosu[None, :, None].expand(X, Y, 1),
                               (4 * v.dyt * v.cost)[None, :, None])):
        for kr in (0, 1):
            for ip in (0, 1):
                hi = _shift(T, ip * di, ip * dj, kr)
                lo = _shift(T, (ip - 1) * di, (ip - 1) * dj, kr)
                wt = _shift(w, 0, (ip - 1) * dj, 0)
                ft = ft + K2 * B[..., ip, kr] * wt * (hi - lo) / den
    keep = torch.zeros((X, Y, nz), dtype=F64, device=T.device)
    keep[2:-2, 2:-2, :-1] = 1.0
    return out[0], out[1], ft * keep


def _iso_step(v, s, tensor, T0, T1, K, iso):
    """(T[taup1] after one step, the tendency's increment, the fluxes)."""
    fe, fn, ft = _fluxes(v, tensor, T0, K if iso else -K, K)
    m = _wet(v, T0.shape[2])
    below = torch.cat([torch.zeros_like(ft[..., :1]), ft[..., :-1]], -1)
    cost = v.cost[None, :, None]
    div = m * ((fe - _shift(fe, -1, 0, 0)) / (cost * v.dxt[:, None, None])
               + (fn - _shift(fn, 0, -1, 0)) / (cost * v.dyt[None, :, None]) + (ft - below) / v.dzt)
    core = torch.zeros(T0.shape[:2] + (1,), dtype=F64, device=T0.device)
    core[2:-2, 2:-2] = 1.0
    div = div * core
    new = T1 + s.dt_tracer * div
    if not iso:
        return new, div, (fe, fn, ft)
    dl = s.dt_tracer / v.dzw * _set_top(tensor[6], 0.0)
    dlm = torch.cat([torch.zeros_like(dl[..., :1]), dl[..., :-1]], -1)
    kb = torch.zeros_like(v.kbot)
    kb[2:-2, 2:-2] = v.kbot[2:-2, 2:-2]
    sol = _thomas(-dlm / v.dzt, 1 + (dl + dlm) / v.dzt, -dl / v.dzt, new, kb, b_edge=1 + dl / v.dzt)
    sol = torch.where(_masks(kb, T0.shape[2])[0], sol, new)
    return sol, div + (sol - new) / s.dt_tracer, (fe, fn, ft)


def _dissipation(v, s, I, fluxes, tensor, new, iso):
    """What one tracer's step adds to P_diss."""
    fe, fn, ft = fluxes
    X, Y, nz = I.shape
    g = 0.5 * s.grav / s.rho_0
    Ix, Iy = (_shift(I, 1, 0, 0) - I) * fe, (_shift(I, 0, 1, 0) - I) * fn
    d = (g * (Ix + _shift(I - _shift(I, -1, 0, 0), 0, 0, 0) * _shift(fe, -1, 0, 0)) / (v.dxt[:, None, None]
         * v.cost[None, :, None]) + g * (Iy + (I - _shift(I, 0, -1, 0)) * _shift(fn, 0, -1, 0))
         / (v.dyt * v.cost)[None, :, None])
    ring = torch.zeros((X, Y, 1), dtype=F64, device=I.device)
    ring[1:-1, 1:-1] = 1.0
    d = d * ring
    water, edge = _masks(v.kbot, nz)
    dzl = torch.cat([v.dzw[:1], v.dzw[:-1]])
    avg = 0.5 * (d + _shift(d, 0, 0, 1))
    w = avg * water + 0.5 * d * dzl / v.dzw * edge
    w[..., -1] = (d * water)[..., -1]
    m = _wet(v, nz)
    mW = _set_top(m * _shift(m, 0, 0, 1), 0.0)
    core = torch.zeros((X, Y, 1), dtype=F64, device=I.device)
    core[2:-2, 2:-2] = 1.0
    flux = ft + (tensor[6] * (_shift(new, 0, 0, 1) - new) / v.dzw if iso else 0.0)
    return w - s.grav / s.rho_0 * (I - _shift(I, 0, 0, 1)) / v.dzw * flux * mW * core


def _with_level(t, value, lev=TAUP1):
    t = t.clone()
    t[..., lev] = value
    return t


def _exact_iso(case, st):
    v, s = st.variables, st.settings
    tensor = _iso_tensor(v, s)
    P, res = 0.0, {}
    for n, I in (("temp", v.int_drhodT), ("salt", v.int_drhodS)):
        f = getattr(v, n)
        new, dtr, fl = _iso_step(v, s, tensor, f[..., TAU], f[..., TAUP1], v.K_iso, True)
        P = P + _dissipation(v, s, I[..., TAU], fl, tensor, new, True)
        res[n], res["d" + n] = new, dtr
    out = [*tensor]
    if case["kind"] == "iso_calls" and case["skew"]:
        Q, K = 0.0, v.K_gm
        for n, I in (("temp", v.int_drhodT), ("salt", v.int_drhodS)):
            f = getattr(v, n)
            new, dtr, fl = _iso_step(v, s, tensor, f[..., TAU], res[n], K, False)
            Q = Q + _dissipation(v, s, I[..., TAU], fl, tensor, new, False)
            res[n], res["d" + n] = new, res["d" + n] + dtr
        B = []
        X, Y, _ = K.shape
        Kb = torch.cat([K[..., :1], K[..., :-1]], -1)
        for di, dj, A, sign, cols in ((0, 1, tensor[1], -1.0, (slice(2, X - 2), slice(1, Y - 2))),
                                      (1, 0, tensor[0], 1.0, (slice(1, X - 2), slice(2, Y - 2)))):
            f = torch.zeros_like(K)
            full = sign * 0.0625 * (K + Kb + _shift(K, di, dj, 0) + _shift(Kb, di, dj, 0)) * A.sum((3, 4))
            f[cols] = full[cols]
            B.append(f)
        more = [Q, B[0], B[1]]
    else:
        more = []
    out += [_with_level(v.temp, res["temp"]), _with_level(v.salt, res["salt"]), res["dtemp"], res["dsalt"], P]
    return out + more


def _exact_vertical(st):
    v, s = st.variables, st.settings
    X, Y, nz = v.kappaH.shape
    dt, res = s.dt_tracer, []
    kb = torch.zeros_like(v.kbot)
    kb[2:-2, 2:-2] = v.kbot[2:-2, 2:-2]
    dl = dt / v.dzw * _set_top(v.kappaH, 0.0)
    dlm = torch.cat([torch.zeros_like(dl[..., :1]), dl[..., :-1]], -1)
    for n in ("temp", "salt"):
        old = getattr(v, n)[..., TAUP1]
        d = _set_top(old, old[..., -1] + dt * getattr(v, "forc_%s_surface" % n) / v.dzt[-1])
        sol = _thomas(-dlm / v.dzt, 1 + (dl + dlm) / v.dzt, -dl / v.dzt, d, kb, b_edge=1 + dl / v.dzt)
        new = torch.where(_masks(kb, nz)[0], sol, old)
        res += [(new - old) / dt, _with_level(getattr(v, n), _cyclic(new.clone()))]
    dt, K, m, out, dm = s.dt_mom, torch.zeros_like(v.kappaM), _wet(v, nz), [], []
    faces = (slice(1, X - 2), slice(1, Y - 2))
    for n, di, dj in (("u", 1, 0), ("v", 0, 1)):
        f = getattr(v, n)
        kss = torch.zeros_like(v.kbot)
        kss[faces] = torch.maximum(v.kbot, torch.roll(v.kbot, (-di, -dj), (0, 1)))[faces]
        mf = m * _shift(m, di, dj, 0)
        fxa = 0.5 * (v.kappaM + _shift(v.kappaM, di, dj, 0))
        mw = _set_top(mf * _shift(mf, 0, 0, 1), 0.0)
        dl = dt / v.dzw * fxa * mw
        dlm = torch.cat([torch.zeros_like(dl[..., :1]), dl[..., :-1]], -1)
        sol = _thomas(-dlm / v.dzt, 1 + (dl + dlm) / v.dzt, -dl / v.dzt, f[..., TAU], kss, b_edge=1 + dl / v.dzt)
        new = torch.where(_masks(kss, nz)[0], sol, f[..., TAUP1])
        tend = torch.zeros_like(K)
        tend[faces] = ((new - f[..., TAU]) / dt)[faces]
        old = f[..., TAU]
        full = (_shift(old, 0, 0, 1) - old) * fxa * (_shift(new, 0, 0, 1) - new) * mw / v.dzw ** 2
        ds = torch.zeros_like(K)
        ds[faces] = full[faces]
        t = ds.clone()
        if di:
            t[2:-2] = ((v.dxu[:, None, None] * ds + _shift(v.dxu[:, None, None] * ds, -1, 0, 0))
                       / (2 * v.dxt[:, None, None]))[2:-2]
        else:
            w = v.area_v[:, :, None] * ds
            t[:, 2:-2] = ((w + _shift(w, 0, -1, 0)) / (2 * v.area_t[:, :, None]))[:, 2:-2]
        K = K + t
        out.append(_with_level(f, new))
        dm.append(tend)
    return res + out + dm + [K]


def _lateral(v, F, coef, nz):
    m = _wet(v, nz)
    fe = coef(1, 0) * (_shift(F, 1, 0, 0) - F) / (v.cost[None, :, None] * v.dxu[:, None, None]) * m * _shift(m, 1, 0, 0)
    fn = (coef(0, 1) * (_shift(F, 0, 1, 0) - F) / v.dyu[None, :, None] * m * _shift(m, 0, 1, 0)
          * v.cosu[None, :, None])
    cost = v.cost[None, :, None]
    div = m * ((fe - _shift(fe, -1, 0, 0)) / (cost * v.dxt[:, None, None])
               + (fn - _shift(fn, 0, -1, 0)) / (cost * v.dyt[None, :, None]))
    core = torch.zeros(F.shape[:2] + (1,), dtype=F64, device=F.device)
    core[2:-2, 2:-2] = 1.0
    return div * core


def _energy_solve(v, kap, diss, rhs, old, dt_scale, dt_bottom=None, kmul=None):
    """The energies' vertical system: half cells at the top, diffusivity kap * dt_scale between levels."""
    nz = kap.shape[2]
    kb = torch.zeros_like(v.kbot)
    kb[2:-2, 2:-2] = v.kbot[2:-2, 2:-2]
    dzl = torch.cat([v.dzt[1:], v.dzt[-1:]])
    dl = _set_top(dt_scale / dzl * 0.5 * (kap + _shift(kap, 0, 0, 1)), 0.0)
    dlm = torch.cat([torch.zeros_like(dl[..., :1]), dl[..., :-1]], -1)
    k0, kp, km = (1.0, 1.0, 1.0) if kmul is None else (kmul, _shift(kmul, 0, 0, 1), _shift(kmul, 0, 0, -1))
    dz = v.dzw.clone()
    dz[-1] *= 0.5
    edge = rhs if dt_bottom is None else rhs + dt_bottom / v.dzw
    sol = _thomas(-dlm * km / dz, 1 + (dl + dlm) * k0 / dz + diss, -dl * kp / dz, rhs, kb,
                  b_edge=1 + dl / v.dzw * k0 + diss, d_edge=edge)
    return torch.where(_masks(kb, nz)[0], sol, old)


def _exact_turbulence(st):
    v, s = st.variables, st.settings
    nz, dt = v.kappaM.shape[2], s.dt_mom
    f = (v.K_diss_v - v.P_diss_v - v.P_diss_adv - v.P_diss_nonlin + v.eke_diss_tke + v.iw_diss)
    rate = s.c_eps / v.mxl * v.sqrttke
    rhs = v.tke[..., TAU] + dt * f
    rhs = _set_top(rhs, rhs[..., -1] + dt * v.forc_tke_surface / (0.5 * v.dzw[-1]))
    new = _energy_solve(v, v.kappaM, dt * rate, rhs, v.tke[..., TAUP1], dt * s.alpha_tke)
    diss = rate * new
    top, corr = new[2:-2, 2:-2, -1], torch.zeros_like(v.tke_surf_corr)
    corr[2:-2, 2:-2] = torch.where(top < 0, -top * 0.5 * v.dzw[-1] / dt, torch.zeros_like(top))
    new[2:-2, 2:-2, -1] = torch.clamp(top, min=0.0)
    if s.enable_tke_hor_diffusion:
        new = new + dt * _lateral(v, v.tke[..., TAU], lambda di, dj: s.K_h_tke, nz)
    out = [_with_level(v.tke, new), corr, diss]
    dt = s.dt_tracer
    f = v.K_diss_gm + v.K_diss_h - v.P_diss_skew - v.P_diss_hmix - v.P_diss_iso
    rate = s.eke_c_eps * v.sqrteke / v.eke_len * _wet(v, nz)
    new = _energy_solve(v, v.kappaM, dt * rate, v.eke[..., TAU] + dt * f, v.eke[..., TAUP1], dt * s.alpha_eke)
    iw = rate * new
    new = new + dt * _lateral(v, v.eke[..., TAU],
                              lambda di, dj: 0.5 * torch.clamp(v.K_gm + _shift(v.K_gm, di, dj, 0), min=500.0), nz)
    out += [_with_level(v.eke, new), iw, torch.zeros_like(iw)]
    E = v.E_iw[..., TAU]
    rate = v.alpha_c * torch.clamp(E, min=0.0)
    rhs = E + dt * (iw + v.K_diss_bot)
    top = rhs[..., -1] + dt * v.forc_iw_surface / (0.5 * v.dzw[-1])
    one = v.kbot == nz  # a single wet level takes the bottom flux in place of the surface's
    bottom = dt * v.forc_iw_bottom[..., None]
    new = _energy_solve(v, v.c0, dt * rate, _set_top(rhs, torch.where(one, rhs[..., -1], top)),
                        v.E_iw[..., TAUP1], dt * s.tau_v, dt_bottom=bottom, kmul=v.c0)
    iw_diss = rate * new
    if s.enable_idemix_hor_diffusion:
        new = new + dt * _lateral(v, v.v0 * E, lambda di, dj: s.tau_h * 0.5 * (v.v0 + _shift(v.v0, di, dj, 0)), nz)
    return out + [_with_level(v.E_iw, new), iw_diss]


def exact(case, seed):
    kind, data = case["kind"], _inputs(case, seed)
    if kind in ("solve", "solve_masks"):
        return _thomas(data.a, data.b, data.c, data.d, data.kbot, b_edge=data.b_edge)
    if kind == "batch":
        return [_thomas(p.a, p.b, p.c, p.d, p.kbot) for p in data]
    if kind == "solve_grad":
        leaves = [t.requires_grad_(True) for t in (data.a, data.b, data.c, data.d, data.b_edge) if t is not None]
        x = _thomas(data.a, data.b, data.c, data.d, data.kbot, b_edge=data.b_edge)
        return [x.detach(), *torch.autograd.grad(x, leaves, data.w)]
    if kind == "step_grad":
        st, p, w = data
        v = st.variables
        tensor = _iso_tensor(v, st.settings)
        T, K = v.temp[..., TAU].contiguous(), v.K_iso.clone()
        leaves = [t.requires_grad_(True) for t in (p.a, p.b, p.c, p.d, T, K, p.b_edge)]
        x = _thomas(p.a, p.b, p.c, p.d, p.kbot, b_edge=p.b_edge)
        T1 = v.temp[..., TAUP1].clone()
        T1[2:-2, 2:-2] = x
        new = _iso_step(v, st.settings, tensor, T, T1, K, True)[0]
        return [new.detach(), *torch.autograd.grad(new, leaves, w)]
    if kind == "vertical":
        return _exact_vertical(data)
    if kind == "turbulence":
        return _exact_turbulence(data)
    return _exact_iso(case, data)
