"""Quotients by grid spacings and the time step, which the column kernels form from
reciprocals, are those of the reference's divisions: without mixing and dissipation
the systems are the identity, and what is left of a call (the surface forcing in the
top level, the tendencies, TKE's surface correction) equals the oracle bit for bit."""
import numpy as np
import pytest

import test_gpu_friction as TF
import test_gpu_rounding as TR
import test_gpu_turbulence as TT
import test_gpu_vertmix as TV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [9, 20, 45, 80])
def test_vertmix(nz):
    from veros_amd import thermodynamics
    st = TV._state(nz, 40, 30, nz)
    st.variables.kappaH[...] = 0
    out = TR._as_dict(thermodynamics.vertmix_tempsalt(TV._dev(st, "outer")))
    ref = TV.V.vertmix_tempsalt(st)
    for k in TV.KEYS:
        assert np.array_equal(out[k], getattr(ref, k)), k


@pytest.mark.parametrize("nz", [9, 20, 45, 80])
def test_friction(nz):
    from veros_amd import friction
    st = TF._state(nz, 40, 30, nz)
    st.variables.kappaM[...] = 0
    out = TR._as_dict(friction.implicit_vert_friction(TF._dev(st, "outer")))
    ref = TF.F.implicit_vert_friction(st)
    for k in TF.KEYS:
        assert np.array_equal(out[k], getattr(ref, k)), k


@pytest.mark.parametrize("nz", [9, 20, 45, 80])
@pytest.mark.parametrize("sign", [1, -1])
def test_tke_surface(nz, sign):
    st = TT._state(nz, 40, 30, nz)
    vs = st.variables
    for k, v in vars(vs).items():
        if "diss" in k.lower() or k in ("kappaM", "sqrttke", "tke"):
            v[...] = 0
    vs.forc_tke_surface[...] = sign * np.random.default_rng(nz).uniform(1e-6, 1e-4, vs.forc_tke_surface.shape)
    out = TT._gpu("tke", st, "outer")
    ref = TT.ORACLE["tke"](st)
    assert np.any(ref.tke_surf_corr[2:-2, 2:-2]) or np.any(ref.tke[..., vs.taup1])
    for k, r in ref._asdict().items():
        assert np.array_equal(out[k], r), k
