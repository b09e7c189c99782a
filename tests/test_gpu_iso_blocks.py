"""Isoneutral pre and face-flux kernels where their blocks can go wrong: blocks
of 4 to 32 columns whose rows end inside a block, columns without a wet or
without a dry level, shallow and deep columns, both time-level layouts, with
the tracer step on either side of the fused call. Bar: 1e-12 relative per
output over the whole array, as for the other isoneutral tests; the stepped
fields sum terms that cancel (noise tracers on thin levels: moving half of the
inputs by one ulp moves the oracle's own temperature by 2.7e-12 of its maximum
on 260x140x5), so theirs is 1e-12 plus four times that movement. The one call and
the separate calls agree value for value."""
import numpy as np
import pytest
import torch

from conftest import rel_err
from oracle import isoneutral as O
from veros_amd import workloads as W

pytestmark = pytest.mark.gpu
TOL = 1e-12
PRE_KEYS = ("Ai_ez", "Ai_nz", "Ai_bx", "Ai_by", "K_11", "K_22", "K_33")
STEP_KEYS = ("temp", "salt", "dtemp_iso", "dsalt_iso", "P_diss_iso")


def _oracle(st):
    for k, v in O.isoneutral_diffusion_pre(st)._asdict().items():
        setattr(st.variables, k, v)
    O.isoneutral_diffusion(st, "temp", True)
    O.isoneutral_diffusion(st, "salt", False)
    return st.variables


@pytest.mark.parametrize("levels", ["inner", "outer"])
@pytest.mark.parametrize("shape,land", [((260, 140, 5), 0.4),   # 32 columns a block
                                        ((150, 131, 2), 0.0),   # no land, two levels
                                        ((97, 66, 64), 0.5),    # 7 columns, whole rounds of lanes
                                        ((23, 19, 65), 0.9),    # 4 columns, hardly any wet
                                        ((40, 61, 128), 0.2)])  # deepest columns
def test_blocks_against_oracle(shape, land, levels):
    from veros_amd import isoneutral
    from veros_amd.state import to_device_state
    rng = np.random.default_rng(17 + sum(shape))
    st = W.iso_state(rng, *shape, dx_deg=1.0, dy_deg=0.5, y_origin=-30.0, dz_top=10.0, dz_bottom=80.0,
                     land_frac=land, cyclic=shape[0] % 2 == 0, stratified=False, random_k_iso=True, jitter=0.02,
                     random_aux=True, tau=1, taup1=0)
    st.settings.K_iso_steep = 20.0
    one, sep = to_device_state(st, levels=levels), to_device_state(st, levels=levels)
    isoneutral.isoneutral_pre_and_diffusion_temp_salt(one)
    isoneutral.isoneutral_diffusion_pre(sep)
    isoneutral.isoneutral_diffusion(sep, sep.variables.temp, True)
    isoneutral.isoneutral_diffusion(sep, sep.variables.salt, False)
    moved = W.state_to_numpy_copy(st)
    for k in ("temp", "salt", "K_iso"):
        v = getattr(moved.variables, k)
        setattr(moved.variables, k, np.where(rng.random(v.shape) < 0.5, np.nextafter(v, np.inf), v))
    ref, near = _oracle(st), _oracle(moved)
    for k in PRE_KEYS + STEP_KEYS:
        a, b = getattr(one.variables, k), getattr(sep.variables, k)
        assert torch.equal(a, b), k
        r = getattr(ref, k)
        bar = TOL + (4 * rel_err(getattr(near, k), r) if k in STEP_KEYS else 0.0)
        assert rel_err(a.cpu().numpy(), r) <= bar, k
