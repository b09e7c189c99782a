"""How the isoneutral kernels round: the root mean square error of every output of
the one call against the oracle run in extended precision (80 bits) on the same
float64 inputs, next to that of the oracle in float64. The kernels' operations round
no more often than the oracle's (reciprocals of metric factors in place of divisions
are made up for by fused multiply-adds, or carry what their rounding cut off): the bar
is the oracle's own error, but for 3% of scatter."""
import numpy as np
import pytest

import test_gpu_rounding as TR
from oracle import isoneutral as O
from veros_amd import workloads as W

pytestmark = TR.pytestmark
KEYS = ("Ai_ez", "Ai_nz", "Ai_bx", "Ai_by", "K_11", "K_22", "K_33", "temp", "salt", "dtemp_iso", "dsalt_iso",
        "P_diss_iso")
BAR = 1.03


def _oracle(m, st):
    for k, v in m.isoneutral_diffusion_pre(st)._asdict().items():
        setattr(st.variables, k, v)
    m.isoneutral_diffusion(st, "temp", True)
    m.isoneutral_diffusion(st, "salt", False)
    return st.variables


def _rms(x, ref):
    """The largest 1% left out: slopes over nearly neutral levels, whose condition decides."""
    d = np.sort(np.abs(np.asarray(x) - ref).ravel())
    d = d[d > 0]
    return float(np.sqrt(np.mean(d[:len(d) - len(d) // 100] ** 2)))


@pytest.mark.parametrize("shape", [(40, 30, 9), (60, 50, 45), (30, 40, 100)])
def test_one_call(shape):
    from veros_amd import isoneutral
    from veros_amd.state import to_device_state
    st = W.iso_state(np.random.default_rng(sum(shape)), *shape, dx_deg=1.0, dy_deg=0.5, y_origin=-30.0, dz_top=10.0,
                     dz_bottom=80.0, land_frac=0.3, random_k_iso=True, random_aux=True, tau=1, taup1=0)
    ds = to_device_state(st, levels="outer")
    isoneutral.isoneutral_pre_and_diffusion_temp_salt(ds)
    wide = TR._wide(st)
    exact = _oracle(TR._extended("isoneutral"), wide)
    plain = _oracle(O, W.state_to_numpy_copy(st))
    ratios = {k: _rms(getattr(ds.variables, k).cpu().numpy(), getattr(exact, k))
              / _rms(getattr(plain, k), getattr(exact, k)) for k in KEYS}
    print({k: round(r, 3) for k, r in ratios.items()})
    assert all(r <= BAR for r in ratios.values()), ratios
