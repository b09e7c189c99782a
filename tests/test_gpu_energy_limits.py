"""TKE where the mixing length is infinite: c_eps sqrttke / mxl vanishes there,
in the rows and in the diagnostic alike."""
import numpy as np
import pytest

import test_gpu_turbulence as TT
from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz,levels", [(12, "inner"), (45, "outer")])
def test_infinite_mixing_length(nz, levels):
    st = TT._state(nz, 14, 11, nz, enable_tke_hor_diffusion=True)
    mxl = st.variables.mxl
    mxl[np.random.default_rng(nz).random(mxl.shape) < 0.2] = np.inf
    ref = TT.ORACLE["tke"](st)
    out = TT._gpu("tke", st, levels)
    for k, r in ref._asdict().items():
        assert rel_err(out[k], r) <= 1e-12, k
