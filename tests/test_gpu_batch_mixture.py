"""Plans over systems of one depth class whose arrays allow 16-byte copies in part
(one or most of five off alignment): every system as its own solve gives it, bit for
bit, whichever kernel the class takes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _system(rng, nz, shift, low=7, high=40):
    nx, ny = rng.integers(low, high, size=2)
    s = dict(kbot=torch.from_numpy(rng.integers(0, nz + 1, size=(nx, ny)).astype(np.int32)).cuda())
    for k, scale, add in (("a", 0.1, 0.0), ("b", 1.0, 3.0), ("c", 0.1, 0.0), ("d", 1.0, 0.0), ("x", 0.0, 7.0)):
        t = torch.empty(nx * ny * nz + 1, dtype=torch.float64, device="cuda")[shift:shift + nx * ny * nz].view(nx, ny, nz)
        s[k] = t.copy_(torch.from_numpy(rng.random((nx, ny, nz)) * scale + add))
    return s


@pytest.mark.parametrize("nz", [16, 32, 48, 64, 66, 80, 82, 96, 112, 128])
@pytest.mark.parametrize("shifts", [(0, 0, 1, 0, 0), (1, 1, 0, 1, 1)])
def test_plan_equals_single_solves(nz, shifts):
    from veros_amd.batched import TdmaBatch
    from veros_amd.utilities import solve_implicit_kbot
    systems = [_system(np.random.default_rng(10 * nz + q), nz, s) for q, s in enumerate(shifts)]
    for precision in ("fp64", "mixed"):
        TdmaBatch(systems, precision=precision).run()
        for q, s in enumerate(systems):
            ref = solve_implicit_kbot(s["a"], s["b"], s["c"], s["d"], s["kbot"], precision=precision)
            assert torch.equal(s["x"], ref), (precision, q)


# 588 tiles at least: more than two per CU of 256, all resident at up to 12 levels per lane,
# five of six systems aligned: taken system by system
@pytest.mark.parametrize("nz", [12, 16, 30, 32, 48, 50, 64, 66, 80, 82, 96])
def test_class_taken_system_by_system(nz):
    from veros_amd.batched import TdmaBatch
    from veros_amd.utilities import solve_implicit_kbot
    systems = [_system(np.random.default_rng(20 * nz + q), nz, s, 28, 37) for q, s in enumerate((0, 0, 1, 0, 0, 0))]
    for precision in ("fp64", "mixed"):
        TdmaBatch(systems, precision=precision).run()
        for q, s in enumerate(systems):
            ref = solve_implicit_kbot(s["a"], s["b"], s["c"], s["d"], s["kbot"], precision=precision)
            assert torch.equal(s["x"], ref), (precision, q)
