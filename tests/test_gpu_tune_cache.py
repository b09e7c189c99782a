"""What a plan's tuning leaves for later plans: block and grid sizes timed on one
kernel are not taken over for systems that run another (arrays off 16-byte
alignment take flat loads instead of copies into LDS)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _plan(nz, shift):
    from veros_amd.batched import TdmaBatch
    g = torch.Generator(device="cuda")
    g.manual_seed(nz)
    n = 200 * 100 * nz
    arrs = []
    for scale, add in ((0.1, 0.0), (1.0, 3.0), (0.1, 0.0), (1.0, 0.0), (0.0, 0.0)):
        t = torch.empty(n + 1, dtype=torch.float64, device="cuda")[shift:shift + n].view(200, 100, nz)
        t.copy_(torch.rand((200, 100, nz), generator=g, dtype=torch.float64, device="cuda") * scale + add)
        arrs.append(t)
    kb = torch.randint(0, nz + 1, (200, 100), generator=g, dtype=torch.int32, device="cuda")
    return TdmaBatch([dict(zip("abcdx", arrs), kbot=kb)])


@pytest.mark.parametrize("nz", [16, 32, 48, 80, 96])
def test_tuning_stays_with_its_kernel(nz):
    for tuned, other in ((0, 1), (1, 0)):
        before = _plan(nz, other).info()["buckets"]
        plan = _plan(nz, tuned)
        chosen = plan.tune()["buckets"]
        assert _plan(nz, other).info()["buckets"] == before
        assert _plan(nz, tuned).info()["buckets"] == chosen
