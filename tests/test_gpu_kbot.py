"""kbot from an edge mask (utilities.kbot_from_masks) against NumPy's argmax:
column counts around the 64 columns of a block, byte runs that are and are not
a multiple of 16, a mask off 16-byte alignment, columns without an edge, and
masks with several marked levels (the first one counts)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 1), (1, 63, 1), (8, 8, 16), (5, 13, 7), (13, 10, 45), (3, 43, 128)])
@pytest.mark.parametrize("form", ["aligned", "offset", "strided"])
def test_kbot_from_masks(shape, form):
    from veros_amd.utilities import kbot_from_masks
    rng = np.random.default_rng(sum(shape))
    edge = rng.random(shape) < 1.5 / shape[2]
    edge[0, 0] = False
    edge[-1, -1] = False
    edge[-1, -1, -1] = True
    t = torch.from_numpy(edge)
    if form == "offset":
        buf = torch.zeros(edge.size + 1, dtype=torch.bool, device="cuda")
        buf[1:] = t.cuda().reshape(-1)
        dev = buf[1:].view(shape)
    elif form == "strided":
        dev = t.permute(2, 0, 1).contiguous().cuda().permute(1, 2, 0)
    else:
        dev = t.cuda()
    ref = np.where(edge.any(-1), edge.argmax(-1) + 1, 0)
    got = kbot_from_masks(dev, dev)
    assert got.dtype == torch.int32 and got.is_contiguous()
    assert np.array_equal(got.cpu().numpy(), ref)
