"""kbot of edge masks around the deepest that the mask kernel takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [(1 << 20) - 1, 1 << 20, (1 << 20) + 1])
def test_deep_masks(nz):
    from veros_amd.utilities import kbot_from_masks
    edge = torch.zeros((3, 1, nz), dtype=torch.bool, device="cuda")
    edge[0, 0, nz - 1] = True
    edge[2, 0, 5] = True
    assert kbot_from_masks(edge, edge).flatten().tolist() == [nz, 0, 6]
