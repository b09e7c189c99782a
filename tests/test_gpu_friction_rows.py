"""Friction's walk over several rows per block: the u faces' dissipation carried
from row to row, the early row of every chunk but the first, the two buffers of
the v faces' and a ragged last chunk, at every number of levels per lane on 8
and 16 lanes per column, against the oracle at the bars of test_gpu_friction."""
import pytest
import torch

import test_gpu_friction as TF

pytestmark = pytest.mark.gpu


def _rows(nx, ny, nz):
    """Rows per block and rows of the last chunk on this device (the rule of fric_rows)."""
    lanes = 8 if nz <= 32 else 16
    S = max(2, -(-nz // lanes))
    per_cu = 4 if S <= 3 else 3 if S == 4 and lanes == 16 else 2
    strips, n = -(-(ny + 1) // (2 * (64 // lanes) - 1)), nx + 1
    slots = per_cu * torch.cuda.get_device_properties(0).multi_processor_count
    rows = min(range(1, 25), key=lambda r: (-(-(strips * -(-n // r)) // slots) * (r + 1), -r))
    return rows, n % rows


@pytest.mark.parametrize("shape,levels", [((1500, 30, 5), "outer"), ((300, 140, 9), "inner"), ((700, 64, 17), "outer"),
                                          ((600, 140, 24), "inner"), ((260, 75, 32), "inner"), ((2400, 7, 33), "outer"),
                                          ((270, 30, 60), "inner"), ((220, 30, 80), "inner"), ((150, 40, 96), "outer"),
                                          ((140, 40, 112), "inner"), ((140, 41, 128), "outer")])
def test_rows_against_oracle(shape, levels):
    from veros_amd import friction
    rows, last = _rows(*shape)
    assert rows > 1 and last > 0  # several rows, the last chunk short
    st = TF._state(sum(shape), *shape)
    TF._check(friction.implicit_vert_friction(TF._dev(st, levels)), TF.F.implicit_vert_friction(st), st)
