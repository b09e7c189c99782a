"""Isoneutral kernels over the widths of their blocks and strips, held to
test_gpu_iso_blocks's oracle and bars: blocks of 32 columns, the most there are,
in pre, flux and step (8 blocks per CU and more on 260x250), blocks of an odd
number of columns, rows that fill one block only and rows of a single column."""
import pytest

import test_gpu_iso_blocks as TB

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("levels", ["inner", "outer"])
@pytest.mark.parametrize("shape,land", [((260, 250, 9), 0.3),    # 32 columns
                                        ((120, 115, 40), 0.35),  # 7 and 7
                                        ((500, 2, 12), 0.2),     # one block a row
                                        ((301, 1, 40), 0.1),
                                        ((4, 700, 6), 0.3)])     # few rows, several strips
def test_strips_against_oracle(shape, land, levels):
    TB.test_blocks_against_oracle(shape, land, levels)
