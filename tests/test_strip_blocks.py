"""The strips that the isoneutral kernels' blocks are numbered in (strip_blocks of
vx_common.hpp, compiled here for the CPU): every row is covered, no strip is wider
than allowed, and less than one block a strip is padding, so that the strips, and with
them the XCDs, have the same work."""
import os
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "veros_amd" / "csrc"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCE = """
#include <cstdio>
#include "vx_common.hpp"
int main() {
    for (int cols : {1, 5, 96, 192, 223})
        for (int ncb = 1; ncb <= 64; ++ncb)
            for (int nj = 1; nj <= 2500; ++nj) {
                const int sb = vx::strip_blocks(cols, ncb, nj), row = (nj + ncb - 1) / ncb;
                const int n = (nj + sb * ncb - 1) / (sb * ncb);  // strips, as the kernels count them
                const int most = cols / ncb > 1 ? cols / ncb : 1;
                if (sb < 1 || sb > most || n * sb < row || n * sb - row >= n || n != (row + most - 1) / most) {
                    std::printf("cols=%d ncb=%d nj=%d: %d strips of %d blocks\\n", cols, ncb, nj, n, sb);
                    return 1;
                }
            }
    return 0;
}
"""


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="no hipcc")
def test_rows_in_equal_strips(tmp_path):
    src, exe = tmp_path / "strips.hip", tmp_path / "strips"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "--offload-host-only", "-O2", "-std=c++17", "-I", str(CSRC), str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
