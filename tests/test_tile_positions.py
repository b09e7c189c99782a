"""The image positions that the column tiles' flat elements read, enumerated on
the host from the kernels' own code (col_tile.hpp, compiled here for the CPU):
every position of an element and of its neighbours lies in the tile's image, and
for a cell of the run it is that cell's, for every depth, column count and first
wet level, the lanes past the run included."""
import os
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "veros_amd" / "csrc"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCE = """
#include <cstdio>
#include "col_tile.hpp"
using namespace vx;

template <int S, int P> int check() {
    using T = Tile<S, P>;
    int bad = 0;
    for (int nz = S == 2 ? 1 : P * (S - 1) + 1 - (P == 8 ? P : 0); nz <= P * S && nz <= kMaxNz; ++nz) {
        const uint32_t m = depth_reciprocal(nz);
        for (int ncol = 0; ncol <= T::C; ++ncol)
            for (int k0 = 0; k0 <= nz; ++k0)
                for (uint32_t e = 0; e < 64u * S; ++e) {
                    const FlatCell f = flat_cell<S, P>(e, ncol, nz, (uint32_t)nz, m);
                    int below, above;
                    flat_neighbours<S, P>(f, k0, nz, below, above);
                    bool ok = f.pos >= 0 && f.pos < T::IMG && below >= 0 && below < T::IMG && above >= 0 && above < T::IMG;
                    if (f.off != kNoAccess) {
                        auto pos = [&](int k) { return f.c * T::CS + k / S * T::SP + k % S; };
                        ok = ok && e == (uint32_t)(f.c * nz + f.k) && f.off == 8u * e && f.pos == pos(f.k);
                        ok = ok && below == pos(f.k > k0 ? f.k - 1 : f.k);
                        ok = ok && above == pos(f.k >= k0 && f.k < nz - 1 ? f.k + 1 : f.k);
                    }
                    if (!ok && bad++ == 0)
                        std::printf("S=%d P=%d nz=%d ncol=%d k0=%d e=%u: pos %d below %d above %d of %d\\n", S, P, nz, ncol,
                                    k0, e, f.pos, below, above, T::IMG);
                }
    }
    return bad;
}

int main() {
    int bad = 0;
    bad += check<2, 8>() + check<4, 8>() + check<6, 8>() + check<8, 8>();
    bad += check<10, 8>() + check<12, 8>() + check<14, 8>() + check<16, 8>();
    bad += check<3, 16>() + check<4, 16>() + check<5, 16>() + check<6, 16>() + check<7, 16>() + check<8, 16>();
    return bad != 0;
}
"""


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="no hipcc")
def test_flat_positions_stay_in_the_image(tmp_path):
    src, exe = tmp_path / "positions.hip", tmp_path / "positions"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "--offload-host-only", "-O2", "-std=c++17", "-I", str(CSRC), str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
