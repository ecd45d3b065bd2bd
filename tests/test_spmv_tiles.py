"""Row bounds that the split SpMV form reads per tile (csrc/pcg.hpp) compiled
for the host: every read lies inside the n + 1 words of the offset arrays, also
for the empty tiles at row n (the padding of a tile list to a multiple of 8, a
trailing scene without rows), and a tile's rows get their own bounds."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"

SOURCE = r"""
#include "pcg.hpp"
#include <cstdio>
using namespace ppf;

// n + 1 words of which reads outside are counted, not made
struct Words {
    uint32_t n, step;
    int *outside;
    uint32_t operator[](size_t k) const {
        if (k > n) {
            ++*outside;
            return 0;
        }
        return step * (uint32_t)k;
    }
};

int main() {
    int outside = 0, wrong = 0;
    for (uint32_t n : {1u, 63u, 64u, 65u, 200u, 1024u}) {
        const Words rp{n, 3u, &outside}, tp{n, 5u, &outside};
        for (uint32_t rows : {64u, 512u}) {
            for (uint32_t lo = 0; lo <= n; lo += lo < n && lo + rows > n ? n - lo : rows) {
                const uint32_t hi = lo + rows < n ? lo + rows : n; // lo == n: an empty tile
                for (uint32_t i = lo; i < lo + rows + 64; ++i) {
                    uint32_t nb[4] = {9, 9, 9, 9};
                    load_row_bounds(rp, tp, lo, hi, i, nb);
                    const uint32_t r = i < hi ? i : lo;
                    const bool ok = lo < hi ? nb[0] == 3 * r && nb[1] == 3 * r + 3 &&
                                                  nb[2] == 5 * r && nb[3] == 5 * r + 5
                                            : nb[0] == nb[1] && nb[2] == nb[3];
                    wrong += !ok;
                }
                if (lo == n) {
                    break;
                }
            }
        }
    }
    std::printf("%d reads outside, %d wrong bounds\n", outside, wrong);
    return outside || wrong;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_row_bounds_stay_inside(tmp_path):
    src, exe = tmp_path / "tiles.hip", tmp_path / "tiles"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "--offload-host-only", "-std=c++17", "-O2",
                    f"-I{ROOT}/ppf-contact-solver_amd/csrc", f"-I{ROOT}/include", str(src),
                    "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
