"""The child test of a walk record (csrc/bvh_query.hpp) compiled for the host:
an unused place is no hit for any query box, infinite and NaN ones among them,
and every other place is one exactly where the boxes overlap."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"

SOURCE = r"""
#include "bvh_query.hpp"
#include <cstdio>
using namespace ppf;

int main() {
    const float inf = __builtin_inff(), nan = __builtin_nanf("");
    const float ends[] = {-inf, -1.0f, 0.5f, 2.0f, inf, nan};
    // a leaf child (place 0, place 1 unused), then a node's two children
    WalkRec w;
    const float lo[3] = {0.0f, 0.0f, 0.0f}, hi[3] = {1.0f, 1.0f, 1.0f};
    const float all0[3] = {-inf, -inf, -inf}, all1[3] = {inf, inf, inf};
    put_child(w, 0, 5u | kLeafCode, 5u, lo, hi);
    put_none(w, 1);
    put_child(w, 2, 40u, 7u, all0, all1); // one element of infinite margin
    put_child(w, 3, 6u | kLeafCode, 6u, lo, hi);
    int bad = 0, hits = 0;
    auto check = [&](auto pair, const QBox &q, uint32_t own, bool scenes, int bound) {
        constexpr int PAIR = decltype(pair)::value;
        const uint32_t got = record_hits<PAIR>(w.code, w.tag, w.box, q, own, scenes, bound);
        uint32_t want = 0;
        for (int k = 0; k < 4; ++k) {
            bool ok = w.code[k] != kNoCode;
            for (int d = 0; d < 3; ++d) {
                ok = ok && w.box[6 * k + d] <= q.mx[d] && w.box[6 * k + 3 + d] >= q.mn[d];
            }
            if (scenes) {
                ok = ok && w.tag[k] == q.scene;
            }
            if (PAIR && ((w.code[k] & kLeafCode) || bound == PAIR)) {
                const uint32_t key =
                    (w.code[k] & kLeafCode) ? w.code[k] & ~kLeafCode : w.tag[k];
                ok = ok && (PAIR > 0 ? key > own : key < own);
            }
            want |= ok ? 1u << k : 0u;
        }
        hits += got != 0;
        if (got != want && ++bad <= 3) {
            std::printf("pair %d box x [%g, %g] y [%g, %g]: hits %x, want %x\n", PAIR, q.mn[0],
                        q.mx[0], q.mn[1], q.mx[1], got, want);
        }
    };
    for (float x0 : ends) for (float x1 : ends) for (float y0 : ends) for (float y1 : ends) {
        QBox q{{x0, y0, -inf}, {x1, y1, inf}, 5u};
        for (uint32_t own : {0u, 6u, 100u}) {
            for (int bound : {-1, 0, 1}) {
                check(std::integral_constant<int, kPairAll>{}, q, own, false, bound);
                check(std::integral_constant<int, kPairAbove>{}, q, own, false, bound);
                check(std::integral_constant<int, kPairBelow>{}, q, own, false, bound);
            }
            check(std::integral_constant<int, kPairAll>{}, q, own, true, 0);
        }
    }
    std::printf("%d wrong, %d with hits\n", bad, hits);
    return bad || !hits;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_unused_places_are_never_hit(tmp_path):
    src, exe = tmp_path / "walk.hip", tmp_path / "walk"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "--offload-host-only", "-std=c++17", "-O2", "-ffp-contract=off",
                    f"-I{ROOT}/ppf-contact-solver_amd/csrc", f"-I{ROOT}/include", str(src),
                    "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
