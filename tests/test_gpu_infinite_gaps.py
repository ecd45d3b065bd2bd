"""Elements of infinite gap or offset: their query boxes and leaf boxes overlap
every node, unused places of the walk records must stay out of the walks, and
pairs, intersections and the certified step equal the oracle's."""
import numpy as np
import pytest

import oracle
from ppf_amd import scenes
from ppf_amd.ccd import LineSearch, static_to_device
from ppf_amd.narrow import NarrowPhase, mesh_to_device, pairs_to_numpy
from test_gpu_ccd import _to

pytestmark = pytest.mark.gpu
ORDER = ("kind", "a", "b", "count")


@pytest.mark.parametrize("field", ["v_ghat", "e_ghat", "f_ghat", "v_off", "e_off", "f_off"])
@pytest.mark.parametrize("res", [2, 17])
def test_one_element_of_infinite_margin(dev, field, res):
    x, f = scenes.stacked_sheets(res, layers=2, gap=9e-4, noise=1e-4, seed=3)
    m = scenes.contact_mesh(x, f, ghat=1e-3)
    m[field] = m[field].copy()
    m[field][len(m[field]) // 2] = np.inf
    sx, sf = scenes.stacked_sheets(5, layers=1, gap=0.0, noise=1e-4, seed=4)
    sx[:, 2] -= 5e-4
    sm = scenes.static_mesh(sx, sf, ghat=1e-3)
    sm[field] = sm[field].copy()
    sm[field][len(sm[field]) // 2] = np.inf
    one = [np.ones(m[k], np.float32) for k in ("nv", "ne", "nf")]
    t, st, t1 = mesh_to_device(m, dev), static_to_device(sm, dev), _to(dev, *one)
    nph = NarrowPhase()
    nph.build(t)
    with np.errstate(all="ignore"):
        want = oracle.proximity(m), oracle.static_proximity(m, sm, *one)
        hits, _ = oracle.intersection_check(m, *one)
    got = [pairs_to_numpy(p) for p in (nph.proximity(t), nph.static_pairs(t, st, *t1))]
    for g, w in zip(got, want):
        assert np.array_equal(np.sort(g, order=ORDER), np.sort(w, order=ORDER))
    n, _ = nph.intersection_check(t, *t1)
    print(f"{field} {res}: {len(got[0])} + {len(got[1])} pairs, {n} intersections")
    assert n == hits
    nph.close()
    x1 = x.copy()
    x1[:, 2] -= np.where(np.arange(len(x)) >= res * res, 2e-3, 0.0).astype(np.float32)
    ls = LineSearch()
    toi, ov = ls(t, *_to(dev, x1.reshape(-1)), *t1, static=st)
    want, wov = oracle.line_search(m, x1, *one, static=sm)
    assert np.float32(toi).tobytes() == np.float32(want).tobytes() and ov == wov
    ls.close()


@pytest.mark.parametrize("ends", [(-np.inf, np.inf), (np.nan, np.nan), (0.0, np.inf)])
def test_vertices_at_infinity(dev, ends):
    """A triangle whose first edge runs between opposite infinities on all axes
    (its query box overlaps every node), or holds NaN, beside two sheets: walks
    stay inside the trees, and what the other elements find is the oracle's."""
    x, f = scenes.stacked_sheets(17, layers=2, gap=1e-4, noise=2e-4, seed=3)
    n = len(x)
    far = np.array([[ends[0]] * 3, [ends[1]] * 3, [0.0, 0.0, 9.0]], np.float32)
    m = scenes.contact_mesh(np.concatenate([x, far]), np.concatenate([f, [[n, n + 1, n + 2]]]),
                            ghat=1e-3, offset=1e-4)
    one = [np.ones(m[k], np.float32) for k in ("nv", "ne", "nf")]
    t, t1 = mesh_to_device(m, dev), _to(dev, *one)
    nph = NarrowPhase()
    nph.build(t)
    got = pairs_to_numpy(nph.proximity(t))
    count, rec = nph.intersection_check(t, *t1, cap=1 << 16)
    with np.errstate(all="ignore"):
        want = oracle.proximity(m)
        nw, wrec = oracle.intersection_check(m, *one, cap=1 << 16)

    def finite(kind, a, b, types):
        """Rows between elements of the sheets alone."""
        last = {"v": n, "e": int((m["edge"] < n).all(1).sum()), "f": len(f)}
        lim = np.array([[last[c] for c in pair] for pair in types])
        return (a < lim[kind, 0]) & (b < lim[kind, 1])

    pairs = [np.sort(r[finite(r["kind"] & 255, r["a"], r["b"], ("vf", "ve", "vv", "ee"))],
                     order=ORDER) for r in (got, want)]
    assert len(pairs[0]) > 0 and np.array_equal(*pairs)
    # face-edge, edge-edge, (collision face-edge), point-point
    found = []
    for r in (rec, wrec):
        r = r[finite(r["type"], r["elem0"], r["elem1"], ("fe", "ee", "fe", "vv"))]
        found.append(sorted(zip(r["type"].tolist(), r["elem0"].tolist(), r["elem1"].tolist())))
    print(f"{ends}: {len(got)}/{len(want)} pairs, {count}/{nw} intersections, "
          f"{len(found[0])} of the sheets")
    assert len(found[0]) > 0 and found[0] == found[1]
    nph.close()
