"""Walks whose pending nodes outgrow the query stacks of the first pass
(proximity, collision-mesh pairs and intersection check): the pass runs again
with the deep stacks and gives the oracle's result."""
import numpy as np
import pytest
import torch

import oracle
from ppf_amd import _lib, scenes
from ppf_amd.ccd import static_to_device
from ppf_amd.narrow import NarrowPhase, mesh_to_device, pairs_to_numpy
from test_gpu_ccd import _comb_mesh, _to

pytestmark = pytest.mark.gpu

FIRST, DEEP = 32, 96  # stack entries of the two passes


def pending(nodes, root):
    """Most entries a walk that overlaps every node holds: it takes two levels
    at a time, goes on with the rightmost and keeps the others."""
    most, st, v = 0, [], root
    while True:
        if nodes[v][1]:
            kids = []
            for c in (nodes[v][0] - 1, nodes[v][1] - 1):
                kids += [nodes[c][0] - 1, nodes[c][1] - 1] if nodes[c][1] else [c]
            st += kids[:-1]
            v = kids[-1]
            most = max(most, len(st) + 3)
        elif st:
            v = st.pop()
        else:
            return most


def comb_with_span():
    """The Morton comb with one triangle across the whole box: its edges, and
    its first vertex through a large gap, overlap every node."""
    m, _ = _comb_mesh(cluster=600)
    x = m["x"].copy()
    x[-2:] = np.float32([[1024.0, 1024.0, 1023.9], [1024.0, 1023.9, 1024.0]])
    m = scenes.contact_mesh(x, m["face"], ghat=1e-3, offset=1e-3)
    m["v_ghat"][len(x) - 3] = 2100.0
    return m


def test_deep_proximity_and_intersections(dev):
    m = comb_with_span()
    needs = [pending(*oracle.bvh_build(m, k)[::2]) for k in (0, 1, 2)]
    print(f"pending entries (face, edge, vertex trees): {needs}")
    assert min(needs) > FIRST and max(needs) <= DEEP
    t = mesh_to_device(m, dev)
    nph = NarrowPhase()
    nph.build(t)
    got = pairs_to_numpy(nph.proximity(t))
    want = oracle.proximity(m)
    order = ("kind", "a", "b", "count")
    assert np.array_equal(np.sort(got, order=order), np.sort(want, order=order))
    ones = [np.ones(m[k], np.float32) for k in ("nv", "ne", "nf")]
    n, _ = nph.intersection_check(t, *_to(dev, *ones))
    nw, _ = oracle.intersection_check(m, *ones)
    print(f"pairs {len(got)}, intersections {n}/{nw}")
    assert n == nw
    # the same mesh as the collision mesh of one spanning triangle
    sm = scenes.static_mesh(m["x"], m["face"], ghat=1e-3, offset=1e-3)
    m1 = scenes.contact_mesh(m["x"][-3:], np.array([[0, 1, 2]]), ghat=1e-3, offset=1e-3)
    m1["v_ghat"][0] = 2100.0
    t1 = mesh_to_device(m1, dev)
    one1 = [np.ones(m1[k], np.float32) for k in ("nv", "ne", "nf")]
    nph.build(t1)
    gs = pairs_to_numpy(nph.static_pairs(t1, static_to_device(sm, dev), *_to(dev, *one1)))
    ws = oracle.static_proximity(m1, sm, *one1)
    assert np.array_equal(np.sort(gs, order=order), np.sort(ws, order=order))
    nph.close()


@pytest.mark.parametrize("offset", [0.0, 1e-3])
def test_intersections_with_and_without_offsets(dev, offset):
    """Without contact offsets the edge-edge and point-point walks are left
    out; one element with an offset brings them back."""
    x, f = scenes.stacked_sheets(24, layers=2, gap=5e-5, noise=2e-4, seed=4)
    m = scenes.contact_mesh(x, f, ghat=1e-3)
    for k in ("e_off", "v_off"):
        m[k][len(m[k]) // 2] = offset
    t = mesh_to_device(m, dev)
    nph = NarrowPhase()
    nph.build(t)
    ones = [np.ones(m[k], np.float32) for k in ("nv", "ne", "nf")]
    n, rec = nph.intersection_check(t, *_to(dev, *ones), cap=4096)
    nw, want = oracle.intersection_check(m, *ones, cap=4096)
    kinds = np.bincount(rec["type"], minlength=4)
    print(f"offset {offset}: {n} / {nw} by type {kinds}")
    assert n == nw and np.array_equal(kinds, np.bincount(want["type"], minlength=4))
    assert (kinds[1] + kinds[3] > 0) == (offset > 0.0)
    nph.close()


def test_statistics_count_a_deep_walk_once(dev):
    """The statistics walk with the deep stacks from the start: one launch per
    kind and call, every element one query."""
    m = comb_with_span()
    t = mesh_to_device(m, dev)
    nph = NarrowPhase()
    nph.build(t)
    out = torch.empty((len(oracle.proximity(m)), 4), dtype=torch.int32, device=dev)
    _lib.walk_stats_enable(True)
    got = pairs_to_numpy(nph.proximity(t, out))
    st = _lib.walk_stats()
    _lib.walk_stats_enable(False)
    order = ("kind", "a", "b", "count")
    assert np.array_equal(np.sort(got, order=order), np.sort(oracle.proximity(m), order=order))
    seen = [(st[k]["launches"], st[k]["queries"]) for k in _lib.WALK_KINDS[2:]]
    assert seen == [(1, m["nv"]), (1, m["ne"])]
    nph.close()
