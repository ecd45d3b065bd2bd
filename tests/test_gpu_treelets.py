"""Trees whose leaf counts lie around the treelet and block borders (1,024 and
32,768 leaves), with equal codes across borders: nodes and boxes equal the
oracle's, after a build and after a refit; pairs too, for one scene and many."""
import numpy as np
import pytest

import oracle
from ppf_amd import scenes
from ppf_amd.narrow import NarrowPhase, mesh_to_device, pairs_to_numpy

pytestmark = pytest.mark.gpu


def triangles(nf, seed, equal=0):
    """nf independent triangles; the first `equal` share one Morton code."""
    x, f = scenes.random_triangles(nf, seed=seed, jitter=0.3 * nf ** (-1.0 / 3.0))
    x = x.reshape(nf, 3, 3)
    x[:equal] = x[:equal] * 1e-5 + 0.5
    return scenes.contact_mesh(x.reshape(-1, 3), f, ghat=1e-3)


def check_trees(nph, m):
    for kind in (0, 1, 2):
        nodes, boxes, root = nph.tree(kind)
        on, ob, oroot = oracle.bvh_build(m, kind)
        assert root == oroot and np.array_equal(nodes, on)
        assert np.array_equal(boxes[:, [0, 1, 2, 4, 5, 6]].view(np.uint32), ob.view(np.uint32))


# faces: n leaves; edges and vertices: 3 n leaves
@pytest.mark.parametrize("nf,equal", [(1, 0), (2, 0), (341, 0), (342, 0), (1024, 0), (1025, 900),
                                      (2049, 2049), (10922, 0), (10923, 5000), (32769, 1500)])
def test_trees_around_the_treelet_borders(dev, nf, equal):
    m = triangles(nf, seed=nf, equal=equal)
    t = mesh_to_device(m, dev)
    nph = NarrowPhase()
    nph.build(t)
    check_trees(nph, m)
    if equal == 0 and nf <= 2049:
        order = ("kind", "a", "b", "count")
        assert np.array_equal(np.sort(pairs_to_numpy(nph.proximity(t)), order=order),
                              np.sort(oracle.proximity(m), order=order))
    # another mesh of fewer leaves in the same buffers
    if nf > 2:
        m2 = triangles(nf // 2, seed=nf + 1)
        nph.build(mesh_to_device(m2, dev))
        check_trees(nph, m2)
    nph.close()


def test_trees_of_many_scenes(dev):
    """Scenes cut anywhere in the leaf order (treelets hold several): every
    scene's pairs equal those of its own trees."""
    sizes = [1, 700, 324, 1023, 2, 1500]
    parts = [triangles(k, seed=k) for k in sizes]
    x = np.concatenate([p["x"] for p in parts])
    first = np.concatenate([[0], np.cumsum([p["nv"] for p in parts])])
    f = np.concatenate([p["face"].astype(np.int64) + first[c] for c, p in enumerate(parts)])
    m = scenes.contact_mesh(x, f, ghat=1e-3)
    m["vscene"] = np.repeat(np.arange(len(sizes)), np.diff(first)).astype(np.uint32)
    m["nscene"] = len(sizes)
    nph = NarrowPhase()
    t = mesh_to_device(m, dev)
    nph.build(t)
    got = pairs_to_numpy(nph.proximity(t))
    want = [len(oracle.proximity(p)) for p in parts]
    edge = got["kind"] & 255 == 3
    v = got["a"].astype(np.int64)
    v[edge] = m["edge"][v[edge], 0]
    have = np.bincount(m["vscene"][v], minlength=len(sizes))
    print(f"pairs per scene {have.tolist()} / {want}")
    assert have.tolist() == want and sum(want) > 0
    nph.close()
