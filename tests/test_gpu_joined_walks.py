"""Launches that hold walks of several kinds (proximity, collision-mesh pairs,
vertex sweeps): meshes around the sizes at which a kind's workgroups end, with
and without a collision mesh, against the oracle."""
import numpy as np
import pytest

import oracle
from ppf_amd import scenes
from ppf_amd.ccd import LineSearch, static_to_device
from ppf_amd.narrow import NarrowPhase, mesh_to_device, pairs_to_numpy
from test_gpu_ccd import _to

pytestmark = pytest.mark.gpu


def soup(nf, seed):
    """nf triangles of size 0.1 at random in the unit box, and their step."""
    rng = np.random.default_rng(seed)
    x = (rng.random((nf, 1, 3)) + rng.normal(0, 0.1, (nf, 3, 3))).reshape(-1, 3)
    return (x.astype(np.float32), np.arange(3 * nf).reshape(nf, 3),
            (x + rng.normal(0, 0.2, x.shape)).astype(np.float32))


@pytest.mark.parametrize("nf", [1, 21, 22, 170, 171, 342])
@pytest.mark.parametrize("ns", [0, 1, 43])
def test_joined_walks(dev, nf, ns):
    x, face, x1 = soup(nf, nf)
    m = scenes.contact_mesh(x, face, ghat=0.05, offset=0.0)
    one = [np.ones(m[k], np.float32) for k in ("nv", "ne", "nf")]
    sx, sface, _ = soup(max(ns, 1), 1000 + ns)
    sm = scenes.static_mesh(sx, sface, ghat=0.05, offset=0.0) if ns else None
    st = static_to_device(sm, dev) if ns else None
    t, t1 = mesh_to_device(m, dev), _to(dev, *one)
    order = ("kind", "a", "b", "count")
    nph = NarrowPhase()
    nph.build(t)
    assert np.array_equal(np.sort(pairs_to_numpy(nph.proximity(t)), order=order),
                          np.sort(oracle.proximity(m), order=order))
    if ns:
        assert np.array_equal(np.sort(pairs_to_numpy(nph.static_pairs(t, st, *t1)), order=order),
                              np.sort(oracle.static_proximity(m, sm, *one), order=order))
    nph.close()
    ls = LineSearch()
    toi, ov = ls(t, *_to(dev, x1.reshape(-1)), *t1, static=st)
    want, wov = oracle.line_search(m, x1, *one, static=sm)
    assert np.float32(toi).tobytes() == np.float32(want).tobytes() and ov == wov
