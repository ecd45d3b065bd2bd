"""The sort behind the trees and patterns at the sizes where its form changes
(one workgroup to 8,192 pairs, small tiles, large tiles from 1,048,576), with
few and with many equal keys: vertex trees, whose nodes follow the sorted order
and its stability."""
import numpy as np
import pytest

import oracle
from ppf_amd.narrow import NarrowPhase, mesh_to_device
from test_gpu_treelets import triangles

pytestmark = pytest.mark.gpu


# faces: nf leaves, vertices: 3 nf leaves
@pytest.mark.parametrize("nf,equal", [(21, 0), (1365, 0), (1366, 700), (2730, 0), (2731, 0),
                                      (4096, 100), (4097, 4097), (349525, 0), (349526, 20000)])
def test_trees_at_the_sorts_borders(dev, nf, equal):
    m = triangles(nf, seed=nf, equal=equal)
    t = mesh_to_device(m, dev)
    nph = NarrowPhase()
    nph.build(t)
    for kind in (0, 2):
        nodes, _, root = nph.tree(kind)
        on, _, oroot = oracle.bvh_build(m, kind)
        assert root == oroot and np.array_equal(nodes, on)
    nph.close()
