"""A tree build captured into a graph and replayed at other positions, with eager
work between the replays, gives the nodes and boxes of an eager build: meshes
whose trees have border nodes of one and of two classes, one scene and many."""
import numpy as np
import pytest
import torch

from ppf_amd.narrow import NarrowPhase, mesh_to_device
from test_gpu_treelets import triangles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nf,nscene", [(700, 1), (2049, 3), (12000, 1)])
def test_replayed_builds(dev, nf, nscene):
    t = mesh_to_device(triangles(nf, seed=nf), dev)
    if nscene > 1:
        ids = np.arange(3 * nf) // 3 * nscene // nf
        t["vscene"] = torch.from_numpy(ids.astype(np.int32)).to(dev)
        t["nscene"] = nscene
    nph, eager = NarrowPhase(), NarrowPhase()
    nph.build(t)  # allocates
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        nph.build(t)
    gen = torch.Generator(device=dev).manual_seed(nf)
    for _ in range(4):
        x = torch.rand((nf, 1, 3), generator=gen, device=dev)
        x = x + 0.01 * torch.rand((nf, 3, 3), generator=gen, device=dev)
        t["x"].copy_(x.reshape(-1))
        g.replay()
        eager.build(t)
        assert eager.count(t) == nph.count(t)
        for kind in (0, 1, 2):
            nodes, boxes, root = nph.tree(kind)
            want, wboxes, wroot = eager.tree(kind)
            assert root == wroot and np.array_equal(nodes, want)
            assert np.array_equal(boxes.view(np.uint32), wboxes.view(np.uint32))
    nph.close()
    eager.close()
