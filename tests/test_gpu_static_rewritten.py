"""Collision meshes whose arrays are rewritten in place between calls on one
handle (positions, whole meshes of the same size, scene ids and counts): pairs,
intersections, certified steps and time steps are those of the present
contents, as the oracle or a fresh handle gives them."""
import copy

import numpy as np
import pytest
import torch

import oracle
from ppf_amd import scenes
from ppf_amd.ccd import LineSearch, static_to_device
from ppf_amd.narrow import NarrowPhase, mesh_to_device, pairs_to_numpy
from ppf_amd.stepper import Stepper, scene_to_device
from test_gpu_ccd import _to

pytestmark = pytest.mark.gpu
ORDER = ("kind", "a", "b", "count")


def sheet(res, z, seed, shift=0.0):
    x, f = scenes.stacked_sheets(res, layers=1, gap=0.0, noise=1e-4, seed=seed, size=0.08)
    return x + np.float32([shift, 0.0, z]), f


def rewrite(st, sm):
    """The mesh sm into the device arrays of st (same sizes)."""
    for k, v in static_to_device(sm, torch.device("cpu")).items():
        if torch.is_tensor(v):
            assert st[k].shape == v.shape
            st[k].copy_(v)


def meshes(res):
    """Collision meshes of one size: under the sheet, far away, crossing it,
    and the first again with its triangles and vertices renumbered."""
    x, f = sheet(res, -8e-4, 11)
    yield scenes.static_mesh(x, f, ghat=1e-3)
    yield scenes.static_mesh(x + np.float32([0.0, 0.0, 0.5]), f, ghat=1e-3)
    y = x.copy()
    y[:, 2] = (y[:, 0] - 0.04) * 0.05
    yield scenes.static_mesh(y, f, ghat=1e-3)
    rng = np.random.default_rng(5)
    p = rng.permutation(len(x))
    inv = np.argsort(p)
    yield scenes.static_mesh(x[p], inv[np.asarray(f)[rng.permutation(len(f))]], ghat=2e-3)


@pytest.mark.parametrize("res", [3, 24])
def test_rewritten_meshes_on_one_handle(dev, res):
    x, f = sheet(20, 0.0, 3)
    m = scenes.contact_mesh(x, f, ghat=1e-3)
    one = [np.ones(m[k], np.float32) for k in ("nv", "ne", "nf")]
    x1 = x - np.float32([0.0, 0.0, 2e-3])
    t, t1, x1d = mesh_to_device(m, dev), _to(dev, *one), _to(dev, x1.reshape(-1))
    nph, ls, st = NarrowPhase(), LineSearch(), None
    nph.build(t)
    seen = []
    for k, sm in enumerate(meshes(res)):
        if st is None:
            st = static_to_device(sm, dev)
        else:
            rewrite(st, sm)
        got = pairs_to_numpy(nph.static_pairs(t, st, *t1))
        want = oracle.static_proximity(m, sm, *one)
        n, _ = nph.intersection_check(t, *t1, static=st)
        nw, _ = oracle.intersection_check(m, *one, static=sm)
        toi, ov = ls(t, *x1d, *t1, static=st, rebuild=k == 0)
        tw, ow = oracle.line_search(m, x1, *one, static=sm)
        print(f"mesh {k}: pairs {len(got)}/{len(want)}, intersections {n}/{nw}, toi {toi}/{tw}")
        assert np.array_equal(np.sort(got, order=ORDER), np.sort(want, order=ORDER))
        assert n == nw
        assert np.float32(toi).tobytes() == np.float32(tw).tobytes() and ov == ow
        seen.append((len(got), n, toi))
    assert len(set(seen)) == len(seen)  # the meshes do differ
    nph.close()
    ls.close()


def test_scene_ids_and_counts_of_one_handle(dev):
    """The same collision mesh for one scene, for two, and with its scene ids
    exchanged, against a handle of its own each time."""
    x, f = sheet(12, 0.0, 3)
    y, _ = sheet(12, 2e-4, 4)
    m = scenes.contact_mesh(np.concatenate([x, y]), np.concatenate([f, np.asarray(f) + len(x)]),
                            ghat=1e-3)
    vscene = np.repeat([0, 1], len(x)).astype(np.int32)
    sx, sf = sheet(9, -6e-4, 11)
    sm = scenes.static_mesh(np.concatenate([sx, sx]),
                            np.concatenate([sf, np.asarray(sf) + len(sx)]), ghat=1e-3)
    st = static_to_device(sm, dev)
    st["vscene"] = torch.from_numpy(np.repeat([0, 1], len(sx)).astype(np.int32)).to(dev)
    t = mesh_to_device(m, dev)
    one = _to(dev, *[np.ones(m[k], np.float32) for k in ("nv", "ne", "nf")])
    t["vscene"] = torch.from_numpy(vscene).to(dev)
    keep, seen = NarrowPhase(), []
    for nscene, swap in ((1, False), (2, False), (2, True), (1, True)):
        t["nscene"] = nscene
        if swap:
            st["vscene"].copy_(1 - st["vscene"])
        out = []
        for nph in (keep, NarrowPhase()):
            nph.build(t)
            out.append(np.sort(pairs_to_numpy(nph.static_pairs(t, st, *one)), order=ORDER))
        nph.close()
        assert np.array_equal(*out)
        seen.append(len(out[0]))
    print(f"pairs {seen}")
    assert seen[0] > seen[1] > 0
    keep.close()


def test_collider_moved_between_time_steps(dev):
    sc = scenes.drape_scene(res=12, height=8e-4)
    t = scene_to_device(sc, dev)
    p = scenes.step_params(cg_tol=1e-5)
    gpu = Stepper(t)
    pairs = []
    # the sphere out of reach, just below the falling sheet, out of reach again
    for drop in (0.05, 8e-4, 0.05):
        low = float(t["mesh"]["x"].view(-1, 3)[:, 1].min())
        sx = sc["static"]["x"]
        sx = sx + np.float32([0.0, low - drop - sx[:, 1].max(), 0.0])
        sc["static"]["x"] = sx.astype(np.float32)
        t["static"]["x"].copy_(torch.from_numpy(sc["static"]["x"].reshape(-1)))
        start = copy.deepcopy(sc)
        start["mesh"]["x"] = t["mesh"]["x"].cpu().numpy().reshape(-1, 3).copy()
        start["prev"] = t["prev"].cpu().numpy().reshape(-1, 3).copy()
        rg, ro = gpu.advance(p), oracle.OracleStepper(start).advance(p)
        err = np.abs(t["mesh"]["x"].cpu().numpy().reshape(-1, 3) - start["mesh"]["x"]).max()
        print(f"drop {drop}: pairs {rg['pairs_max']}/{ro['pairs_max']}, position error {err:.2e}")
        assert rg["status"] == ro["status"] == 0 and rg["pairs_max"] == ro["pairs_max"]
        assert err <= 1e-5 * np.abs(start["mesh"]["x"]).max()
        pairs.append(rg["pairs_max"])
    assert pairs[0] == pairs[2] == 0 < pairs[1]
    gpu.close()
