"""Iterations whose product forms p itself against iterations with a kernel for
it: a scene stopped after k iterations, around the eight of a captured graph,
has the same bits beside a small scene (fused) and beside one that takes the
plan's blocks past the limits (not fused), and follows the oracle."""
import numpy as np
import pytest
import torch

import oracle
from ppf_amd import scenes
from ppf_amd.solver import BatchPCG, BlockJacobiPCG, stack_systems
from test_gpu_batch import cloth, to_dev

pytestmark = pytest.mark.gpu

CAPS = (1, 2, 7, 8, 9, 16, 17)


def capped(dev, syss, form, tiles):
    st, rows = stack_systems(syss)
    t = to_dev(st, dev)
    plan = BatchPCG(t["row_offset"], t["col_index"], rows)
    plan.set_tiles(*tiles)
    assert plan.set_form(form) == form
    out = []
    for k in CAPS:
        x = torch.zeros_like(t["b"])
        r = plan.solve(t["value"], t["cdiag"], t["b"], x, tol=1e-9, max_iter=k)[0]
        out.append((r.iter, r.resid, r.status, x[:3 * rows[1]].cpu().numpy()))
    plan.close()
    return out


@pytest.mark.parametrize("form", ["ell", "split"])
@pytest.mark.parametrize("tiles", [(64, 256), (256, 512)])
def test_fused_equals_unfused(dev, form, tiles):
    s = cloth(21, 1)
    g = scenes.grid_spd_system(640)
    big = {k: g[k] for k in s}
    assert 36 * len(big["col_index"]) > 48 << 20
    for a, b in zip(capped(dev, [s, cloth(9, 0)], form, tiles),
                    capped(dev, [s, big], form, tiles)):
        assert a[:3] == b[:3] and np.array_equal(a[3], b[3])


@pytest.mark.parametrize("form", ["ell", "split", "sym"])
def test_fused_caps_follow_the_oracle(dev, form):
    s = dict(cloth(21, 1))
    s["n"] = len(s["row_offset"]) - 1
    t = {k: v for k, v in to_dev({k: s[k] for k in s if k != "n"}, dev).items()}
    plan = BlockJacobiPCG(t["row_offset"], t["col_index"])
    assert plan.set_form(form) == form
    for k in CAPS:
        x = torch.zeros_like(t["b"])
        r = plan.solve(t["value"], t["cdiag"], t["b"], x, tol=1e-9, max_iter=k)
        o = oracle.pcg(s, tol=1e-9, max_iter=k)
        assert (r.iter, r.status) == (o["iter"], o["status"])
        # other summation orders only: the 1e-3 that residual curves of the first
        # 20 iterations agree to
        assert abs(r.resid - o["resid"]) <= 1e-3 * o["resid"]
        assert np.abs(x.cpu().numpy() - o["x"]).max() <= 1e-3 * np.abs(o["x"]).max()
    plan.close()


@pytest.mark.parametrize("ordered", [False, True])
def test_a_refused_pattern_leaves_the_plan_usable(dev, ordered):
    """The checks of a pattern are read once, behind the kernels they gate."""
    s = cloth(21, 1)
    t = to_dev(s, dev)
    n = len(s["row_offset"]) - 1
    plan = BlockJacobiPCG(t["row_offset"], t["col_index"])
    if ordered:
        plan.set_order(torch.arange(n - 1, -1, -1, dtype=torch.int32, device=dev))
        plan.repattern(t["row_offset"], t["col_index"])
    x0 = torch.zeros_like(t["b"])
    first = plan.solve(t["value"], t["cdiag"], t["b"], x0)
    ro, ci = t["row_offset"].clone(), t["col_index"].clone()
    ro[5] = t["col_index"].numel() + 7  # beyond the pattern: nothing may follow it
    ci[3] = n + 100
    for bad in ((ro, t["col_index"]), (t["row_offset"], ci), (ro, ci)):
        with pytest.raises(RuntimeError):
            plan.repattern(*bad)
    plan.repattern(t["row_offset"], t["col_index"])
    x = torch.zeros_like(t["b"])
    again = plan.solve(t["value"], t["cdiag"], t["b"], x)
    assert (again.iter, again.resid) == (first.iter, first.resid) and torch.equal(x, x0)
    plan.close()
