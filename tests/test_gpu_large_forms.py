"""Large one-scene plans in each SpMV form: sheets coupled to one another and a
single grid, whose split and symmetric forms agree bit for bit and with fp64;
and the form that a plan takes by itself on both sides of the lines (14 entries
a row on average, 16 MiB of blocks) at which short rows become symmetric."""
import numpy as np
import pytest
import torch

from ppf_amd import scenes
from ppf_amd.solver import BlockJacobiPCG

pytestmark = pytest.mark.gpu


def coupled_sheets(res, layers, seed=0):
    """layers grids of res x res rows, every vertex coupled to two of the next
    sheet: a Laplacian-like SPD system with unsymmetric off-diagonal blocks."""
    per, n = res * res, res * res * layers
    e = scenes.unique_edges(scenes.rect_faces(res, res)).astype(np.int64)
    pairs = [e + k * per for k in range(layers)]
    v = np.arange((layers - 1) * per)
    pairs += [np.stack([v, v + per], 1), np.stack([v[1:], v[1:] + per - 1], 1)]
    pairs = np.concatenate(pairs)
    rng = np.random.default_rng(seed)
    g = rng.normal(0, 1, (len(pairs), 3, 6))
    blk = np.einsum("pki,pkj->pij", g[:, :, :3], g[:, :, 3:])
    diag = np.zeros((n, 3, 3))
    for c in range(2):
        h = g[:, :, 3 * c:3 * c + 3]
        np.add.at(diag, pairs[:, c], np.einsum("pki,pkj->pij", h, h))
    ro, ci, val = scenes.upper_bsr(n, pairs, blk, diag)
    cd = np.tile(np.eye(3, dtype=np.float32).reshape(-1), (n, 1))
    return dict(n=n, row_offset=ro, col_index=ci, value=val, cdiag=cd,
                b=rng.standard_normal(3 * n).astype(np.float32))


@pytest.mark.parametrize("res,layers", [(223, 2), (131, 6), (314, 1)])
def test_forms_of_large_plans(dev, res, layers):
    s = coupled_sheets(res, layers)
    assert s["n"] >= 98304
    t = {k: torch.from_numpy(np.ascontiguousarray(s[k])).to(dev).reshape(-1)
         for k in ("row_offset", "col_index", "value", "cdiag", "b")}
    plan = BlockJacobiPCG(t["row_offset"], t["col_index"])
    out = {}
    for form in ("split", "sym", "ell", "split"):
        assert plan.set_form(form) == form
        y = plan.spmv(t["value"], t["cdiag"], t["b"]).cpu().numpy()
        x = torch.zeros_like(t["b"])
        r = plan.solve(t["value"], t["cdiag"], t["b"], x, tol=1e-4)
        assert r.status == 0
        if form in out:  # the same again after other forms
            assert np.array_equal(y, out[form][0]) and np.array_equal(x.cpu().numpy(), out[form][1])
        out[form] = (y, x.cpu().numpy(), r.iter)
    assert np.array_equal(out["split"][0], out["sym"][0])
    assert np.array_equal(out["split"][1], out["sym"][1])
    M = scenes.sparse_from_upper(s["n"], s["row_offset"], s["col_index"], s["value"], s["cdiag"])
    ref = M @ s["b"].astype(np.float64)
    absref = abs(M) @ np.abs(s["b"]).astype(np.float64)
    # a row sums at most 60 products: 60 roundings of 2^-24 of their magnitudes
    assert np.all(np.abs(out["sym"][0] - ref) <= 60 * 2.0 ** -24 * absref)
    res_l1 = np.abs(s["b"] - M @ out["sym"][1].astype(np.float64)).sum() / np.abs(s["b"]).sum()
    print(f"{res} x {layers}: {out['sym'][2]} iterations, true residual {res_l1:.2e}")
    assert res_l1 < 1.5e-4
    plan.close()


def banded(n, band, seed=0):
    """Row i coupled to the `band` rows after it: 2 band + 1 entries a row, a
    diagonally dominant system."""
    rng = np.random.default_rng(seed)
    i = np.repeat(np.arange(n), band)
    j = i + np.tile(np.arange(1, band + 1), n)
    keep = j < n
    pairs = np.stack([i[keep], j[keep]], 1)
    blk = rng.normal(0, 1, (len(pairs), 3, 3))
    diag = np.tile(np.eye(3) * (12.0 * band), (n, 1, 1))
    ro, ci, val = scenes.upper_bsr(n, pairs, blk, diag)
    cd = np.tile(np.eye(3, dtype=np.float32).reshape(-1), (n, 1))
    return dict(n=n, row_offset=ro, col_index=ci, value=val, cdiag=cd,
                b=rng.standard_normal(3 * n).astype(np.float32))


# 8 (7) stored blocks of 36 B a row: 16 MiB are 58,255 (66,577) rows
@pytest.mark.parametrize("n,band,want", [(59000, 7, "sym"), (58000, 7, "ell"), (70000, 6, "ell"),
                                         (1000, 7, "ell")])
def test_form_by_rule(dev, n, band, want):
    s = banded(n, band)
    avg = (2 * len(s["col_index"]) - n) / n
    size = 36 * len(s["col_index"])
    print(f"{avg:.3f} entries a row, {size / 2**20:.2f} MiB of blocks")
    assert (want == "sym") == (avg >= 14.0 and size >= 16 << 20)
    t = {k: torch.from_numpy(np.ascontiguousarray(s[k])).to(dev).reshape(-1)
         for k in ("row_offset", "col_index", "value", "cdiag", "b")}
    plan = BlockJacobiPCG(t["row_offset"], t["col_index"])
    out = []
    for form in (None, "split", "sym", "auto"):
        if form is not None:
            assert plan.set_form(form) == (want if form == "auto" else form)
        y = plan.spmv(t["value"], t["cdiag"], t["b"])
        x = torch.zeros_like(t["b"])
        r = plan.solve(t["value"], t["cdiag"], t["b"], x, tol=1e-4)
        assert r.status == 0
        out.append((y.cpu().numpy(), x.cpu().numpy(), r.iter))
    # the three forms sum a row in one order
    for y, x, it in out[1:]:
        assert np.array_equal(y, out[0][0]) and np.array_equal(x, out[0][1]) and it == out[0][2]
    plan.close()
