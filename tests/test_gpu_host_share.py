"""The host's core is free for most of a long solve: the thread that waits for
the iterations neither spins through them nor slows them down."""
import time

import numpy as np
import pytest
import torch

from ppf_amd import scenes
from ppf_amd.solver import BlockJacobiPCG

pytestmark = pytest.mark.gpu


def test_waiting_thread_naps(dev):
    s = scenes.grid_spd_system(800)
    t = {k: torch.from_numpy(np.ascontiguousarray(s[k])).to(dev).reshape(-1)
         for k in ("row_offset", "col_index", "value", "cdiag", "b")}
    plan = BlockJacobiPCG(t["row_offset"], t["col_index"])
    x = torch.zeros_like(t["b"])
    plan.solve(t["value"], t["cdiag"], t["b"], x, tol=1e-5)
    torch.cuda.synchronize()
    wall, cpu, iters = -time.perf_counter(), -time.thread_time(), 0
    for _ in range(20):
        x.zero_()
        iters += plan.solve(t["value"], t["cdiag"], t["b"], x, tol=1e-5).iter
    wall, cpu = wall + time.perf_counter(), cpu + time.thread_time()
    print(f"{iters} iterations of {wall / iters * 1e6:.1f} us, share of a core {cpu / wall:.2f}")
    # four iterations of 70 us lie between two reports, and naps start after
    # 100 us of them; launches and the start of a solve are on top
    assert cpu < 0.7 * wall
    plan.close()
