"""Fused launches of long steps in a dense gas: collisions in the same step as
tet crossings (several tets at once among them), surface hits and exits, in
waves where other lanes take plain steps.  FP64 bit for bit against the CPU
oracle, mixed to its bars."""
from __future__ import annotations

import pytest

from start_amd import workloads

from ._parity import Pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("model", ["HS", "VHS", "VSS"])
@pytest.mark.parametrize("walk,block,persistent", [(1, 256, False), (0, 256, False), (0, 128, False), (1, 256, True)])
def test_collisions_within_long_steps(precision, model, walk, block, persistent):
    w = workloads.large_box(n_particles=4000, cells=5, model=model)
    w.gas.concentration *= 0.1  # about a quarter of the steps collide
    w.dt = 1e-5  # 2 cm of a 10 cm tet
    w.phi *= 1e-3
    w.vel[::9] = 0.0
    pr = Pair(w, steps_per_launch=8, precision=precision)
    pr.eng.set_launch(steps_per_launch=8, block=block, persistent=persistent, sort_interval=16, walk=walk)
    pr.advance(24)
    where = f"{precision} {model} walk={walk} block={block} persistent={persistent}"
    if precision == "fp64":
        res = pr.compare(where)
    else:
        res = pr.compare_mixed(where)
    assert 200 < res["settled"] < 3800
    pr.close()
