"""Lists of deferred particles that fill every lane of the straggler kernel
(4,096 for single steps, 65,536 for fused ones) and shorter ones, from tiles
in which most lanes defer, some of them in later steps of the launch: without
the multi-tet walk every segment through two faces does.  Bit for bit against
the CPU oracle."""
from __future__ import annotations

import pytest

from start_amd import workloads

from ._parity import Pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,K,steps,least", [(500, 3, 9, 300), (20_000, 1, 3, 3 * 4096), (120_000, 5, 5, 65_536)])
def test_long_deferred_lists_match_the_oracle(n, K, steps, least):
    w = workloads.large_box(n_particles=n, cells=16)
    w.dt = 2e-5  # about a tet a step
    w.phi *= 1e-3
    w.gas.concentration *= 0.01
    pr = Pair(w, steps_per_launch=K, sort_interval=0)
    pr.eng.set_launch(steps_per_launch=K, sort_interval=0, walk=0)
    pr.advance(steps)
    res = pr.compare(f"deferred lists n={n} K={K}")
    assert res["deferred"] > least and res["settled"] > 0
    pr.close()
