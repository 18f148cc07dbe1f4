"""The streaming step kernels at the edges of their tiles and decisions, bit
for bit against the CPU oracle: populations around a wave, a workgroup and
several workgroups, single and fused launches, gas densities at which nearly
no step, a share of them, or nearly every step collides (the FP32 test that
skips the exact collision decision must never skip one), and particles at and
around the speed below which they are frozen."""
from __future__ import annotations

import numpy as np
import pytest

from start_amd import workloads

from ._parity import Pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,K", [(1, 7), (63, 1), (64, 8), (65, 5), (255, 1), (256, 16), (257, 1), (1023, 9), (1025, 2)])
@pytest.mark.parametrize("model,density", [("HS", 1e4), ("VHS", 1e3), ("VSS", 30.0), ("VHS", 1e-3)])
def test_tiles_and_collision_densities(n, K, model, density):
    w = workloads.large_box(n_particles=n, cells=4, model=model)
    w.gas.concentration *= density
    w.dt = 2e-8
    w.vel[::7] = 0.0  # frozen from the start
    w.vel[3::11] *= 1e-9
    pr = Pair(w, steps_per_launch=K)
    pr.advance(6 * K + 12)
    pr.compare(f"n={n} K={K} {model} density x{density}")
    pr.close()
