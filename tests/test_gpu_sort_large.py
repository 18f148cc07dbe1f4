"""The sort of large populations at the sizes where its method changes (1M
rows as loaded, 1.5M with fewer than two a tet, 4M) and with a partial last
tile (8,192 rows), for one, two and three passes over the key bits: the same
run never sorted takes every particle to the same state, bit for bit (each row
moved exactly once), the same number of steps (the live prefix holds every
particle that moves), and the same charge."""
from __future__ import annotations

import numpy as np
import pytest

from start_amd import workloads
from start_amd.engine import ParticleInCellStep
from start_amd.species import E_CHARGE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cells,precision", [(999_999, 12, "fp64"), (1_000_000, 12, "fp64"),
                                               (1_007_617, 12, "mixed"), (1_000_001, 6, "mixed"),
                                               (1_499_999, 51, "mixed"), (1_500_000, 51, "fp64"),
                                               (1_500_001, 89, "fp64"), (4_000_001, 12, "mixed")])
def test_sorted_run_equals_the_unsorted_one(n, cells, precision):
    w = workloads.large_box(n_particles=n, cells=cells)
    w.dt = 4e-5 / cells  # a part settles between the sorts
    w.gas.model = "NONE"
    w.phi *= 1e-3
    rng = np.random.default_rng(n)
    k = n // 16
    w.pos[:k] = w.pos[k]  # many rows in one tet
    w.pos[k:2 * k, 0] += 1.0  # outside the mesh
    w.vel[2 * k:3 * k] = 0.0
    order = rng.permutation(n)
    w.pos, w.vel = w.pos[order], w.vel[order]
    out = []
    for interval in (0, 3):
        eng = ParticleInCellStep(w.mesh, w.species, w.gas, w.dt, w.seed, precision=precision, sort_interval=interval)
        eng.set_node_potential(w.phi)
        eng.load_particles(w.pos, w.vel, w.sp_idx)
        eng.process(10)
        out.append((eng.particles(), eng.stats(), eng.tri_counts(), eng.node_charge()))
        eng.close()
    (a, sa, ta, qa), (b, sb, tb, qb) = out
    for c in ("x", "y", "z", "vx", "vy", "vz", "tet", "status", "hit"):
        assert np.array_equal(a[c], b[c]), c
    assert sa["processed"] == sb["processed"] and 0 < sa["settled"] == sb["settled"] < n
    assert np.array_equal(ta, tb)
    # sums of up to n/16 charges in another order: n/16 roundings of 2^-53 each
    tol = (n / 16 + 64) * 2.0 ** -53
    assert np.abs(qa - qb).max() <= tol * max(np.abs(qa).max(), E_CHARGE)
