"""Launches of one step in every shape that can be asked for, whose kernels are
their own: block, persistent and walk settings bit for bit against the CPU
oracle, a batch against its runs one by one, and movement records against
those of fused launches; populations around a wave and a workgroup."""
from __future__ import annotations

import numpy as np
import pytest

from start_amd import workloads
from start_amd.engine import ParticleInCellStep

from ._parity import REL_Q, Pair

pytestmark = pytest.mark.gpu

COLUMNS = ("x", "y", "z", "vx", "vy", "vz", "tet", "status", "hit")


def plasma(n):
    w = workloads.large_box(n_particles=n, cells=5)
    w.gas.concentration *= 0.1
    w.dt = 1e-5
    w.phi *= 1e-3
    w.vel[1::9] = 0.0
    return w


@pytest.mark.parametrize("n", [1, 65, 257, 3000])
@pytest.mark.parametrize("block,persistent,walk", [(128, False, 0), (256, True, 0), (256, True, 1), (128, True, 0)])
def test_shapes_match_the_oracle(n, block, persistent, walk):
    pr = Pair(plasma(n))
    pr.eng.set_launch(steps_per_launch=1, block=block, persistent=persistent, sort_interval=7, walk=walk)
    pr.advance(25)
    pr.compare(f"single steps n={n} block={block} persistent={persistent} walk={walk}")
    pr.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("walk", [0, 1])
def test_batch_equals_its_runs(precision, walk):
    sizes = [1, 900, 63, 1300]
    w = plasma(sum(sizes))
    runs = [dict(n=n, scale=(0.4 * (k + 1), 0.0), concentration=w.gas.concentration, run=k)
            for k, n in enumerate(sizes)]

    def run(which, rows, track):
        e = ParticleInCellStep(w.mesh, w.species, w.gas, w.dt, w.seed, precision=precision, sort_interval=6)
        e.set_launch(steps_per_launch=1, sort_interval=6, walk=walk)
        e.set_field_basis(0, phi=w.phi)
        e.load_batch(which, w.pos[rows], w.vel[rows], w.sp_idx[rows])
        if track:
            e.track_movements(500, 40)
        e.process(20)
        out = e.particles(), e.node_charge_runs(), e.tri_counts_runs(), e.stats()["processed"]
        moves = e.movements() if track else None
        e.close()
        return out, moves

    everything = slice(0, sum(sizes))
    (batch, charge, counts, done), _ = run(runs, everything, False)
    (tracked, _, _, done_tracked), moves = run(runs, everything, True)
    assert done == done_tracked and len(moves) == 500
    assert all(np.array_equal(batch[c], tracked[c]) for c in COLUMNS)
    first = total = 0
    for r, n in enumerate(sizes):
        rows = slice(first, first + n)
        (single, q, t, one), _ = run([runs[r]], rows, False)
        for c in COLUMNS:
            assert np.array_equal(batch[c][rows], single[c]), (r, c)
        assert np.array_equal(counts[r], t[0])
        assert np.abs(charge[r] - q[0]).max() <= REL_Q * max(np.abs(q[0]).max(), 1.6e-19)
        first, total = first + n, total + one
    assert total == done


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_movement_records_equal_those_of_fused_launches(precision):
    w = plasma(700)
    out = []
    for K in (1, 5):
        e = ParticleInCellStep(w.mesh, w.species, w.gas, w.dt, w.seed, precision=precision, steps_per_launch=K,
                               sort_interval=10)
        e.set_node_potential(w.phi)
        e.load_particles(w.pos, w.vel, w.sp_idx)
        e.track_movements(600, 30)
        e.process(20)
        out.append((e.movements(), e.particles()))
        e.close()
    (a, pa), (b, pb) = out
    assert a.keys() == b.keys() and all(np.array_equal(a[i], b[i]) for i in a)
    assert all(np.array_equal(pa[c], pb[c]) for c in COLUMNS)
