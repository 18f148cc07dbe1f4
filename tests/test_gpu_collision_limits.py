"""The FP32 test that lets a step skip the collision decision must never skip
one that would be accepted: at and beyond the limits of the factors it is
trusted for (concentration, time step and cross section 1e-35 to 1e35, the
viscosity exponent), with zero among them, FP64 bit for bit against the CPU
oracle; and in mixed precision, where the decision itself is FP32, over speeds
of four decades."""
from __future__ import annotations

import numpy as np
import pytest

from start_amd import workloads

from ._parity import Pair

pytestmark = pytest.mark.gpu


# concentration, time step and diameter with P of order 1 or far from it
FACTORS = [(0.0, 1e-8, 4e-10), (1e-40, 1e-8, 4e-10), (9.9e-36, 1e-8, 4e-10), (1e24, 0.0, 4e-10),
           (9e34, 1e-8, 1e-17), (1.1e35, 1e-8, 1e-17), (1e36, 1e-8, 1e-17), (1e37, 1e-8, 1e-18),
           (1e38, 1e-8, 1.7e-18), (1e35, 1e-36, 4e-10), (1e38, 1e-24, 4e-10)]


@pytest.mark.parametrize("model", ["HS", "VHS", "VSS"])
@pytest.mark.parametrize("K", [1, 4])
def test_decisions_at_the_limits_of_the_factors(model, K):
    for conc, dt, diameter in FACTORS:
        w = workloads.large_box(n_particles=300, cells=3, model=model)
        w.gas.concentration, w.dt, w.species[0].diameter = conc, dt, diameter
        w.vel *= 10.0 ** np.random.default_rng(5).uniform(-2.0, 2.0, (300, 1))
        pr = Pair(w, steps_per_launch=K)
        pr.advance(8)
        pr.compare(f"{model} K={K} n={conc:g} dt={dt:g} d={diameter:g}")
        pr.close()


@pytest.mark.parametrize("omega", [-0.7, -0.5, 0.5, 1.5, 2.0])
@pytest.mark.parametrize("K", [1, 4])
def test_decisions_over_viscosity_exponents(omega, K):
    for density in (1.0, 1e3, 1e5):
        w = workloads.large_box(n_particles=400, cells=3, model="VHS")
        w.gas.omega = omega
        w.gas.concentration *= density
        w.dt = 1e-8
        pr = Pair(w, steps_per_launch=K)
        pr.advance(8)
        pr.compare(f"omega={omega} K={K} density x{density:g}")
        pr.close()


@pytest.mark.parametrize("model", ["HS", "VHS", "VSS"])
@pytest.mark.parametrize("density", [1.0, 1e2, 1e3, 1e5])
def test_mixed_decisions_follow_fp64(model, density):
    n = 100_000
    w = workloads.large_box(n_particles=n, cells=4, model=model)
    w.gas.concentration *= density
    w.vel *= 10.0 ** np.random.default_rng(6).uniform(-2.0, 2.0, (n, 1))
    w.phi *= 0.0  # no push: a velocity changes in a collision only
    pr = Pair(w, precision="mixed", charge=False)
    pr.advance(1)
    st, g = pr.st, pr.eng.particles()
    ref = st.vx != w.vel[:, 0]
    got = g["vx"] != w.vel[:, 0]
    pr.close()
    # The FP32 probability is within 1e-5 of the FP64 one: a draw falls between
    # them with probability below 1e-5 P.  1e5 draws make at most 1 of those on
    # average; 10 are allowed, and the test that rejects in FP32 alone would
    # lose a thousandth of the collisions if its margin had the wrong sign.
    lost, made = int((ref & ~got).sum()), int((got & ~ref).sum())
    print(f"{model} x{density:g}: {int(ref.sum())} collisions, {lost} lost, {made} made", flush=True)
    assert lost <= 10 and made <= 10
    assert ref.any()
