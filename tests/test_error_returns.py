"""Error returns of the C ABI, on the CPU over a stub HIP runtime: whichever
HIP call of an entry point fails, nothing it queued is left running when it
returns (the staging buffers and the caller's arrays would still be in use),
and the calls after it find their transfers' sources unchanged."""
from __future__ import annotations

import ctypes as C
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

# name -> the entry point, called with the engine, its workload and a number
# that makes the call's data differ from the last call's
CALLS = {
    "load": lambda e, w, k: e.load_particles(w.pos[:300] + 1e-6 * k, w.vel[:300], w.sp_idx[:300]),
    "append": lambda e, w, k: e.append_particles(w.pos[300:340] + 1e-6 * k, w.vel[300:340], w.sp_idx[300:340]),
    "locate": lambda e, w, k: e.locate(w.pos[:100] + 1e-6 * k),
    "step": lambda e, w, k: e.process(1),
    "particles": lambda e, w, k: e.particles(),
    "node_charge": lambda e, w, k: e.node_charge(),
    "density": lambda e, w, k: e.node_charge_density(),
    "tri_counts": lambda e, w, k: e.tri_counts(),
    "settled": lambda e, w, k: e.settled_ids(),
    "hits": lambda e, w, k: e.hits(),
    "adjoint": lambda e, w, k: e.adjoint_push(np.ones((e.n, 3))),
    "stats": lambda e, w, k: e.stats(),
    "potential": lambda e, w, k: e.set_node_potential(w.phi + k),
    "basis": lambda e, w, k: e.set_field_basis(1, phi=w.phi + k),
    "track": lambda e, w, k: e.track_movements(50, 8),
}


def child(stub_path: str) -> None:
    stub = C.CDLL(stub_path, mode=C.RTLD_GLOBAL)  # before the library, whose HIP calls then bind to it
    from start_amd import workloads
    from start_amd.engine import ParticleInCellStep
    for precision in ("fp64", "mixed"):
        w = workloads.small_box(n_particles=400, charge_units=1.0)
        w.gas.model = "NONE"
        for name, call in CALLS.items():
            print(precision, name, flush=True)
            eng = ParticleInCellStep(w.mesh, w.species, w.gas, w.dt, w.seed, precision=precision)
            eng.record_settle(True)
            CALLS["load"](eng, w, 0)
            failures = 0
            for k in range(200):
                stub.stub_fail_after(k)
                try:
                    call(eng, w, k)
                    failed = False
                except RuntimeError:
                    failed = True
                left = stub.stub_pending()
                stub.stub_fail_after(-1)
                failures += failed
                assert not (failed and left), f"{precision} {name}: call {k} failed, {left} transfers left running"
                CALLS["locate"](eng, w, 1000 + k)  # stages other data
                assert stub.stub_torn() == 0, f"{precision} {name}: call {k} failed, its transfer was overwritten"
                if not failed and k > 60:
                    break
                if eng.n == 0 or failed:
                    CALLS["load"](eng, w, 0)
            assert failures > 0, f"{name}: no call was made to fail"
            eng.close()
    print("ok")


@pytest.mark.skipif(shutil.which("gcc") is None, reason="no C compiler")
def test_nothing_is_left_running_after_an_error(tmp_path):
    stub = str(tmp_path / "libhipstub.so")
    subprocess.run(["gcc", "-std=c11", "-O1", "-shared", "-fPIC", "-fvisibility=default", "-o", stub,
                    os.path.join(HERE, "_hip_stub.c")], check=True, capture_output=True, text=True)
    r = subprocess.run([sys.executable, "-c", "import sys; sys.path.insert(0, sys.argv[1]); "
                        "from tests.test_error_returns import child; child(sys.argv[2])", ROOT, stub],
                       cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr
