"""sfx_get_timings: the step's time is the whole run's, the steps without events
and those that sample included.  The host build counts a launch as one
millisecond, so the time is the launches per step.
Usage: check_timings.py LIB.so"""
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path.insert(0, ROOT)

import specfempp_amd._native as nat  # noqa: E402

nat._lib = None
nat.LIB_PATH = sys.argv[1]
nat.load()
from specfempp_amd import Engine2D, Engine3D, meshes  # noqa: E402

failures = []


def check(name, engine, steps, launches):
    engine.initialize()
    engine.run()
    got = engine.timings()["step_ms"] * steps
    engine.close()
    ok = abs(got - launches) < 1e-3 * launches
    print(f"{'ok  ' if ok else 'FAIL'} {name}: {got:.1f} launches counted, {launches} made", flush=True)
    if not ok:
        failures.append(name)


# sources, stiffness, Stacey entries and update, and a sample every third step
w = meshes.config3(n=2, nstep=20, h=100.0, nrec_side=1)
e = Engine3D(w.mesh, w.sources, w.receivers, w.dt, 20, 3, ("velocity",), scatter="atomic")
check("3-D atomic", e, 20, 20 * 4 + 7)
# one launch per step, one for the boundary points; no receivers
mesh = meshes.quad_mesh(6, 5, 0, 300.0, 0, 250.0, materials=[meshes.elastic(2400.0, 3000.0, 1732.0)])
check("2-D patches", Engine2D(mesh, [], [], 1e-3, 20, 3, ()), 20, 21)
print("failures:", failures, flush=True)
sys.exit(1 if failures else 0)
