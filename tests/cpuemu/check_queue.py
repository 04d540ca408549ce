"""Runs of many steps keep a bounded number of launches queued: plain and
recorded ones with checkpoints closer together than the engine's windows of
256 steps, and the combined run.  The bound is two windows and one step at two
launches per step: these runs take less than two on average.
Usage: check_queue.py LIB.so"""
import ctypes
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path.insert(0, ROOT)

import numpy as np  # noqa: E402

import specfempp_amd._native as nat  # noqa: E402

nat._lib = None
nat.LIB_PATH = sys.argv[1]
lib = nat.load()
lib.emu_most_queued.restype = ctypes.c_long
from specfempp_amd import Engine2D, meshes  # noqa: E402

STEPS = 1200
mesh = meshes.quad_mesh(1, 1, 0, 50.0, 0, 50.0, materials=[meshes.elastic(2400.0, 3000.0, 1732.0)])
failures = []


def check(name):
    most = lib.emu_most_queued()
    ok = most <= 2 * 513
    print(f"{'ok  ' if ok else 'FAIL'} {name}: at most {most} launches queued", flush=True)
    if not ok:
        failures.append(name)


e = Engine2D(mesh, [], [], 1e-3, STEPS, 1, ("displacement",))
e.initialize()
lib.emu_most_queued()
e.run()
check("run")
e.initialize()
e.forward_record(55)
check("recorded run, a checkpoint every 55 steps")
e.set_adjoint_sources([dict(x=20.0, z=30.0)], np.zeros((1, STEPS, 2)))
lib.emu_most_queued()
e.adjoint_run()
check("combined run")
e.close()
print("failures:", failures, flush=True)
sys.exit(1 if failures else 0)
