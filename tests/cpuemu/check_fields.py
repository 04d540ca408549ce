"""Field getters and setters on a host build of the library when no device
memory is left for the permutation's staging copy: same values as with it, in
the call in which the allocation fails and in later ones.
Usage: check_fields.py LIB.so"""
import ctypes
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path.insert(0, ROOT)
sys.path.insert(0, os.path.join(ROOT, "tests"))

import numpy as np  # noqa: E402

import specfempp_amd._native as nat  # noqa: E402

nat._lib = None
nat.LIB_PATH = sys.argv[1]
lib = nat.load()
lib.emu_allow_mallocs.argtypes = [ctypes.c_long]
from specfempp_amd import Engine2D, Engine3D, meshes  # noqa: E402

failures = []


def engine(kind):
    if kind == "3d":
        w = meshes.config3(n=2, nstep=4, h=100.0, nrec_side=1)
        e = Engine3D(w.mesh, w.sources, w.receivers, w.dt, 4, 1, ("displacement",), scatter="gather")
    else:
        mesh = meshes.quad_mesh(6, 5, 0, 300.0, 0, 250.0, materials=[meshes.elastic(2400.0, 3000.0, 1732.0)])
        e = Engine2D(mesh, [dict(x=110.0, z=160.0, angle=30.0, f0=15.0, factor=1e10)], [dict(x=200.0, z=50.0)], 1e-3, 4, 1,
                     ("displacement",), scatter=kind)
    e.initialize()
    return e


for kind in ("colored", "gather", "3d"):
    e = engine(kind)
    rng = np.random.default_rng(3)
    u = rng.standard_normal(e.field("displacement").shape).astype(np.float32)
    e.close()
    for left in (0, 1):
        e = engine(kind)
        lib.emu_allow_mallocs(left)
        try:
            e.set_field("displacement", u)
            e.set_field("velocity", 2 * u)
            ok = np.array_equal(e.field("displacement"), u) and np.array_equal(e.field("velocity"), 2 * u)
        except Exception as err:  # noqa: BLE001
            ok = False
            print(err)
        lib.emu_allow_mallocs(-1)
        ok = ok and np.array_equal(e.field("displacement"), u) and np.array_equal(e.field("velocity"), 2 * u)
        e.close()
        print(f"{'ok  ' if ok else 'FAIL'} {kind}, {left} allocations left", flush=True)
        if not ok:
            failures.append((kind, left))
print("failures:", failures, flush=True)
sys.exit(1 if failures else 0)
