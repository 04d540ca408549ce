"""A batch of meshes with 4 and 9 control nodes per element: no geometry form
fits both, so its patches read per-point arrays; every simulation still gives
its engine's traces bit for bit (the forms give the same values)."""
import numpy as np
import pytest

from conftest import load_case

pytestmark = pytest.mark.gpu


def test_batch_of_4_and_9_node_meshes():
    from specfempp_amd import Batch, Engine2D, meshes

    m9, cfg = load_case("elastic_stacey_80x60")
    h = 20.0
    m4 = meshes.quad_mesh(13, 9, 0.0, 13 * h, 0.0, 9 * h, materials=[meshes.elastic(2000.0, 2500.0, 1400.0)])
    args = [(m9, cfg["sources"], cfg["stations"], cfg["dt"], 60),
            (m4, [dict(x=6.4 * h, z=4.3 * h, angle=30.0, f0=40.0, factor=1e10)], [dict(x=6.0 * h, z=4.0 * h)],
             meshes.stable_dt(h, 2500.0), 90)]
    print("[case] batch of 4- and 9-node meshes", flush=True)
    want = []
    for mesh, src, rec, dt, nstep in args:
        e = Engine2D(mesh, src, rec, dt, nstep, 1, ("displacement", "velocity"), scatter="gather")
        e.initialize()
        e.run()
        want.append(e.seismograms())
        e.close()
    assert all(w.any() for w in want)
    hosts = [Engine2D(mesh, src, rec, dt, nstep, 1, ("displacement", "velocity"), host_only=True)
             for mesh, src, rec, dt, nstep in args]
    b = Batch(hosts)
    for e in hosts:
        e.close()
    b.set_config(5, True, "gather")
    b.run()
    assert all(np.array_equal(b.seismograms(i), w) for i, w in enumerate(want))
    b.close()
