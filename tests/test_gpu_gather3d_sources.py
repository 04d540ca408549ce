"""3-D gather path: several sources in one element, on and off an absorbing
face, and all trace kinds at receivers on element corners, edges, faces and
inside, against the FP32 oracle: within 1e-5 relative L2 for the displacement
and velocity and acceleration within 1.5 times its own distance to the FP64
oracle where that is larger (the rule of the parity tests)."""
import numpy as np
import pytest

import oracle
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,corner,types", [((1, 1, 1), True, ("displacement",)),
                                            ((3, 3, 3), False, ("displacement",)),
                                            ((4, 3, 5), True, ("acceleration", "displacement", "velocity")),
                                            ((3, 5, 3), False, ("velocity", "acceleration"))])
def test_sources_and_samples(n, corner, types):
    from specfempp_amd import Engine3D, meshes

    h, dt, nstep = 100.0, 2e-3, 60
    mesh = meshes.hex_mesh(*n, h, np.zeros(n[::-1], np.int32), [2500.0], [3000.0], [1730.0])
    o = np.zeros(3) if corner else np.array([h, h, h])  # the element of the first sources
    src = []
    for i in range(9):
        x, y, z = o + h * np.array([0.15 + 0.09 * i, 0.8 - 0.05 * i, 0.3 + 0.02 * i])
        src.append(dict(type="force", x=x, y=y, z=z, fx=0.3, fy=-0.5, fz=0.1 * i, f0=15.0 + i, factor=1e10))
        if i % 3 == 1:  # another element between them, where there is one
            x, y, z = (np.array(n) - 0.4) * h if corner else o + 0.5 * h
            src.append(dict(type="force", x=x, y=y, z=z, fx=1.0, fy=0.2, fz=0.4, f0=12.0, factor=1e10))
    top = np.array(n) * h
    rec = [dict(zip("xyz", p)) for p in (np.zeros(3), top, top * [0.5, 1, 1], top * [0.3, 0.4, 1], 0.37 * top,
                                         np.array([h, min(h, top[1]), 0.5 * h]))]
    print(f"[case] 3-D gather {n} corner={corner} {types}", flush=True)
    e = Engine3D(mesh, src, rec, dt, nstep, 1, types, scatter="gather")
    e.initialize()
    e.run()
    s = e.seismograms().astype(np.float64)
    e.close()
    r32, _ = oracle.Oracle3D(mesh, 4, dt).forward(src, rec, nstep, dt, 1, types)
    r64, _ = oracle.Oracle3D(mesh, 8, dt).forward(src, rec, nstep, dt, 1, types)
    for it, t in enumerate(types):
        e32, e64, floor = rel_l2(s[:, it], r32[:, it]), rel_l2(s[:, it], r64[:, it]), rel_l2(r32[:, it], r64[:, it])
        print(f"[report] {t} {e32:.2e} {e64:.2e} {floor:.2e}", flush=True)
        assert e32 <= 1e-5 or e64 <= 1.5 * floor
