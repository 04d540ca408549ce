"""3-D database meshes, default scatter: element forces stored and summed per
point.  Sizes at the edges of the launch (one element, a count that is not a
multiple of the five elements a workgroup holds), meshes with only regular and
with irregular elements, without sources, receivers or absorbing faces, and a
source element with several sources on an absorbing corner, against the FP32
oracle (displacement within 1e-5 relative L2, as in the other parity tests) and
the seam calls (final state within FP32 rounding, 1e-6)."""
import numpy as np
import pytest

import oracle
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,perturb,absorbing,nsrc", [((1, 1, 1), 0.0, (1, 1, 1, 1, 1, 0), 3),
                                                      ((3, 2, 2), 0.0, (0, 0, 0, 0, 0, 0), 1),
                                                      ((4, 3, 3), 0.1, (1, 0, 1, 0, 1, 0), 3),
                                                      ((2, 3, 1), 0.1, (1, 1, 1, 1, 1, 0), 0)])
def test_database_sums(n, perturb, absorbing, nsrc):
    from specfempp_amd import Engine3DDatabase, meshes

    h, dt, nstep = 100.0, 1e-3, 60
    db = meshes.hex_database(*n, h, np.zeros(n[::-1], np.int32), [2500.0], [3000.0], [1730.0], absorbing=absorbing,
                             perturb=perturb, seed=1, dt=dt)
    src = [dict(type="force", x=30.0, y=40.0, z=20.0, fx=0.3, fy=-0.5, fz=0.8, f0=30.0, factor=1e10),
           dict(type="moment_tensor", x=15.0, y=20.0, z=35.0, mxx=0.3, myy=-0.5, mzz=0.8, mxy=0.2, mxz=-0.1, myz=0.4,
                f0=30.0, factor=1e12),
           dict(type="force", x=h * n[0] - 12.0, y=30.0, z=45.0, fx=1.0, fy=0.2, fz=0.1, f0=25.0, factor=1e10)][:nsrc]
    rec = [dict(x=55.0, y=60.0, z=h * n[2]), dict(x=h * n[0] - 20.0, y=h * n[1] - 30.0, z=40.0)] if nsrc else []
    print(f"[case] database sums {n} perturb={perturb} absorbing={absorbing} nsrc={nsrc}", flush=True)

    def engine():
        e = Engine3DDatabase(db, src, rec, dt, nstep, 1, ("displacement", "velocity"))
        e.initialize()
        return e

    e = engine()
    e.run()
    seis, u = e.seismograms(), e.field("displacement")
    e.close()
    e = engine()
    for i in range(nstep):
        e.update_wavefields(i)
        e.apply_corrector_phase()
        e.apply_predictor_phase()
    # the fused pass and the separate phases contract their products alike or
    # differ by roundings
    assert not u.any() or rel_l2(e.field("displacement").astype(float), u.astype(float)) <= 1e-6
    e.close()
    if nsrc:
        ref, _ = oracle.Oracle3D.from_database(db, 4, dt).forward(src, rec, nstep, dt, 1, ("displacement",))
        assert rel_l2(seis[:, 0].astype(float), ref[:, 0]) <= 1e-5
    else:
        assert not u.any()
