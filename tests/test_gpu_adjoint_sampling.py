"""Recorded and combined runs that sample every second or third step: the
sample rows of the backward run count from the latest sampled step, whichever
phase of the loop takes them (first step, checkpoint step, runs of combined
steps between).  Numbers of steps whose last is sampled or not, checkpoints on
sampled steps and beside them, receivers inside patches, on shared points of
several elements and on the mesh's edge.

Against the atomic scatter, whose loop runs step by step: both are FP32 sums of
the same terms in another order.  Traces and kernels agree within 1e-4
relative L2, the bar of the combined loop's seam test (the kernels are sums of
products of two wavefields, and the backward field is a reconstruction); a
sample in another row differs by its own size, as the rows are of different
steps."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TYPES = ("displacement", "velocity", "acceleration")


@pytest.mark.parametrize("nstep,every,snapshots", [(120, 1, 0), (121, 2, 0), (120, 2, 7), (121, 3, 0), (120, 3, 9),
                                                   (119, 3, 10), (4, 3, 2), (3, 2, 1), (2, 3, 0)])
def test_sampling_intervals(nstep, every, snapshots):
    from specfempp_amd import Engine2D, meshes

    nx, nz, h = 13, 9, 20.0
    mesh = meshes.quad_mesh(nx, nz, 0.0, nx * h, 0.0, nz * h, materials=[meshes.elastic(2000.0, 2500.0, 1400.0)])
    dt = meshes.stable_dt(h, 2500.0)
    src = [dict(x=6.4 * h, z=4.3 * h, angle=30.0, f0=40.0, factor=1e10, tshift=-0.02)]
    rec = [dict(x=6.0 * h, z=4.0 * h), dict(x=7.3 * h, z=5.0 * h), dict(x=5.5 * h, z=3.5 * h), dict(x=7.3 * h, z=0.0),
           dict(x=8.0 * h, z=4.4 * h)]
    print(f"[case] sampling nstep={nstep} every={every} snapshots={snapshots}", flush=True)
    rng = np.random.default_rng(nstep)
    stf = 1e-6 * rng.standard_normal((len(rec), nstep, 2))
    out = []
    for scatter in ("colored", "atomic"):
        e = Engine2D(mesh, src, rec, dt, nstep, every, TYPES, scatter=scatter)
        u0 = 1e-3 * np.random.default_rng(7).standard_normal(e.field("displacement").shape)
        e.initialize()
        e.set_field("displacement", u0.astype(np.float32))
        e.forward_record(snapshots)
        got = [e.seismograms()]
        e.set_adjoint_sources(rec, stf)
        e.adjoint_run()
        back, k = e.seismograms(), e.kernels()
        got += [back[:, i] for i in range(len(TYPES))] + [k[n] for n in sorted(k)]
        e.close()
        assert got[0].shape[0] == (nstep + every - 1) // every
        out.append([np.asarray(a, np.float64) for a in got])
    for a, b in zip(*out):
        if b.any():
            assert rel_l2(a, b) <= 1e-4
        else:
            assert not a.any()
    # samples of neighbouring rows differ by more than the bar
    rows = out[1][1]
    if rows.shape[0] > 1:
        assert all(rel_l2(rows[i], rows[i + 1]) > 1e-2 for i in range(rows.shape[0] - 1))
