"""Meshes with acoustic elements, default scatter: forces of both media stored
in one launch and summed per point.  Sizes at the edges of the launches (fewer
elements than a workgroup's five, counts that are no multiple of it, a receiver
and source count of one), against the atomic scatter's separate launches: both
are FP32 sums of the same terms in another order, so all trace kinds and the
final fields agree within 1e-5 relative L2, the bar of the parity tests."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TYPES = ("displacement", "velocity", "acceleration", "pressure")


def _mesh(nx, nz, water, h):
    """nz rows of nx elements of side h, the top `water` of them water."""
    from specfempp_amd import meshes

    mat = np.zeros((nz, nx), np.int32)
    mat[nz - water:] = 1
    m = meshes.quad_mesh(nx, nz, 0.0, nx * h, 0.0, nz * h, mat,
                         meshes.MaterialArrays([2500.0, 1020.0], [3000.0, 1500.0], [1700.0, 0.0]))
    m.afs_ispec = ((nz - 1) * nx + np.arange(nx)).astype(np.int32)
    m.afs_type = np.full(nx, 3, np.int32)
    if water < nz:
        m.fs_acoustic = ((nz - water) * nx + np.arange(nx)).astype(np.int32)
        m.fs_elastic = ((nz - water - 1) * nx + np.arange(nx)).astype(np.int32)
    return m


@pytest.mark.parametrize("nx,nz,water,every", [(1, 2, 1, 1), (3, 4, 2, 3), (7, 5, 5, 1), (13, 9, 3, 2)])
def test_coupled_sums(nx, nz, water, every):
    from specfempp_amd import Engine2D

    h, dt, nstep = 25.0, 3e-4, 60
    x, top = nx * h, nz * h
    src = [dict(type="force", x=0.4 * x, z=top - 0.6 * h, angle=0.0, f0=25.0, factor=1e6)]
    rec = [dict(x=0.7 * x, z=top - 0.3 * h)]
    if water < nz:
        src += [dict(type="force", x=0.3 * x, z=0.4 * h, angle=30.0, f0=20.0, factor=1e9),
                dict(type="force", x=0.32 * x, z=0.45 * h, angle=70.0, f0=30.0, factor=1e9)]
        rec += [dict(x=0.6 * x, z=0.7 * h), dict(x=0.2 * x, z=(nz - water) * h - 2.0)]
    print(f"[case] coupled sums {nx}x{nz} water={water} every={every}", flush=True)
    out = []
    for scatter in ("colored", "atomic"):
        e = Engine2D(_mesh(nx, nz, water, h), src, rec, dt, nstep, every, TYPES, scatter=scatter)
        assert e.nspec_acoustic == nx * water
        e.initialize()
        e.run(0, 17)
        e.step(17)
        e.run(18, nstep - 18)
        s = e.seismograms().astype(np.float64)
        f = [e.acoustic_field(k).astype(np.float64) for k in ("displacement", "velocity", "acceleration")]
        if water < nz:
            f += [e.field(k).astype(np.float64) for k in ("displacement", "velocity", "acceleration")]
        out.append(([s[:, it] for it in range(len(TYPES))], f))
        e.close()
    for (a, b) in zip(out[0][0] + out[0][1], out[1][0] + out[1][1]):
        if b.any():
            assert rel_l2(a, b) <= 1e-5
        else:
            assert not a.any()
