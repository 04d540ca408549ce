"""2-D forward steps run patch by patch: sizes at the edges of the partition
(one element, one full small patch, one element more, strips, the first mesh
with large patches), elements listed in random order, several sources in one
element, receivers on shared points, every trace type, and the same run cut
into calls of one and several steps.

Bars, as in the other forward parity tests: displacement within 1e-5 relative
L2 of the FP32 oracle, other types on the FP32 rounding-floor rule; a run cut
into pieces equals the whole run bit for bit."""
import numpy as np
import pytest

import oracle
from conftest import rel_l2
from test_gpu_parity import _check, _report

pytestmark = pytest.mark.gpu

TYPES = ("displacement", "velocity", "acceleration", "pressure")


def _case(nx, nz, shuffle, nstep):
    from specfempp_amd import meshes

    h = 20.0
    mesh = meshes.quad_mesh(nx, nz, 0.0, nx * h, 0.0, nz * h, materials=[meshes.elastic(2000.0, 2500.0, 1400.0),
                                                                       meshes.elastic(2300.0, 3000.0, 1700.0)],
                            material=(np.arange(nx * nz).reshape(nz, nx) % 2).astype(np.int32))
    rng = np.random.default_rng(nx * 1000 + nz)
    if shuffle:
        order = rng.permutation(mesh.nspec)
        place = np.empty_like(order)
        place[order] = np.arange(mesh.nspec)
        mesh.knods, mesh.kmato = mesh.knods[:, order].copy(), mesh.kmato[order].copy()
        mesh.abs_ispec = place[mesh.abs_ispec].astype(np.int32)
    x, z = (nx // 2 + 0.3) * h, (nz // 2 + 0.6) * h
    src = [dict(x=x, z=z, angle=30.0, f0=40.0, factor=1e10), dict(x=x + 2.0, z=z - 3.0, angle=75.0, f0=30.0, factor=2e9),
           dict(type="moment_tensor", x=0.4 * h, z=0.7 * h, mxx=1.0, mzz=-0.5, mxz=0.3, f0=40.0, factor=1e10)]
    # corners, edges and interiors of elements near the sources
    rec = [dict(x=float(np.clip(x + dx * h, 0, nx * h)), z=float(np.clip(z + dz * h, 0, nz * h)))
           for dx, dz in ((-0.3, 0.4), (0.7, -0.6), (-0.3, -0.1), (0.2, 0.4), (-1.3, -0.6), (0.1, 0.1))]
    return mesh, src, rec, meshes.stable_dt(h, 3000.0), nstep


@pytest.mark.parametrize("scatter", ["gather", "colored"])
@pytest.mark.parametrize("nx,nz,shuffle", [(1, 1, False), (5, 5, False), (26, 1, False), (1, 30, True), (13, 9, True),
                                           (161, 150, False)])
def test_patches_match_oracle(nx, nz, shuffle, scatter):
    from specfempp_amd import Engine2D

    mesh, src, rec, dt, nstep = _case(nx, nz, shuffle, 90)
    print(f"[case] patches {nx}x{nz} shuffle={shuffle} {scatter}", flush=True)

    def engine():
        e = Engine2D(mesh, src, rec, dt, nstep, 2, TYPES, scatter=scatter)
        e.initialize()
        return e

    e = engine()
    e.run()
    ours, last = e.seismograms(), e.field("displacement")
    e.close()
    e = engine()
    e.run(0, 1)
    e.run(1, 2)
    e.step(3)
    e.run(4, 31)
    e.run(35)
    assert np.array_equal(e.seismograms(), ours)
    assert np.array_equal(e.field("displacement"), last)
    e.close()
    s32, _ = oracle.Oracle2D(mesh, 4, 1, dt).forward(src, rec, nstep, dt, 2, TYPES)
    s64, _ = oracle.Oracle2D(mesh, 8, 1, dt).forward(src, rec, nstep, dt, 2, TYPES)
    for it, t in enumerate(TYPES):
        a, b32, b64 = ours[:, it].astype(np.float64), s32[:, it], s64[:, it]
        e32, e64, floor = rel_l2(a, b32), rel_l2(a, b64), rel_l2(b32, b64)
        _report(f"patches_{nx}x{nz}_{scatter}/{t}", vs_oracle_fp32=e32, vs_oracle_fp64=e64, fp32_floor=floor)
        if t == "displacement":
            assert e32 <= 1e-5
        else:
            _check(e32, e64, floor)
