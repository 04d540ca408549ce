"""A force held in the stored acceleration between predictor and update joins
the step's own forces: the update phase sums into the acceleration before the
mass division (domain_kernels.hpp:69-126), and a fused step or run starts from
what the predictor left and the caller set.  The default scatter (2-D patches
of both sizes, 3-D database sums) against the atomic one, whose kernels add to
the stored array itself.  Both are FP32 sums of the same terms in another
order, so fields, traces and records agree within 1e-5 relative L2, the bar of
the parity tests; the force is as large as the step's own, so that leaving it
out changes the result by its own size."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

NSTEP = 6
FIELDS = ("displacement", "velocity", "acceleration")


def _engine(kind, scatter):
    from specfempp_amd import Engine2D, Engine3DDatabase, meshes

    if kind == "database":
        db = meshes.hex_database(4, 3, 3, 100.0, np.zeros((3, 3, 4), np.int32), [2500.0], [3000.0], [1730.0],
                                 perturb=0.1, seed=2, dt=1e-3)
        src = [dict(type="force", x=140.0, y=160.0, z=130.0, fx=0.3, fy=-0.5, fz=0.8, f0=30.0, factor=1e10)]
        rec = [dict(x=150.0, y=150.0, z=150.0)]
        e = Engine3DDatabase(db, src, rec, 1e-3, NSTEP, 1, FIELDS, scatter=scatter)
    else:
        nx, nz = (13, 9) if kind == "small" else (161, 150)
        h = 20.0
        mesh = meshes.quad_mesh(nx, nz, 0.0, nx * h, 0.0, nz * h, materials=[meshes.elastic(2000.0, 2500.0, 1400.0)])
        src = [dict(x=6.4 * h, z=4.3 * h, angle=30.0, f0=40.0, factor=1e10)]
        rec = [dict(x=6.0 * h, z=4.0 * h), dict(x=7.3 * h, z=0.0)]
        e = Engine2D(mesh, src, rec, meshes.stable_dt(h, 2500.0), NSTEP, 1, FIELDS, scatter=scatter)
    e.initialize()
    return e


def _call(e, call):
    if call == "update":
        e.update_wavefields(1)
        return []
    if call == "step":
        e.step(1)
        e.run(2, 2)
    elif call == "run":
        e.run(0, 4)
    else:
        e.forward_record(2 if call == "record" else 1)
        return [e.seismograms(), e.stacey_record()]
    return [e.seismograms()]


@pytest.mark.parametrize("kind,call", [(k, c) for k in ("small", "large") for c in ("update", "step", "run", "record", "record_every")]
                         + [("database", c) for c in ("update", "step", "run")])
def test_stored_force_joins_the_step(kind, call):
    print(f"[case] stored force {kind} {call}", flush=True)
    rng = np.random.default_rng(5)
    e = _engine(kind, "atomic")
    u = (1e-3 * rng.standard_normal(e.field("displacement").shape)).astype(np.float32)
    e.set_field("displacement", u)
    e.update_wavefields(0)
    own = e.field("acceleration") / e.field("mass_inverse")
    e.close()
    force = (own.std() * rng.standard_normal(u.shape)).astype(np.float32)
    out = {}
    for scatter, with_force in (("colored", True), ("atomic", True), ("atomic", False)):
        e = _engine(kind, scatter)
        e.set_field("displacement", u)
        e.apply_predictor_phase()
        if with_force:
            e.set_field("acceleration", force)
        got = _call(e, call)
        out[scatter, with_force] = [np.asarray(a, np.float64) for a in got + [e.field(k) for k in FIELDS]]
        e.close()
    for i, (a, b, c) in enumerate(zip(out["colored", True], out["atomic", True], out["atomic", False])):
        if not b.any():
            assert not a.any()
            continue
        print(f"  output {i}: {rel_l2(a, b):.2e}, the force makes {rel_l2(c, b):.2e}", flush=True)
        assert rel_l2(a, b) <= 1e-5
    assert max(rel_l2(c, b) for b, c in zip(out["atomic", True], out["atomic", False]) if b.any()) > 1e-2


@pytest.mark.parametrize("kind", ["small", "database"])
def test_a_stored_zero_keeps_the_bits(kind):
    """A run that goes on from read and written fields (a restart) is the run."""
    print(f"[case] stored zero {kind}", flush=True)
    out = []
    for restart in (False, True):
        e = _engine(kind, "colored")
        e.run(0, 3)
        if restart:
            for k in FIELDS:
                e.set_field(k, e.field(k))
        e.run(3, 3)
        out.append([e.seismograms()] + [e.field(k) for k in FIELDS])
        e.close()
    assert all(np.array_equal(a, b) for a, b in zip(*out))
