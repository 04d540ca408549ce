"""The work a user of this library has it do, as measurable cases.

Every case is one pass of a wave-propagation program through the public entry
points: forward simulations (2-D quads, structured 3-D cubes, 3-D mesh
databases, elastic-acoustic meshes), wavefield snapshots, the solver's loop
driven seam by seam, an adjoint gradient, a batch of events.  Engines are
built by ``prepare`` (a program builds one and steps it); ``run`` steps it and
reads the results back.

All meshes are grids of quads or hexahedra whose corner nodes may be moved.
Sources (a finite fault of forces or moment tensors) and receivers are drawn
within a few elements of each other, and the Ricker frequency is set by the
element size (about 3.5 elements per P wavelength), so that the recorded
waves are fully developed within a pass.

``exact`` integrates the same Newmark / spectral-element equations (NGLL = 5)
in float64 with torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from specfempp_amd import Batch, Engine2D, Engine3D, Engine3DDatabase, meshes
from specfempp_amd.io.database3d import Faces, Mesh3DDatabase
from specfempp_amd.io.fortran_db import EDGE_TOP
from specfempp_amd.solver import Newmark, TimeMarching

GLL_X = np.array([-1.0, -math.sqrt(3.0 / 7.0), 0.0, math.sqrt(3.0 / 7.0), 1.0])
GLL_W = np.array([0.1, 49.0 / 90.0, 32.0 / 45.0, 49.0 / 90.0, 0.1])
FIELDS = ("displacement", "velocity", "acceleration")
DVA = ",".join(FIELDS)
# float64 point-steps (points x steps x components) one exact() may integrate
EXACT_LIMIT = 6.0e9


def _case(name, kind, n, steps, h=50.0, medium="homogeneous", distort=0.0, scatter="default", types="displacement",
          every=1, nsrc=4, nrec=32, source="force", **more):
    return dict(name=name, kind=kind, n="x".join(map(str, n)), steps=steps, h=h, medium=medium, distort=distort,
                scatter=scatter, types=types, every=every, nsrc=nsrc, nrec=nrec, source=source, **more)


def listed():
    return [
        # the smallest calls: a SPECFEM++ solver driving predictor, update,
        # corrector and sampling one by one on a toy mesh (latency only)
        _case("seams_2d_11x9", "seams", (11, 9), 40, types=DVA, nsrc=1, nrec=3),
        # the usual first simulation: homogeneous 80x80 quads, one vertical
        # force, a line of receivers, every option left at its default
        _case("forward_2d_80x80", "forward", (80, 80), 400, nsrc=1, nrec=50),
        # a meshed domain that is not affine, layers, all trace types, every
        # third step sampled, moment tensors, deterministic gather sums
        _case("forward_2d_moved_177x131", "forward", (177, 131), 240, h=20.0, medium="layers", distort=0.2,
              scatter="gather", types=DVA, every=3, nsrc=3, nrec=41, source="moment_tensor"),
        # a large heterogeneous medium, one material per element
        _case("forward_2d_random_1000x900", "forward", (1000, 900), 100, h=2.5, medium="random", scatter="gather",
              nsrc=64, nrec=200),
        # run to a time and keep the whole wavefield (movie, checkpoint)
        _case("snapshot_2d_301x203", "snapshot", (301, 203), 80, medium="layers", nsrc=8, nrec=16),
        # a small 3-D model with all trace types and its final wavefield
        _case("snapshot_3d_9x11x7", "snapshot", (9, 11, 7), 160, h=100.0, medium="layers", types=DVA, nsrc=2, nrec=9,
              source="moment_tensor"),
        # a medium 3-D model of odd sides, velocity traces
        _case("forward_3d_37x29x41", "forward", (37, 29, 41), 100, h=100.0, medium="random", types="velocity",
              nsrc=8, nrec=60, source="force"),
        # the headline: the layered 64^3 cube
        _case("forward_3d_64x64x64", "forward", (64, 64, 64), 100, h=100.0, medium="layers", nsrc=16, nrec=400,
              source="moment_tensor"),
        # a general hexahedral mesh from a 3-D database, half of it irregular
        _case("database_3d_26x22x18", "database", (26, 22, 18), 100, h=100.0, medium="layers", distort=0.12,
              types="displacement,velocity", nsrc=3, nrec=20, source="moment_tensor"),
        # marine model: water over rock, free surface, an air gun, hydrophones
        # and ocean-bottom receivers
        _case("coupled_2d_120x80", "coupled", (120, 80), 300, h=25.0, nsrc=2, nrec=40, types="displacement,pressure"),
        # one gradient of an inversion: recorded forward run, adjoint run with
        # checkpoints, all six kernels
        _case("gradient_2d_100x100", "gradient", (100, 100), 300, h=20.0, medium="layers", nsrc=8, nrec=100,
              snapshots=55),
        # many small events at once
        _case("batch_2d_16_events", "batch", (20, 120), 200, nsrc=1, nrec=32, events=16),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["seams", "forward", "forward", "forward", "snapshot", "forward3", "forward3", "snapshot3",
                       "database", "coupled", "gradient", "batch"])
    medium = rng.choice(["homogeneous", "layers", "random"])
    types = rng.choice(["displacement", "velocity", "displacement,velocity", DVA])
    every = rng.choice([1, 1, 2, 5])
    source = rng.choice(["force", "moment_tensor"])
    opt = dict(medium=medium, types=types, every=every, source=source, nsrc=rng.randint(1, 12),
               nrec=rng.randint(1, 120))
    if kind == "seams":
        return _case("", "seams", (size(3, 30), size(3, 30)), rng.randint(20, 60),
                     **dict(opt, scatter=rng.choice(["default", "gather"])))
    if kind in ("forward", "snapshot"):
        nx, nz = size(4, 900), size(4, 900)
        steps = max(20, min(rng.randint(80, 400), int(9.0e7 / (nx * nz))))
        return _case("", kind, (nx, nz), steps, h=rng.choice([2.5, 20.0, 50.0]),
                     distort=rng.choice([0.0, 0.0, 0.2]), scatter=rng.choice(["default", "gather", "gather", "atomic"]),
                     **opt)
    if kind in ("forward3", "snapshot3"):
        n = (size(2, 60), size(2, 60), size(2, 60))
        steps = max(20, min(rng.randint(60, 200), int(2.6e7 / (n[0] * n[1] * n[2]))))
        return _case("", kind[:-1], n, steps, h=100.0, **opt)
    if kind == "database":
        n = (size(2, 26), size(2, 22), size(2, 18))
        return _case("", "database", n, rng.randint(60, 100), h=100.0, distort=rng.choice([0.0, 0.12]),
                     scatter=rng.choice(["default", "atomic"]), **opt)
    if kind == "coupled":
        return _case("", "coupled", (size(8, 160), size(8, 100)), rng.randint(80, 200), h=25.0, types=types, every=every,
                     nsrc=rng.randint(1, 3), nrec=rng.randint(2, 60))
    if kind == "gradient":
        nx, nz = size(6, 130), size(6, 110)
        return _case("", "gradient", (nx, nz), rng.randint(80, 250), h=20.0, medium=medium, nsrc=rng.randint(1, 8),
                     nrec=rng.randint(1, 100), snapshots=rng.choice([0, 40, 55]))
    lo = rng.randint(6, 40)
    return _case("", "batch", (lo, lo + rng.randint(1, 80)), rng.randint(80, 200), types=rng.choice(["displacement", DVA]),
                 nsrc=rng.randint(1, 2), nrec=rng.randint(1, 32), events=rng.randint(2, 16))


# ---------------------------------------------------------------------------
# The model of a case: grid, materials, sources, receivers (float64, host)
# ---------------------------------------------------------------------------
class Model:
    """A grid of nx (x ny) x nz elements of size h, elements x fastest, z up.
    The free surface is the top; the other sides absorb."""

    def __init__(self, case, rng, n=None):
        self.n = n if n is not None else tuple(int(s) for s in case["n"].split("x"))
        self.dim, self.h = len(self.n), case["h"]
        self.nspec = int(np.prod(self.n))
        self.regular = case["distort"] == 0.0
        self.types = tuple(case["types"].split(","))
        self.every, self.steps = case["every"], case["steps"]
        self.water = case["kind"] == "coupled"
        # corner nodes (..., z, [y,] x, component), x first; the interior ones
        # may be moved: all of them in 2-D, the lower half along x in 3-D
        axes = [np.arange(m + 1) * self.h for m in self.n]
        self.nodes = np.stack(np.meshgrid(*axes[::-1], indexing="ij")[::-1], axis=-1)
        if not self.regular:
            inner = tuple(slice(1, m) for m in self.n[::-1])
            if self.dim == 3:
                inner = inner[:2] + (slice(1, self.n[0] // 2 + 1) if self.n[0] > 2 else slice(1, self.n[0]),)
            d = case["distort"] * self.h
            self.nodes[inner] += rng.uniform(-d, d, size=self.nodes[inner].shape)
        self._materials(case["medium"], rng)
        dt = 0.4 * 0.5 * (GLL_X[1] - GLL_X[0]) * self.h / self.vp.max()
        self.dt = float(np.float32(dt if self.regular else 0.6 * dt))
        self._points(case, rng)

    def _materials(self, medium, rng):
        n = self.n
        z = np.broadcast_to(np.arange(n[-1]).reshape((-1,) + (1,) * (self.dim - 1)), n[::-1])
        vp0 = rng.uniform(2500.0, 4000.0)
        if self.water:
            # the upper third is water: one horizontal interface
            self.wet = z >= n[-1] - max(1, n[-1] // 3)
            vp = np.where(self.wet, 1500.0, vp0)
            vs, rho = np.where(self.wet, 0.0, vp / math.sqrt(3.0)), np.where(self.wet, 1020.0, 2500.0)
            index = self.wet.astype(np.int32)
            pick = [tuple(int(i) for i in np.argwhere(~self.wet)[0]), tuple(int(i) for i in np.argwhere(self.wet)[0])]
        elif medium == "random":
            # smooth random velocity, one material per element
            g = np.zeros(n[::-1])
            grid = np.meshgrid(*[np.arange(m) * 1.0 for m in n[::-1]], indexing="ij")
            for _ in range(6):
                k = rng.normal(size=self.dim) * 0.3
                g += np.cos(sum(a * b for a, b in zip(k, grid)) + rng.uniform(0, 2 * np.pi)) / 6
            vp = vp0 * (1.0 + 0.2 * g)
            vs, rho = vp / math.sqrt(3.0), 310.0 * vp ** 0.25
            index, pick = np.arange(self.nspec, dtype=np.int32).reshape(n[::-1]), None
        else:
            layers = 1 if medium == "homogeneous" else min(4, n[-1])
            v = np.sort(rng.uniform(2000.0, 5000.0, size=layers))[::-1] if layers > 1 else np.array([vp0])
            index = (z * layers // n[-1]).astype(np.int32)
            vp = v[index]
            vs, rho = vp / 1.73, 2000.0 + 0.15 * vp
            pick = [tuple(int(i) for i in np.argwhere(index == m)[0]) for m in range(layers)]
        self.vp, self.vs, self.rho = vp.astype(np.float64), vs.astype(np.float64), rho.astype(np.float64)
        self.material = np.ascontiguousarray(index)
        # material table (rho, vp, vs)
        self.table = [(a.ravel() if pick is None else np.array([a[p] for p in pick])) for a in (self.rho, self.vp, self.vs)]

    def _points(self, case, rng):
        """Sources and receivers at seeded reference coordinates of elements;
        receivers within three elements of a source."""
        n, dim = np.array(self.n), self.dim

        def local():
            return rng.uniform(-0.85, 0.85, size=dim)

        f0 = float(np.median(self.vp)) / (3.5 * self.h)
        self.sources, self.receivers = [], []
        low = np.zeros(dim, int)
        if self.water:
            # air guns in the water
            low[-1] = int(np.argmax(self.wet[:, 0]))
            f0 = 1500.0 / (3.5 * self.h)
        for _ in range(case["nsrc"]):
            e = np.array([rng.integers(lo, m) for lo, m in zip(low, n)])
            r = local()
            s = dict(zip("xyz" if dim == 3 else "xz", (float(v) for v in self.position(e, r))))
            s.update(type=case["source"], f0=f0 * float(rng.uniform(0.8, 1.2)), tshift=0.0, factor=1e10)
            if case["source"] == "moment_tensor":
                m = rng.normal(size=6)
                names = ("mxx", "mzz", "mxz") if dim == 2 else ("mxx", "myy", "mzz", "mxy", "mxz", "myz")
                s.update({k: float(v) for k, v in zip(names, m)})
            elif dim == 2:
                s["angle"] = float(rng.uniform(0.0, 360.0))
            else:
                s.update({k: float(v) for k, v in zip(("fx", "fy", "fz"), rng.normal(size=3))})
            self.sources.append((s, e, r))
        for _ in range(case["nrec"]):
            c = self.sources[rng.integers(len(self.sources))][1]
            e = np.clip(c + rng.integers(-3, 4, size=dim), 0, n - 1)
            r = local()
            self.receivers.append((dict(zip("xyz" if dim == 3 else "xz", (float(v) for v in self.position(e, r)))), e, r))

    def corners(self, e):
        """(2^dim, dim) corner nodes of element e = (ex, [ey,] ez); corner c
        has bit s set on the upper side of axis s."""
        return np.array([self.nodes[tuple(int(e[s]) + ((c >> s) & 1) for s in reversed(range(self.dim)))]
                         for c in range(1 << self.dim)])

    def position(self, e, r):
        sign = np.array([[((c >> s) & 1) * 2 - 1 for s in range(self.dim)] for c in range(1 << self.dim)])
        return np.prod(0.5 * (1 + sign * r), axis=1) @ self.corners(e)

    # ---- meshes of the public entry points ----
    def mesh2d(self):
        nx, nz = self.n
        rho, vp, vs = self.table
        m = meshes.quad_mesh(nx, nz, 0.0, nx * self.h, 0.0, nz * self.h, self.material,
                             meshes.MaterialArrays(rho, vp, vs))
        if not self.regular:
            m.coorg = np.ascontiguousarray(self.nodes.reshape(-1, 2).T)
        if self.water:
            top = (nz - 1) * nx + np.arange(nx, dtype=np.int32)
            m.afs_ispec, m.afs_type = top.astype(np.int32), np.full(nx, EDGE_TOP, np.int32)
            iz = int(np.argmax(self.wet[:, 0]))
            m.fs_acoustic = (iz * nx + np.arange(nx)).astype(np.int32)
            m.fs_elastic = ((iz - 1) * nx + np.arange(nx)).astype(np.int32)
        return m

    def mesh3d(self):
        rho, vp, vs = self.table
        return meshes.hex_mesh(*self.n, self.h, self.material, rho, vp, vs)

    def database(self):
        """The arrays read_3d_mesh holds, from the float64 geometry."""
        g = Geometry(self, "cpu")
        nspec, f4 = self.nspec, (self.nspec, 5, 5, 5)
        moved = np.zeros(self.nodes.shape[:3], bool)
        base = np.stack(np.meshgrid(*[np.arange(m + 1) * self.h for m in self.n][::-1], indexing="ij")[::-1], -1)
        moved[np.any(self.nodes != base, axis=-1)] = True
        irr = np.zeros(self.n[::-1], bool)
        for c in range(8):
            irr |= moved[(c >> 2) & 1:, (c >> 1) & 1:, c & 1:][:self.n[2], :self.n[1], :self.n[0]]
        inv = np.broadcast_to(g.inv.numpy(), (nspec, 125, 3, 3))
        jac = np.broadcast_to(g.jac.numpy(), (nspec, 125))
        d = {a + b: inv[:, :, s, r].reshape(f4).astype(np.float32) for s, a in enumerate(("xi", "eta", "gamma"))
             for r, b in enumerate("xyz")}
        d["jacobian"] = jac.reshape(f4).astype(np.float32)

        def point(v):
            return np.repeat(v.ravel(), 125).reshape(f4).astype(np.float32)

        rho, vp, vs = self.rho, self.vp, self.vs
        xyz = np.zeros((g.nglob, 3), np.float32)
        xyz[g.gather.numpy().ravel()] = g.xyz.reshape(-1, 3)
        db = Mesh3DDatabase(dict(nspec=nspec, nglob=g.nglob), g.gather.numpy().reshape(f4).astype(np.int32), xyz[:, 0],
                            xyz[:, 1], xyz[:, 2], np.flatnonzero(irr.ravel()).astype(np.int32), np.float32(2.0 / self.h),
                            np.float32((self.h / 2) ** 3), d, point(rho * (vp ** 2 - 4.0 / 3.0 * vs ** 2)),
                            point(rho * vs ** 2), point(rho), np.ones(nspec, np.int32))
        db.rho_vp, db.rho_vs = point(rho * vp), point(rho * vs)
        nf = len(g.face_elem) // 25
        p = g.face_point.reshape(nf, 25)
        db.absorbing = Faces(g.face_elem.reshape(nf, 25)[:, 0].astype(np.int32),
                             np.stack([p % 5, p // 5 % 5, p // 25], axis=1).astype(np.int32),
                             (g.face_area * g.face_weight).reshape(nf, 25).astype(np.float32),
                             g.face_normal.reshape(nf, 25, 3).transpose(0, 2, 1).astype(np.float32))
        return db

    def engine(self, case):
        src, rec = [s for s, _, _ in self.sources], [r for r, _, _ in self.receivers]
        opt = {} if case["scatter"] == "default" else {"scatter": case["scatter"]}
        args = (src, rec, self.dt, self.steps, self.every, self.types)
        if case["kind"] == "database":
            return Engine3DDatabase(self.database(), *args, **opt)
        return Engine3D(self.mesh3d(), *args, **opt) if self.dim == 3 else Engine2D(self.mesh2d(), *args, **opt)


def _models(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] != "batch":
        return [Model(case, rng)]
    # sides spread over the range, the larger events with the fewer steps
    lo, hi = (int(s) for s in case["n"].split("x"))
    out = []
    for i in range(case["events"]):
        f = i / max(case["events"] - 1, 1)
        side, steps = int(round(lo + f * (hi - lo))), int(round(case["steps"] * (1.0 - 0.5 * f)))
        out.append(Model(dict(case, steps=steps), rng, (side, side)))
    return out


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def prepare(case, seed):
    ms = _models(case, seed)
    engines = [m.engine(case) for m in ms]
    state = dict(case=case, models=ms, engine=engines[0])
    if case["kind"] == "batch":
        state["batch"] = Batch(engines)
    return state


def _traces(seismograms):
    """The recorded traces by type, each (samples, receivers, components)."""
    return [seismograms[:, i] for i in range(seismograms.shape[1])]


def run(state):
    case, eng, kind = state["case"], state["engine"], state["case"]["kind"]
    steps = case["steps"]
    if kind == "batch":
        batch = state["batch"]
        batch.run()
        return [_traces(batch.seismograms(i)) for i in range(len(state["models"]))]
    if kind == "seams":
        ts = Newmark(steps, case["every"], eng.dt, "forward")
        ts.link_assembly(eng)
        TimeMarching(eng, ts).run()
        return dict({t: eng.field(t) for t in FIELDS}, seismograms=_traces(eng.seismograms()))
    eng.initialize()
    if kind == "snapshot":
        eng.run(0, steps - 1)
        eng.update_wavefields(steps - 1)
        eng.apply_corrector_phase()
        if (steps - 1) % case["every"] == 0:
            eng.compute_seismograms((steps - 1) // case["every"])
        return dict({t: eng.field(t) for t in FIELDS}, seismograms=_traces(eng.seismograms()))
    if kind == "gradient":
        m = state["models"][0]
        eng.forward_record(case["snapshots"])
        u = eng.seismograms()
        # the gradient of the energy sum(u^2) / 2 dt at the receivers
        eng.set_adjoint_sources([r for r, _, _ in m.receivers], np.transpose(u[:, 0], (1, 0, 2)) / np.float32(m.dt))
        eng.adjoint_run()
        return dict(eng.kernels(), seismograms=_traces(u))
    eng.run()
    return _traces(eng.seismograms())


def work(case):
    """Per step and point: u and v read and written once, one M^-1; per
    element: its kappa and mu (a database's irregular elements: 10 geometry
    values per point).  Operations of the weak form per element point."""
    if case["kind"] == "batch":
        lo, hi = (int(s) for s in case["n"].split("x"))
        side = 0.5 * (lo + hi)
        n, steps = (side, side), 0.75 * case["steps"] * case["events"]
    else:
        n, steps = tuple(int(s) for s in case["n"].split("x")), case["steps"]
    dim = len(n)
    nspec, nglob = float(np.prod(n)), float(np.prod([4 * m + 1 for m in n]))
    per_point, per_local = 16.0 * dim + 4.0, {2: 110.0, 3: 220.0}[dim]
    nbytes, flops = nglob * per_point + nspec * 8.0, nspec * 5.0 ** dim * per_local + nglob * 6.0 * dim
    if case["kind"] == "database" and case["distort"]:
        nbytes, flops = nbytes + 0.5 * nspec * 125 * 40.0, flops + nspec * 125 * 75.0
    if case["kind"] == "gradient":
        # the forward run, then the adjoint and the backward field and the
        # two strain kernels per element point, the rho product per point
        nbytes, flops = 3 * nbytes + nspec * 25 * 16.0 + nglob * 8.0, 3 * flops
    return {"bytes": nbytes * steps, "flops": flops * steps}


# ---------------------------------------------------------------------------
# The same equations in float64
# ---------------------------------------------------------------------------
def _lagrange(r):
    """Values and derivatives of the five Lagrange polynomials at r."""
    h, hp = np.ones(5), np.zeros(5)
    for i in range(5):
        for j in range(5):
            if j != i:
                h[i] *= (r - GLL_X[j]) / (GLL_X[i] - GLL_X[j])
        for k in range(5):
            if k != i:
                t = 1.0 / (GLL_X[i] - GLL_X[k])
                for j in range(5):
                    if j not in (i, k):
                        t *= (r - GLL_X[j]) / (GLL_X[i] - GLL_X[j])
                hp[i] += t
    return h, hp


HPRIME = np.array([_lagrange(x)[1] for x in GLL_X])  # [point][polynomial]


class Geometry:
    """GLL points, inverse Jacobians, absorbing faces of a Model."""

    def __init__(self, m, device):
        dim, n, npe = m.dim, m.n, 5 ** m.dim
        self.npe = npe
        idx = np.stack(np.meshgrid(*[np.arange(5)] * dim, indexing="ij")[::-1], -1).reshape(npe, dim)  # (p, axis)
        self.idx = idx
        el = np.stack(np.meshgrid(*[np.arange(k) for k in n[::-1]], indexing="ij")[::-1], -1).reshape(-1, dim)
        side = [4 * k + 1 for k in n]
        self.nglob = int(np.prod(side))
        stride = np.cumprod([1] + side[:-1])
        self.gather = torch.from_numpy((4 * el @ stride)[:, None] + (idx @ stride)[None, :]).to(device)
        if m.regular and m.dim == 3 and m.h and device != "cpu":
            inv, jac = np.eye(dim)[None, None] * 2.0 / m.h, np.full((1, 1), (m.h / 2) ** dim)
            self.xyz = None
        else:
            cor = np.stack([m.nodes[tuple(slice((c >> s) & 1, (c >> s & 1) + n[s]) for s in reversed(range(dim)))]
                            .reshape(-1, dim) for c in range(1 << dim)])          # (corner, e, comp)
            sgn = np.array([[((c >> s) & 1) * 2 - 1 for s in range(dim)] for c in range(1 << dim)])
            f = 0.5 * (1 + sgn[:, None, :] * GLL_X[idx][None])                  # (corner, p, axis)
            self.xyz = np.tensordot(np.prod(f, axis=2).T, cor, 1).transpose(1, 0, 2)
            dx = np.zeros((len(el), npe, dim, dim))                               # d x_r / d xi_s
            for s in range(dim):
                d = 0.5 * sgn[:, None, s] * np.prod(np.delete(f, s, axis=2), axis=2)
                dx[..., s] = np.tensordot(d.T, cor, 1).transpose(1, 0, 2)
            inv, jac = np.linalg.inv(dx), np.linalg.det(dx)                       # inv[s][r] = d xi_s / d x_r
        self.inv, self.jac = torch.from_numpy(inv).to(device), torch.from_numpy(jac).to(device)
        # absorbing faces: in 2-D an element point on two of its edges keeps
        # the last one (bottom, right, top, left), in 3-D both
        order = [(1, 0), (0, 1), (0, 0)] if dim == 2 else [(0, 0), (0, 1), (1, 0), (1, 1), (2, 0)]
        fe, fp, fn, fa, fw = [], [], [], [], []
        for axis, up in order:
            es = np.flatnonzero(el[:, axis] == (n[axis] - 1 if up else 0))
            ps = np.flatnonzero(idx[:, axis] == 4 * up)
            e, p = np.repeat(es, len(ps)), np.tile(ps, len(es))
            ie, ip = (e if inv.shape[0] > 1 else 0 * e), (p if inv.shape[1] > 1 else 0 * p)
            v = (1.0 if up else -1.0) * jac[ie, ip][:, None] * inv[ie, ip, axis, :]
            a = np.linalg.norm(v, axis=1)
            fe.append(e), fp.append(p), fn.append(v / a[:, None]), fa.append(a)
            fw.append(np.prod(GLL_W[np.delete(idx[p], axis, axis=1)], axis=1))
        self.face_elem, self.face_point, self.face_normal, self.face_area, self.face_weight = (
            np.concatenate(v) for v in (fe, fp, fn, fa, fw))
        if dim == 2:
            key = self.face_elem * npe + self.face_point
            keep = np.sort(len(key) - 1 - np.unique(key[::-1], return_index=True)[1])
            for name in ("elem", "point", "normal", "area", "weight"):
                setattr(self, "face_" + name, getattr(self, "face_" + name)[keep])


class Reference:
    """Newmark time loop of one Model in float64."""

    def __init__(self, m, device):
        self.m, self.dev = m, device
        g = self.g = Geometry(m, device)
        dim, npe = m.dim, g.npe
        self.dt = float(np.float32(m.dt))
        self.shape = (m.nspec,) + (5,) * dim
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=device)  # noqa: E731
        per = lambda a: t(a.ravel()).view((-1,) + (1,) * dim)  # noqa: E731
        self.rho, self.mu = per(m.rho), per(m.rho * m.vs ** 2)
        self.lam = per(m.rho * (m.vp ** 2 - 2 * m.vs ** 2))
        self.hp = t(HPRIME)
        self.hpw = t(HPRIME.T * GLL_W[None, :])           # [i][l] = hprime[l][i] w[l]
        grid = lambda a: a.view((a.shape[0],) + ((5,) * dim if a.shape[1] > 1 else (1,) * dim))  # noqa: E731
        self.jac = grid(g.jac)
        self.inv = [[grid(g.inv[:, :, s, r]) for r in range(dim)] for s in range(dim)]
        self.w = t(GLL_W)
        self.wall = t(np.prod(GLL_W[g.idx], axis=1)).view((1,) + (5,) * dim)
        wet = m.wet.ravel() if m.water else np.zeros(m.nspec, bool)
        self.dry = torch.from_numpy(~wet).to(device).view((-1,) + (1,) * dim)
        # absorbing faces: solid and fluid
        solid = ~wet[g.face_elem]
        fe, fp = torch.from_numpy(g.face_elem).to(device), torch.from_numpy(g.face_point).to(device)
        fg = g.gather[fe, fp]
        area = t(g.face_area * g.face_weight * solid)
        rvp, rvs = t((m.rho * m.vp).ravel()[g.face_elem]), t((m.rho * m.vs).ravel()[g.face_elem])
        self.face = (fg, t(g.face_normal).T.contiguous(), area, rvp, rvs)
        ng = g.nglob
        mass = torch.zeros(ng, dtype=torch.float64, device=device)
        mass.index_add_(0, g.gather.reshape(-1), (self.rho * self.dry * self.jac * self.wall).expand(self.shape).reshape(-1))
        one = torch.ones((dim, 1), dtype=torch.float64, device=device)
        self.minv = mass[None].repeat(dim, 1)
        self.minv.index_add_(1, fg, -self.dt / 2 * self.traction(one.expand(dim, len(fg))))
        self.minv = torch.where(self.minv > 0, 1.0 / self.minv.clamp_min(1e-300), torch.zeros_like(self.minv))
        if m.water:
            self._fluid(t, wet, fg)
        self.stf, self.src = self._sources(t)
        rec = [(self._element(e), np.prod(np.array([_lagrange(r[s])[0][g.idx[:, s]] for s in range(dim)]), axis=0))
               for _, e, r in m.receivers]
        self.rec_elem = np.array([e for e, _ in rec])
        self.rec_h = t(np.array([h for _, h in rec]))
        self.rec_gather = g.gather[torch.from_numpy(self.rec_elem).to(device)]

    def _element(self, e):
        return int(e @ np.cumprod([1] + list(self.m.n[:-1])))

    def _fluid(self, t, wet, fg):
        """Potential formulation: 1/kappa mass, 1/rho stiffness, free surface
        on top, the horizontal interface below."""
        m, g = self.m, self.g
        kap = t((m.rho * m.vp ** 2).ravel()).view(-1, 1, 1)
        wetd = torch.from_numpy(wet).to(self.dev).view(-1, 1, 1)
        self.irho, self.kap = wetd / self.rho, kap
        mass = torch.zeros(g.nglob, dtype=torch.float64, device=self.dev)
        mass.index_add_(0, g.gather.reshape(-1), (wetd / kap * self.jac * self.wall).expand(self.shape).reshape(-1))
        # a point on the free surface takes no element contribution
        top = torch.from_numpy((np.arange(m.nspec) // m.n[0]) == m.n[1] - 1).to(self.dev).view(-1, 1, 1)
        edge = torch.zeros((1, 5, 5), dtype=torch.bool, device=self.dev)
        edge[:, 4] = True
        self.free = top & edge
        rvpi = np.sqrt(1.0 / (m.rho * m.rho * m.vp ** 2)).ravel()[g.face_elem]
        coef = t(g.face_area * g.face_weight * wet[g.face_elem] * rvpi)
        mass.index_add_(0, fg, self.dt / 2 * coef)
        fe, fp = torch.from_numpy(g.face_elem).to(self.dev), torch.from_numpy(g.face_point).to(self.dev)
        self.fcoef = torch.where(self.free.expand(self.shape).reshape(m.nspec, -1)[fe, fp], torch.zeros_like(coef), coef)
        self.fgather = fg
        self.minv_f = torch.where(mass > 0, 1.0 / mass.clamp_min(1e-300), torch.zeros_like(mass))
        iz = int(np.argmax(m.wet[:, 0]))
        e = torch.arange(m.n[0], device=self.dev) + (iz - 1) * m.n[0]
        self.if_gather = g.gather[e][:, 20:]                     # top row of the solid elements
        self.if_coef = (self.w * m.h / 2)[None, :].expand(m.n[0], 5)  # their normal is (0, 1)

    def _sources(self, t):
        m, g, dim = self.m, self.g, self.m.dim
        t0 = np.array([-1.2 / s["f0"] for s, _, _ in m.sources])
        time = t0.min() + self.dt * np.arange(m.steps)[:, None] - (t0 - t0.min())[None, :]
        a = (np.pi * np.array([s["f0"] for s, _, _ in m.sources])) ** 2
        stf = -1e10 * (1 - 2 * a * time ** 2) * np.exp(-a * time ** 2)
        arrays, gath = [], []
        for s, e, r in m.sources:
            h, hp = zip(*[_lagrange(r[k]) for k in range(dim)])
            hl = np.prod(np.array([h[k][g.idx[:, k]] for k in range(dim)]), axis=0)
            el = self._element(e)
            ge = el if g.inv.shape[0] > 1 else 0
            if m.water:
                arr = np.zeros((dim, g.npe))
                arr[0] = hl / (m.rho * m.vp ** 2).ravel()[el]
            elif s["type"] == "force":
                f = ((math.sin(math.radians(s["angle"])), -math.cos(math.radians(s["angle"]))) if dim == 2
                     else (s["fx"], s["fy"], s["fz"]))
                arr = np.outer(f, hl)
            else:
                inv = g.inv[ge].cpu().numpy() * np.ones((g.npe, 1, 1))
                dav = np.einsum("p,psr->sr", hl, inv)
                dref = [np.prod(np.array([(hp if k == q else h)[k][g.idx[:, k]] for k in range(dim)]), axis=0)
                        for q in range(dim)]
                d = np.einsum("sp,sr->rp", np.array(dref), dav)
                M = (np.array([[s["mxx"], s["mxz"]], [s["mxz"], s["mzz"]]]) if dim == 2 else
                     np.array([[s["mxx"], s["mxy"], s["mxz"]], [s["mxy"], s["myy"], s["myz"]],
                               [s["mxz"], s["myz"], s["mzz"]]]))
                arr = M @ d
            arrays.append(arr)
            gath.append(g.gather[el])
        return t(stf), (torch.cat(gath), t(np.array(arrays)).permute(1, 0, 2).contiguous())

    def numbering(self):
        """Lattice point of each field index: points numbered at their first
        visit, in 2-D the elements without absorbing edges first and z fastest."""
        m = self.m
        order = np.arange(m.nspec)
        if m.dim == 2:
            absorbs = np.zeros(m.nspec, bool)
            absorbs[self.g.face_elem] = True
            order = np.concatenate([np.flatnonzero(~absorbs), np.flatnonzero(absorbs)])
        pts = self.g.gather.cpu().numpy()[order]
        if m.dim == 2:
            pts = pts.reshape(-1, 5, 5).transpose(0, 2, 1)
        pts = pts.ravel()
        uniq, first = np.unique(pts, return_index=True)
        return uniq[np.argsort(first)]

    def derive(self, U, s):
        return torch.movedim(torch.movedim(U, -1 - s, -1) @ self.hp.T, -1, -1 - s)

    def collect(self, F, s):
        """Weighted divergence part along reference axis s."""
        r = torch.movedim(torch.movedim(F, -1 - s, -1) @ self.hpw.T, -1, -1 - s)
        for k in range(self.m.dim):
            if k != s:
                r = r * self.w.view((5,) + (1,) * k)
        return r

    def gradient(self, u):
        """du[c][r] = d u_c / d x_r at the element points."""
        dim = self.m.dim
        out = []
        for c in range(u.shape[0]):
            U = u[c][self.g.gather].view(self.shape)
            dr = [self.derive(U, s) for s in range(dim)]
            out.append([sum(dr[s] * self.inv[s][r] for s in range(dim) if not (self.inv[s][r].numel() == 1 and s != r))
                        for r in range(dim)])
        return out

    def assemble(self, sigma, ncomp):
        dim = self.m.dim
        a = torch.zeros((ncomp, self.g.nglob), dtype=torch.float64, device=self.dev)
        flat = self.g.gather.reshape(-1)
        for c in range(ncomp):
            r = 0.0
            for s in range(dim):
                F = self.jac * sum(sigma(c, k) * self.inv[s][k] for k in range(dim)
                                   if not (self.inv[s][k].numel() == 1 and s != k))
                r = r - self.collect(F, s)
            if ncomp == 1:
                r = r.masked_fill(self.free, 0.0)
            a[c].index_add_(0, flat, r.reshape(-1))
        return a

    def traction(self, v):
        _, n, area, rvp, rvs = self.face
        return -((v * n).sum(0) * n * (rvp - rvs) + v * rvs) * area

    def force(self, u, v):
        du = self.gradient(u)
        tr = sum(du[c][c] for c in range(self.m.dim)) * self.lam * self.dry
        mu = self.mu
        a = self.assemble(lambda c, k: mu * (du[c][k] + du[k][c]) + (tr if c == k else 0.0), self.m.dim)
        fg = self.face[0]
        return a.index_add_(1, fg, self.traction(v[:, fg]))

    def fluid_force(self, x, xd):
        gr = self.gradient(x[None])[0]
        a = self.assemble(lambda c, k: self.irho * gr[k], 1)[0]
        return a.index_add_(0, self.fgather, -self.fcoef * xd[self.fgather])

    def sample(self, u, v, a, fluid=None):
        out = []
        for t in self.m.types:
            k = ("displacement", "velocity", "acceleration", "pressure").index(t)
            if k < 3:
                x = (u, v, a)[k][:, self.rec_gather]
            else:
                x = torch.zeros((self.m.dim,) + tuple(self.rec_gather.shape), dtype=torch.float64, device=self.dev)
                du = self.gradient(u)
                p = -(self.lam + 2.0 / 3.0 * self.mu) * (du[0][0] + du[1][1])
                x[0] = p.reshape(self.m.nspec, -1)[torch.from_numpy(self.rec_elem).to(self.dev)]
            if fluid is not None:
                wet = torch.from_numpy(self.m.wet.ravel()[self.rec_elem]).to(self.dev)[:, None]
                f = fluid[min(k, 2)]
                if k < 3:
                    e = torch.from_numpy(self.rec_elem).to(self.dev)
                    y = torch.stack([(self.irho * d).reshape(self.m.nspec, -1)[e] for d in self.gradient(f[None])[0]])
                else:
                    y = torch.zeros_like(x)
                    y[0] = -f[self.rec_gather]
                x = torch.where(wet, y, x)
            out.append((x * self.rec_h).sum(-1).T)
        return torch.stack(out)

    def forward(self, keep=False):
        """(seismograms, (u, v, a) after the last corrector, all u)."""
        m, dt = self.m, self.dt
        z = lambda *s: torch.zeros(s, dtype=torch.float64, device=self.dev)  # noqa: E731
        ng = self.g.nglob
        u, v, a = z(m.dim, ng), z(m.dim, ng), z(m.dim, ng)
        x, xd, xdd = z(ng), z(ng), z(ng)
        seis, us = [], []
        sg, sa = self.src
        for i in range(m.steps):
            u += dt * v + 0.5 * dt * dt * a
            v += 0.5 * dt * a
            amp = self.stf[i].repeat_interleave(self.g.npe)
            if m.water:
                x += dt * xd + 0.5 * dt * dt * xdd
                xd += 0.5 * dt * xdd
                xdd = self.fluid_force(x, xd)
                # the fluid's outward normal on the interface is -z
                xdd.index_add_(0, self.if_gather.reshape(-1), (-self.if_coef * u[1][self.if_gather]).reshape(-1))
                xdd.index_add_(0, sg, sa[0].reshape(-1) * amp)
                xdd *= self.minv_f
                xd += 0.5 * dt * xdd
            a = self.force(u, v)
            if m.water:
                a[1].index_add_(0, self.if_gather.reshape(-1), (self.if_coef * xdd[self.if_gather]).reshape(-1))
            else:
                a.index_add_(1, sg, sa.reshape(m.dim, -1) * amp)
            a *= self.minv
            v += 0.5 * dt * a
            if i % m.every == 0:
                seis.append(self.sample(u, v, a, (x, xd, xdd) if m.water else None))
            if keep:
                us.append(u.clone())
        return torch.stack(seis), (u, v, a), us

    def kernels(self, seis, us):
        """The six kernels of the adjoint run driven by the traces / dt."""
        m, dt = self.m, self.dt
        z = lambda *s: torch.zeros(s, dtype=torch.float64, device=self.dev)  # noqa: E731
        u, v, a = (z(2, self.g.nglob) for _ in range(3))
        kr, kk, km = z(self.g.nglob), z(*self.shape), z(*self.shape)
        for i in reversed(range(m.steps)):
            u += dt * v + 0.5 * dt * dt * a
            v += 0.5 * dt * a
            a = self.force(u, v)
            for c in range(2):
                a[c].index_add_(0, self.rec_gather.reshape(-1), (self.rec_h * (seis[i, 0, :, c] / dt)[:, None]).reshape(-1))
            a *= self.minv
            v += 0.5 * dt * a
            p, b = self.gradient(u), self.gradient(us[i])
            div = (p[0][0] + p[1][1]) * (b[0][0] + b[1][1])
            dot = p[0][0] * b[0][0] + p[1][1] * b[1][1] + 0.5 * (p[0][1] + p[1][0]) * (b[0][1] + b[1][0])
            kk += dt * div
            km += dt * (dot - div / 3.0)
            kr += dt * (a * us[i]).sum(0)
        bulk = self.lam + self.mu
        rho = (-self.rho * kr[self.g.gather].view(self.shape))
        mu, kap = -2.0 * self.mu * km, -bulk * kk
        q = 4.0 / 3.0 * self.mu / bulk
        return dict(rho=rho, mu=mu, kappa=kap, rhop=rho + kap + mu, alpha=2.0 * (1.0 + q) * kap, beta=2.0 * (mu - q * kap))


def exact(case, seed):
    w = work(case)
    dim = len(case["n"].split("x"))
    if w["bytes"] / (16.0 * dim + 4.0) * dim > EXACT_LIMIT:
        return None
    device = "cuda" if torch.cuda.is_available() else "cpu"
    out = []
    for m in _models(case, seed):
        ref = Reference(m, device)
        kind = case["kind"]
        seis, last, us = ref.forward(keep=kind == "gradient")
        if kind == "gradient":
            k = {n: v.cpu().numpy() for n, v in ref.kernels(seis, us).items()}
            return dict(k, seismograms=_traces(seis.cpu().numpy()))
        seis = _traces(seis.cpu().numpy())
        if kind in ("snapshot", "seams"):
            order = ref.numbering()
            return dict({t: f.cpu().numpy()[:, order] for t, f in zip(FIELDS, last)}, seismograms=seis)
        out.append(seis)
    return out if case["kind"] == "batch" else out[0]
