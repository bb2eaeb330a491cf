"""The tracking work whose speed counts, and what its results should be.

Every case goes through the package's public entry points the way a program
uses them: particle rows in host memory (elegant's own layout), a lattice, and
a call that tracks, downloads or differentiates.  Kinds of case:

  track    a beam through a ring for some turns (tracking.Beam, tracking.track,
           Beam.download), fused or element by element ("plain", the drop-in path
           in which every element is a routine call of its own)
  matrix   transport maps on a resident beam, as elegant's matrix elements call
           them (Beam.track_particles)
  batch    error-seeded variants of one ring with uneven beams (tracking.Batch)
  adjoint  tracking and its reverse-mode gradient (adjoint.track_turns)
  seeds    the same gradient summed over error seeds (BatchAdjointTracker)

exact() restates the maps in plain torch, in 64 bits and in well-conditioned
forms, without the package's tracking code.  The package only supplies the
description of the lattice there (element parameters).
"""
import copy
import functools
import math

import numpy as np
import torch

from elegant_amd import adjoint, census, configs, optics, tracking
from elegant_amd import structs as S

P_FODO = configs.p_central_from_mev(1000.0)
P_MBA = configs.p_central_from_mev(3000.0)
MULTIPOLES = (S.T_KQUAD, S.T_KSEXT, S.T_KOCT)
SEXTUPOLES = ["S%d" % i for i in range(6)]


# --------------------------------------------------------------------------
# the cases

def listed():
    return [
        # a handful of particles once around: closed-orbit and one-turn-map probes,
        # issued by the hundred in a matching loop; all latency and launches
        dict(name="orbit_fodo_16", kind="track", ring="fodo", cells=10, n=16, turns=1, beam="matched", mode="fused"),
        # the ordinary study: ten thousand matched particles, many turns
        dict(name="study_fodo_1e4", kind="track", ring="fodo", cells=10, n=10000, turns=40, beam="matched",
             mode="fused"),
        # the drop-in path: every element and every aperture sweep a call of its own
        dict(name="plain_fodo_1e4", kind="track", ring="fodo", cells=10, n=10000, turns=2, beam="matched",
             mode="plain"),
        # the dynamic-aperture grid, the largest
        dict(name="grid_mba_1e6", kind="track", ring="mba", cells=40, n=1000000, turns=2, beam="grid", mode="fused"),
        # a quick look at the aperture on a coarse, ragged grid
        dict(name="grid_mba_30401", kind="track", ring="mba", cells=40, n=30401, turns=2, beam="grid", mode="fused"),
        # a grid that reaches past the vacuum chamber: most particles are lost
        dict(name="lossy_mba_1e5", kind="track", ring="mba", cells=40, n=99855, turns=2, beam="wide", mode="fused"),
        # synchrotron radiation on, bends with pole-face edges
        dict(name="radiating_mba_5e4", kind="track", ring="mba_rad", cells=40, n=50000, turns=1, beam="matched",
             mode="fused"),
        # a line of matrix elements on a beam that comes from and returns to the host
        dict(name="matrix_2e5", kind="matrix", n=200000, maps=8, order=2),
        # error seeds in one batch, uneven beams
        dict(name="batch_mba_12", kind="batch", cells=40, variants=12, median=16000, turns=1),
        # gradient with every anchor kept
        dict(name="adjoint_mba_1e4", kind="adjoint", cells=40, n=10000, turns=2, every=1, what="strengths"),
        # gradient with checkpoints and re-tracking, a last segment cut short,
        # misalignments among the parameters
        dict(name="adjoint_cells_5001", kind="adjoint", cells=10, n=5001, turns=3, every=2, what="offsets"),
        # sextupole families over error seeds
        dict(name="seeds_mba_6", kind="seeds", cells=8, variants=6, n=2000, turns=2, every=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    k = rng.choice(["fodo", "fodo", "plain", "grid", "grid", "wide", "rad", "matrix", "batch", "adjoint", "adjoint",
                    "seeds"])
    if k == "fodo":
        n = _log(rng, 8, 200000)
        t = max(1, min(_log(rng, 1, 60), int(4e7 / (100 * n))))
        return dict(kind="track", ring="fodo", cells=rng.choice([1, 5, 10]), n=n, turns=t, beam="matched",
                    mode="fused")
    if k == "plain":
        ring = rng.choice(["fodo", "mba"])
        return dict(kind="track", ring=ring, cells=10 if ring == "fodo" else 1, n=_log(rng, 64, 200000), turns=1,
                    beam="matched", mode="plain")
    if k in ("grid", "wide", "rad"):
        n = _log(rng, 1000, 600000 if k == "grid" else 150000)
        return dict(kind="track", ring="mba_rad" if k == "rad" else "mba", cells=40, n=n,
                    turns=1 if k == "rad" or n > 300000 else rng.randint(1, 2),
                    beam="matched" if k == "rad" else k, mode="fused")
    if k == "matrix":
        return dict(kind="matrix", n=_log(rng, 1000, 400000), maps=rng.randint(1, 10), order=rng.choice([1, 2]))
    if k == "batch":
        return dict(kind="batch", cells=rng.choice([4, 10, 40]), variants=rng.randint(2, 12),
                    median=_log(rng, 200, 16000), turns=1)
    if k == "adjoint":
        return dict(kind="adjoint", cells=rng.choice([4, 10]), n=_log(rng, 200, 8000), turns=rng.randint(1, 3),
                    every=rng.randint(1, 2), what=rng.choice(["strengths", "offsets", "bends"]))
    return dict(kind="seeds", cells=rng.choice([2, 4]), variants=rng.randint(2, 6), n=_log(rng, 100, 2000),
                turns=rng.randint(1, 2), every=rng.randint(1, 2))


# --------------------------------------------------------------------------
# lattices and inputs

@functools.lru_cache(maxsize=None)
def _ring(ring, cells):
    if ring == "fodo":
        return configs.fodo_ring(cells)
    lat = configs.mba_ring(P_MBA, cells)
    if ring == "mba_rad":
        for e in lat.elements:
            if e.type in MULTIPOLES:
                e.params["SYNCH_RAD"] = 1
            elif e.type == S.T_CSBEND:
                half = e.params["ANGLE"] / 2
                e.params.update(SYNCH_RAD=1, EDGE1_EFFECTS=1, EDGE2_EFFECTS=1, E1=half, E2=half, HGAP=0.01)
    return lat


def _variants(cells, count, seed):
    """error-seeded copies (strength error and offsets on quadrupoles and
    sextupoles, as configs.mba_variants draws them)"""
    base = _ring("mba", cells)
    rng = np.random.default_rng([seed, 17])
    out = []
    for _ in range(count):
        lat = copy.deepcopy(base)
        where = [e for e in lat.elements if e.type in (S.T_KQUAD, S.T_KSEXT)]
        err = np.clip(rng.standard_normal((len(where), 3)), -2, 2) * np.array([1e-3, 30e-6, 30e-6])
        for e, (f, dx, dy) in zip(where, err.tolist()):
            e.params.update(FSE=f, DX=dx, DY=dy)
        out.append(lat)
    return out


@functools.lru_cache(maxsize=None)
def _twiss(ring):
    return optics.periodic_twiss(configs.Lattice(configs.fodo_cell()) if ring == "fodo" else configs.mba_period())


def _matched(ring, n, seed):
    return configs.gaussian_beam(n, _twiss("fodo" if ring == "fodo" else "mba"), 5e-9, 50e-12, 1e-3, 3e-3, seed=seed)


def _rows(case, seed):
    n = case["n"]
    if case["beam"] == "matched":
        return _matched(case["ring"], n, seed)
    u = np.random.default_rng([seed, 3]).uniform(0.9, 1.1, 2)
    xmax, ymax = (0.015, 0.005) if case["beam"] == "grid" else (0.030, 0.025)
    nx = max(1, int(math.sqrt(n * 1.5)))
    ny = -(-n // nx)
    return np.ascontiguousarray(configs.da_grid(nx, ny, xmax * u[0], ymax * u[1])[:n])


def _counts(case):
    return configs.variant_counts(case["variants"], seed=case["median"], lo=max(1, case["median"] // 16),
                                  hi=6 * case["median"], median=float(case["median"])).tolist()


def _matrices(case, seed):
    """maps of quadrupole-like elements, with their chromatic second-order terms"""
    rng = np.random.default_rng([seed, 5])
    out = []
    for _ in range(case["maps"]):
        k, L = rng.uniform(0.2, 1.5), rng.uniform(0.1, 0.4)
        a = math.sqrt(k) * L
        R = np.eye(6)
        R[:2, :2] = [[math.cos(a), math.sin(a) / math.sqrt(k)], [-math.sqrt(k) * math.sin(a), math.cos(a)]]
        R[2:4, 2:4] = [[math.cosh(a), math.sinh(a) / math.sqrt(k)], [math.sqrt(k) * math.sinh(a), math.cosh(a)]]
        T = np.zeros((6, 6, 6))
        T[0, 5, 0], T[1, 5, 0], T[2, 5, 2], T[3, 5, 2] = a * a / 2, k * L, -a * a / 2, -k * L
        T[4, 1, 1] = T[4, 3, 3] = L / 2
        C0 = np.array([0, 0, 0, 0, L, 0.0])
        out.append((C0, R, T if case["order"] == 2 else None))
    return out


def _spec(lat, what):
    if what == "strengths":
        return adjoint.ParamSpec.strengths(lat)
    if what == "offsets":
        return adjoint.ParamSpec.strengths(lat) + adjoint.ParamSpec.offsets(lat)
    return adjoint.ParamSpec.bends(lat) + adjoint.ParamSpec.strengths(lat, (S.T_KQUAD,))


def _gradient_inputs(case, seed):
    """(lattices, rows per lattice, spec, cotangent of the final coordinates)"""
    if case["kind"] == "adjoint":
        lats = [copy.deepcopy(_ring("mba", case["cells"]))]
        rows = [_matched("mba", case["n"], seed)]
        spec = _spec(lats[0], case["what"])
    else:
        lats = _variants(case["cells"], case["variants"], seed)
        ns = [max(1, case["n"] - 37 * v) for v in range(case["variants"])]
        rows = [_matched("mba", n, seed * 1009 + v) for v, n in enumerate(ns)]
        spec = adjoint.ParamSpec.split_families(lats[0], SEXTUPOLES)
    # the derivative of a mean of squares and of a linear term in every coordinate
    scale = np.array([1e3, 1e4, 1e3, 1e4, 1.0, 10.0])
    rng = np.random.default_rng([seed, 7])
    cot = [rng.standard_normal((len(r), 6)) * scale / len(r) for r in rows]
    return lats, rows, spec, cot


def prepare(case, seed):
    tracking.init(0)
    if case["kind"] == "track":
        lat = copy.deepcopy(_ring(case["ring"], case["cells"]))
        lat.c_beamline()
        return dict(case=case, lat=lat, rows=_rows(case, seed))
    if case["kind"] == "matrix":
        return dict(case=case, rows=_matched("mba", case["n"], seed),
                    maps=[S.vmatrix(*m) for m in _matrices(case, seed)])
    if case["kind"] == "batch":
        lats = _variants(case["cells"], case["variants"], seed)
        for lat in lats:
            lat.c_beamline()
        rows = [_matched("mba", n, seed * 1009 + v) for v, n in enumerate(_counts(case))]
        return dict(case=case, lats=lats, rows=rows)
    lats, rows, spec, cot = _gradient_inputs(case, seed)
    for lat in lats:
        lat.c_beamline()
    if case["kind"] == "adjoint":
        trk = adjoint.AdjointTracker(lats[0], spec, P_MBA, case["turns"], case["every"])
        return dict(case=case, tracker=trk,
                    theta=torch.tensor(spec.values(lats[0]), device="cuda", requires_grad=True),
                    z0=torch.tensor(rows[0][:, :6], device="cuda", requires_grad=True),
                    cot=torch.tensor(cot[0], device="cuda"))
    trk = adjoint.BatchAdjointTracker(lats, spec, P_MBA, case["turns"], case["every"])
    return dict(case=case, tracker=trk, theta=spec.values(lats[0]), rows=rows, cot=cot)


def _parts(a):
    """coordinates by size (the path length would hide the rest), then particle
    identity and pass of loss where rows carry them"""
    out = {"transverse": a[:, :4], "s": a[:, 4], "delta": a[:, 5]}
    if a.shape[1] > 6:
        out["id_pass"] = a[:, 6:8]
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "track":
        lat = state["lat"]
        lat.reset_state()  # a run of its own: RF phases are found from its beam
        beam = tracking.Beam(state["rows"])
        n, _, _ = tracking.track(beam, lat, case["turns"], P_FODO if case["ring"] == "fodo" else P_MBA,
                                 mode=case["mode"], turns_per_launch=16)
        out = beam.download()
        beam.free()
        return {"rows": _parts(out), "survivors": n}
    if kind == "matrix":
        beam = tracking.Beam(state["rows"])
        for m in state["maps"]:
            beam.track_particles(m)
        out = beam.download()
        beam.free()
        return {"rows": _parts(out)}
    if kind == "batch":
        for lat in state["lats"]:
            lat.reset_state()
        b = tracking.Batch(state["rows"])
        n, _ = b.track(state["lats"], case["turns"], P_MBA)
        out = [b.download(v) for v in range(case["variants"])]
        b.free()
        return {"rows": [_parts(r) for r in out], "survivors": n}
    if kind == "adjoint":
        final, alive = adjoint.track_turns(state["theta"], state["z0"], state["tracker"])
        gt, gz = torch.autograd.grad(final, (state["theta"], state["z0"]), state["cot"])
        return {"final": _parts(final.detach()), "alive": alive, "grad_theta": gt, "grad_z0": gz}
    res = state["tracker"].forward(state["rows"], state["theta"])
    gp, gz = state["tracker"].backward(state["cot"])
    return {"final": [_parts(f) for f, _ in res], "alive": [a for _, a in res], "grad_theta": gp, "grad_z0": gz}


# --------------------------------------------------------------------------
# work and tolerance

def work(case):
    kind = case["kind"]
    row = 8 * S.NPROP
    if kind == "matrix":
        per = 36 * 2 + (126 * 2 if case["order"] == 2 else 0)
        return {"bytes": 2 * row * case["n"], "flops": per * case["n"] * case["maps"]}
    ring = case.get("ring", "mba")
    c = census.lattice_census(_ring(ring, case["cells"]))
    turn = c["flops"] + c["T"]
    if kind == "track":
        return {"bytes": 2 * row * case["n"], "flops": turn * case["turns"] * case["n"]}
    if kind == "batch":
        n = sum(_counts(case))
        return {"bytes": 2 * row * n, "flops": turn * case["turns"] * n}
    n = case["n"] if kind == "adjoint" else sum(max(1, case["n"] - 37 * v) for v in range(case["variants"]))
    # a reverse sweep does the forward map's work once more and about as much
    # again for the adjoint of each sub-step
    return {"bytes": 4 * 48 * n, "flops": 3 * turn * case["turns"] * n}


def tolerance(case):
    """Double precision throughout.  A ring amplifies the rounding of its thousands
    of sub-steps: rho0 (f - 1) in the exact bend drift, with rho0 about 25 m against
    beams of 10 to 100 microns, costs six digits.  About four times the error
    measured against exact(), which avoids that cancellation: 7.5e-9 (2-norm,
    transverse) for grids reaching out to the aperture, 2e-9 for matched beams and
    for the coordinates and gradients of the adjoint, 2.3e-16 for matrices."""
    if case["kind"] == "matrix":
        return {"rel": 1e-15, "max": 1e-13}
    if case["kind"] == "track" and case["beam"] != "matched":
        return {"rel": 3e-8, "max": 1e-5, "differ": 0.0}
    return {"rel": 8e-9, "max": 1e-6, "differ": 0.0}


# --------------------------------------------------------------------------
# the same in plain 64-bit torch

BETA = 2.0 ** (1.0 / 3.0)
DRIFT4 = [0.5 / (2 - BETA), (1 - BETA) / (2 - BETA) / 2, (1 - BETA) / (2 - BETA) / 2, 0.5 / (2 - BETA)]
KICK4 = [1 / (2 - BETA), -BETA / (2 - BETA), 1 / (2 - BETA)]
C_MKS = 2.99792458e8
E_MKS, EPS0, ME_MKS = 1.602176634e-19, 8.8541878128e-12, 9.1093837015e-31


def _operations(lat):
    """about how many torch operations one turn of a lattice takes"""
    ops = 0
    for e, s in zip(lat.elements, lat.structs()):
        if e.type == S.T_CSBEND:
            ops += s.nSlices * (4 * 24 + 3 * (45 if s.k1 else 12) + 4)
        elif e.type in MULTIPOLES:
            ops += _slices(s) * 4 * 24
        else:
            ops += 12
    return ops


def _slices(s):
    return max(1, -(-s.n_kicks // s.integration_order)) if s.n_kicks > 0 else s.nSlices


def _bend_field(k1, h):
    """(i, j, coefficient) lists of the mid-plane field 1 + K1/h * (h x) of a bend of
    curvature h carried off the mid-plane to total order 4: with psi the scalar
    potential, psi = sum a_n(x) y^n / n!, a_1 the mid-plane field and
    a_(n+2) = -((1 + h x) a_n')' / (1 + h x); By = d psi/dy, Bx = d psi/dx.
    Per unit K1, since the field is linear in it; the dipole part is constant."""
    N = 8
    inv = [(-h) ** k for k in range(N)]

    def mul(a, b):
        out = [0.0] * N
        for i, u in enumerate(a):
            for j, v in enumerate(b):
                if i + j < N:
                    out[i + j] += u * v
        return out

    def der(a):
        return [(k + 1) * a[k + 1] for k in range(N - 1)] + [0.0]

    a = {1: [0.0, 1.0] + [0.0] * (N - 2)}
    for n in (3, 5):
        a[n] = [-v for v in mul(inv, der(mul([1.0, h] + [0.0] * (N - 2), der(a[n - 2]))))]
    fx, fy = [], []
    for n in (1, 3, 5):
        d = der(a[n])
        for i in range(5):
            if i + n < 5 and d[i]:
                fx.append((i, n, d[i] / math.factorial(n)))
            if i + n - 1 < 5 and a[n][i]:
                fy.append((i, n - 1, a[n][i] / math.factorial(n - 1)))
    return fx, fy


class _Exact:
    """A beam of one or several lattice variants, one tensor per coordinate, all
    variants one after the other.  Parameters that differ between variants are
    tensors with one value per particle."""

    def __init__(self, lats, rows, p_central, theta=None, slots=None):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.dev = dev
        self.lats, self.Po, self.theta, self.slots = lats, p_central, theta, slots
        self.counts = torch.tensor([len(r) for r in rows], device=dev)
        allrows = torch.tensor(np.concatenate(rows), device=dev)
        self.z = {k: allrows[:, i].clone() for i, k in enumerate(("x", "xp", "y", "yp", "s", "dp"))}
        self.z["id"] = torch.arange(len(allrows), device=dev)
        self.structs = [lat.structs() for lat in lats]
        self.watch = theta is None  # apertures; gradients are taken on surviving beams
        self.amp = None
        self.events = []  # (event, ids, loss rows)
        self.fields = {}

    # ---- parameters and losses
    def par(self, i, name, kind=None):
        if kind is not None and self.theta is not None and self.slots[i][kind] >= 0:
            return self.theta[int(self.slots[i][kind])]
        v = [getattr(s[i], name) for s in self.structs]
        if all(u == v[0] for u in v):
            return v[0]
        return torch.repeat_interleave(torch.tensor(v, dtype=torch.float64, device=self.dev), self.counts)

    def lose(self, bad, event, row):
        """take the particles of `bad` out with the coordinates row() gives them"""
        if not bool(bad.any()):
            return False
        if len(self.lats) > 1:
            raise ArithmeticError("losses in a batch")
        vals = torch.stack([torch.as_tensor(v, dtype=torch.float64, device=self.dev).expand(len(bad))[bad]
                            for v in row()], 1)
        self.events.append((event, self.z["id"][bad].cpu().numpy(), vals.cpu().numpy()))
        keep = ~bad
        self.z = {k: v[keep] for k, v in self.z.items()}
        return True

    def outside(self, x, y):
        return (x.abs() > self.amp[0]) | (y.abs() > self.amp[1])

    def sweep(self, event, z_end, extrapolate):
        if self.amp is None or not self.watch:
            return
        z = self.z
        bad = self.outside(z["x"], z["y"])

        def row():
            dz = torch.zeros_like(z["x"])
            if extrapolate:
                big = torch.full_like(dz, -1.7976931348623157e308)
                dzx, dzy = (torch.where((z[c].abs() > lim) & (z[p] != 0),
                                        (z[c] - torch.where(z[p] < 0, -1.0, 1.0) * lim) / z[p], big)
                            for c, p, lim in (("x", "xp", self.amp[0]), ("y", "yp", self.amp[1])))
                dz = -torch.maximum(dzx, dzy)
                dz = torch.where(dz.abs() > 1e300, torch.zeros_like(dz), dz)
            return (z["x"] + dz * z["xp"], z["xp"], z["y"] + dz * z["yp"], z["yp"], z_end + dz,
                    self.Po * (1 + z["dp"]))

        self.lose(bad, event, row)

    # ---- elements
    @staticmethod
    def slopes(qx, qy, dp):
        d = torch.sqrt((1 + dp) ** 2 - qx * qx - qy * qy)
        return qx / d, qy / d

    @staticmethod
    def momenta(xp, yp, dp):
        f = (1 + dp) / torch.sqrt(1 + xp * xp + yp * yp)
        return xp * f, yp * f

    def drift(self, L):
        z = self.z
        z["x"], z["y"] = z["x"] + L * z["xp"], z["y"] + L * z["yp"]
        z["s"] = z["s"] + L + L / 2 * (z["xp"] ** 2 + z["yp"] ** 2)

    def multipole(self, i, t, event, z_start):
        s = self.structs[0][i]
        order = {S.T_KQUAD: 1, S.T_KSEXT: 2, S.T_KOCT: 3}[t]
        K = self.par(i, "k%d" % order, 0) * s.length * (1 + self.par(i, "fse"))
        dx, dy = self.par(i, "dx", 1), self.par(i, "dy", 2)
        ns, z = _slices(s), self.z
        rad = E_MKS ** 2 * self.Po ** 3 / (6 * math.pi * EPS0 * C_MKS ** 2 * ME_MKS) if s.synch_rad else 0.0
        drift = s.length / ns
        z["x"], z["y"] = z["x"] - dx, z["y"] - dy
        z["x0p"], z["y0p"], z["s0"], z["dp0"] = z["xp"], z["yp"], z["s"], z["dp"]
        z["qx"], z["qy"] = self.momenta(z["xp"], z["yp"], z["dp"])
        path, done = torch.zeros_like(z["x"]), 0.0
        z["path"] = path

        def check():
            if self.watch and self.amp is not None:
                z = self.z
                self.lose(self.outside(z["x"] + dx, z["y"] + dy), event,
                          lambda: (z["x"] + dx, z["x0p"], z["y"] + dy, z["y0p"], z_start + done,
                                   self.Po * (1 + z["dp0"])))

        for _ in range(ns):
            check()
            z = self.z
            for j in range(4):
                h = drift * DRIFT4[j]
                z["x"], z["y"] = z["x"] + h * z["xp"], z["y"] + h * z["yp"]
                z["path"] = z["path"] + h * torch.sqrt(1 + z["xp"] ** 2 + z["yp"] ** 2)
                done += h
                if j == 3:
                    break
                x, y = z["x"], z["y"]
                if order == 1:
                    by, bx = x, y
                elif order == 2:
                    by, bx = (x * x - y * y) / 2, x * y
                else:
                    by, bx = x * (x * x - 3 * y * y) / 6, y * (3 * x * x - y * y) / 6
                k = K / ns * KICK4[j]
                z["qx"], z["qy"] = z["qx"] - k * by, z["qy"] + k * bx
                z["xp"], z["yp"] = self.slopes(z["qx"], z["qy"], z["dp"])
                if rad:
                    f2 = (K / ns / drift) ** 2 * (bx * bx + by * by)
                    w = torch.sqrt(1 + z["xp"] ** 2 + z["yp"] ** 2)
                    new = z["dp"] - rad * (1 + z["dp"]) ** 2 * f2 * w * drift * KICK4[j]
                    g = (1 + new) / (1 + z["dp"])
                    z["qx"], z["qy"], z["dp"] = z["qx"] * g, z["qy"] * g, new
                    z["xp"], z["yp"] = self.slopes(z["qx"], z["qy"], z["dp"])
        check()
        z = self.z
        if rad:
            b0, b1 = self.beta(z["dp0"]), self.beta(z["dp"])
            z["s"] = b1 * (z["s"] / b0 + 2 * z["path"] / (b0 + b1))
        else:
            z["s"] = z["s"] + z["path"]
        z["x"], z["y"] = z["x"] + dx, z["y"] + dy
        for k in ("x0p", "y0p", "s0", "dp0", "qx", "qy", "path"):
            del z[k]

    def beta(self, dp):
        p = self.Po * (1 + dp)
        return p / torch.sqrt(p * p + 1)

    def field(self, k1, h, x, y):
        """(Bx, By) in units of the dipole field: 1 in the mid-plane on axis"""
        if k1 is None:
            return torch.zeros_like(x), torch.ones_like(x)
        if h not in self.fields:
            self.fields[h] = _bend_field(1.0, h)
        px, py = [None, x], [None, y]
        for _ in range(3):
            px.append(px[-1] * x)
            py.append(py[-1] * y)

        def total(terms):
            out = None
            for i, j, c in terms:
                v = c * px[i] if i else c
                v = v * py[j] if j else v
                out = v if out is None else out + v
            return out

        fx, fy = self.fields[h]
        return k1 * total(fx), 1 + k1 * total(fy)

    def bend(self, i, event, z_start):
        s, z = self.structs[0][i], self.z
        fse = self.par(i, "fse", 3)
        k1 = self.par(i, "k1", 0)
        rho0 = s.length / s.angle
        h = 1 / rho0
        rho_a = rho0 / (1 + fse)
        if not torch.is_tensor(k1) and k1 == 0:
            kf = None
        else:  # the gradient scales with the magnet, the dipole part with 1 + FSE through rho_a
            kf = k1 * rho0
        psi = [2 * s.hgap * s.fint / rho_a / math.cos(e) * (1 + math.sin(e) ** 2) for e in (s.e1, s.e2)]
        rad = (E_MKS ** 2 * self.Po ** 3 * (1 + fse) ** 2 / (6 * math.pi * EPS0 * C_MKS ** 2 * ME_MKS * rho0 ** 2)
               if s.synch_rad else 0.0)

        def edge(z, e, ps):
            op = 1 + z["dp"]
            z["xp"] = z["xp"] + math.tan(e) / (op * rho_a) * z["x"]
            z["yp"] = z["yp"] - torch.tan(e - ps / op) / (op * rho_a) * z["y"]

        def adjust(z, e, sign):
            bx, by = self.field(kf, h, z["x"], z["y"])
            loss = -rad * (bx * bx + by * by) * (1 + z["dp"]) ** 2 * torch.sqrt(
                (1 + z["x"] * h) ** 2 + z["xp"] ** 2 + z["yp"] ** 2)
            z["dp"] = z["dp"] + sign * loss * z["x"] * math.tan(e)

        z["dp0"] = z["dp"]
        if s.edgeFlags & 1 and s.edge1_effects:
            edge(z, s.e1, psi[0])
        if rad and s.edgeFlags & 1 and s.e1:
            adjust(z, s.e1, -1)
        z["qx"], z["qy"] = self.momenta(z["xp"], z["yp"], z["dp"])
        z["path"] = torch.zeros_like(z["x"])
        sl, done = s.length / s.nSlices, 0.0

        def check():
            if self.watch and self.amp is not None:
                def row():
                    z = self.z
                    xp, yp = self.slopes(z["qx"], z["qy"], z["dp"])
                    return z["x"], xp, z["y"], yp, z_start + done, self.Po * (1 + z["dp"])
                self.lose(self.outside(self.z["x"], self.z["y"]), event, row)

        for _ in range(s.nSlices):
            check()
            z = self.z
            op = 1 + z["dp"]
            for j in range(4):
                th = sl * DRIFT4[j] / rho0
                f = torch.sqrt(op * op - z["qy"] * z["qy"])
                phi = torch.asin(z["qx"] / f)
                ang = phi + th
                c = torch.cos(ang)
                R = rho0 + z["x"]
                F = R * math.sin(th) / (f * c)
                # rho0 (cos phi / cos ang - 1) without the cancellation
                g = 2 * math.sin(th / 2) * torch.sin(phi + th / 2) / c
                z["x"] = z["x"] + R * g
                z["y"] = z["y"] + z["qy"] * F
                z["path"] = z["path"] + F * op
                z["qx"] = f * torch.sin(ang)
                done += sl * DRIFT4[j]
                if j == 3:
                    break
                bx, by = self.field(kf, h, z["x"], z["y"])
                h1 = 1 + z["x"] * h
                ds = sl * KICK4[j]
                z["qx"] = z["qx"] - ds * h1 * by / rho_a
                z["qy"] = z["qy"] + ds * h1 * bx / rho_a
                if rad:
                    xp, yp = self.slopes(z["qx"], z["qy"], z["dp"])
                    w = h1 * torch.sqrt(1 + xp ** 2 + yp ** 2)
                    new = z["dp"] - rad * op ** 2 * (bx * bx + by * by) * ds * w
                    g = (1 + new) / op
                    z["qx"], z["qy"], z["dp"] = z["qx"] * g, z["qy"] * g, new
                    op = 1 + new
        done = s.length
        check()
        z = self.z
        z["xp"], z["yp"] = self.slopes(z["qx"], z["qy"], z["dp"])
        if rad:
            if s.edgeFlags & 2 and s.e2:
                adjust(z, s.e2, -1)
            z["s"] = self.beta(z["dp"]) * z["s"] / self.beta(z["dp0"]) + z["path"]
        else:
            z["s"] = z["s"] + z["path"]
        if s.edgeFlags & 2 and s.edge2_effects:
            edge(z, s.e2, psi[1])
        for k in ("dp0", "qx", "qy", "path"):
            del z[k]

    def cavity(self, i, phases):
        s, z = self.structs[0][i], self.z
        L, omega, volt = s.length, 2 * math.pi * s.freq, s.volt / (1e6 * S.ME_MEV)
        P = self.Po * (1 + z["dp"])
        gamma = torch.sqrt(P * P + 1)
        beta = P / gamma
        if i not in phases:  # each variant's phase is fixed by the mean arrival time of its beam
            t = (z["s"] + L / 2) / (C_MKS * beta)
            parts = torch.split(t.detach(), self.counts.tolist()) if len(self.lats) > 1 else [t.detach()]
            mean = torch.stack([p.mean() if len(p) else p.sum() for p in parts])
            phases[i] = torch.repeat_interleave(mean, self.counts) if len(self.lats) > 1 else mean[0]
        half = L / 2 * torch.sqrt(1 + z["xp"] ** 2 + z["yp"] ** 2)
        t = (z["s"] + half) / (C_MKS * beta)
        dgamma = volt * torch.sin(omega * (t - phases[i]) + s.phase * math.pi / 180)
        g1 = gamma + dgamma
        P1 = torch.sqrt(g1 * g1 - 1)
        u = dgamma * (g1 + gamma) / (P * (P1 + P))  # (P1 - P) / P
        R12 = L * torch.log1p(u) / u
        z["x"], z["y"] = z["x"] + R12 * z["xp"], z["y"] + R12 * z["yp"]
        z["xp"], z["yp"] = z["xp"] / (1 + u), z["yp"] / (1 + u)
        path = z["s"] + half + L / 2 * torch.sqrt(1 + z["xp"] ** 2 + z["yp"] ** 2)
        z["dp"] = (P * (1 + u) - self.Po) / self.Po
        z["s"] = P1 / g1 * path / beta

    def turn(self, t, phases):
        pos = 0.0
        lat = self.lats[0]
        for i, e in enumerate(lat.elements):
            s = self.structs[0][i]
            start, pos = pos, pos + e.length()
            if e.type == S.T_DRIF:
                self.drift(s.length)
            elif e.type in MULTIPOLES:
                self.multipole(i, e.type, (t, i, 0), start)
            elif e.type == S.T_CSBEND:
                self.bend(i, (t, i, 0), start)
            elif e.type == S.T_RFCA:
                self.cavity(i, phases)
            elif e.type == S.T_MAXAMP:
                self.amp = (s.x_max, s.y_max)
            else:
                raise NotImplementedError(e.type)
            self.sweep((t, i, 1), pos, e.type == S.T_DRIF)

    def track(self, turns, phases=None):
        phases = {} if phases is None else phases
        for t in range(turns):
            self.turn(t, phases)
        return self

    def coordinates(self):
        return torch.stack([self.z[k] for k in ("x", "xp", "y", "yp", "s", "dp")], 1)

    def rows(self, start):
        """the rows as elegant leaves them: each routine call moves a particle it
        loses to the end of the rows it still has"""
        n = len(start)
        out = start.copy()
        live = self.coordinates().cpu().numpy()
        out[self.z["id"].cpu().numpy(), :6] = live
        order, where, left = np.arange(n), np.arange(n), n
        k = 0
        while k < len(self.events):
            event, lost = self.events[k][0], []
            while k < len(self.events) and self.events[k][0] == event:
                ids, vals = self.events[k][1:]
                out[ids, :6] = vals
                out[ids, S.LOSS_PASS_INDEX] = event[0]
                lost.extend(ids.tolist())
                k += 1
            gone = set(lost)
            for p in sorted(where[lost].tolist()):
                while p < left and order[p] in gone:
                    left -= 1
                    a, b = order[p], order[left]
                    order[p], order[left] = b, a
                    where[a], where[b] = left, p
        return out[order], left


def exact(case, seed):
    kind = case["kind"]
    if kind == "matrix":
        rows = _matched("mba", case["n"], seed)
        v = torch.tensor(rows[:, :6])
        for C0, R, T in _matrices(case, seed):
            w = torch.tensor(C0) + v @ torch.tensor(R).T
            if T is not None:
                tri = [(i, j, k, T[i, j, k]) for i in range(6) for j in range(6) for k in range(j + 1) if T[i, j, k]]
                for i, j, k, c in tri:
                    w[:, i] += c * v[:, j] * v[:, k]
            v = w
        rows[:, :6] = v.numpy()
        return {"rows": _parts(rows)}
    if kind == "track":
        lat = copy.deepcopy(_ring(case["ring"], case["cells"]))
        # launches of about 8 microseconds, or the memory traffic of a large beam
        if _operations(lat) * case["turns"] * max(8e-6, case["n"] * 1e-11) > 18:
            return None
        rows = _rows(case, seed)
        with torch.no_grad():
            b = _Exact([lat], [rows], P_FODO if case["ring"] == "fodo" else P_MBA).track(case["turns"])
            out, left = b.rows(rows)
        return {"rows": _parts(out), "survivors": left}
    if kind == "batch":
        lats = _variants(case["cells"], case["variants"], seed)
        rows = [_matched("mba", n, seed * 1009 + v) for v, n in enumerate(_counts(case))]
        n = sum(len(r) for r in rows)
        if _operations(lats[0]) * case["turns"] * max(9e-6, n * 1e-11) > 18:
            return None
        with torch.no_grad():
            b = _Exact(lats, rows, P_MBA).track(case["turns"])
            final = b.coordinates().cpu().numpy()
        out, k = [], 0
        for r in rows:
            r = r.copy()
            r[:, :6] = final[k:k + len(r)]
            k += len(r)
            out.append(_parts(r))
        return {"rows": out, "survivors": n}
    lats, rows, spec, cot = _gradient_inputs(case, seed)
    n = sum(len(r) for r in rows)
    ops = _operations(lats[0]) * case["turns"]
    if ops * 22e-6 > 18 or ops * n * 16 > 1.5e11:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    theta = torch.tensor(spec.values(lats[0]), device=dev, requires_grad=True)
    b = _Exact(lats, rows, P_MBA, theta, spec.slot_array(lats[0]))
    z0 = b.coordinates().detach().requires_grad_(True)
    # the cavity's phase is the one the first pass of the unchanged beam fixes
    phases = {}
    with torch.no_grad():
        b.track(1, phases)
    b = _Exact(lats, rows, P_MBA, theta, spec.slot_array(lats[0]))
    for q, k in enumerate(("x", "xp", "y", "yp", "s", "dp")):
        b.z[k] = z0[:, q]
    final = b.track(case["turns"], phases).coordinates()
    gt, gz = torch.autograd.grad(final, (theta, z0), torch.tensor(np.concatenate(cot), device=dev))
    final = final.detach()
    if kind == "adjoint":
        return {"final": _parts(final), "alive": torch.ones(n, dtype=torch.bool, device=dev), "grad_theta": gt, "grad_z0": gz}
    sizes = [len(r) for r in rows]
    return {"final": [_parts(f) for f in torch.split(final, sizes)], "alive": [np.ones(m, dtype=bool) for m in sizes],
            "grad_theta": gt, "grad_z0": list(torch.split(gz, sizes))}
