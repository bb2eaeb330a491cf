"""The integrators for regular particles against the oracle, where they can go
wrong: at and beyond every limit at which a particle leaves them for the general
ones, at zeros of either sign and near underflow.  Bit for bit, signs of zeros
included; no tolerance."""
import ctypes as C

import numpy as np
import pytest

from elegant_amd import configs, structs as S, tracking
from elegant_amd.lattice import Element, Lattice
from oracle import oracle
from tests.test_batch_host import _host_track, harness

Po = configs.p_central_from_mev(3000.0)
BEND = dict(L=0.8, ANGLE=0.0314, N_KICKS=3, EDGE1_EFFECTS=0, EDGE2_EFFECTS=0)

# element, and the regular path its descriptor asks for
ELEMENTS = {
    "bend": (Element("B", "CSBEND", **BEND), True),
    "bend_edges": (Element("B", "CSBEND", **{**BEND, "EDGE1_EFFECTS": 1, "EDGE2_EFFECTS": 1, "E1": 0.01, "HGAP": 0.01}),
                   True),
    "bend_k1": (Element("B", "CSBEND", K1=-0.5, FSE=1e-3, **BEND), True),
    "bend_k1_order2": (Element("B", "CSBEND", K1=0.5, INTEGRATION_ORDER=2, **BEND), True),
    "bend_k1_order6": (Element("B", "CSBEND", K1=0.5, INTEGRATION_ORDER=6, **BEND), True),
    "bend_k1_k2": (Element("B", "CSBEND", K1=0.5, K2=3.0, **BEND), True),
    "bend_k3": (Element("B", "CSBEND", K3=30.0, **BEND), True),
    "bend_wide_angle": (Element("B", "CSBEND", **{**BEND, "ANGLE": 0.15}), True),
    "bend_steep_steps": (Element("B", "CSBEND", **{**BEND, "ANGLE": 0.5}), False),
    "bend_negative": (Element("B", "CSBEND", K1=0.3, **{**BEND, "ANGLE": -0.0314}), False),
    "bend_tilted": (Element("B", "CSBEND", K1=0.3, TILT=0.1, **BEND), False),
    "quad": (Element("Q", "KQUAD", L=0.25, K1=2.9, N_KICKS=8), True),
    "quad_offset_kicks": (Element("Q", "KQUAD", L=0.25, K1=-1.4, N_KICKS=8, DX=3e-5, DY=-2e-5, DZ=1e-5, FSE=1e-3,
                                  HKICK=1e-5, VKICK=-2e-5), True),
    "quad_order2": (Element("Q", "KQUAD", L=0.25, K1=1.0, N_KICKS=3, INTEGRATION_ORDER=2), True),
    "quad_order6": (Element("Q", "KQUAD", L=0.25, K1=1.0, N_KICKS=12, INTEGRATION_ORDER=6), True),
    "quad_tilted": (Element("Q", "KQUAD", L=0.25, K1=1.0, N_KICKS=8, TILT=0.2), False),
    "quad_thin": (Element("Q", "KQUAD", L=0.0, K1=1.0, N_KICKS=8), False),
    "quad_off": (Element("Q", "KQUAD", L=0.25, K1=0.0, N_KICKS=8), False),
    "sext": (Element("X", "KSEXT", L=0.2, K2=-25.0, N_KICKS=4), True),
    "sext_k1": (Element("X", "KSEXT", L=0.2, K2=-25.0, K1=0.1, N_KICKS=4), False),
    "bend_rad": (Element("B", "CSBEND", SYNCH_RAD=1, **BEND), True),
    "bend_k1_rad_edges": (Element("B", "CSBEND", K1=0.5, SYNCH_RAD=1, **{
        **BEND, "EDGE1_EFFECTS": 1, "EDGE2_EFFECTS": 1, "E1": 0.015, "E2": 0.015, "HGAP": 0.01}), True),
    "bend_k2_rad": (Element("B", "CSBEND", K2=4.0, SYNCH_RAD=1, **BEND), True),
    "quad_rad": (Element("Q", "KQUAD", L=0.25, K1=2.9, N_KICKS=8, SYNCH_RAD=1, HKICK=1e-5, VKICK=-2e-5, DX=1e-4),
                 True),
    "quad_rad_order6": (Element("Q", "KQUAD", L=0.25, K1=2.9, N_KICKS=6, SYNCH_RAD=1, INTEGRATION_ORDER=6), False),
    "sext_rad": (Element("X", "KSEXT", L=0.2, K2=-25.0, N_KICKS=4, SYNCH_RAD=1), True),
    "oct_rad": (Element("O", "KOCT", L=0.2, K3=-1000.0, SYNCH_RAD=1), True),
    "oct": (Element("O", "KOCT", L=0.2, K3=-1000.0), True),
}
APERTURE = 0.02


def particles():
    """ordinary particles, and one or a pair beyond the limits at a time"""
    rng = np.random.default_rng(2)
    z = [[3e-3 * u[0], 5e-4 * u[1], 2e-3 * u[2], 5e-4 * u[3], 1e-3 * u[4], 2e-3 * u[5]]
         for u in rng.standard_normal((48, 6))]
    base = [1.3e-3, 2.1e-4, -7e-4, 3.3e-4, 1e-3, 4e-4]
    nxt = np.nextafter

    def put(k, values):
        for v in values:
            p = list(base)
            p[k] = v
            z.append(p)

    around = lambda v: [nxt(v, 0), v, nxt(v, 1e9)]  # noqa: E731
    lim = around(APERTURE) + around(10.0)
    put(0, lim + [-v for v in lim] + [0.0, -0.0, 1e-300, 5e-324, np.inf, np.nan])
    put(2, lim + [0.0, -0.0, -1e-300, 5e-324, -np.inf, np.nan])
    slope = around(2.0 ** -8) + around(0.0117) + around(0.05) + around(0.0625) + [0.0116, 0.0118, 0.3]
    tiny = [0.0, -0.0, 1e-300, -1e-300, 2e-103, 4e-103, 5e-324, np.inf, np.nan]
    put(1, slope + [-v for v in slope] + tiny)
    put(3, slope + [-v for v in slope] + tiny)
    put(5, around(-0.125) + around(0.25) + [-0.3, 0.5, -0.999, -1.0, -1.5, 0.0, 2.0 ** -53, -2.0 ** -53, np.nan])
    for p in ([0.0] * 6, [-0.0] * 6, [1e-3, 0, 0, 0, 0, 0], [0, 0, 1e-3, 0, 0, 0], [1e-3, -0.0, -0.0, -0.0, 0, 0],
              [1e-3, 1e-4, 1e-300, 0, 0, 0], [1e-3, 1e-4, 0, 1e-300, 0, 0], [1e-3, 1e-4, 1e-160, 1e-200, 0, 1e-3],
              [2e-310, 1e-310, 3e-310, 1e-310, 0, 0]):
        z.append(list(p))
    rows = np.zeros((len(z), S.NPROP))
    rows[:, :6] = z
    rows[:, 6] = np.arange(1, len(z) + 1)
    return rows


def line(name):
    return Lattice([Element("AP", "MAXAMP", X_MAX=APERTURE, Y_MAX=APERTURE), ELEMENTS[name][0]])


def identical(got, ref):
    """doubles equal, NaN for NaN, zeros of one sign"""
    return ((got == ref) & (np.signbit(got) == np.signbit(ref))) | (np.isnan(got) & np.isnan(ref))


def check(got, ref, what):
    bad = np.argwhere(~identical(got, ref))
    assert not len(bad), "%s: %d entries differ, first at id %d column %d: %r, oracle %r" % (
        what, len(bad), ref[bad[0][0], 6] if ref.shape[1] > 6 else -1, bad[0][1], got[tuple(bad[0])],
        ref[tuple(bad[0])])


def test_quotients_and_roots_are_correctly_rounded():
    assert harness().bh_regular_arithmetic(400000, 5) == 0


def test_quotients_and_roots_of_radiating_particles_are_correctly_rounded():
    assert harness().bh_regular_radiation(200000, 7) == 0


@pytest.mark.parametrize("name", sorted(ELEMENTS))
def test_host_build_matches_oracle(name):
    rows = particles()
    r, out6, lpass, _ = _host_track([rows], [line(name)], 2, Po, None, 1)
    ref, n, _, _ = oracle.do_tracking(rows, line(name), 2, Po)
    assert r == n
    got = ref.copy()
    where = ref[:, 6].astype(int) - 1
    got[:, :6] = out6[where]
    # the position of a loss at entry, or in an element with an exit offset, is settled on download
    settled = (lpass[where] != -1) & ((lpass[where] & 0x40000000 != 0) | ("DX" in ELEMENTS[name][0].params))
    got[settled, 4] = ref[settled, 4]
    check(got, ref, name)


@pytest.mark.parametrize("name", sorted(ELEMENTS))
def test_who_is_regular(name):
    """ordinary particles take the regular path of every element that has one,
    particles beyond a limit do not"""
    el, has = ELEMENTS[name]
    arr, keep = Lattice([el]).c_beamline()
    rows = particles()
    z = np.ascontiguousarray(rows[:, :6])
    taken = np.zeros(len(z), dtype=np.int32)
    f = harness().bh_regular_taken
    f.argtypes = [C.c_void_p, C.c_long, C.c_void_p, C.c_double, C.c_double, C.c_double, C.c_void_p]
    f.restype = C.c_long
    n = f(z.ctypes.data, len(z), C.cast(arr, C.c_void_p), APERTURE, APERTURE, Po, taken.ctypes.data)
    assert n == taken.sum()
    if not has:
        assert n == 0
        return
    assert taken[:48].all()
    out = (~np.isfinite(z[:, [0, 1, 2, 3, 5]]).all(1)) | (np.abs(z[:, 3]) > 0.0125) | (z[:, 5] < -0.126) | (
        z[:, 5] > 0.2501) | (np.abs(z[:, 0]) > APERTURE + 1e-4) | (np.abs(z[:, 2]) > APERTURE + 1e-4)
    assert out.sum() > 20 and not taken[out].any()


def regular_path(el, P, z):
    """(whether the element asks for the regular path, how many particles it takes)"""
    arr, keep = Lattice([el]).c_beamline()
    z = np.ascontiguousarray(z)
    taken = np.zeros(len(z), dtype=np.int32)
    h = harness()
    h.bh_regular_taken.argtypes = [C.c_void_p, C.c_long, C.c_void_p, C.c_double, C.c_double, C.c_double, C.c_void_p]
    h.bh_regular_taken.restype = C.c_long
    h.bh_regular_asked.argtypes = [C.c_void_p, C.c_double]
    h.bh_regular_asked.restype = C.c_long
    asked = h.bh_regular_asked(C.cast(arr, C.c_void_p), P)
    assert asked >= 0
    return asked > 0, h.bh_regular_taken(z.ctypes.data, len(z), C.cast(arr, C.c_void_p), 0.0, 0.0, P,
                                         taken.ctypes.data)


@pytest.mark.parametrize("rad", [0, 1])
@pytest.mark.parametrize("order", [2, 4, 6])
def test_no_bend_asks_for_what_it_cannot_pass(order, rad):
    """the design orbit swings by the sub-step angles and radiates at every kick: a bend
    whose swing or energy loss no particle can follow does not ask for the regular path,
    and one that asks passes a small beam whole"""
    rng = np.random.default_rng(6)
    z = rng.standard_normal((64, 6)) * [5e-5, 5e-5, 5e-5, 5e-5, 1e-4, 2e-4]
    seen = set()
    for mev in (300.0, 3000.0, 7000.0):
        for rho in (2.0, 6.4, 25.0, 39.0):
            for degrees in (0.5, 4.5, 18.0, 40.0):
                for kicks in (4, 5, 6, 8, 12, 30):
                    angle = np.radians(degrees)
                    el = Element("B", "CSBEND", L=rho * angle, ANGLE=angle, N_KICKS=kicks, INTEGRATION_ORDER=order,
                                 SYNCH_RAD=rad, EDGE1_EFFECTS=0, EDGE2_EFFECTS=0)
                    asked, n = regular_path(el, configs.p_central_from_mev(mev), z)
                    assert n == (len(z) if asked else 0), (mev, rho, degrees, kicks, n)
                    seen.add(asked)
    assert seen == {False, True}


@pytest.mark.parametrize("kick", [0.0, 1e-3, 0.02])
def test_no_corrector_asks_for_what_it_cannot_pass(kick):
    z = np.random.default_rng(6).standard_normal((64, 6)) * 5e-5
    for plane in ("HKICK", "VKICK"):
        el = Element("Q", "KQUAD", L=0.25, K1=1.0, N_KICKS=8, **{plane: kick})
        assert regular_path(el, Po, z) == ((True, len(z)) if kick < 0.01 else (False, 0))


@pytest.mark.gpu
@pytest.mark.parametrize("lane", [0, 17, 63])
@pytest.mark.parametrize("slope", [0.0115, 0.013])  # leaves the limits inside the quadrupole, at its entry
def test_one_irregular_particle_in_a_wavefront(ehlib, lane, slope):
    rng = np.random.default_rng(lane)
    rows = np.zeros((192, S.NPROP))  # the first and the last wavefront are regular
    rows[:, :6] = rng.standard_normal((192, 6)) * [1e-3, 2e-4, 1e-3, 2e-4, 1e-3, 1e-3]
    rows[64 + lane, :4] = [2e-3, slope, -3e-3, -slope]
    rows[:, 6] = np.arange(1, 193)
    lat = Lattice([ELEMENTS[k][0] for k in ("quad", "bend_k1", "sext", "quad_rad")])
    ref, nref, _, _ = oracle.do_tracking(rows, lat, 2, Po)
    beam = tracking.Beam(rows)
    n, _, _ = tracking.track(beam, lat, 2, Po, mode="fused", turns_per_launch=2)
    got = beam.download()
    beam.free()
    assert n == nref == 192
    check(got, ref, "lane %d slope %g" % (lane, slope))


UNBOUNDED = [(np.inf, 0.02), (0.02, np.inf), (np.inf, np.inf), (np.nan, 0.02), (np.finfo(float).max, 0.02)]


def overflowing():
    """an aperture's limit may be infinite, a coordinate that overflows is lost all
    the same: (line, rows) per limits, drifts and a bend whose entry is at 1e308"""
    rows = np.zeros((4, S.NPROP))
    rows[1, 1] = rows[2, 3] = 1e307
    rows[3, 0] = rows[3, 2] = 1e308
    rows[:, 6] = np.arange(1, 5)
    for x, y in UNBOUNDED:
        for els in ([Element("D", "EDRIFT", L=1000.0)], [Element("D", "DRIF", L=1000.0), ELEMENTS["bend"][0]]):
            yield Lattice([Element("AP", "MAXAMP", X_MAX=x, Y_MAX=y)] + els), rows, "%g %g" % (x, y)


def test_infinite_limits_keep_no_infinite_coordinate():
    for lat, rows, what in overflowing():
        r, out6, lpass, _ = _host_track([rows], [lat], 1, Po, None, 1)
        ref, n, _, _ = oracle.do_tracking(rows, lat, 1, Po)
        alive = set(np.flatnonzero(lpass == -1) + 1)
        assert r == n and alive == set(ref[:n, 6].astype(int)), what
        check(out6[ref[:n, 6].astype(int) - 1], ref[:n, :6], what)


@pytest.mark.gpu
def test_infinite_limits_on_the_gpu(ehlib):
    for lat, rows, what in overflowing():
        ref, nref, _, _ = oracle.do_tracking(rows, lat, 1, Po)
        for mode in ("fused", "plain"):
            beam = tracking.Beam(rows)
            n, _, _ = tracking.track(beam, lat, 1, Po, mode=mode)
            got = beam.download()
            beam.free()
            assert n == nref, what
            check(got, ref, what + " " + mode)


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(ELEMENTS))
def test_gpu_matches_oracle(ehlib, name):
    rows = np.concatenate([particles()] * 3)
    rows[:, 6] = np.arange(1, len(rows) + 1)
    ref, nref, _, _ = oracle.do_tracking(rows, line(name), 2, Po)
    for mode in ("fused", "plain"):  # registers through the line; in place, element by element
        beam = tracking.Beam(rows)
        n, st, _ = tracking.track(beam, line(name), 2, Po, mode=mode, turns_per_launch=2)
        got = beam.download()
        beam.free()
        assert n == nref
        check(got, ref, name + " " + mode)
