"""A beam taken through a line by the entry points one after another, as the adapter
calls them from elegant's own loop: the element's routine, the aperture sweep, the
sweep of invalid particles.  Rows, loss order, loss passes and settled loss positions
bit for bit with the oracle's do_tracking."""
import ctypes as C
import sys

import numpy as np
import pytest

from elegant_amd import _lib, configs, structs as S, tracking
from elegant_amd.lattice import Element, Lattice
from oracle import oracle
from tests.helpers import assert_rows_identical

pytestmark = pytest.mark.gpu
Po = configs.p_central_from_mev(3000.0)


def line(offset):
    rf = dict(L=0.3, VOLT=2.0e6, PHASE=170.0, FREQ=6e8, N_KICKS=0)
    return Lattice([
        Element("AP", "MAXAMP", X_MAX=0.02, Y_MAX=0.015), Element("D1", "DRIF", L=0.8),
        Element("Q1", "KQUAD", L=0.3, K1=1.2, N_KICKS=8, DX=offset, DZ=2 * offset),
        Element("B1", "CSBEND", L=0.8, ANGLE=0.0314, K1=-0.4, N_KICKS=8, EDGE1_EFFECTS=0, EDGE2_EFFECTS=0),
        Element("RF", "RFCA", **rf), Element("X1", "KSEXT", L=0.2, K2=40.0, N_KICKS=4, DY=offset),
        Element("E1", "EDRIFT", L=0.6), Element("AQ", "MAXAMP", X_MAX=0.012, Y_MAX=0.02),
        Element("O1", "KOCT", L=0.2, K3=-2e4), Element("B2", "CSBEND", L=0.6, ANGLE=-0.02, N_KICKS=4, E1=0.01,
                                                       HGAP=0.01),
        Element("Q2", "KQUAD", L=0.3, K1=-1.3, N_KICKS=8), Element("D2", "DRIF", L=1.1)])


def by_entry_points(beam, lat, passes):
    L, h = tracking.lib(), beam.handle
    arr, keep = lat.c_beamline()
    structs = lat.structs()
    pc = C.c_double(Po)
    big = np.finfo(float).max
    n = _lib.check(L.eh_limit_amplitudes(h, big, big, beam.n_alive(), 0.0, Po, 0, 0))
    amp = None
    for p in range(passes):
        L.eh_beam_set_pass(h, p)
        z = 0.0
        for i, e in enumerate(lat.elements):
            z0, z = z, z + e.length()
            el = C.cast(C.byref(arr[i]), C.POINTER(S.EH_ELEMENT_LIST))
            limits = C.byref(amp) if amp is not None else None
            if e.type == S.T_MAXAMP:
                amp = structs[i]
            elif e.type == S.T_DRIF:
                n = L.eh_drift_beam(h, n, e.length(), 2)
            elif e.type == S.T_EDRIFT:
                n = L.eh_exactDrift(h, n, e.length())
            elif e.type == S.T_CSBEND:
                n = L.eh_track_through_csbend(h, n, C.byref(structs[i]), 0.0, Po, z0, limits, -1)
            elif e.type == S.T_RFCA:
                n = L.eh_simple_rf_cavity(h, n, C.byref(structs[i]), C.byref(pc), z)
            else:
                n = L.eh_multipole_tracking2(h, n, el, 0.0, Po, z0, limits, -1)
            _lib.check(n)
            if amp is not None:
                n = _lib.check(L.eh_limit_amplitudes(h, amp.x_max, amp.y_max, n, z, Po, e.type == S.T_DRIF, 0))
            n = _lib.check(L.eh_limit_amplitudes(h, big, big, n, z, Po, 0, 0))
    return n


@pytest.mark.parametrize("spread", [3e-4, 4e-3, 2e-2])  # none, some, nearly all lost
@pytest.mark.parametrize("offset", [0.0, 2e-3])  # entry losses inherit their position
def test_entry_points_one_after_another(ehlib, oracle_mod, spread, offset):
    print("entry points", spread, offset, flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(8)
    rows = np.zeros((3000, S.NPROP))
    rows[:, :6] = rng.standard_normal((3000, 6)) * [spread, spread / 3, spread, spread / 3, 1e-3, 2e-3]
    rows[5, 1], rows[6, 0], rows[7, 3], rows[8, 2] = 1.5, 12.0, np.nan, np.inf
    rows[:, 6] = np.arange(1, 3001)
    ref, nref, _, _ = oracle.do_tracking(rows, line(offset), 3, Po)
    beam = tracking.Beam(rows)
    n = by_entry_points(beam, line(offset), 3)
    got = beam.download()
    beam.free()
    assert_rows_identical(got, ref, n, nref, "spread %g offset %g" % (spread, offset))
    assert nref < 3000
    beam = tracking.Beam(rows)
    m, _, _ = tracking.track(beam, line(offset), 3, Po, mode="plain")
    plain = beam.download()
    beam.free()
    assert_rows_identical(plain, ref, m, nref, "plain mode, spread %g offset %g" % (spread, offset))
