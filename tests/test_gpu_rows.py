"""Rows up and down: taken apart and put together on the device, in chunks of
262144, with losses moved to the reference's places.  Bit for bit with the oracle."""
import ctypes as C

import numpy as np
import pytest

from elegant_amd import _lib, configs, structs as S, tracking
from elegant_amd.lattice import Element, Lattice
from tests.helpers import assert_rows_identical

pytestmark = pytest.mark.gpu
Po = configs.p_central_from_mev(3000.0)


def line():
    return Lattice([Element("AP", "MAXAMP", X_MAX=0.01, Y_MAX=0.008), Element("D", "DRIF", L=1.0),
                    Element("Q", "KQUAD", L=0.2, K1=1.0, N_KICKS=4, DX=1e-4), Element("D", "DRIF", L=0.7)])


def rows_of(n, spread):
    rng = np.random.default_rng(n)
    rows = rng.standard_normal((n, S.NPROP)) * [spread, 1e-3, spread, 1e-3, 1e-3, 1e-3, 1, 1, 1, 1]
    rows[:, 6] = np.arange(1, n + 1)
    return rows


@pytest.mark.parametrize("n", [1, 2, 63, 1000, 262144, 262145, 600001])
@pytest.mark.parametrize("spread", [1e-4, 6e-3, 1.0])  # none, some, nearly all lost
def test_rows_round_trip(ehlib, oracle_mod, n, spread):
    rows = rows_of(n, spread)
    beam = tracking.Beam(rows)
    assert_rows_identical(beam.download(), rows, beam.n_alive(), n, "untracked")
    na, _, _ = tracking.track(beam, line(), 2, Po, mode="fused", turns_per_launch=1)
    got = beam.download()
    ref, nref, _, _ = oracle_mod.do_tracking(rows, line(), 2, Po)
    assert_rows_identical(got, ref, na, nref, "n=%d spread=%g" % (n, spread))
    order = beam.row_order()
    assert np.array_equal(rows[order, 6], got[:, 6])
    beam.free()


@pytest.mark.parametrize("n", [5, 262150])
def test_rows_by_pointer(ehlib, oracle_mod, n):
    """rows scattered in memory, as a caller may hand them over"""
    rows = rows_of(n, 6e-3)
    place = np.random.default_rng(1).permutation(n)
    store = np.zeros((n, S.NPROP + 3))
    store[place, :S.NPROP] = rows
    ptr = (store.ctypes.data + place.astype(np.uint64) * np.uint64(store.strides[0])).astype(np.uint64)
    L = tracking.lib()
    L.eh_beam_upload.argtypes = [C.c_void_p, C.c_void_p, C.c_long]
    L.eh_beam_download.argtypes = [C.c_void_p, C.c_void_p, C.c_long]
    beam = tracking.Beam(rows_of(n, 1e-4), capacity=n + 17)
    _lib.check(L.eh_beam_upload(beam.handle, ptr.ctypes.data, n))
    na, _, _ = tracking.track(beam, line(), 1, Po, mode="plain")
    store[:] = -7.0
    _lib.check(L.eh_beam_download(beam.handle, ptr.ctypes.data, n))
    ref, nref, _, _ = oracle_mod.do_tracking(rows, line(), 1, Po)
    assert_rows_identical(store[place, :S.NPROP], ref, na, nref, "by pointer")
    assert (store[:, S.NPROP:] == -7.0).all()
    beam.free()


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 128, 129, 200])
def test_line_lengths(ehlib, oracle_mod, n):
    """positions are read 64 at a time: lines of about that many elements and of
    multiples, spans that begin inside a line (after a cavity), losses all along"""
    rng = np.random.default_rng(n)
    kinds = [("DRIF", dict(L=0.3)), ("KQUAD", dict(L=0.2, K1=0.6, N_KICKS=2)), ("EDRIFT", dict(L=0.2)), ("MARK", {}),
             ("KSEXT", dict(L=0.1, K2=4.0, N_KICKS=2)), ("MAXAMP", dict(X_MAX=4e-3, Y_MAX=3e-3)),
             ("RFCA", dict(L=0.1, VOLT=1e5, FREQ=5e8, PHASE=90.0))]
    els = [Element("%s%d" % (kinds[k][0], k), kinds[k][0], **kinds[k][1])
           for k in np.append(rng.integers(0, 6, n - 1), 0 if n < 63 else 6)]
    rng.shuffle(els)
    rows = rows_of(400, 1e-3)
    ref, nref, _, _ = oracle_mod.do_tracking(rows, Lattice(els), 3, Po)
    for turns in (16, 1):
        beam = tracking.Beam(rows)
        na, _, st = tracking.track(beam, Lattice(els), 3, Po, mode="fused", turns_per_launch=turns)
        assert_rows_identical(beam.download(), ref, na, nref, "fused n=%d" % n)
        beam.free()
    batch = tracking.Batch([rows, rows[:65]])
    batch.track([Lattice(els), Lattice(els)], 3, Po, span_elements=70)
    assert_rows_identical(batch.download(0), ref, batch.n_alive(0), nref, "batch n=%d" % n)
    batch.free()


@pytest.mark.parametrize("counts", [[1], [0, 1, 64, 65], [300000, 5, 0, 129]])
def test_batch_rows(ehlib, oracle_mod, counts):
    """a variant's rows go up and down through memory that all variants share: chunks,
    empty variants, losses in some of them, a cavity's fiducial in each"""
    lat = [Lattice(line().elements + [Element("RF", "RFCA", L=0.1, VOLT=1e5, FREQ=5e8, PHASE=90.0)]) for _ in counts]
    ref_lat = [Lattice(line().elements + [Element("RF", "RFCA", L=0.1, VOLT=1e5, FREQ=5e8, PHASE=90.0)]) for _ in counts]
    rows = [rows_of(n, (6e-3, 1e-4)[v % 2]) if n else np.zeros((0, S.NPROP)) for v, n in enumerate(counts)]
    batch = tracking.Batch(rows)
    batch.track(lat, 2, Po)
    for v in reversed(range(len(counts))):
        ref, nref, _, _ = oracle_mod.do_tracking(rows[v], ref_lat[v], 2, Po)
        assert_rows_identical(batch.download(v), ref, batch.n_alive(v), nref, "variant %d" % v)
    batch.free()


@pytest.mark.parametrize("n", [1, 63, 262145])
@pytest.mark.parametrize("flat", [True, False])
def test_columns_on_the_host(ehlib, oracle_mod, n, flat):
    """a beam whose columns 6 to 9 did not fit on the device: rows consecutive or by
    pointer, up again after a run"""
    rows = rows_of(n, 6e-3)
    place = np.arange(n) if flat else np.random.default_rng(1).permutation(n)
    store = np.zeros((n, S.NPROP + (0 if flat else 2)))
    ptr = (store.ctypes.data + place.astype(np.uint64) * np.uint64(store.strides[0])).astype(np.uint64)
    L = tracking.lib()
    L.eh_beam_upload.argtypes = [C.c_void_p, C.c_void_p, C.c_long]
    L.eh_beam_download.argtypes = [C.c_void_p, C.c_void_p, C.c_long]
    beam = tracking.Beam(np.zeros((0, S.NPROP)), capacity=n + 5)
    _lib.check(L.eh_diag_host_columns(beam.handle, None))
    ref, nref, _, _ = oracle_mod.do_tracking(rows, line(), 1, Po)
    for _ in range(2):
        store[place, :S.NPROP] = rows
        _lib.check(L.eh_beam_upload(beam.handle, ptr.ctypes.data, n))
        na, _, _ = tracking.track(beam, line(), 1, Po)
        store[:] = -7.0
        _lib.check(L.eh_beam_download(beam.handle, ptr.ctypes.data, n))
        assert_rows_identical(store[place, :S.NPROP], ref, na, nref, "n=%d flat=%d" % (n, flat))
    assert L.eh_diag_host_columns(beam.handle, None) < 0
    beam.free()


def test_batch_columns_on_the_host(ehlib, oracle_mod):
    counts = [300, 0, 262150, 65]
    rows = [rows_of(n, (6e-3, 1e-4)[v % 2]) if n else np.zeros((0, S.NPROP)) for v, n in enumerate(counts)]
    batch = tracking.Batch(rows)
    L = tracking.lib()
    _lib.check(L.eh_diag_host_columns(None, batch._h))
    for v, r in enumerate(rows):
        r = np.ascontiguousarray(r)
        _lib.check(L.eh_batch_upload(batch._h, v, r.ctypes.data, len(r)))
    batch.track([line() for _ in counts], 2, Po)
    for v in reversed(range(len(counts))):
        ref, nref, _, _ = oracle_mod.do_tracking(rows[v], line(), 2, Po)
        assert_rows_identical(batch.download(v), ref, batch.n_alive(v), nref, "variant %d" % v)
    batch.free()
