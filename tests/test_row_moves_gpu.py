"""Rows on their way to the device and back: adjacent rows (one copy) and
rows that are not, few rows (ordered on the host) and many (on the device),
with and without losses, wider rows, accepted rows."""
import ctypes as C

import numpy as np
import pytest

from elegant_amd import _abi as A
from elegant_amd import elements as E
from elegant_amd import native
from oracle import oracle_ctypes as O
from tests.helpers import assert_rows_bitwise
from tests.test_elements_gpu import PO, beam

pytestmark = pytest.mark.gpu


def pointers(block, w, adjacent):
    """row pointers over block (n, w), or over the same rows two apart"""
    if adjacent:
        return A.rows_pointer(block) + (block,)
    wide = np.full((2 * block.shape[0], w), 7.5)
    wide[::2] = block
    ptr, keep = A.rows_pointer(wide)
    every = np.ascontiguousarray(keep[::2])
    return every.ctypes.data_as(C.POINTER(C.POINTER(C.c_double))), every, wide


def rows_of(holder, adjacent):
    if adjacent:
        return holder
    assert (holder[1::2] == 7.5).all()  # what lies between the rows is not ours
    return holder[::2]


@pytest.mark.parametrize("adjacent", [True, False])
@pytest.mark.parametrize("n,w,loss", [(1, 8, True), (255, 8, False), (257, 11, True), (14563, 8, True),
                                      (14564, 8, False), (14564, 8, True), (20011, 10, True)])
def test_element_rows(tracker, n, w, loss, adjacent):
    """an aperture check over rows of w columns (14563 rows of 8 columns with
    their loss records are the most that take the small copy): survivors and
    order as the checker's, other columns and accepted rows follow"""
    r = np.zeros((n, w))
    r[:, :8] = beam(n, 5)[:, :8]
    r[:, 7:] = np.arange(n)[:, None] + np.arange(w - 7) / 64
    xmax, ymax = (0.004, 0.002) if loss else (10.0, 10.0)
    c = r[:, :8].copy()
    cp, keep = A.rows_pointer(c)
    nc = O.lib("glibc").or_limit_amplitudes(cp, xmax, ymax, n, 9.0, PO, 1, 0)
    assert (nc < n) == (loss and n > 1)
    ptr, k1, held = pointers(r.copy(), w, adjacent)
    acc, k2, aheld = pointers(-r, w, adjacent)
    tracker.set_particle_properties(w)
    try:
        ng = native.lib().eh_limit_amplitudes(tracker._ctx, ptr, xmax, ymax, n, acc, 9.0, PO, 1, 0)
    finally:
        tracker.set_particle_properties(8)
    g = rows_of(held, adjacent)
    assert ng == nc
    assert_rows_bitwise(np.ascontiguousarray(g[:, :7]), np.ascontiguousarray(c[:, :7]), "rows")
    src = g[:, 6].astype(np.int64) - 1  # IDs are 1..n
    assert_rows_bitwise(np.ascontiguousarray(g[:, 7:]), np.ascontiguousarray(r[src, 7:]), "other columns")
    assert_rows_bitwise(np.ascontiguousarray(rows_of(aheld, adjacent)), np.ascontiguousarray(-r[src]), "accepted")


@pytest.mark.parametrize("adjacent", [True, False])
@pytest.mark.parametrize("n", [1, 256, 14565])
def test_upload_track_download(tracker, n, adjacent):
    """do_tracking's calls over both kinds of rows, with rows culled for NaN
    and infinity before the first element, against the one-call entry"""
    r = beam(n, 6)[:, :8].copy()
    if n > 1:
        r[n // 2, 0] = np.nan
        r[n - 1, 2] = np.inf
    bl = E.Beamline([E.MAXAMP(X_MAX=0.004, Y_MAX=0.003), E.DRIF(L=0.7), E.KQUAD(L=0.3, K1=0.9, N_KICKS=4)])
    o = O.Oracle("emath")
    c = r.copy()
    o_left = o.do_tracking(c, bl, PO, 3)
    tracker.load(bl, PO)
    ptr, k1, held = pointers(r.copy(), 8, adjacent)
    native.check(tracker._ctx, native.lib().eh_upload(tracker._ctx, ptr, n, 8))
    tracker.n = n
    held[:] = 7.5  # the rows are the caller's again once eh_upload returns
    st = tracker.track(0, 3)
    left = C.c_int64()
    native.check(tracker._ctx, native.lib().eh_download(tracker._ctx, ptr, n, 8, C.byref(left)))
    assert left.value == o_left == st.n_left
    assert_rows_bitwise(np.ascontiguousarray(rows_of(held, adjacent)[:, :7]),
                        np.ascontiguousarray(c[:, :7]), "tracked")


def test_columns_taken_by_a_batch(tracker):
    """a batch of the context leaves its own particles on the device: the
    upload before it is refused, not read as if it were still there"""
    bl = E.Beamline([E.DRIF(L=0.7)])
    tracker.load(bl, PO)
    tracker.upload(beam(300, 8))
    b = native.Batch(tracker)
    b.add_variant(bl, PO, beam(500, 9))
    b.track(0, 1)
    b.close()
    for call in (lambda: tracker.track(0, 1), tracker.download):
        with pytest.raises(native.EHError) as e:
            call()
        assert e.value.code == A.EH_ERR_STATE


def refused(call):
    with pytest.raises(native.EHError) as e:
        call()
    assert e.value.code == A.EH_ERR_STATE


@pytest.mark.parametrize("sizes", [(300,), (500, 300)])
def test_columns_taken_by_a_batch_of_the_same_size(tracker, sizes):
    """the count of particles does not tell whose they are: a batch as large
    as the upload, also after a larger one for which the columns were
    allocated anew"""
    bl = E.Beamline([E.DRIF(L=0.7)])
    tracker.load(bl, PO)
    tracker.upload(beam(300, 8))
    for n in sizes:
        b = native.Batch(tracker)
        b.add_variant(bl, PO, beam(n, 9))
        b.track(0, 1)
        b.close()
    for call in (lambda: tracker.track(0, 1), tracker.download, tracker.loss_records):
        refused(call)
    r = beam(300, 8)[:, :8]
    tracker.upload(r)
    assert tracker.track(0, 1).n_left == 300
    assert np.array_equal(tracker.download()[0][:, 6], r[:, 6])


def test_batch_whose_columns_are_taken(tracker):
    """an element call, an upload and another batch, each with as many
    particles as the batch: its own are gone; another context's are not"""
    bl = E.Beamline([E.MAXAMP(X_MAX=1.0, Y_MAX=1.0), E.DRIF(L=0.7)])
    r = np.ascontiguousarray(beam(300, 8)[:, :8])

    def batch(t):
        b = native.Batch(t)
        b.add_variant(bl, PO, r)
        b.set_tuning(1, 64, 4)
        b.track(0, 1)
        return b

    other = native.Tracker(0)
    for take in (lambda: tracker.track_particles_drift(r.copy(), E.DRIF(L=0.1).p.drift), lambda: tracker.upload(r),
                 lambda: batch(tracker).close()):
        b, o = batch(tracker), batch(other)
        take()
        for call in (lambda: b.track(1, 1), lambda: b.download(0), lambda: b.loss_passes(0), b.autotune,
                     lambda: b.set_tuning(2, 64, 4)):
            refused(call)
        assert o.track(1, 1).n_left == 300 and o.download(0)[1] == 300
        b.close()
        o.close()
    other.close()


@pytest.mark.parametrize("adjacent", [True, False])
@pytest.mark.parametrize("n,w,loss", [(257, 20, True), (257, 21, True), (256, 33, False), (20011, 20, True),
                                      (20011, 21, True), (14564, 21, False)])
def test_element_wide_rows(tracker, n, w, loss, adjacent):
    """rows of up to 20 columns move whole, wider ones send eight"""
    test_element_rows(tracker, n, w, loss, adjacent)


@pytest.mark.parametrize("w", [9, 20, 21, 40])
def test_wide_rows_through_do_tracking(tracker, w):
    """the first eight columns as without the others, which follow their
    particle, as the accepted rows do"""
    n = 5003
    bl = E.Beamline([E.MAXAMP(X_MAX=0.004, Y_MAX=0.003), E.DRIF(L=0.7), E.KQUAD(L=0.3, K1=0.9, N_KICKS=4)])
    r = np.zeros((n, w))
    r[:, :8] = beam(n, 6)[:, :8]
    r[:, 8:] = np.arange(n)[:, None] + np.arange(w - 8) / 64
    g8, gw = np.ascontiguousarray(r[:, :8]), r.copy()
    a8, aw = np.zeros_like(g8), np.zeros_like(gw)
    left8, _ = tracker.do_tracking(g8, bl, PO, 3, accepted=a8)
    tracker.set_particle_properties(w)
    try:
        leftw, _ = tracker.do_tracking(gw, bl, PO, 3, accepted=aw)
    finally:
        tracker.set_particle_properties(8)
    assert left8 == leftw and 0 < left8 < n
    assert_rows_bitwise(np.ascontiguousarray(gw[:, :8]), g8, "rows")
    src = gw[:, 6].astype(np.int64) - 1
    assert_rows_bitwise(np.ascontiguousarray(gw[:, 8:]), np.ascontiguousarray(r[src, 8:]), "other columns")
    assert_rows_bitwise(aw, np.ascontiguousarray(r[src]), "accepted")


@pytest.fixture
def staged(tracker):
    """1000 rows at a time to and from the device"""
    tracker.set_stage_rows(1000)
    yield tracker
    tracker.set_stage_rows(0)


@pytest.mark.parametrize("adjacent", [True, False])
@pytest.mark.parametrize("n,w,loss", [(1000, 8, True), (1001, 8, True), (2000, 11, True), (20011, 8, False),
                                      (20011, 21, True)])
def test_element_rows_in_stages(staged, n, w, loss, adjacent):
    test_element_rows(staged, n, w, loss, adjacent)


@pytest.mark.parametrize("adjacent", [True, False])
@pytest.mark.parametrize("n", [1000, 2001, 14565])
def test_upload_track_download_in_stages(staged, n, adjacent):
    test_upload_track_download(staged, n, adjacent)


@pytest.mark.parametrize("w", [9, 21])
def test_wide_rows_in_stages(staged, w):
    test_wide_rows_through_do_tracking(staged, w)


def test_cavity_in_stages(staged):
    """the fiducial mean over arrival times that come back in stages, and an
    impedance step's rows"""
    bl = E.Beamline([E.MAXAMP(X_MAX=0.004, Y_MAX=0.003), E.DRIF(L=0.7), E.RFCA(VOLT=1e6, FREQ=352e6, PHASE=90.0)])
    z = E.ZLONGIT(BROAD_BAND=1, RS=1e4, Q=1.0, FREQ=20e9, N_BINS=1024, BIN_SIZE=1e-12, ALLOW_LONG_BEAM=1)
    r = np.ascontiguousarray(beam(3500, 6)[:, :8])
    out = []
    for stage in (1000, 0):
        staged.set_stage_rows(stage)
        a, b = r.copy(), r.copy()
        left, _ = staged.do_tracking(a, bl, PO, 2)
        phase = staged.rfca_fiducial(2)
        staged.track_through_zlongit(b, z.p.zlongit, PO, 0, 1e-12)
        out.append((left, phase, a, b))
    assert out[0][:2] == out[1][:2] and 0 < out[0][0] < 3500
    assert_rows_bitwise(out[0][2], out[1][2], "tracked")
    assert_rows_bitwise(out[0][3], out[1][3], "impedance")
