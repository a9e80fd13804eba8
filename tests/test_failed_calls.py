"""What the library's host code does when a call of the HIP runtime fails:
every allocation, copy and event of a call is made to fail in turn, on the
CPU, against the runtime of fake_hip.c (in a process of its own; no kernel
runs)."""
import ctypes
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="session")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "fake_hip.so")
    subprocess.run(["gcc", "-O1", "-Wall", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "fake_hip.c")], check=True)
    return so


def run(fake, call):
    """call(F, native) in a process where fake's functions are the runtime"""
    code = "from tests import test_failed_calls as t; t.child(%r, t.%s)" % (fake, call.__name__)
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, text=True, timeout=120, stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT)
    assert r.returncode == 0, r.stdout[-2000:]


def child(fake, call):
    F = ctypes.CDLL(fake, mode=ctypes.RTLD_GLOBAL)
    for f in ("failed", "live", "nulls", "launches", "calls", "h2d_bytes", "device_bytes", "queued"):
        getattr(F, "fake_" + f).restype = ctypes.c_long
    F.fake_fail_at.argtypes = [ctypes.c_long]
    from elegant_amd import native
    native.Tracker(0).close()  # what the first context of a process makes and keeps
    call(F, native)


def each_failure(F, native, fresh, call, after=lambda s: None, most=200):
    """call(state) with its k-th runtime call failing, for every k, then once
    more unharmed on the same state"""
    seen = 0
    for k in range(1, most):
        before = F.fake_live()
        s = fresh()
        F.fake_fail_at(k)
        try:
            call(s)
            ok = True
        except native.EHError:
            ok = False
        hit = bool(F.fake_failed())
        F.fake_fail_at(0)
        assert ok != hit, "call %d failed unnoticed" % k
        assert F.fake_queued() == 0, "call %d: work left on a stream" % k
        after(s)
        call(s)
        assert F.fake_nulls() == 0, "call %d: NULL used after its failure" % k
        s[-1].close()
        assert F.fake_live() == before, "call %d: %d allocations left" % (k, F.fake_live() - before)
        if not hit:
            assert seen, "nothing was made to fail"
            return
        seen += 1
    raise AssertionError("more than %d runtime calls" % most)


def net(native):
    from elegant_amd import learned
    t = native.Tracker(0)
    return learned.MLP(t, hidden=16), t


def rows(n, w=8):
    import numpy as np
    r = np.zeros((n, w))
    r[:, 6] = np.arange(n)
    return r


def prediction(F, native):
    import numpy as np
    for n in (100, 70000):  # one chunk; three on two streams
        X = np.zeros((n, 19), np.float32)
        each_failure(F, native, lambda: net(native), lambda s: s[0].predict(X))


def gradient(F, native):
    import numpy as np
    X, y = np.zeros((1000, 19), np.float32), np.zeros(1000, np.float32)
    each_failure(F, native, lambda: net(native), lambda s: s[0].gradient(X, y))


def element(F, native):
    from elegant_amd import elements as E
    q = E.KQUAD(L=0.3, K1=1.0)
    for n in (100, 20000):  # the small copy back and the other one
        each_failure(F, native, lambda: (native.Tracker(0),),
                     lambda s: s[0].multipole_tracking2(rows(n), q, 1e4, 0.0))


def impedance(F, native):
    from elegant_amd import elements as E
    z = E.ZLONGIT(BROAD_BAND=1, RS=1e4, Q=1.0, FREQ=20e9, N_BINS=1024, BIN_SIZE=1e-12)
    each_failure(F, native, lambda: (native.Tracker(0),),
                 lambda s: s[0].track_through_zlongit(rows(1000), z.p.zlongit, 1e4, 0, 1e-12))


def tracking(F, native):
    from elegant_amd import elements as E
    from elegant_amd import lattices as Lt
    bl = E.Beamline([E.CHARGE(TOTAL=1e-9), E.KQUAD(L=0.3, K1=1.0), E.RFCA(L=0.1, VOLT=1e5, FREQ=352e6, PHASE=90.0),
                     E.WAKE(Lt.resonator_wake(points=200)), E.DRIF(L=0.5)])
    for n, w in ((300, 8), (300, 11)):
        def fresh():
            t = native.Tracker(0)
            t.set_particle_properties(w)
            return (t,)
        each_failure(F, native, fresh, lambda s: s[0].do_tracking(rows(n, w), bl, 1e4, 2), most=1000)


def test_prediction(fake):
    """a stream, event or buffer that could not be made is made by the next
    call, not used as if it were there"""
    run(fake, prediction)


@pytest.mark.parametrize("call", [gradient, element, impedance, tracking])
def test_nothing_in_flight(fake, call):
    """no copy from or to the caller's arrays outlives a failed call"""
    run(fake, call)


def wide_rows(F, native):
    from elegant_amd import elements as E
    bl = E.Beamline([E.DRIF(L=0.5)])
    q = E.KQUAD(L=0.3, K1=1.0)
    for n in (50, 20000):
        moved = {}
        for w in (8, 21, 64):
            t = native.Tracker(0)
            t.set_particle_properties(w)
            before = F.fake_h2d_bytes()
            t.do_tracking(rows(n, w), bl, 1e4, 1)
            between = F.fake_h2d_bytes()
            t.multipole_tracking2(rows(n, w), q, 1e4, 0.0)
            moved[w] = between - before, F.fake_h2d_bytes() - between
            t.close()
        assert moved[21] == moved[64] == moved[8], (n, moved)


def test_wide_rows_move_as_eight_columns(fake):
    """the device reads seven columns of a row: wide rows send eight"""
    run(fake, wide_rows)


def device_memory(F, native):
    from elegant_amd import elements as E
    bl = E.Beamline([E.DRIF(L=0.5), E.RFCA(VOLT=1e5, FREQ=352e6, PHASE=90.0)])
    q = E.KQUAD(L=0.3, K1=1.0)
    n, w = 6000011, 8
    r = rows(n, w)
    t = native.Tracker(0)
    before = F.fake_device_bytes()
    t.do_tracking(r, bl, 1e4, 1)
    t.multipole_tracking2(r, q, 1e4, 0.0)
    used = F.fake_device_bytes() - before
    t.close()
    assert used <= 64 * n + (2 << 28) + (1 << 26), (used, 64 * n)


def test_device_memory_per_particle(fake):
    """64 bytes per particle in the columns; rows pass through buffers of
    bounded size (256 MiB each)"""
    run(fake, device_memory)


def few_rows(F, native):
    import numpy as np
    n, t = net(native)
    X = np.zeros((100, 19), np.float32)
    before = F.fake_calls()
    n.predict(X)
    first = F.fake_calls() - before
    n.predict(X)
    again = F.fake_calls() - before - first
    t.close()
    # in, a launch looked after, out; the first time two buffers more
    assert (first, again) == (5, 3), (first, again)


def test_prediction_of_few_rows(fake):
    """no second stream and no events where there is one chunk"""
    run(fake, few_rows)


def contexts(F, native):
    live, calls = F.fake_live(), F.fake_calls()
    native.Tracker(0).close()
    each = F.fake_calls() - calls
    many = [native.Tracker(0) for _ in range(100)]
    while many:
        many.pop(len(many) // 2).close()
    native.Tracker(0).close()
    assert F.fake_live() == live
    assert each == 6, each  # a stream and five events, no memory


def test_context_makes_no_memory(fake):
    """creating a context allocates nothing once the process has had one, also
    after more of them than there are places for"""
    run(fake, contexts)
