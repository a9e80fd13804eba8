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
    for f in ("failed", "live", "nulls", "launches", "calls", "h2d_bytes", "queued"):
        getattr(F, "fake_" + f).restype = ctypes.c_long
    F.fake_fail_at.argtypes = [ctypes.c_long]
    from elegant_amd import native
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


def prediction(F, native):
    import numpy as np
    from elegant_amd import learned

    def fresh():
        t = native.Tracker(0)
        return learned.MLP(t, hidden=16), t

    X = np.zeros((70000, 19), np.float32)
    each_failure(F, native, fresh, lambda s: s[0].predict(X))


def test_prediction_set_up(fake):
    """a stream, event or buffer that could not be made is made by the next
    call, not used as if it were there"""
    run(fake, prediction)
