"""The kernels' branch-free common paths at the edges of the ranges that
select them, against the checker bit for bit."""
import ctypes as C

import numpy as np
import pytest

from elegant_amd import _abi as A
from elegant_amd import elements as E
from oracle import oracle_ctypes as O
from tests.helpers import assert_rows_bitwise
from tests.test_elements_gpu import PO, assert_same_survivors, beam, csbend_edge_rows, rows_ptr

pytestmark = pytest.mark.gpu


def near_midpoint_squares(n, rng):
    """doubles whose square roots lie as close to a midpoint between two
    doubles as any: N = M^2 + M + d, |d| small, with N a multiple of 2^52
    (Hensel lifting of M^2 + M = -d modulo 2^52, d even)"""
    out = []
    for _ in range(n):
        d = 2 * int(rng.integers(-64, 64))
        m = int(rng.integers(0, 2))
        for k in range(1, 52):
            if (m * m + m + d) >> k & 1:
                m += 1 << k
        m |= 1 << 52
        N = m * m + m + d
        if N & ((1 << 52) - 1) == 0 and N >> 52 < 1 << 53:
            out.append(float(N >> 52) * 2.0 ** 2)  # sqrt's exponent parity is that of 2^52 (even)
        if len(out) >= n:
            break
    return np.array(out)


@pytest.mark.parametrize("fn", ["sqrt", "quotient", "by_cosine"])
def test_reciprocal_sequences_match_ieee(tracker, fn):
    """sqrt with its reciprocal, quotients by it, and quotients by a cosine
    on the narrow band: correctly rounded on 2^21 operands, the hard cases of
    the square root among them"""
    rng = np.random.default_rng(31)
    n = 1 << 21
    a = rng.uniform(1, 2, n) * np.exp2(rng.integers(-600, 600, n)) * rng.choice([-1.0, 1.0], n)
    a[::5] = 0.0
    if fn == "by_cosine":
        b = rng.uniform(-1, 1, n) * np.exp2(-5.0 - 8 * rng.random(n))
        c = O.math_eval(1, b, b, mode="emath")
        gpu = tracker.math_probe(13, a, b)
        cpu = a / c
    else:
        b = rng.uniform(1, 2, n) * np.exp2(rng.integers(-128, 128, n))
        b[: n // 4] = 1 + rng.random(n // 4) * 2.0 ** -rng.integers(1, 60, n // 4)
        hard = near_midpoint_squares(2000, rng)
        b[: hard.size] = hard
        root = np.sqrt(b)
        q = n // 2
        mid = root[q:] * rng.uniform(1, 2, n - q)
        a[q:] = mid  # quotients that come near representable values
        gpu = tracker.math_probe(11 if fn == "sqrt" else 12, a, b)
        cpu = root if fn == "sqrt" else a / root
    assert (gpu == cpu).all(), (fn, int((gpu != cpu).sum()))


# substep angles just below and above 2^-6 (both squares watched from there
# on) and 2^-5 (the general code from there on); 0.6756 of a slice is the
# fourth-order integrator's longest substep, 0.5 the second-order one's
@pytest.mark.parametrize("angle,order", [(0.3699, 4), (0.3701, 4), (0.7399, 4), (0.7402, 4), (0.01, 2), (0.9, 2),
                                         (0.05, 6), (0.4, 6)])
def test_csbend_substep_angles(tracker, angle, order):
    b = E.CSBEND(L=1.0, ANGLE=angle, N_KICKS=16, INTEGRATION_ORDER=order).p.csbend
    ap = A.EH_MAXAMP(0.05, 0.04, 0, 2, 2, 0)
    r = csbend_edge_rows(1500, 41)
    r[700::3, 3] = 0.0
    r[701::3, 3] = -0.0
    r[702::3, 5] = 0.0
    r[1100::2, 1] *= 60.0  # slopes up to the band's edge on both sides
    g, c = r.copy(), r.copy()
    ng = tracker.track_through_csbend(g, b, PO, 3.0, ap)
    ptr, keep = rows_ptr(c)
    nc = O.lib("emath").or_track_through_csbend(ptr, c.shape[0], C.byref(b), PO, 3.0, C.byref(ap))
    assert_same_survivors(r, g, ng, c, nc)
    assert_rows_bitwise(g[:, :7], c[:, :7], "csbend angle %g order %d" % (angle, order))


# strong kicks that carry slopes past the bound of the common path (2) and
# past the end of the slope range, kicks so weak that momenta go below its
# smallest dividend, thin elements, several orders at once, each integrator
@pytest.mark.parametrize("make", [
    lambda: E.KQUAD(L=0.5, K1=400.0, N_KICKS=4), lambda: E.KQUAD(L=0.5, K1=1e-300, N_KICKS=16),
    lambda: E.KSEXT(L=0.2, K2=4e5, N_KICKS=4), lambda: E.KSEXT(L=0.3, K2=-30.0, K1=0.4, J1=0.1, N_KICKS=8),
    lambda: E.KQUAD(L=0.4, K1=1.8, N_KICKS=5, INTEGRATION_ORDER=2, HKICK=1e-3, VKICK=-2e-3),
    lambda: E.KOCT(L=0.1, K3=4e4, N_KICKS=12, INTEGRATION_ORDER=6, DX=1e-4, DY=-2e-4, DZ=1e-3, TILT=0.2),
    lambda: E.KQUAD(L=0.0, K1=3.0, N_KICKS=4), lambda: E.KQUAD(L=0.4, K1=0.0, N_KICKS=4),
])
def test_multipole_common_path_bounds(tracker, make):
    e = make()
    # within the entry limits: a row beyond them is lost with the path length
    # that the row before it reached, as the reference leaves that variable
    r = beam(1500, 43, halo=0.0)
    r[600:700, 1] = np.linspace(-1.0, 1.0, 100)
    r[700:800, 3] = np.linspace(-1.0, 1.0, 100)
    r[800:900, 0] = np.linspace(-0.05, 0.05, 100)
    r[900:920, 5] = np.linspace(-0.9999, -0.98, 20)
    r[920:940, 5] = 10.0 ** np.arange(20)
    r[940:990, 0] = 10.0 ** -np.linspace(250, 320, 50)
    r[990:1000, 1] = 10.0 ** -np.linspace(170, 190, 10)
    r[1000:1010, :4] = 0.0
    r[1010:1020, :4] = -0.0
    for ap in (A.EH_MAXAMP(0.05, 0.04, 0, 2, 2, 0), None):
        g, c = r.copy(), r.copy()
        ng = tracker.multipole_tracking2(g, e, PO, 12.5, ap)
        ptr, keep = rows_ptr(c)
        nc = O.lib("emath").or_multipole_tracking2(ptr, c.shape[0], C.byref(e), PO, 12.5,
                                                    C.byref(ap) if ap is not None else None)
        assert ng == nc
        assert_rows_bitwise(g[:, :7], c[:, :7], "multipole bounds")


@pytest.mark.parametrize("make", [lambda: E.KQUAD(L=0.3, K1=1.1, N_KICKS=4), lambda: E.KSEXT(L=0.2, K2=40.0),
                                  lambda: E.KOCT(L=0.1, K3=200.0)])
def test_slopes_of_a_few_ulps(tracker, make):
    """1 + x'^2 + y'^2 of one or a few ulps above 1, where the root lies within
    2^-55 of a midpoint between doubles: the path length decides its rounding"""
    e = make()
    rng = np.random.default_rng(47)
    r = beam(60000, 47, halo=0.0)
    r[:, 1] = rng.choice([-1.0, 1.0], 60000) * 10.0 ** rng.uniform(-8.5, -6.5, 60000)
    r[:, 3] = rng.choice([-1.0, 1.0, 0.0], 60000) * 10.0 ** rng.uniform(-8.5, -6.5, 60000)
    r[:, [0, 2]] *= 1e-6
    r[::3, 5] = 0.0
    g, c = r.copy(), r.copy()
    ng = tracker.multipole_tracking2(g, e, PO, 12.5)
    ptr, keep = rows_ptr(c)
    assert ng == O.lib("emath").or_multipole_tracking2(ptr, c.shape[0], C.byref(e), PO, 12.5, None)
    assert_rows_bitwise(g[:, :7], c[:, :7], "small slopes")


# edges, fringe angles (a tangent per particle), kick limits, error tilt,
# misalignment with DZ, a bore along the aperture's edge
@pytest.mark.parametrize("kw", [
    dict(E1=0.03, E2=-0.02), dict(E1=0.02, E2=0.03, HGAP=0.02), dict(E1=0.02, E2=0.03, HGAP=0.02, FINT=0.4, FSE=2e-3),
    dict(E1=0.05, E2=0.05, EDGE1_KICK_LIMIT=1e-5, EDGE2_KICK_LIMIT=2e-5), dict(EDGE1_EFFECTS=0, EDGE2_EFFECTS=0),
    dict(E1=0.01, ETILT=1e-3, TILT=0.3, DX=1e-4, DY=-2e-4, DZ=3e-4), dict(TILT=1.5707963267948966),
])
def test_csbend_whole_element_common_path(tracker, kw):
    b = E.CSBEND(L=1.0, ANGLE=0.08, N_KICKS=16, **kw).p.csbend
    r = csbend_edge_rows(1500, 45)
    r[800:850, 0] = np.linspace(-0.0062, 0.0062, 50)
    r[850:900, 4] = 10.0 ** -np.linspace(100, 300, 50)
    r[900:950, 5] = np.linspace(-1.0, 1.0, 50)
    for ap in (A.EH_MAXAMP(0.006, 0.004, 0, 2, 2, 0), A.EH_MAXAMP(0.006, 0.004, 1, 2, 4, 0),
               A.EH_MAXAMP(0.006, 0.004, 0, 2, 2, A.EH_OPEN_PLUS_X)):
        g, c = r.copy(), r.copy()
        ng = tracker.track_through_csbend(g, b, PO, 3.0, ap)
        ptr, keep = rows_ptr(c)
        nc = O.lib("emath").or_track_through_csbend(ptr, c.shape[0], C.byref(b), PO, 3.0, C.byref(ap))
        assert_same_survivors(r, g, ng, c, nc)
        assert_rows_bitwise(g[:, :7], c[:, :7], "csbend whole element")


def test_quotients_of_powers_of_two(tracker):
    """divisors 1 - k 2^-53 (all mantissa bits set for k = 1) under powers of
    two and their neighbours: the reciprocal that ends on a rounding tie"""
    k = np.arange(1, 8193)
    g = (1 - k * 2.0 ** -53)[None, :] * 2.0 ** np.array([-60, -1, 0, 1, 60])[:, None]
    for a in (1.0, -(2.0 ** -26), 2.0 ** 500, 1 + 2.0 ** -52, 1.5, 2 - 2.0 ** -52):
        b = np.concatenate([(g * g).ravel(), (2.0 ** np.array([-120, 0, 2, 120])[:, None] *
                                              (1 - k * 2.0 ** -53)[None, :]).ravel()])
        aa = np.full(b.size, a)
        assert (tracker.math_probe(12, aa, b) == aa / np.sqrt(b)).all(), a


@pytest.mark.parametrize("make", [
    lambda: E.KQUAD(L=0.3, K1=1.1, N_KICKS=4), lambda: E.KOCT(L=0.1, K3=10.0, N_KICKS=4),
    lambda: E.CSBEND(L=1.0, ANGLE=0.08, N_KICKS=16), lambda: E.CSBEND(L=0.3, ANGLE=4e-7, N_KICKS=4),
    lambda: E.CSBEND(L=1.0, ANGLE=0.08, K1=0.3, NONLINEAR=0, N_KICKS=16)])
def test_slopes_near_sqrt_epsilon(tracker, make):
    """slopes of 2^-26 and around it on the reference energy, where momenta
    are powers of two and roots 1 - 2^-53, and a scan that crosses such slopes
    at a bend's exit"""
    el = make()
    h = 2.0 ** -26
    r = np.zeros((6001, 8))
    r[:, 6] = np.arange(1, 6002)
    r[:, 1] = np.linspace(-1.5e-7, 1.5e-7, 6001)
    edge = [(a, b) for a in (0, h, -h, h / 2, 2 * h, h * (1 + 2.0 ** -52)) for b in (0, h, -h, h / 2)]
    for i, (a, b) in enumerate(edge):
        r[10 * i:10 * i + 5, 1] = a
        r[10 * i:10 * i + 5, 3] = b
        r[10 * i + 1, 5] = 1.0
        r[10 * i + 2, 5] = -0.5
        r[10 * i + 3, 0] = 1e-3
        r[10 * i + 4, 2] = 1e-9
    g, c = r.copy(), r.copy()
    ptr, keep = rows_ptr(c)
    if el.type == A.EH_T_CSBEND:
        ng = tracker.track_through_csbend(g, el.p.csbend, PO, 3.0)
        nc = O.lib("emath").or_track_through_csbend(ptr, c.shape[0], C.byref(el.p.csbend), PO, 3.0, None)
    else:
        ng = tracker.multipole_tracking2(g, el, PO, 3.0)
        nc = O.lib("emath").or_multipole_tracking2(ptr, c.shape[0], C.byref(el), PO, 3.0, None)
    assert ng == nc == r.shape[0]
    assert_rows_bitwise(g[:, :7], c[:, :7], "slopes near 2^-26")


# expansion order 4 with the 4th-order integrator (the common path), and next
# to it what stays with the general code: orders 5 and 6, another integrator;
# kicks so strong that slopes leave the bands, so weak that kicks fall below
# the smallest dividend; wide substep angles; XKICK alone
@pytest.mark.parametrize("kw", [
    dict(K1=-0.4, K2=2.0), dict(K1=0.6, E1=0.02, E2=0.03, HGAP=0.02), dict(K2=200.0, ANGLE=-0.08), dict(XKICK=1e-4),
    dict(K1=0.3, NONLINEAR=0), dict(K1=400.0), dict(K1=1e-250), dict(K1=-0.4, ANGLE=0.5), dict(K1=-0.4, FSE=1e-3,
    ETILT=1e-3, DX=1e-4, DZ=2e-4), dict(K1=0.2, K3=30.0), dict(K4=900.0), dict(K1=-0.4, INTEGRATION_ORDER=2),
    dict(K1=-0.4, INTEGRATION_ORDER=6)])
def test_combined_function_bend(tracker, kw):
    b = E.CSBEND(L=1.0, N_KICKS=16, **{"ANGLE": 0.08, **kw}).p.csbend
    r = csbend_edge_rows(1500, 47)
    r[700::3, 3] = 0.0
    r[701::3, 3] = -0.0
    r[800:850, 0] = np.linspace(-0.0062, 0.0062, 50)
    r[850:900, 2] = 10.0 ** -np.linspace(100, 320, 50)
    r[900:950, 5] = np.linspace(-1.0, 1.0, 50)
    r[1100::2, 1] *= 60.0
    for ap in (A.EH_MAXAMP(0.05, 0.04, 0, 2, 2, 0), A.EH_MAXAMP(0.006, 0.004, 1, 2, 4, 0)):
        g, c = r.copy(), r.copy()
        ng = tracker.track_through_csbend(g, b, PO, 3.0, ap)
        ptr, keep = rows_ptr(c)
        nc = O.lib("emath").or_track_through_csbend(ptr, c.shape[0], C.byref(b), PO, 3.0, C.byref(ap))
        assert_same_survivors(r, g, ng, c, nc)
        assert_rows_bitwise(g[:, :7], c[:, :7], "combined-function bend")


# substep angles around 2^-20, where the instance for small bends begins
# (0.1756 of a slice is the fourth-order integrator's shortest substep, 0.5
# the second-order one's), and down to the largest radius
@pytest.mark.parametrize("L,angle,kw", [
    (0.2, 2.17e-5, {}), (0.2, 2.18e-5, {}), (0.2, 2.1e-7, {}), (0.001, 1.1e-9, {}), (0.1, 7.6e-6, dict(INTEGRATION_ORDER=2)),
    (0.1, 7.7e-6, dict(INTEGRATION_ORDER=2)), (0.3, 1e-6, dict(INTEGRATION_ORDER=6)), (0.3, -1e-5, dict(TILT=1.5)),
    (0.2, 1e-6, dict(E1=0.03, E2=-0.02, HGAP=0.02, FSE=0.5, DX=1e-4, DZ=3e-4, ETILT=1e-3)),
    (0.2, 1e-6, dict(E1=0.2, E2=0.2, EDGE1_KICK_LIMIT=1e-9)), (0.2, 1e-6, dict(K1=0.3)), (0.2, 2.0 ** -22, {}),
])
def test_csbend_small_angles(tracker, L, angle, kw):
    b = E.CSBEND(L=L, ANGLE=angle, N_KICKS=4, **kw).p.csbend
    r = csbend_edge_rows(3000, 51)
    h = 2.0 ** -26
    rng = np.random.default_rng(51)
    r[600:1200, 1] = rng.choice([-1.0, 1.0], 600) * 10.0 ** rng.uniform(-9.5, -5.5, 600)  # cosines 1 - n 2^-53
    r[600:1200, [3, 5]] = 0.0
    r[600:1200:2, 3] = rng.choice([-1.0, 1.0], 300) * 10.0 ** rng.uniform(-9.5, -6.0, 300)
    r[1200:1300, 1] = rng.choice([0.0, -0.0, h, -h, h / 2, 2 * h, h * (1 + 2.0 ** -52)], 100)
    r[1200:1300, 3] = rng.choice([0.0, -0.0, h, -h, h / 2], 100)
    r[1200:1300, 5] = rng.choice([0.0, 1.0, -0.5], 100)
    r[1200:1300:3, 0] = 0.0
    r[1300:1350, 1] = -angle * np.linspace(0.0, 1.2, 50)  # c + phi through zero
    r[1350:1400, 1] = 10.0 ** -np.linspace(150, 320, 50)
    r[1400:1450, 0] = 10.0 ** -np.linspace(150, 320, 50)
    r[1450:1500, 5] = np.linspace(-1.0, 1.0, 50)
    r[1500:1550, 5] = 10.0 ** np.linspace(0, 30, 50)
    r[1550:1600, 1] = np.linspace(-0.04, 0.04, 50)  # the band's edge
    r[1600:1650, 0] = np.linspace(-0.0062, 0.0062, 50)
    for ap in (A.EH_MAXAMP(0.006, 0.004, 0, 2, 2, 0), A.EH_MAXAMP(0.006, 0.004, 1, 2, 4, 0)):
        g, c = r.copy(), r.copy()
        ng = tracker.track_through_csbend(g, b, PO, 3.0, ap)
        ptr, keep = rows_ptr(c)
        nc = O.lib("emath").or_track_through_csbend(ptr, c.shape[0], C.byref(b), PO, 3.0, C.byref(ap))
        assert_same_survivors(r, g, ng, c, nc)
        assert_rows_bitwise(g[:, :7], c[:, :7], "csbend angle %g" % angle)


def test_small_bends_take_a_common_path(tracker):
    """a ring of correctors modelled as bends of 1e-6 rad against one of 1e-3
    (1.2 times the kernel's time; the general code takes 2.9), tracked alone
    and in a batch with the same result"""
    r = np.ascontiguousarray(beam(20000, 53, halo=0.0)[:, :8])
    r[:, [0, 2]] *= 0.05
    r[:, [1, 3]] *= 0.05
    ms, rows = {}, {}
    for angle in (1e-6, 1e-3):
        els = [E.MAXAMP(X_MAX=0.02, Y_MAX=0.02)]
        for i in range(20):
            els += [E.DRIF(L=0.5), E.CSBEND(L=0.2, ANGLE=angle, N_KICKS=4)]
        bl = E.Beamline(els)
        tracker.load(bl, PO)
        times = []
        for k in range(5):
            tracker.upload(r)
            times.append(tracker.track(0, 20).track_ms)
        ms[angle], rows[angle] = min(times), tracker.download()[0]
    assert ms[1e-6] < 2.0 * ms[1e-3], ms
    els = [E.MAXAMP(X_MAX=0.02, Y_MAX=0.02)]
    for i in range(20):
        els += [E.DRIF(L=0.5), E.CSBEND(L=0.2, ANGLE=1e-6, N_KICKS=4)]
    bl = E.Beamline(els)
    from elegant_amd import native
    for ppl in (1, 2):
        b = native.Batch(tracker)
        b.add_variant(bl, PO, r)
        b.set_tuning(ppl, 64, 8)
        b.track(0, 20)
        got, _ = b.download(0)
        b.close()
        assert_rows_bitwise(got, rows[1e-6], "batch, %d per lane" % ppl)


# lanes beyond the box of 0.7 of an ellipse's half-axes: inside its circle,
# between the circle and a higher power's curve, on the curve and outside
@pytest.mark.parametrize("ap", [
    A.EH_MAXAMP(0.006, 0.004, 1, 2, 0, 0), A.EH_MAXAMP(0.006, 0.004, 1, 2, 4, 0), A.EH_MAXAMP(0.004, 0.006, 1, 8, 2, 0),
    A.EH_MAXAMP(0.006, 0.004, 1, 2, 0, A.EH_OPEN_PLUS_X), A.EH_MAXAMP(0.006, 1e32, 1, 2, 0, 0),
    A.EH_MAXAMP(1e-40, 0.006, 1, 2, 0, 0), A.EH_MAXAMP(0.006, 0.004, 1, 2, 0, A.EH_OPEN_MINUS_Y)])
@pytest.mark.parametrize("make", [
    lambda: E.KQUAD(L=0.3, K1=0.4, N_KICKS=16), lambda: E.KSEXT(L=0.2, K2=3.0, TILT=0.3, DX=1e-4, DY=-2e-4),
    lambda: E.KQUAD(L=0.2, K1=0.1, N_KICKS=4, HKICK=1e-5, INTEGRATION_ORDER=2), lambda: E.KOCT(L=0.1, K3=10.0),
    lambda: E.CSBEND(L=0.2, ANGLE=1e-3, N_KICKS=4), lambda: E.CSBEND(L=0.2, ANGLE=1e-6, N_KICKS=4, TILT=0.2),
    lambda: E.CSBEND(L=0.2, ANGLE=0.05, N_KICKS=1, INTEGRATION_ORDER=2), lambda: E.CSBEND(L=0.2, ANGLE=0.01, K1=0.2)])
def test_lanes_beyond_an_ellipses_box(tracker, ap, make):
    e = make()
    n = 4000
    rng = np.random.default_rng(57)
    r = beam(n, 57, halo=0.0)
    a, b = min(ap.x_max, 0.006), min(ap.y_max, 0.006)
    t, f = rng.uniform(0, 2 * np.pi, n), rng.choice([0.5, 0.72, 0.9, 0.99, 1.0, 1 - 1e-14, 1 + 1e-14, 1.001, 1.1], n)
    r[:, 0], r[:, 2] = a * f * np.cos(t), b * f * np.sin(t)
    r[:200, 2] = 0.0
    r[100:300, 0] = 0.0
    r[:, [1, 3]] *= rng.choice([0.0, 1e-3, 1.0], (n, 1))
    if e.type == A.EH_T_CSBEND:
        # (a multipole's entry limits lose such a row with the path length that
        # the row before it reached, as the reference leaves that variable)
        r[3000:3010, 0] = np.nan
        r[3010:3020, 2] = np.inf
    g, c = r.copy(), r.copy()
    ptr, keep = rows_ptr(c)
    if e.type == A.EH_T_CSBEND:
        ng = tracker.track_through_csbend(g, e.p.csbend, PO, 3.0, ap)
        nc = O.lib("emath").or_track_through_csbend(ptr, n, C.byref(e.p.csbend), PO, 3.0, C.byref(ap))
    else:
        ng = tracker.multipole_tracking2(g, e, PO, 3.0, ap)
        nc = O.lib("emath").or_multipole_tracking2(ptr, n, C.byref(e), PO, 3.0, C.byref(ap))
    assert ng == nc and (nc > 0 or ap.x_max < 1e-6)
    assert_rows_bitwise(g[:, :7], c[:, :7], "ellipse")


def test_a_beam_that_fills_an_ellipse(tracker):
    """particles beyond the box take the common path twice at most (2.8 times
    the kernel's time inside it; with the general code 4.8)"""
    els = [E.MAXAMP(X_MAX=0.02, Y_MAX=0.02, ELLIPTICAL=1)]
    for i in range(20):
        els += [E.DRIF(L=0.1), E.KSEXT(L=0.2, K2=1e-6)]
    tracker.load(E.Beamline(els), PO)
    ms = []
    for lo, hi in ((0.1, 0.6), (0.75, 0.95)):
        r = np.zeros((20000, 8))
        r[:, 0] = 0.02 * np.random.default_rng(3).uniform(lo, hi, 20000)
        r[:, 6] = np.arange(1, 20001)
        times = []
        for k in range(5):
            tracker.upload(r)
            st = tracker.track(0, 20)
            times.append(st.track_ms)
        assert st.n_left == 20000
        ms.append(min(times))
    assert ms[1] < 3.7 * ms[0], ms
