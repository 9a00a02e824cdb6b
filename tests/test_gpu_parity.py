"""Bit-for-bit parity of the HIP path against the oracle (run on the GPU).

Every comparison here is exact (integer or float64 bit patterns): the plain
FP64 path follows the reference's operation order, so any difference is a
defect."""
import numpy as np
import pytest

from tests.helpers import bits_equal, oracle_state

pytestmark = pytest.mark.gpu

NGS = [32, 64]


@pytest.fixture(scope="module")
def hyd_cache():
    from hydra_amd import Hydra
    cache = {}

    def get(ng):
        if ng not in cache:
            cache[ng] = Hydra(ng)
        return cache[ng]
    return get


@pytest.mark.parametrize("ng", NGS)
def test_tables_match_oracle(ng, hyd_cache):
    from oracle.hyo import Oracle
    o = Oracle(ng)
    h = hyd_cache(ng)
    for name, n in [("green", None), ("flo", None), ("fhi", None), ("qdiss", None),
                    ("hrkx", ng), ("hrky", ng), ("rkx", ng), ("xtrig", 2 * ng)]:
        a = h.table(name)
        b = o.d(name, n).ravel() if n else o.d(name).ravel()
        assert bits_equal(a, b), name


@pytest.mark.parametrize("ng", NGS + [256])
def test_fft_bitwise(ng, hyd_cache):
    from oracle.hyo import Oracle
    o = Oracle(ng)
    h = hyd_cache(ng)
    rng = np.random.default_rng(ng)
    f = rng.standard_normal((ng, ng))
    assert bits_equal(h.ptospc(f), o.ptospc(f))
    s = rng.standard_normal((ng, ng))
    assert bits_equal(h.spctop(s), o.spctop(s))


@pytest.mark.parametrize("ng", NGS)
def test_invert_and_gradient_bitwise(ng, hyd_cache):
    from oracle.hyo import Oracle
    o = Oracle(ng)
    h = hyd_cache(ng)
    rng = np.random.default_rng(7 + ng)
    s = rng.standard_normal((ng, ng))
    for a, b in zip(h.main_invert(s), o.main_invert(s)):
        assert bits_equal(a, b)
    for a, b in zip(h.gradient(s), o.gradient(s)):
        assert bits_equal(a, b)


@pytest.mark.parametrize("ng", NGS)
def test_velint_bitwise(ng, hyd_cache):
    o, qq, c = oracle_state(ng)
    h = hyd_cache(ng)
    rng = np.random.default_rng(3)
    uu, vv = rng.standard_normal((2, ng, ng))
    a = h.velint(uu, vv, c["x"], c["y"])
    b = o.velint(uu, vv)
    assert bits_equal(a[0], b[0]) and bits_equal(a[1], b[1])


@pytest.mark.parametrize("ng", NGS)
def test_con2grid_bitwise(ng, hyd_cache):
    o, qq, c = oracle_state(ng)
    h = hyd_cache(ng)
    qc_h, cnt_h = h.con2grid(c["x"], c["y"], c["nextq"], c["qjump"], with_counts=True)
    qc_o, cnt_o = o.con2grid(with_counts=True)
    assert np.array_equal(cnt_h.ravel(), cnt_o.ravel())
    assert bits_equal(qc_h, qc_o)


def test_sum_sequential_bitwise(hyd_cache):
    h = hyd_cache(64)
    rng = np.random.default_rng(11)
    cases = [rng.standard_normal(4096 * 4) * 10 + 3, rng.standard_normal(4096 * 4),
             np.round(rng.standard_normal(12345) * 64) / 64 + 2.0 ** -30,
             rng.integers(-5, 6, 9999) * 0.1, rng.standard_normal(777) ** 2,
             np.full(5000, 0.1), np.array([1.0, 1e-16, 1e-16, 1e-16, -1.0]),
             rng.standard_normal(5000) * 1e-300,
             np.array([1e16 if i % 2 == 0 else -1e16 + 1.5 for i in range(3001)]),
             np.r_[rng.standard_normal(8000) * 1e8, -rng.standard_normal(8000) * 1e8],
             np.r_[[2.0 ** 40], np.tile([0.5 ** 12 * 3, -0.5 ** 12], 6000)],
             np.r_[[-0.0, 0.0, -0.0], rng.standard_normal(600)], np.array([-0.0]),
             np.array([0.0, -0.0, -0.0]), np.zeros(0)]
    for a in cases:
        ref = 0.0
        for x in a:
            ref = ref + float(x)
        got = h.sum_sequential(a)
        assert np.float64(got).view(np.int64) == np.float64(ref).view(np.int64), (len(a), got, ref)


def test_sum_sequential_long_bitwise():
    """Long sums (up to the 4 ng^2 work space at ng=256) of zero-mean,
    tie-rich data shaped like the con2grid field: many binade changes,
    exact ties, chunk counts that are not multiples of 64."""
    from hydra_amd import Hydra
    h = Hydra(256)
    rng = np.random.default_rng(5)
    ng = 256
    x = np.linspace(-np.pi, np.pi, ng, endpoint=False)
    f = np.add.outer(np.sin(3 * x), np.cos(2 * x)) * 5 + rng.standard_normal((ng, ng)) * 0.1
    qj = 0.37
    lev = np.round(f / qj) * qj  # level steps: many exact ties
    cases = [lev.ravel(), (lev - lev.mean()).ravel(), f.ravel(),
             np.tile(lev.ravel(), 4)[: 4 * ng * ng - 77], rng.standard_normal(4 * ng * ng)]
    for a in cases:
        ref = 0.0
        for v in a.tolist():
            ref = ref + v
        got = h.sum_sequential(a)
        assert np.float64(got).view(np.int64) == np.float64(ref).view(np.int64), (len(a), got, ref)
    h.close()


def test_sum_sequential_binade_walks_bitwise():
    """Running sums that wander across powers of two inside the windows of
    1024 values (crossings up and down, several binades, sign changes, exact
    ties), the case the per-window class tables resolve; bit for bit."""
    from hydra_amd import Hydra
    h = Hydra(256)
    rng = np.random.default_rng(21)
    n = 4 * 256 * 256
    steps = rng.standard_normal(n)
    cases = []
    for level in (1024.0, 1.0, 2.0 ** -20, 3.0e5):
        a = steps * level * 0.02
        a[0] = level * 0.99  # start just below the power of two
        cases.append(a)
    walk = np.cumsum(rng.standard_normal(n) * 0.5)
    cases.append(np.diff(np.r_[0.0, np.sin(walk) * 700.0 + 1024.0 * np.cos(walk / 50.0)]))
    ties = np.round(rng.standard_normal(n) * 8.0) * 0.25
    ties[0] = 511.875
    cases.append(ties)
    sign = rng.standard_normal(n) * 3.0
    sign[::4096] += np.where(np.arange(len(sign[::4096])) % 2 == 0, 5e4, -5e4)
    cases.append(sign)
    for a in cases:
        ref = 0.0
        for v in a.tolist():
            ref = ref + v
        got = h.sum_sequential(a)
        assert np.float64(got).view(np.int64) == np.float64(ref).view(np.int64), (got, ref)
    h.close()


@pytest.fixture(scope="module")
def hyd_2048():
    from hydra_amd import Hydra
    h = Hydra(2048)
    yield h
    h.close()


# one launch up to 4096 values, one chained level up to 64 segments of 4096,
# then one and two folded levels; beyond 512 segments prefixed totals
@pytest.mark.parametrize("n", [1, 64, 4095, 4096, 4097, 64 * 4096, 64 * 4096 + 1, 512 * 4096 + 1,
                               1024 * 4096, 1024 * 4096 + 1, 4 * 2048 * 2048])
def test_sum_sequential_level_edges_bitwise(n, hyd_2048):
    import ctypes as C
    from oracle.hyo import lib
    ol = lib()
    ol.hyo_sum_seq.restype = C.c_double
    ol.hyo_sum_seq.argtypes = [np.ctypeslib.ndpointer(dtype=np.float64), C.c_int64]
    rng = np.random.default_rng(n)
    walk = rng.standard_normal(n) * 10.0 ** rng.integers(-3, 3, n)
    level = np.full(n, 0.1)                       # no crossing for long
    jumps = rng.standard_normal(n)
    jumps[::1021] *= 1e12                         # starts far from any guess
    for a in (walk, level, jumps):
        want = np.float64(ol.hyo_sum_seq(a, n))
        got = np.float64(hyd_2048.sum_sequential(a))
        assert got.view(np.int64) == want.view(np.int64), (got, want)
    for bad in (np.inf, -np.inf, np.nan):
        a = walk.copy()
        a[n // 2] = bad
        want, got = ol.hyo_sum_seq(a, n), hyd_2048.sum_sequential(a)
        assert (np.isnan(got) and np.isnan(want)) or got == want


def test_sum_sequential_unfolded_start_after_another_sum(hyd_2048):
    """A first group of segments that does not fold (a run up to 1e300 and
    back in its second segment) under two folded levels, in a work area that
    another sum of the same length, alike from the third segment on, has
    filled: nothing of that sum may be taken for this one's start."""
    import ctypes as C
    from oracle.hyo import lib
    ol = lib()
    ol.hyo_sum_seq.restype = C.c_double
    ol.hyo_sum_seq.argtypes = [np.ctypeslib.ndpointer(dtype=np.float64), C.c_int64]
    n = (1 << 22) + 8 * 4096
    a = np.full(n, 0.75)
    b = a.copy()
    b[5000:5003] = [1e300, -1e300, 2.25]
    for x in (a, b, a):
        assert hyd_2048.sum_sequential(x) == ol.hyo_sum_seq(x, n)


@pytest.mark.parametrize("ng", [32, 64])
def test_advance_bitwise(ng):
    """Several RK4 steps of the device-resident state, every field and node
    position bit for bit."""
    from hydra_amd import Hydra
    from oracle.hyo import Oracle
    from hydra_amd.ic import random_pv
    qq = random_pv(ng, seed=12345)
    o = Oracle(ng)
    o.init_from_field(qq)
    o.recontour(o.d("qr").copy())
    c = o.contours()
    o.evolution_init()
    h = Hydra(ng)
    h.set_field(qq)
    assert h.scalar("qjump") == o.getd("qjump")
    h.set_contours(c)
    h.evolution_init()
    for name in ("qc", "qd", "qs"):
        assert bits_equal(h.field(name), o.d(name)), name
    for step in range(4):
        o.advance()
        h.advance()
        for name in ("qs", "qd", "qq", "uu", "vv", "pp"):
            assert bits_equal(h.field(name), o.d(name)), (step, name)
        cg = h.contours()
        n = o.get("nptq")
        assert bits_equal(cg["x"], o.d("xq", n)) and bits_equal(cg["y"], o.d("yq", n)), step
        assert h.scalar("t") == o.getd("t") and h.scalar("twist") == o.getd("twist")
    h.close()


@pytest.mark.parametrize("ng", NGS)
def test_renode_bitwise(ng, hyd_cache):
    o, qq, c = oracle_state(ng)
    h = hyd_cache(ng)
    rng = np.random.default_rng(ng)
    for j in list(range(4)) + list(rng.integers(0, len(c["i1q"]), 6)):
        i1, i2 = c["i1q"][j], c["i2q"][j]
        # perturb so that the contour is not already renoded
        xd = c["x"][i1 - 1:i2] + 1e-3 * np.sin(7 * c["y"][i1 - 1:i2])
        yd = c["y"][i1 - 1:i2]
        a = h.renode(xd, yd)
        b = o.renode(xd, yd)
        assert bits_equal(a[0], b[0]) and bits_equal(a[1], b[1]), j
    # a triangle: several corners
    verts = np.array([[-0.6, -0.4], [0.7, -0.3], [0.0, 0.6]])
    pts = np.concatenate([verts[a] + np.arange(40)[:, None] / 40.0 * (verts[(a + 1) % 3] - verts[a])
                          for a in range(3)])
    a = h.renode(pts[:, 0], pts[:, 1])
    b = o.renode(pts[:, 0], pts[:, 1])
    assert bits_equal(a[0], b[0]) and bits_equal(a[1], b[1])


# stretches between corners at the edges of what a lane and a wavefront take
# (64 nodes) and of a block of the chain (256), corners beyond one pass of
# their list (2048), no corner and one corner
@pytest.mark.parametrize("stretches", [[64, 65], [1, 2, 3, 63, 64, 65, 128, 255, 256, 257, 511, 513],
                                       [1] * 5000, [2, 70] * 30, [3000, 1], [700], []])
def test_renode_stretches_bitwise(stretches, hyd_cache):
    from oracle.hyo import Oracle
    h, o = hyd_cache(64), Oracle(64)
    nc = len(stretches)
    if nc > 1:   # a star with alternating radii: every vertex is a corner
        if nc % 2:
            stretches, nc = stretches + [5], nc + 1
        th = 2 * np.pi * np.arange(nc) / nc
        r = np.where(np.arange(nc) % 2 == 0, 2.5, 0.5)
        vx, vy = r * np.cos(th), r * np.sin(th)
        if nc == 2:
            vy = vy + [0.0, 0.3]
        x, y = [], []
        for k, m in enumerate(stretches):
            f = np.arange(m) / m
            k1 = (k + 1) % nc
            bow = 0.02 * np.sin(np.pi * f) * (1 if m > 8 else 0)
            x.append(vx[k] + f * (vx[k1] - vx[k]) - bow * (vy[k1] - vy[k]))
            y.append(vy[k] + f * (vy[k1] - vy[k]) + bow * (vx[k1] - vx[k]))
        x, y = np.concatenate(x), np.concatenate(y)
    else:        # a circle, or a drop with its tip at the first node
        n = stretches[0] if nc else 4099
        th = 2 * np.pi * np.arange(n) / n
        r = 1.0 - (0.8 * np.exp(-th * 3) + 0.8 * np.exp(-(2 * np.pi - th) * 3) if nc else 0.0)
        x, y = r * np.cos(th), r * np.sin(th)
    a, b = h.renode(x, y, cap=1 << 20), o.renode(x, y, cap=1 << 20)
    assert len(a[0]) == len(b[0])
    assert bits_equal(a[0], b[0]) and bits_equal(a[1], b[1])


@pytest.mark.parametrize("ng", NGS)
def test_recontour_from_field_bitwise(ng):
    """congen from the initial field: contour count, node count, topology and
    positions identical to the oracle."""
    from hydra_amd import Hydra
    from hydra_amd.ic import random_pv
    from oracle.hyo import Oracle
    qq = random_pv(ng, seed=12345)
    o = Oracle(ng)
    o.init_from_field(qq)
    o.recontour(o.d("qr").copy())
    c = o.contours()
    h = Hydra(ng)
    h.set_field(qq)
    h.recontour()
    g = h.contours()
    assert len(g["x"]) == len(c["x"]) and len(g["i1q"]) == len(c["i1q"])
    for k in ("nextq", "i1q", "i2q", "npq", "indq"):
        assert np.array_equal(g[k], c[k]), k
    assert bits_equal(g["x"], c["x"]) and bits_equal(g["y"], c["y"])
    h.close()


def test_recontour_cycle_bitwise():
    """prepare + recontour with existing contours (the con2ugrid branch)
    after a few steps, then evolution_init: identical to the oracle."""
    from hydra_amd import Hydra
    from hydra_amd.ic import random_pv
    from oracle.hyo import Oracle
    ng = 32
    qq = random_pv(ng, seed=7)
    o = Oracle(ng)
    o.init_from_field(qq)
    o.recontour(o.d("qr").copy())
    c = o.contours()
    o.evolution_init()
    h = Hydra(ng)
    h.set_field(qq)
    h.set_contours(c)
    h.evolution_init()
    for _ in range(3):
        o.advance()
        h.advance()
    o.L.hyo_prepare(o.m)
    h.prepare()
    assert bits_equal(h.field("qr"), o.d("qr"))
    o.recontour(o.d("qr").copy())
    h.recontour()
    c2, g2 = o.contours(), h.contours()
    for k in ("nextq", "i1q", "i2q", "npq", "indq"):
        assert np.array_equal(g2[k], c2[k]), k
    assert bits_equal(g2["x"], c2["x"]) and bits_equal(g2["y"], c2["y"])
    o.evolution_init()
    h.evolution_init()
    for name in ("qc", "qd", "qs"):
        assert bits_equal(h.field(name), o.d(name)), name
    h.close()


def test_recontour_with_contours_ng256_bitwise():
    """Two recontourings with contours at ng=256, whose ultra-fine mean is a
    sum with two folded levels, in one work area."""
    from hydra_amd import Hydra
    from hydra_amd.ic import random_pv
    from oracle.hyo import Oracle
    ng = 256
    o, h = Oracle(ng, ncontq=15), Hydra(ng, ncontq=15)
    q = random_pv(ng, seed=7)
    o.init_from_field(q)
    h.set_field(q)
    o.recontour(o.d("qr").copy())
    h.recontour()
    for _ in range(2):
        for m in (o, h):
            m.evolution_init()
            m.advance()
            m.prepare()
        o.recontour(o.d("qr").copy())
        h.recontour()
        c, g = o.contours(), h.contours()
        for k in ("nextq", "i1q", "i2q", "npq", "indq"):
            assert np.array_equal(g[k], c[k]), k
        assert bits_equal(g["x"], c["x"]) and bits_equal(g["y"], c["y"])
    h.close()


def _hairpins(ng, nest=4):
    """Closed thin loops whose crossings of one fine x-gridline fall in one
    fine cell with both signs, `nest` of each: order-dependent cells
    (summed in node order from the buckets), inside the grid and on the
    bottom row (loops wrapping the periodic y boundary), plus one large
    circle so that the grid has ordinary cells too."""
    h = 2 * np.pi / (4 * ng)  # fine cell
    xs, ys, npq = [], [], []

    def loop(pts):
        xs.extend(p[0] for p in pts)
        ys.extend(p[1] for p in pts)
        npq.append(len(pts))
    # interior: rectangles across a few gridlines, both long sides in one fine row
    for cx, cy in ((0.3, -1.1), (-2.0, 0.7), (1.7, 2.2)):
        x0 = -np.pi + h * (round((cx + np.pi) / h) + 0.5)
        y0 = -np.pi + h * (round((cy + np.pi) / h) + 0.2)
        for k in range(nest):
            ya, yb = y0 + 0.05 * h * k, y0 + 0.55 * h - 0.05 * h * k
            loop([(x0 - 0.1 * k * h, ya), (x0 + 3 * h + 0.1 * k * h, ya),
                  (x0 + 3 * h + 0.1 * k * h, yb), (x0 - 0.1 * k * h, yb)])
    # bottom row: loops through y = +-pi, both vertical sides in one fine column
    for cx in (-0.9, 2.6):
        x0 = -np.pi + h * (round((cx + np.pi) / h) + 0.2)
        for k in range(nest):
            xa, xb = x0 + 0.05 * h * k, x0 + 0.55 * h - 0.05 * h * k
            d = 3 * h + 0.1 * h * k
            loop([(xa, np.pi - d), (xa, -np.pi + d), (xb, -np.pi + d), (xb, np.pi - d)])
    # one circle
    t = np.linspace(0.0, 2 * np.pi, 400, endpoint=False)
    loop(list(zip(1.3 * np.cos(t) - 0.2, 1.1 * np.sin(t) + 0.1)))
    n = len(xs)
    i1 = np.cumsum([0] + npq[:-1]) + 1
    nxt = np.empty(n, dtype=np.int32)
    for a, m in zip(i1, npq):
        idx = np.arange(a, a + m)
        nxt[idx - 1] = np.roll(idx, -1)
    nq = len(npq)
    return dict(x=np.array(xs), y=np.array(ys), nextq=nxt, i1q=i1.astype(np.int32),
                i2q=(i1 + np.array(npq) - 1).astype(np.int32), npq=np.array(npq, np.int32),
                indq=np.ones(nq, np.int32), qjump=0.1234567891234)


def _order_dependent(c, ng):
    """Fine cells and bottom-row counters with both signs and at least
    three of one (crossings located as contours.f90:206-269 does)."""
    import math
    nxf, ell, hl = 4 * ng, 2 * np.pi, np.pi
    glxfi = nxf / ell
    xg = -hl + (ell / nxf) * np.arange(nxf)
    cells, bottom = {}, {}
    x, y, nx = c["x"], c["y"], c["nextq"]
    for i in range(len(x)):
        xi, yi = x[i], y[i]
        xa, ya = x[nx[i] - 1], y[nx[i] - 1]
        ixci, ixca = 1 + int(glxfi * (xi + hl)), 1 + int(glxfi * (xa + hl))
        dx = (xa - xi) - ell * int((xa - xi) / hl)
        yy = ya - yi
        dy = yy - ell * int(yy / hl)
        if abs(yy) > hl:
            cc = math.copysign(1.0, dy)
            p = -(yi - hl * cc) / (dy + 1e-12)
            ix = 1 + int(glxfi * math.fmod(ell + hl + xi + p * dx, ell))
            bottom.setdefault(ix, []).append(-1 if cc > 0 else 1)
        ixdif = ixca - ixci
        nxc = ixdif - nxf * int(2 * ixdif / nxf)
        jump = 1 if nxc > 0 else -1
        for ncr in range(0, nxc, jump):
            ix = 1 + (ixci + (0 if jump == 1 else -1) + nxf + ncr) % nxf
            x2 = xg[ix - 1] - xi
            y2 = yi + (x2 - ell * int(x2 / hl)) / dx * dy
            iy = 2 + int(glxfi * (y2 - ell * int(y2 / hl) + hl))
            cells.setdefault((ix, iy), []).append(1 if dx > 0 else -1)

    def flagged(d):
        return sum(1 for v in d.values() if v.count(1) and v.count(-1)
                   and max(v.count(1), v.count(-1)) >= 3)
    return flagged(cells), flagged(bottom)


@pytest.mark.parametrize("ng", NGS)
def test_con2grid_order_dependent_cells_bitwise(ng, hyd_cache):
    """Fine cells and bottom-row counters holding both signs with several of
    each (summed in node order) give the oracle's grid, through the
    diagnostic sweep (with counts) and through the step's fused sweep."""
    from oracle.hyo import Oracle
    c = _hairpins(ng)
    o = Oracle(ng)
    o.set_contours(c)
    qc_o, cnt_o = o.con2grid(with_counts=True)
    cells, bottom = _order_dependent(c, ng)
    assert cells >= 6 and bottom >= 2  # the case is exercised
    h = hyd_cache(ng)
    for rep in range(2):  # the second sweep starts from the counters the first cleared
        qc_h, cnt_h = h.con2grid(c["x"], c["y"], c["nextq"], c["qjump"], with_counts=True)
        assert np.array_equal(cnt_h.ravel(), cnt_o.ravel())
        assert bits_equal(qc_h, qc_o)
        assert bits_equal(h.con2grid(c["x"], c["y"], c["nextq"], c["qjump"]), o.con2grid())


def _crowded(ng, kind):
    """Contours that fill cells' buckets: "chords", long random segments, so
    that most fine cells become order-dependent, more of them per block of
    nodes than its list holds; "ringsN", rings about one fine cell wide
    inside N x N cells, so that buckets hold from a few entries to a thousand."""
    rng = np.random.default_rng(len(kind))
    h = 2 * np.pi / (4 * ng)
    npq, xs, ys = [], [], []
    if kind == "chords":
        npq = [60] * 50
        xs.append(rng.uniform(-np.pi, np.pi, 3000))
        ys.append(rng.uniform(-np.pi, np.pi, 3000))
    else:
        side = int(kind[5:]) * h
        for _ in range(2500 if kind == "rings1" else 400):
            m = int(rng.integers(5, 60))
            t = np.sort(rng.uniform(0, 2 * np.pi, m))[::int(rng.choice([-1, 1]))]
            cx, cy = rng.uniform(0, side, 2) + 0.1
            xs.append(cx + 0.9 * h * np.cos(t))
            ys.append(cy + 0.9 * h * np.sin(t))
            npq.append(m)
    npq = np.array(npq, np.int32)
    i2 = np.cumsum(npq).astype(np.int32)
    nxt = np.arange(2, i2[-1] + 2, dtype=np.int32)
    nxt[i2 - 1] = i2 - npq + 1
    return dict(x=np.concatenate(xs), y=np.concatenate(ys), nextq=nxt, i1q=i2 - npq + 1, i2q=i2,
                npq=npq, indq=np.ones(len(npq), np.int32), qjump=0.1234567891234)


@pytest.mark.parametrize("kind,least", [("chords", 10000), ("rings1", 6), ("rings3", 10),
                                        ("rings10", 60)])
def test_con2grid_crowded_cells_bitwise(kind, least, hyd_cache):
    """Buckets of every size, and more order-dependent cells in a block of
    nodes than its list holds, against the oracle's grid."""
    from oracle.hyo import Oracle
    ng = 32
    c = _crowded(ng, kind)
    o = Oracle(ng)
    o.set_contours(c)
    qc_o, cnt_o = o.con2grid(with_counts=True)
    cells, _ = _order_dependent(c, ng)
    assert cells >= least  # the case is exercised
    h = hyd_cache(ng)
    for rep in range(2):
        qc_h, cnt_h = h.con2grid(c["x"], c["y"], c["nextq"], c["qjump"], with_counts=True)
        assert np.array_equal(cnt_h, cnt_o)
        assert bits_equal(qc_h, qc_o)
        assert bits_equal(h.con2grid(c["x"], c["y"], c["nextq"], c["qjump"]), qc_o)


def test_recontour_of_nan_is_refused():
    """A field with one NaN gives boxes that a contour enters and does not
    leave: an error, after which the context contours a sound field."""
    from hydra_amd import Hydra, HydraError
    from hydra_amd.ic import random_pv
    ng = 32
    q = random_pv(ng, seed=5)
    h = Hydra(ng)
    h.set_field(q)
    h.recontour()
    want = h.contours()
    bad = q.copy()
    bad[11, 17] = np.nan
    h.set_field(bad)
    with pytest.raises(HydraError, match="inconsistent crossing tables"):
        h.recontour()
    h.set_field(q)
    h.recontour()
    got = h.contours()
    for k in ("x", "y", "nextq", "i1q", "i2q", "npq", "indq"):
        assert np.array_equal(got[k], want[k]), k
    h.close()


# more entries of order-dependent cells than the buckets hold (2^22), and
# more such cells (2^20; each has at least four entries) besides
@pytest.mark.parametrize("ng,nodes", [(32, 150000), (512, 90000)])
def test_con2grid_overflow_is_reported_once(ng, nodes, hyd_cache):
    """A sweep whose order-dependent cells exceed the buckets is refused; the
    next one is right again."""
    from hydra_amd import HydraError
    from oracle.hyo import Oracle
    h = hyd_cache(ng)
    rng = np.random.default_rng(nodes)
    x, y = rng.uniform(-np.pi, np.pi, (2, nodes))
    nxt = np.r_[np.arange(2, nodes + 1), 1].astype(np.int32)
    with pytest.raises(HydraError, match="error -3"):
        h.con2grid(x, y, nxt, 0.37)
    c = _hairpins(ng)
    o = Oracle(ng)
    o.set_contours(c)
    assert bits_equal(h.con2grid(c["x"], c["y"], c["nextq"], c["qjump"]), o.con2grid())


@pytest.mark.parametrize("ng", [64, 256])
def test_recontour_of_noise_bitwise(ng):
    """White noise: tens of thousands of short contours (a level hardly ever
    passes through a saddle: chains that close on themselves)."""
    from hydra_amd import Hydra
    from oracle.hyo import Oracle
    q = np.random.default_rng(ng).standard_normal((ng, ng))
    o = Oracle(ng, ncontq=3)
    o.init_from_field(q)
    o.recontour(o.d("qr").copy())
    h = Hydra(ng, ncontq=3)
    h.set_field(q)
    h.recontour()
    c, g = o.contours(), h.contours()
    for k in ("nextq", "i1q", "i2q", "npq", "indq"):
        assert np.array_equal(g[k], c[k]), k
    assert bits_equal(g["x"], c["x"]) and bits_equal(g["y"], c["y"])
    h.close()


def _saddle_boxes(q, level):
    """Boxes of the 16 times finer bilinear field whose corners alternate
    about a level."""
    i = np.arange(16 * len(q))
    i, p = i // 16, i % 16 / 16.0
    j = (i + 1) % len(q)
    a = q[i] * (1 - p)[:, None] + q[j] * p[:, None]
    s = a[:, i] * (1 - p) + a[:, j] * p >= level
    r, t = np.roll(s, -1, 0), np.roll(s, -1, 1)
    return int(np.sum((s == np.roll(r, -1, 1)) & (r == t) & (s != r)))


@pytest.mark.parametrize("ng,in_lds", [(64, True), (128, False)])
def test_recontour_through_saddles_bitwise(ng, in_lds):
    """A product of two alternating sequences has a saddle at the same value
    in every grid box, off the fine grid's vertices; shifted so that a level
    has that value, each is a box that two chains enter: the ordered walk
    through them, with the level's chains in LDS and beyond its capacity of
    12000 in global memory."""
    from hydra_amd import Hydra
    from oracle.hyo import Oracle
    rng = np.random.default_rng(ng)
    sign = (-1.0) ** np.arange(ng)
    q = np.outer(sign * rng.uniform(0.6, 1.4, ng), sign * rng.uniform(0.6, 1.4, ng))
    q += (q.max() - q.min()) / 6  # half of the level spacing
    chains = 2 * _saddle_boxes(q, (q.max() - q.min()) / 6)
    assert 0 < chains <= 12000 if in_lds else chains > 12000
    o = Oracle(ng, ncontq=3)
    o.init_from_field(q)
    o.recontour(o.d("qr").copy())
    h = Hydra(ng, ncontq=3)
    h.set_field(q)
    h.recontour()
    c, g = o.contours(), h.contours()
    for k in ("nextq", "i1q", "i2q", "npq", "indq"):
        assert np.array_equal(g[k], c[k]), k
    assert bits_equal(g["x"], c["x"]) and bits_equal(g["y"], c["y"])
    h.close()
