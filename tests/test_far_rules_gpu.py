"""What the factored far field may take: pairs whose weights keep their bits, whatever the
core radii, the shape of a block or the values of its strengths, and calls that it is
chosen for."""
import ctypes as C

import numpy as np
import pytest

from omega3d_amd import scenes
from omega3d_amd.metrics import rel_errors

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def infl():
    pytest.importorskip("torch")   # before the library, as the other modules have it
    from omega3d_amd import _lib, influence
    assert _lib.lib.o3d_init(-1) == 0, _lib.last_error()
    return influence


@pytest.mark.parametrize("over", [1.0, 0.3, 0.1, 0.03])
@pytest.mark.parametrize("core,grads,n", [("rm", True, 30001), ("wl", True, 44801), ("v2", True, 44801),
                                          ("rm", False, 47001), ("wl", False, 54901), ("v2", False, 54901)])
def test_cores_wider_than_the_gap(infl, core, grads, n, over):
    """a cube `over` core radii wide, which AUTO sends to the far field: the gaps between
    tiles are small beside the cores.  Within the compensated bar of the FP64 sums"""
    rng = np.random.default_rng(n)
    pos = rng.random((3, n)).astype(np.float32)
    st = (rng.normal(size=(3, n)) / n).astype(np.float32)
    rad = (rng.uniform(0.8, 1.25, n) / over).astype(np.float32)
    k = np.arange(0, n, n // 500)
    v, g = infl.p2p(core, pos, st, rad, pos, rad, grads, "comp")
    d, dg = infl.p2p(core, pos, st, rad, pos[:, k], rad[k], grads, "fp64")
    e = [rel_errors(v[:, k], d), rel_errors(g[:, k], dg) if grads else None]
    print(core, grads, over, e)
    assert e[0][0] <= 2e-6 and (not grads or e[1][0] <= 2e-6)


def _pair_sums(core, sp, ss, sr, t, grads):
    """sums of |K alpha x d| (and of |Bp d (alpha x d)| + |K alpha|) of one target in FP64"""
    d = t[:, None].astype(np.float64) - sp
    q = (d * d).sum(0)
    s2 = sr.astype(np.float64) ** 2
    if core == "rm":
        K, B = (q + s2) ** -1.5, 3 * (q + s2) ** -2.5
    elif core == "wl":
        K = (q + 2.5 * s2) * (q + s2) ** -2.5
        B = 3 * (q + 3.5 * s2) * (q + s2) ** -3.5
    elif core == "v2":
        K, B = (q * q + s2 * s2) ** -0.75, 3 * q * (q * q + s2 * s2) ** -1.75
    else:
        K, B = q ** -1.5, 3 * q ** -2.5   # beyond the core; within it less
    a, c = np.linalg.norm(ss, axis=0), np.linalg.norm(np.cross(ss, d, axis=0), axis=0)
    return (K * c).sum(), (B * np.sqrt(q) * c + K * a).sum() if grads else 0.0


@pytest.mark.parametrize("sigma", [0.05, 0.003])
@pytest.mark.parametrize("core,grads", [("rm", True), ("wl", True), ("v2", True), ("exp", True), ("rm", False),
                                        ("wl", False), ("v2", False), ("exp", False)])
def test_blocks_without_extent(infl, core, grads, sigma):
    """65 blocks of 256 coincident points and a block of one, inside a dense ring: a tile may
    lie as near to such a block as its own sphere ends.  Each point for itself against FP64:
    a pair keeps 22 bits of its weight and moments, at most four times its own size, 1e-6 of
    the sum of its pairs' sizes in all"""
    rng = np.random.default_rng(5)
    ns, nb = 200000, 65
    ph, th, r = 6.2831853 * rng.random(ns), 6.2831853 * rng.random(ns), 0.1 * np.sqrt(rng.random(ns))
    sp = np.stack([(1 + r * np.cos(ph)) * np.cos(th), (1 + r * np.cos(ph)) * np.sin(th), r * np.sin(ph)]).astype(np.float32)
    ss = (rng.normal(size=(3, ns)) / ns).astype(np.float32)
    sr = np.full(ns, sigma, np.float32)
    at = sp[:, rng.choice(ns, nb, replace=False)] + np.float32(1e-4)
    tp = np.concatenate([np.repeat(at, 256, 1), at[:, -1:]], 1)
    v, g = infl.p2p(core, sp, ss, sr, tp, None, grads, "comp")
    d, dg = infl.p2p(core, sp, ss, sr, at, None, grads, "fp64")
    for b in range(nb):
        size = _pair_sums(core, sp, ss, sr, at[:, b], grads)
        for t in (256 * b, 256 * b + 255) + ((256 * nb,) if b == nb - 1 else ()):
            e = [np.linalg.norm(v[:, t] - d[:, b]) / size[0], np.linalg.norm(g[:, t] - dg[:, b]) / size[1] if grads else 0.0]
            assert max(e) <= 1e-6, (core, grads, sigma, b, t, e)


@pytest.mark.parametrize("core,grads,prec", [("wl", True, "comp"), ("v2", True, "fp32"), ("rm", False, "comp"),
                                             ("exp", False, "fp32"), ("rm", True, "fp64"), ("exp", True, "fp64")])
def test_profile_refuses_what_factored_refuses(infl, core, grads, prec):
    """the profile is of method FACTORED whatever the method field says: calls that it does not
    serve are refused, and the outputs stay as they were"""
    from omega3d_amd import _lib
    p, D = scenes.ring(2048), _lib.DeviceArray.from_host
    x, s, r = D(p.pos), D(p.str), D(p.rad)
    out = D(np.full((12, p.n), 0.5, np.float32))
    q = _lib.Points()
    q.n, q.r = p.n, r.ptr
    for d in range(3):
        q.x[d], q.s[d], q.u[d] = x.row(d), s.row(d), out.row(d)
    for k in range(9):
        q.ug[k] = out.row(3 + k)
    for method in ("auto", "direct"):
        o = _lib.make_opts(core, grads, prec, method=method)
        assert _lib.lib.o3d_factored_profile_dev(C.byref(q), C.byref(q), C.byref(o), C.byref(_lib.FactoredProfile())) == 1
    assert (out.to_host() == 0.5).all()


@pytest.mark.parametrize("what", ["strength inf", "strength nan", "radius inf", "place 3e19"])
@pytest.mark.parametrize("core,grads", [("rm", True), ("wl", True), ("v2", True), ("exp", True), ("rm", False), ("wl", False)])
def test_values_that_are_no_numbers(infl, core, grads, what):
    """a strength component that is infinite or no number, an infinite core or a distance whose
    square overflows touches the components that it touches in the direct sums, no others"""
    n = 56001
    p = scenes.colliding_rings((n + 1) // 2, sigma=0.03)
    pos, st, rad = p.pos[:, :n].copy(), p.str[:, :n].copy(), p.rad[:n].copy()
    tp = pos[:, ::3].copy()
    if what.startswith("strength"):
        st[0, 5] = float(what.split()[1])
    elif what == "radius inf":
        rad[5] = np.inf
    else:
        pos[0, 5] = 3e19
    for t, tr in ((pos, rad), (tp, None)):
        ns = n if tr is not None else 6 * n
        s = (pos, st, rad) if tr is not None else tuple(np.concatenate([a] * 6, -1) for a in (pos, st / 6, rad))
        v, g = infl.p2p(core, *s, t, tr, grads, "comp")
        w, h = infl.p2p(core, *s, t, tr, grads, "comp", method="direct", tile=256, tpt=1)
        for a, b in [(v, w)] + ([(g, h)] if grads else []):
            fa, fb = np.isfinite(a), np.isfinite(b)
            assert np.array_equal(fa, fb), (what, ns, fa.mean(1), fb.mean(1))
            rows = fb.all(1)
            if rows.any():
                assert rel_errors(a[rows], b[rows])[0] <= 4e-6


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_panel_strengths_that_are_no_numbers(infl, bad):
    """the same of a panel's strength by both rules and of a particle's on panels"""
    from omega3d_amd import _lib
    pan, D = scenes.icosphere_panels(levels=3), _lib.DeviceArray.from_host
    ts = pan.ts.astype(np.float32).copy()
    ts[1, 7] = bad
    tp = scenes.shell_points(3000, 1.02, 3.0, seed=4).astype(np.float32)
    nodes, idx, ar = D(pan.nodes.astype(np.float32)), D(pan.idx.astype(np.uint32)), D(pan.area.astype(np.float32))
    dts, dtp = D(ts), D(tp)
    p, q = _lib.Panels(), _lib.Points()
    p.np, p.nn, p.idx, p.area, q.n = pan.np, pan.nodes.shape[1], idx.ptr, ar.ptr, tp.shape[1]
    out = _lib.DeviceArray((12, q.n))
    for d in range(3):
        p.x[d], p.ts[d], q.x[d], q.u[d] = nodes.row(d), dts.row(d), dtp.row(d), out.row(d)
    for k in range(9):
        q.ug[k] = out.row(3 + k)
    for method in ("auto", "gauss7"):
        res = []
        for tile in (0, 128):
            out.zero()
            o = _lib.make_opts("rm", True, "comp", method=method, tile=tile)
            _lib.check(_lib.lib.o3d_panels_affect_points_dev(C.byref(p), C.byref(q), C.byref(o), None))
            res.append(np.isfinite(out.to_host()))
        assert np.array_equal(*res), (method, [r.mean(1) for r in res])
    st = np.full((3, 40000), 1e-5, np.float32)
    st[1, 7] = bad
    sp = D(scenes.shell_points(40000, 1.05, 3.0, seed=5).astype(np.float32))
    dst = D(st)
    q.n = 40000
    for d in range(3):
        q.x[d], q.s[d] = sp.row(d), dst.row(d)
    few = scenes.icosphere_panels(levels=2)
    nodes, idx, ar = D(few.nodes.astype(np.float32)), D(few.idx.astype(np.uint32)), D(few.area.astype(np.float32))
    p.np, p.nn, p.idx, p.area = few.np, few.nodes.shape[1], idx.ptr, ar.ptr
    for d in range(3):
        p.x[d] = nodes.row(d)
    vel = _lib.DeviceArray((3, few.np))
    pv = (C.c_void_p * 3)(*[vel.row(d) for d in range(3)])
    res = []
    for tile in (0, 256):
        vel.zero()
        o = _lib.make_opts("rm", False, "comp", tile=tile)
        _lib.check(_lib.lib.o3d_points_affect_panels_dev(C.byref(q), C.byref(p), pv, C.byref(o), None))
        res.append(np.isfinite(vel.to_host()))
    assert np.array_equal(*res), [r.mean(1) for r in res]


def _far_fraction(pos):
    """share of the pairs that one factored RM evaluation of particles on themselves takes far"""
    from omega3d_amd import _lib
    n, D = pos.shape[1], _lib.DeviceArray.from_host
    x, s, r, out = D(pos.astype(np.float32)), D(np.full((3, n), 1e-3, np.float32)), D(np.full(n, 0.02, np.float32)), _lib.DeviceArray((12, n))
    q = _lib.Points()
    q.n, q.r = n, r.ptr
    for d in range(3):
        q.x[d], q.s[d], q.u[d] = x.row(d), s.row(d), out.row(d)
    for k in range(9):
        q.ug[k] = out.row(3 + k)
    prof, o = _lib.FactoredProfile(), _lib.make_opts("rm", True, "comp", method="factored")
    _lib.check(_lib.lib.o3d_factored_profile_dev(C.byref(q), C.byref(q), C.byref(o), C.byref(prof)))
    return prof.far_tile_fraction


@pytest.mark.parametrize("share,far", [(1e-4, 100), (1e-3, 1000), (0.05, 300)])
def test_few_particles_far_away_leave_the_order(infl, share, far):
    """a few particles many radii away widen the box, not the blocks of the rest: at most 5% of
    the pairs less are far, beside those of blocks that a stray particle is in"""
    p = scenes.colliding_rings(30000)
    pos, rng = p.pos.copy(), np.random.default_rng(3)
    base, m = _far_fraction(pos), int(share * p.n)
    pos[:, rng.choice(p.n, m, replace=False)] = far * rng.normal(size=(3, m))
    got = _far_fraction(pos)
    print(share, far, base, got)
    assert got >= base - 0.05 - 2 * share


def test_rings_far_apart_keep_their_order(infl):
    """two rings 300 radii apart, a few cells of the grid across each: the pairs that the
    far field takes are at least those of blocks cut from a Hilbert order of 2^10 cells per axis"""
    from test_panfar_gpu import _hilbert_order
    p, q = scenes.ring(100000), scenes.ring(100000, seed=3)
    pos = np.concatenate([p.pos, q.pos + np.float32(300) * np.array([[1], [0.3], [0.1]], np.float32)], 1).astype(np.float32)
    n, s = pos.shape[1], pos[:, _hilbert_order(pos)].astype(float)
    c, r = [], []
    for i in range(0, n, 256):
        b = s[:, i:i + 256]
        c.append(0.5 * (b.min(1) + b.max(1)))
        r.append(np.linalg.norm(b - c[-1][:, None], axis=0).max())
    c, r, m = np.array(c), np.array(r), np.minimum(256, n - 256 * np.arange(len(r)))
    gap = np.linalg.norm(c[:, None] - c[None], axis=2) - r[:, None] - r[None]
    want = (m[:, None] * m[None] * (gap > np.maximum(r[:, None], r[None]))).sum() / float(n) ** 2
    got = _far_fraction(pos)
    print(got, want)
    assert got >= want - 0.002


def test_auto_without_room_for_the_far_field(infl):
    """a call whose far field would need more memory than the GPU has is the direct kernel's
    (7e8 targets in one place: outputs of 34 GB, 290 GB of scratch), bit for bit;
    the method asked for by name has no other way and says so"""
    from omega3d_amd import _lib
    n, p, D = 700_000_000, scenes.ring(8192, sigma=0.05), _lib.DeviceArray.from_host
    x, s, r = D(p.pos), D(p.str), D(p.rad)
    zero, out = C.c_void_p(), C.c_void_p()
    for a, rows in ((zero, 1), (out, 12)):
        if _lib.lib.o3d_dev_malloc(C.byref(a), 4 * n * rows):
            pytest.skip("no room for the outputs")
        _lib.check(_lib.lib.o3d_memset_dev(a, 0, 4 * n * rows))
    src, t = _lib.Points(), _lib.Points()
    src.n, src.r, t.n = p.n, r.ptr, n
    for d in range(3):
        src.x[d], src.s[d], t.x[d], t.u[d] = x.row(d), s.row(d), zero.value, out.value + 4 * n * d
    for k in range(9):
        t.ug[k] = out.value + 4 * n * (3 + k)
    _lib.synchronize()   # the stream below does not wait for the fills
    stream = C.c_void_p()
    _lib.check(_lib.lib.o3d_stream_create(C.byref(stream)))
    try:
        o = _lib.make_opts("rm", True, "fp32", method="factored", stream=stream)
        assert _lib.lib.o3d_points_affect_points_dev(C.byref(src), C.byref(t), C.byref(o), None) == 2
        o = _lib.make_opts("wl", True, "comp", stream=stream)
        _lib.check(_lib.lib.o3d_points_affect_points_dev(C.byref(src), C.byref(t), C.byref(o), None))
        _lib.check(_lib.lib.o3d_stream_synchronize(stream))
        got = np.empty((12, 2), np.float32)
        for k in range(12):
            for e, i in enumerate((0, n - 1)):
                _lib.check(_lib.lib.o3d_memcpy_dtoh(got[k, e:].ctypes.data, out.value + 4 * (n * k + i), 4))
    finally:
        _lib.lib.o3d_stream_destroy(stream)
        for a in (zero, out):
            _lib.lib.o3d_dev_free(a)
    v, g = infl.p2p("wl", p.pos, p.str, p.rad, np.zeros((3, 1)), None, True, "comp", method="direct", tile=256, tpt=1)
    for e in (0, 1):
        assert np.array_equal(got[:3, e:e + 1], v) and np.array_equal(got[3:, e:e + 1], g)


def test_factored_counts_whose_sum_passes_the_int_range(infl):
    """FACTORED takes up to INT_MAX sources and targets each, also where both together are more
    (one sort orders both): sources and targets in one place, whose gradient is that of the
    summed strengths, N K(0) alpha with RM's K(0) = 1 / sigma^3, within the compensated bar"""
    from omega3d_amd import _lib
    ns, nt = 2**31 - 601, 1000
    bufs, fill = [], (0, 0x3d, 0x2e)   # places 0, radii 0.0462, strengths 4e-11
    out, D = _lib.DeviceArray.from_host(np.zeros((12, nt), np.float32)), None
    sigma, alpha = (float(np.frombuffer(bytes([b] * 4), np.float32)[0]) for b in fill[1:])
    try:
        for b in fill:
            p = C.c_void_p()
            if _lib.lib.o3d_dev_malloc(C.byref(p), 4 * ns):
                pytest.skip("no room for the sources")
            bufs.append(p)
            _lib.check(_lib.lib.o3d_memset_dev(p, b, 4 * ns))
        _lib.synchronize()
        s, t = _lib.Points(), _lib.Points()
        s.n, s.r, t.n = ns, bufs[1].value, nt
        for d in range(3):
            s.x[d], s.s[d], t.x[d], t.u[d] = bufs[0].value, bufs[2].value, bufs[0].value, out.row(d)
        for k in range(9):
            t.ug[k] = out.row(3 + k)
        stream = C.c_void_p()
        _lib.check(_lib.lib.o3d_stream_create(C.byref(stream)))
        try:
            o = _lib.make_opts("rm", True, "comp", method="factored", stream=stream)
            rc = _lib.lib.o3d_points_affect_points_dev(C.byref(s), C.byref(t), C.byref(o), None)
            if rc == 2:
                pytest.skip("no room for the scratch")
            _lib.check(rc)
            _lib.check(_lib.lib.o3d_stream_synchronize(stream))
        finally:
            _lib.lib.o3d_stream_destroy(stream)
        got = out.to_host().astype(np.float64)
    finally:
        for p in bufs:
            _lib.lib.o3d_dev_free(p)
    W = ns * alpha / sigma ** 3
    want = np.array([0, W, -W, -W, 0, W, W, -W, 0])[:, None]   # skew of (W, W, W)
    assert not got[:3].any()
    assert np.abs(got[3:] - want).max() <= 2e-6 * W


@pytest.mark.parametrize("levels,np_,below,beyond", [(3, 1280, 255999, 256001), (3, 640, 127999, 128001), (4, 5120, 351562, 351563)])
def test_line_of_particles_on_panels(infl, levels, np_, below, beyond):
    """200 particles per panel or 1.8e9 pairs: the direct kernel's bits below, others beyond"""
    from omega3d_amd import _lib
    pan, D = scenes.icosphere_panels(levels=levels), _lib.DeviceArray.from_host
    sp, st = D(scenes.shell_points(beyond, 1.02, 1.5, seed=4).astype(np.float32)), D(np.full((3, beyond), 1e-5, np.float32))
    nodes, idx, ar = D(pan.nodes.astype(np.float32)), D(pan.idx.astype(np.uint32)), D(pan.area.astype(np.float32))
    q, p, vel = _lib.Points(), _lib.Panels(), _lib.DeviceArray((3, np_))
    p.np, p.nn, p.idx, p.area = np_, pan.nodes.shape[1], idx.ptr, ar.ptr
    for d in range(3):
        p.x[d], q.x[d], q.s[d] = nodes.row(d), sp.row(d), st.row(d)
    pv = (C.c_void_p * 3)(*[vel.row(d) for d in range(3)])
    for n in (below, beyond):
        q.n, res = n, []
        for tile in (0, 256):
            vel.zero()
            o = _lib.make_opts("rm", False, "comp", tile=tile)
            _lib.check(_lib.lib.o3d_points_affect_panels_dev(C.byref(q), C.byref(p), pv, C.byref(o), None))
            res.append(vel.to_host())
        assert np.array_equal(*res) == (n == below)
        assert rel_errors(*res)[0] <= 4e-6


@pytest.mark.parametrize("core,ns,nt,far", [("rm", 65535, 65535, False), ("exp", 65535, 65535, False), ("exp", 32768, 32768, False),
                                            ("rm", 110000, 65535, False), ("exp", 65535, 70000, False),
                                            ("rm", 65536, 65536, True), ("exp", 65536, 66000, True)])
def test_line_of_plain_sums(infl, core, ns, nt, far):
    """plain FP32 takes the far field from 65,536 sources and targets on: the direct bits below"""
    p = scenes.ring(ns, seed=5)
    t = (p.pos, p.rad) if ns == nt else (scenes.ring(nt, a=0.2, seed=6).pos, None)
    args = (core, p.pos, p.str, p.rad, *t, True, "fp32")
    (v, g), (w, h) = infl.p2p(*args), infl.p2p(*args, method="direct")
    assert (np.array_equal(v, w) and np.array_equal(g, h)) != far


@pytest.mark.parametrize("core,ns", [("rm", 33), ("rm", 64), ("rm", 111), ("wl", 97), ("v2", 80), ("exp", 33), ("exp", 48)])
def test_fewest_sources_take_one_pass(infl, core, ns):
    """so few sources are not cut: the bits of the one-pass kernel"""
    p = scenes.ring(ns, seed=7)
    t = (2.4 * np.random.default_rng(9).random((3, 1000)) - 1.2).astype(np.float32)
    for grads, prec in ((True, "comp"), (False, "comp"), (True, "fp32")):
        a = infl.p2p(core, p.pos, p.str, p.rad, t, None, grads, prec)
        b = infl.p2p(core, p.pos, p.str, p.rad, t, None, grads, prec, tile=256, tpt=1)
        assert np.array_equal(a[0], b[0]) and (not grads or np.array_equal(a[1], b[1]))


@pytest.mark.parametrize("core,grads,below,nt", [("exp", True, 24494, 0), ("rm", True, 29999, 0), ("wl", True, 44721, 0),
                                                 ("v2", True, 44721, 0), ("exp", False, 31622, 0), ("rm", False, 46904, 0),
                                                 ("wl", False, 54772, 0), ("v2", False, 54772, 0), ("exp", True, 104999, 10000),
                                                 ("wl", True, 213636, 16383), ("rm", False, 320833, 12000),
                                                 ("rm", True, 109863, 8192), ("exp", True, 73242, 8191)])
def test_both_sides_of_autos_lines(infl, core, grads, below, nt):
    """compensated calls a particle below AUTO's line have the direct kernel's bits, a particle
    beyond it others (nt 0: on themselves; fewer than 8,192 targets are direct at any count)"""
    for ns in (below, below + 1):
        p = scenes.ring(ns, seed=12)
        t = (p.pos, p.rad) if nt == 0 else (scenes.ring(nt, a=0.3, seed=13).pos, None)
        args = (core, p.pos, p.str, p.rad, *t, grads, "comp")
        (v, g), (w, h) = infl.p2p(*args), infl.p2p(*args, method="direct")
        same = np.array_equal(v, w) and (not grads or np.array_equal(g, h))
        assert same == (ns == below or nt == 8191)


def test_field_points_do_not_widen_the_sources_grid(infl):
    """rings among field points of a box 30 times as wide: each set is ordered on a grid of its
    own, so as many pairs are far as with the points in a box that just holds the rings"""
    from omega3d_amd import _lib
    p, D = scenes.colliding_rings(30000), _lib.DeviceArray.from_host
    box, f = 4.0 * np.random.default_rng(6).random((3, 20000)) - 2.0, []
    x, s, r, out = D(p.pos.astype(np.float32)), D(p.str.astype(np.float32)), D(p.rad.astype(np.float32)), _lib.DeviceArray((12, 20000))
    for wide in (1, 30):
        tp = D((wide * box).astype(np.float32))
        q, t = _lib.Points(), _lib.Points()
        q.n, q.r, t.n = p.n, r.ptr, 20000
        for d in range(3):
            q.x[d], q.s[d], t.x[d], t.u[d] = x.row(d), s.row(d), tp.row(d), out.row(d)
        for k in range(9):
            t.ug[k] = out.row(3 + k)
        prof, o = _lib.FactoredProfile(), _lib.make_opts("rm", True, "comp", method="factored")
        _lib.check(_lib.lib.o3d_factored_profile_dev(C.byref(q), C.byref(t), C.byref(o), C.byref(prof)))
        f.append(prof.far_tile_fraction)
    print(f)
    assert f[1] >= f[0]
