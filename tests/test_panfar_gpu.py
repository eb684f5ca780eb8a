"""Panel sums whose separated pairs go to the matrix cores (panfar.hip): large calls with
the tile left open, against the oracle on some targets and against the direct kernels (a
tile given) on all.

Bars, in units of the largest value: the oracle's as for the direct kernels
(test_pan_gpu.py: max(2e-6, 3 x the float reference's own distance from FP64); 7-point
rule 2e-6); between the two GPU paths, which take the same decision for every pair, twice
2e-6 in compensated precision, and in FP32, whose direct kernel adds up to `np` (7 np)
terms in one float, 2e-6 + 4e-6 as for a random walk of 2,500 roundings of 6e-8.
"""
import ctypes as C

import numpy as np
import pytest

import oracle
from omega3d_amd import scenes
from omega3d_amd.metrics import rel_errors

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mods():
    torch = pytest.importorskip("torch")
    from omega3d_amd import _lib, influence
    assert _lib.lib.o3d_init(-1) == 0, _lib.last_error()
    return torch, _lib, influence


def _call(mods, pan, n, tp, grads, prec, method, tile, ss=True, maxlev=-1, scale=1.0, area=None):
    """panels_affect_points on device arrays: velocity and gradient (12 or 3, nt)"""
    torch, _lib, influence = mods
    dev = lambda x: torch.tensor(np.ascontiguousarray(x), device="cuda")
    nodes, idx = dev(pan.nodes.astype(np.float32)), dev(pan.idx[:3 * n].astype(np.int32))
    ts = dev((pan.ts[:, :n] * scale).astype(np.float32))
    ar = dev((pan.area if area is None else area)[:n].astype(np.float32))
    s = dev((pan.ss[:n] * scale).astype(np.float32)) if ss else None
    t, out = dev(tp.astype(np.float32)), torch.zeros(12 if grads else 3, tp.shape[1], device="cuda")
    p, q = _lib.Panels(), _lib.Points()
    p.np, p.nn, p.idx, p.area = n, nodes.shape[1], idx.data_ptr(), ar.data_ptr()
    p.ss = s.data_ptr() if ss else None
    q.n = tp.shape[1]
    for d in range(3):
        p.x[d], p.ts[d], q.x[d], q.u[d] = (a[d].data_ptr() for a in (nodes, ts, t, out))
    for k in range(9 if grads else 0):
        q.ug[k] = out[3 + k].data_ptr()
    o = _lib.make_opts("rm", grads, prec, method=method, tile=tile, maxlev=maxlev)
    _lib.check(_lib.lib.o3d_panels_affect_points_dev(C.byref(p), C.byref(q), C.byref(o), None))
    torch.cuda.synchronize()
    return out.cpu().numpy()


def _surface():
    pan = scenes.icosphere_panels(levels=3)   # 1,280 panels
    pan.ss = (0.3 * np.random.default_rng(3).normal(size=pan.np)).astype(np.float32)
    return pan


def _bar(a, b, tol):
    for rows in ([slice(0, 3)] if a.shape[0] == 3 else [slice(0, 3), slice(3, 12)]):
        assert rel_errors(a[rows], b[rows])[0] <= tol


@pytest.mark.parametrize("method", ["auto", "gauss7"])
@pytest.mark.parametrize("n,nt,grads,ss,prec,maxlev", [
    (1280, 2048, True, True, "comp", -1),     # whole tiles and blocks
    (1280, 2049, True, False, "comp", 2),     # a block of one target
    (1281 - 256, 2303, False, True, "comp", -1),   # a tile of one panel
    (1024, 5000, False, False, "comp", 0),
    (1153, 2304, True, True, "fp32", -1),
    (1279, 2100, False, False, "fp32", 1)])
def test_separated_panels(mods, method, n, nt, grads, ss, prec, maxlev):
    pan = _surface()
    tp = scenes.shell_points(nt, 1.02, 3.0, seed=nt)
    a = _call(mods, pan, n, tp, grads, prec, method, 0, ss, maxlev)
    b = _call(mods, pan, n, tp, grads, prec, method, 128, ss, maxlev)
    assert not np.array_equal(a, b)   # the far field took part
    _bar(a, b, 6e-6 if prec == "fp32" else 4e-6)
    k = np.random.default_rng(1).choice(nt, 150, replace=False)
    if method == "gauss7":
        o = oracle.pan_g7(pan.nodes, pan.idx[:3 * n], pan.ts[:, :n], pan.area[:n], pan.ss[:n] if ss else None, tp[:, k],
                          grads=grads)
        _bar(a[:, k], np.concatenate(o[:2] if grads else o[:1]), 6e-6 if prec == "fp32" else 2e-6)
    else:
        args = ("rm", pan.nodes, pan.idx[:3 * n], pan.ts[:, :n], pan.area[:n], pan.ss[:n] if ss else None, tp[:, k], grads)
        o64, o32 = (np.concatenate([x for x in oracle.pan(*args, mode, maxlev=3 if maxlev < 0 else maxlev) if x is not None])
                    for mode in ("f64", "f32d"))
        for rows in ([slice(0, 3), slice(3, 12)] if grads else [slice(0, 3)]):
            bar = max(2e-6 if prec == "comp" else 6e-6, 3 * rel_errors(o32[rows], o64[rows])[0])
            assert rel_errors(a[rows][:, k], o64[rows])[0] <= bar


@pytest.mark.parametrize("method", ["auto", "gauss7"])
def test_scaling_and_places(mods, method):
    """strengths times -1 and times powers of two give just that, and points far away, all in
    one place or beside panels whose area is no number are summed as the direct kernels do"""
    pan = _surface()
    n, tp = pan.np, scenes.shell_points(3000, 1.02, 1.5, seed=9)
    a = _call(mods, pan, n, tp, True, "comp", method, 0)
    for f in (-1.0, 2.0, -2.0 ** -20, 2.0 ** 80):
        assert np.array_equal(_call(mods, pan, n, tp, True, "comp", method, 0, scale=f), a * np.float32(f))
    for far in (tp + 50.0, np.repeat(tp[:, :1], 2500, 1), np.concatenate([tp[:, :1300], 1e4 * tp[:, :1300]], 1)):
        _bar(_call(mods, pan, n, far, True, "comp", method, 0), _call(mods, pan, n, far, True, "comp", method, 128), 4e-6)
    if method == "auto":
        area = pan.area.copy()
        area[77] = -area[77]
        x = _call(mods, pan, n, tp, True, "comp", method, 0, area=area, maxlev=1)
        y = _call(mods, pan, n, tp, True, "comp", method, 128, area=area, maxlev=1)
        _bar(x, y, 4e-6)


def _hilbert_order(p):
    """numpy restatement of the sort: positions along the Hilbert curve of a 2^10 grid"""
    lo = p.min(1, keepdims=True)
    q = ((p - lo) * (np.float32(1023) / (p.max(1, keepdims=True) - lo).max())).astype(np.uint32)
    x = [q[d].copy() for d in range(3)]
    for b in range(9, 0, -1):
        low = np.uint32((1 << b) - 1)
        for d in range(3):
            up = (x[d] >> np.uint32(b)) & np.uint32(1) == 1
            t = np.where(up, np.uint32(0), (x[0] ^ x[d]) & low)
            x[0] = np.where(up, x[0] ^ low, x[0] ^ t)
            if d:
                x[d] = x[d] ^ t
    x[1] ^= x[0]
    x[2] ^= x[1]
    t = np.zeros_like(x[0])
    for b in range(9, 0, -1):
        t ^= np.where((x[2] >> np.uint32(b)) & np.uint32(1) == 1, np.uint32((1 << b) - 1), np.uint32(0))
    key = np.zeros(p.shape[1], np.int64)
    for b in range(9, -1, -1):
        for d in range(3):
            key = 2 * key + (((x[d] ^ t) >> np.uint32(b)) & np.uint32(1))
    return np.argsort(key, kind="stable")


@pytest.mark.parametrize("n", [20000, 65537])
def test_blocks_follow_the_hilbert_curve(mods, n):
    """the pairs that the far field takes are at least those of blocks cut from a Hilbert
    order (a box of random points; blocks cut from a Morton order miss 2 to 4%)"""
    torch, _lib, _ = mods
    p = np.random.default_rng(n).random((3, n)).astype(np.float32)
    s = p[:, _hilbert_order(p)]
    c, r = [], []
    for i in range(0, n, 256):
        b = s[:, i:i + 256].astype(float)
        c.append(0.5 * (b.min(1) + b.max(1)))
        r.append(np.linalg.norm(b - c[-1][:, None], axis=0).max())
    c, r, m = np.array(c), np.array(r), np.minimum(256, n - 256 * np.arange(len(r)))
    gap = np.linalg.norm(c[:, None] - c[None], axis=2) - r[:, None] - r[None]
    want = (m[:, None] * m[None] * (gap > r[:, None])).sum() / float(n) ** 2
    dev = [torch.tensor(x, device="cuda") for x in (p, np.full((3, n), 1e-3, np.float32), np.full(n, 1e-3, np.float32))]
    out = torch.zeros(12, n, device="cuda")
    q = _lib.Points()
    q.n, q.r = n, dev[2].data_ptr()
    for d in range(3):
        q.x[d], q.s[d], q.u[d] = dev[0][d].data_ptr(), dev[1][d].data_ptr(), out[d].data_ptr()
    for k in range(9):
        q.ug[k] = out[3 + k].data_ptr()
    prof = _lib.FactoredProfile()
    o = _lib.make_opts("rm", True, "comp", method="factored")
    _lib.check(_lib.lib.o3d_factored_profile_dev(C.byref(q), C.byref(q), C.byref(o), C.byref(prof)))
    print(n, prof.far_tile_fraction, want)
    assert prof.far_tile_fraction >= want - 0.002


@pytest.mark.parametrize("core,grads", [("rm", True), ("exp", True), ("wl", True), ("v2", True), ("rm", False),
                                        ("v2", False)])
def test_tiles_smaller_than_the_block(mods, core, grads):
    """points spread wide over dense sources: most far tiles are nearer than the block is
    wide and summed about their own centres.  Against the direct FP64 sums; the bar is the
    22 bits of a product, 2.4e-7, for the whole and 2e-6 for the worst point"""
    torch, _lib, influence = mods
    rng = np.random.default_rng(11)
    ns, nt = 70001, 65537
    th, r, ph = 6.2831853 * rng.random(ns), 0.1 * np.sqrt(rng.random(ns)), 6.2831853 * rng.random(ns)
    sp = np.stack([(1 + r * np.cos(ph)) * np.cos(th), (1 + r * np.cos(ph)) * np.sin(th), r * np.sin(ph)]).astype(np.float32)
    ss = (rng.normal(size=(3, ns)) / ns).astype(np.float32)
    sr = np.full(ns, 0.03, np.float32)
    tp = (4.0 * rng.random((3, nt)) - 2.0).astype(np.float32)
    k = rng.choice(nt, 2000, replace=False)
    v, g = influence.p2p(core, sp, ss, sr, tp, None, grads, "comp")[:2]
    d, dg = influence.p2p(core, sp, ss, sr, tp[:, k], None, grads, "fp64")[:2]
    for a, b in [(v[:, k], d)] + ([(g[:, k], dg)] if grads else []):
        e = rel_errors(a, b)
        print(core, grads, e)
        assert e[0] <= 2e-6 and e[1] <= 2.4e-7


def _ptpan(mods, pan, sp, ss, prec, method, tile, maxlev):
    """points_affect_panels on device arrays: velocities (3, np)"""
    torch, _lib, _ = mods
    dev = lambda x: torch.tensor(np.ascontiguousarray(x), device="cuda")
    nodes, idx, ar = dev(pan.nodes.astype(np.float32)), dev(pan.idx.astype(np.int32)), dev(pan.area)
    pos, a, out = dev(sp), dev(ss), torch.zeros(3, pan.np, device="cuda")
    p, q = _lib.Panels(), _lib.Points()
    p.np, p.nn, p.idx, p.area, q.n = pan.np, nodes.shape[1], idx.data_ptr(), ar.data_ptr(), sp.shape[1]
    for d in range(3):
        p.x[d], q.x[d], q.s[d] = nodes[d].data_ptr(), pos[d].data_ptr(), a[d].data_ptr()
    vel = (C.c_void_p * 3)(*[out[d].data_ptr() for d in range(3)])
    o = _lib.make_opts("rm", False, prec, method=method, tile=tile, maxlev=maxlev)
    _lib.check(_lib.lib.o3d_points_affect_panels_dev(C.byref(q), C.byref(p), vel, C.byref(o), None))
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("levels,ns,prec,maxlev", [(1, 8192, "comp", -1), (2, 32769, "comp", 2), (2, 40001, "fp32", -1),
                                                   (0, 8193, "comp", 8)])
def test_separated_particles_on_panels(mods, levels, ns, prec, maxlev):
    """few panels, many particles, a good part of them near: against the direct kernel and,
    with the first particles alone, the oracle"""
    pan = scenes.icosphere_panels(levels=levels)
    sp = scenes.shell_points(ns, 1.01, 2.5, seed=ns).astype(np.float32)
    ss = (np.random.default_rng(5).normal(size=(3, ns)) / ns).astype(np.float32)
    a = _ptpan(mods, pan, sp, ss, prec, "auto", 0, maxlev)
    b = _ptpan(mods, pan, sp, ss, prec, "auto", 256, maxlev)
    assert not np.array_equal(a, b)
    assert rel_errors(a, b)[0] <= (6e-6 if prec == "fp32" else 4e-6)
    assert np.array_equal(_ptpan(mods, pan, sp, -2 * ss, prec, "auto", 0, maxlev), -2 * a)
    m = 2000
    lev = 3 if maxlev < 0 else maxlev
    o64, o32 = (oracle.ptpan("rm", sp[:, :m], ss[:, :m], pan.nodes, pan.idx, pan.area, mode, maxlev=lev)
                for mode in ("f64", "f32d"))
    ss[:, m:] = 0
    bar = max(2e-6 if prec == "comp" else 6e-6, 3 * rel_errors(o32, o64)[0])
    assert rel_errors(_ptpan(mods, pan, sp, ss, prec, "auto", 0, maxlev), o64)[0] <= bar


@pytest.mark.parametrize("maxlev,tile", [(1, 128), (3, 128), (6, 0), (8, 128), (8, 0)])
def test_deep_trees(mods, maxlev, tile):
    """points so near the surface that trees reach every level (the stack of nodes at its
    fullest), direct and separated, against the oracle"""
    pan = _surface()
    k = np.arange(40)
    tp = scenes.shell_points(1100, 1.0002, 1.02, seed=maxlev)
    v = _call(mods, pan, pan.np, tp, True, "comp", "auto", tile, True, maxlev)
    args = ("rm", pan.nodes, pan.idx, pan.ts, pan.area, pan.ss, tp[:, k], True)
    o64, o32 = (np.concatenate(oracle.pan(*args, mode, maxlev=maxlev)) for mode in ("f64", "f32d"))
    for rows in (slice(0, 3), slice(3, 12)):
        bar = max(2e-6, 3 * rel_errors(o32[rows], o64[rows])[0])
        assert rel_errors(v[rows][:, k], o64[rows])[0] <= bar


@pytest.mark.parametrize("core,n", [("wl", 32768), ("v2", 33001), ("exp", 12288)])
def test_batch_takes_other_cores_factored(mods, core, n):
    """instances from the line on leave the queue, one below it stays; both within the
    compensated bar of the FP64 sums on some targets"""
    torch, _lib, influence = mods
    from omega3d_amd import batch
    inst = [scenes.ring(n, seed=21), scenes.ring(n - 1 if n != 33001 else 32767, seed=22), scenes.ring(300, seed=23)]
    b = batch.Batch(inst, core=core, precision="comp")
    try:
        assert b.config()["factored_instances"] == 1
        b.run()
        for (v, g), p in zip(b.results(), inst):
            k = np.arange(0, p.n, max(1, p.n // 300))
            ov, og = oracle.p2p(core, p.pos, p.str, p.rad, p.pos[:, k], p.rad[k], True, "f64")
            assert rel_errors(v[:, k], ov)[0] <= 1e-6 and rel_errors(g[:, k], og)[0] <= 1e-6
    finally:
        b.close()


@pytest.mark.parametrize("core,grads,ns,nt", [("exp", True, 24495, 24495), ("exp", True, 8192, 73300), ("rm", True, 30001, 30001),
                                              ("exp", False, 31700, 31700), ("rm", True, 110000, 8192)])
def test_auto_line(mods, core, grads, ns, nt):
    """calls just beyond AUTO's line between the methods: not the direct bits, within the
    compensated bar of FP64; and just before it the direct bits"""
    torch, _lib, influence = mods
    p = scenes.ring(ns, seed=31)
    t = (p.pos, p.rad) if nt == ns else ((3 * np.random.default_rng(2).random((3, nt)) - 1.5).astype(np.float32), None)
    call = lambda m: influence.p2p(core, p.pos, p.str, p.rad, t[0], t[1], grads, "comp", method=m)
    v, g = call("auto")
    w, h = call("direct")
    assert not np.array_equal(v, w)
    k = np.arange(0, nt, nt // 300)
    ov, og = oracle.p2p(core, p.pos, p.str, p.rad, t[0][:, k], None if t[1] is None else t[1][k], grads, "f64")
    assert rel_errors(v[:, k], ov)[0] <= 1e-6 and (not grads or rel_errors(g[:, k], og)[0] <= 1e-6)
    m = 8191
    a = influence.p2p(core, p.pos[:, :m], p.str[:, :m], p.rad[:m], t[0], t[1], grads, "comp")
    b = influence.p2p(core, p.pos[:, :m], p.str[:, :m], p.rad[:m], t[0], t[1], grads, "comp", method="direct")
    assert np.array_equal(a[0], b[0]) and (not grads or np.array_equal(a[1], b[1]))


@pytest.mark.parametrize("n,maxlev,nunk", [(1, 3, 3), (33, 3, 2), (65, 3, 3), (257, 3, 3), (120, 1, 3), (120, 2, 2), (70, 4, 3)])
def test_bem_matrix_ragged(mods, n, maxlev, nunk):
    """the influence matrix of a patch of n coarse panels, most pairs near: list remainders,
    quarters without a pair, gathered leaves full and partial.  Against the oracle's FP64 leaves
    on the same trees: leaf kernels in float (1e-7 each) and one rounding, 1e-6"""
    torch, _lib, influence = mods
    pan = scenes.icosphere_panels(levels=2)
    S = oracle.surface(np.ascontiguousarray(pan.nodes, np.float32), np.asarray(pan.idx, np.uint32).reshape(-1, 3)[:n])
    a = influence.bem_matrix(S[:3], None, nunk, maxlev)
    b = oracle.bem_matrix("wl", S, S, nunk, True, maxlev, mode="f64t")
    assert np.abs(a - b).max() <= 1e-6 * np.abs(b).max()


@pytest.mark.parametrize("core", ["rm", "exp"])
@pytest.mark.parametrize("ns,nt", [(1, 1), (32, 5), (33, 300), (65, 257), (1025, 1), (1000, 16129), (4095, 255)])
def test_short_slices(mods, core, ns, nt):
    """the smallest calls, whose sources are cut below a tile: one source over a slice, the
    last slice short, one target; within the compensated bar of the oracle"""
    torch, _lib, influence = mods
    p = scenes.ring(ns, seed=41)
    t = (2.4 * np.random.default_rng(6).random((3, nt)) - 1.2).astype(np.float32)
    v, g = influence.p2p(core, p.pos, p.str, p.rad, t, None, True, "comp")
    k = np.arange(0, nt, max(1, nt // 400))
    ov, og = oracle.p2p(core, p.pos, p.str, p.rad, t[:, k], None, True, "f64")
    assert rel_errors(v[:, k], ov)[0] <= 2e-6 and rel_errors(g[:, k], og)[0] <= 2e-6


@pytest.mark.parametrize("prec", ["comp", "fp32"])
@pytest.mark.parametrize("core,ns,nt", [("rm", 257, 64), ("rm", 1024, 65), ("wl", 8192, 63), ("v2", 8449, 1),
                                        ("exp", 16641, 129), ("rm", 20000, 1000)])
def test_slices_added_by_column(mods, core, ns, nt, prec):
    """slice counts at and about whole rounds of loads, last blocks of few targets, sums added
    into values that are there, the self pair taken out.  Compensated: the oracle's bar.  Plain
    FP32 adds up to 512 terms of a slice one after another, 512 roundings of 2^-24 of sums that
    pass the result by less than a factor of three: 1e-4"""
    torch, _lib, influence = mods
    bar = 2e-6 if prec == "comp" else 1e-4
    p = scenes.ring(ns, seed=43)
    t = (2.4 * np.random.default_rng(8).random((3, nt)) - 1.2).astype(np.float32)
    v0, g0 = np.full((3, nt), 0.25, np.float32), np.full((9, nt), -0.5, np.float32)
    v, g = influence.p2p(core, p.pos, p.str, p.rad, t, None, True, prec, vel=v0.copy(), grad=g0.copy())
    u, _ = influence.p2p(core, p.pos, p.str, p.rad, t, None, False, prec)
    ov, og = oracle.p2p(core, p.pos, p.str, p.rad, t, None, True, "f64")
    assert rel_errors(v, ov + v0)[0] <= bar and rel_errors(g, og + g0)[0] <= bar
    assert rel_errors(u, ov)[0] <= bar
    if ns <= 1024:
        v, g = influence.p2p(core, p.pos, p.str, p.rad, p.pos, p.rad, True, prec, self_term=1)
        w, h = influence.p2p(core, p.pos, p.str, p.rad, p.pos, p.rad, True, prec, self_term=1, tile=256, tpt=1)
        assert rel_errors(v, w)[0] <= bar and rel_errors(g, h)[0] <= bar


@pytest.mark.parametrize("core,n", [("rm", 12300), ("rm", 40000), ("rm", 65534), ("exp", 12300), ("exp", 32768)])
def test_factored_no_less_exact_than_direct(mods, core, n):
    """below 65,536 particles the factored sum stands where the direct one stood: its normwise
    errors against FP64 are no larger (a twentieth for the draw of a seed)"""
    torch, _lib, influence = mods
    p = scenes.colliding_rings(n // 2, sigma=0.05)
    k = np.arange(0, p.pos.shape[1], 8)
    ov, og = oracle.p2p(core, p.pos, p.str, p.rad, p.pos[:, k], p.rad[k], True, "f64")
    err = {}
    for m in ("direct", "factored"):
        v, g = influence.p2p(core, p.pos, p.str, p.rad, p.pos, p.rad, True, "comp", method=m)
        err[m] = [np.linalg.norm(x[:, k].astype(np.float64) - y) / np.linalg.norm(y) for x, y in ((v, ov), (g, og))]
    print(core, n, err)
    assert all(f <= 1.05 * d for f, d in zip(err["factored"], err["direct"])), err
