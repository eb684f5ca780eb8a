"""GPU parity of the factored method (Morton order, far tiles through the matrix
cores, near tiles direct) against the oracle, through the C ABI.

Bars (normwise, omega3d_amd.metrics), the same as for the direct kernels:
  * compensated FP32 against the FP64 oracle: max rel <= 1e-6 on ring workloads,
    <= 2e-6 on random clouds;
  * plain FP32: no worse than twice the one-pass direct plain-FP32 kernel's own error
    plus 1e-6 (both sum in FP32 per target; the orders differ; an explicit tile keeps
    the direct kernel from splitting its sources, whose slices add in FP64);
  * the factored and direct methods agree to 2e-6 on every case.
"""
import ctypes as C

import numpy as np
import pytest

import oracle
from omega3d_amd import scenes
from omega3d_amd.metrics import rel_errors, self_term_gradient

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def infl():
    from omega3d_amd import _lib, influence
    assert _lib.lib.o3d_init(-1) == 0, _lib.last_error()
    return influence


def _sel(n, k, seed=3):
    return np.sort(np.random.default_rng(seed).choice(n, size=min(k, n), replace=False))


@pytest.mark.parametrize("core", ["rm", "exp"])
@pytest.mark.parametrize("prec", ["comp", "fp32"])
def test_factored_ring_matches_oracle(infl, core, prec):
    """Two colliding rings, N = 131,072 (the full two-ring geometry at 1/8 size): every
    target evaluated, 2,048 of them checked against the FP64 oracle."""
    p = scenes.colliding_rings(n_each=65536)
    print(f"case: {core} {prec} N={p.n}", flush=True)
    v, g = infl.p2p(core, p.pos, p.str, p.rad, p.pos, p.rad, True, prec, method="factored")
    vd, gd = infl.p2p(core, p.pos, p.str, p.rad, p.pos, p.rad, True, prec, method="direct", tile=512, tpt=1)
    sel = _sel(p.n, 2048)
    ov, og = oracle.p2p(core, p.pos, p.str, p.rad, p.pos[:, sel], p.rad[sel], True, "f64")
    ev, eg = rel_errors(v[:, sel], ov), rel_errors(g[:, sel], og)
    edv, edg = rel_errors(vd[:, sel], ov), rel_errors(gd[:, sel], og)
    print(f"factored vs fp64 vel {ev} grad {eg}; direct vel {edv} grad {edg}")
    if prec == "comp":
        assert ev[0] <= 1e-6 and eg[0] <= 1e-6
        assert rel_errors(v, vd)[0] <= 2e-6 and rel_errors(g, gd)[0] <= 2e-6
    else:
        assert ev[0] <= 2 * edv[0] + 1e-6 and eg[0] <= 2 * edg[0] + 1e-6
    # the far-field path ran: the summation order differs from the direct kernel
    assert not np.array_equal(g, gd)


def test_factored_full_two_rings_subset(infl):
    """The full two-ring workload (N = 1,048,576, EXP, sigma 0.02, compensated) by the
    default method (factored at this size): 512 targets against the FP64 oracle."""
    c = scenes.colliding_rings()
    v, g = infl.p2p("exp", c.pos, c.str, c.rad, c.pos, c.rad, True, "comp")
    sel = np.arange(0, c.n, c.n // 512)[:512]
    ov, og = oracle.p2p("exp", c.pos, c.str, c.rad, c.pos[:, sel], c.rad[sel], True, "f64")
    ev, eg = rel_errors(v[:, sel], ov), rel_errors(g[:, sel], og)
    print("c1 factored comp vs fp64", ev, eg)
    assert ev[0] <= 1e-6 and eg[0] <= 1e-6


@pytest.mark.parametrize("core", ["rm", "exp"])
@pytest.mark.parametrize("thick", [True, False])
def test_factored_separate_targets(infl, core, thick):
    """Targets a different collection from the sources (sorted separately on the
    common box), counts not multiples of the block or tile, point targets."""
    c = scenes.colliding_rings(n_each=40000)
    ns = c.n - 77
    sp, ss, sr = c.pos[:, :ns], c.str[:, :ns], c.rad[:ns]
    tp = scenes.ring(70001, R=1.2, a=0.3, seed=9).pos
    tp[2] += 0.5
    tr = np.full(tp.shape[1], 0.03, np.float32) if thick else None
    print(f"case: {core} thick={thick} ns={ns} nt={tp.shape[1]}", flush=True)
    v, g = infl.p2p(core, sp, ss, sr, tp, tr, True, "comp", method="factored")
    vd, gd = infl.p2p(core, sp, ss, sr, tp, tr, True, "comp", method="direct")
    sel = _sel(tp.shape[1], 1024)
    ov, og = oracle.p2p(core, sp, ss, sr, tp[:, sel], None if tr is None else tr[sel], True, "f64")
    assert rel_errors(v[:, sel], ov)[0] <= 1e-6 and rel_errors(g[:, sel], og)[0] <= 1e-6
    assert rel_errors(v, vd)[0] <= 2e-6 and rel_errors(g, gd)[0] <= 2e-6


@pytest.mark.parametrize("core", ["rm", "exp"])
def test_factored_self_excluded(infl, core):
    p = scenes.colliding_rings(n_each=50000)
    v, g = infl.p2p(core, p.pos, p.str, p.rad, p.pos, p.rad, True, "comp", self_term=1, method="factored")
    sel = _sel(p.n, 1024)
    ov, og = oracle.p2p(core, p.pos, p.str, p.rad, p.pos[:, sel], p.rad[sel], True, "f64")
    og = og - self_term_gradient(core, p.str[:, sel], p.rad[sel])
    assert rel_errors(v[:, sel], ov)[0] <= 1e-6 and rel_errors(g[:, sel], og)[0] <= 1e-6


@pytest.mark.parametrize("n", [1, 2, 63, 257, 1000, 5000])
def test_factored_small_and_ragged(infl, n):
    p = scenes.ring(n, sigma=0.02, seed=n)
    for core in ("rm", "exp"):
        for tile in (64, 128, 256):
            v, g = infl.p2p(core, p.pos, p.str, p.rad, p.pos, p.rad, True, "comp", tile=tile, method="factored")
            ov, og = oracle.p2p(core, p.pos, p.str, p.rad, p.pos, p.rad, True, "f64")
            assert rel_errors(v, ov)[0] <= 2e-6 and rel_errors(g, og)[0] <= 2e-6, (core, tile)


def test_factored_accumulates(infl):
    p = scenes.colliding_rings(n_each=40000)
    v0 = np.random.default_rng(1).normal(size=(3, p.n)).astype(np.float32)
    g0 = np.random.default_rng(2).normal(size=(9, p.n)).astype(np.float32)
    v, g = infl.p2p("rm", p.pos, p.str, p.rad, p.pos, p.rad, True, "comp", vel=v0.copy(), grad=g0.copy(),
                    method="factored")
    vz, gz = infl.p2p("rm", p.pos, p.str, p.rad, p.pos, p.rad, True, "comp", method="factored")
    np.testing.assert_allclose(v, v0 + vz, rtol=1e-6, atol=1e-6 * np.abs(vz).max())
    np.testing.assert_allclose(g, g0 + gz, rtol=1e-6, atol=1e-6 * np.abs(gz).max())


def test_factored_repeatable_and_device_entry(infl):
    """Same bits on repeated calls, through the host and the device entry points."""
    from omega3d_amd import _lib
    p = scenes.colliding_rings(n_each=40000)
    a = infl.p2p("exp", p.pos, p.str, p.rad, p.pos, p.rad, True, "comp", method="factored")
    b = infl.p2p("exp", p.pos, p.str, p.rad, p.pos, p.rad, True, "comp", method="factored")
    np.testing.assert_array_equal(a[0], b[0])
    np.testing.assert_array_equal(a[1], b[1])
    D = _lib.DeviceArray.from_host
    dp, ds, dr = D(p.pos), D(p.str), D(p.rad)
    dv, dg = _lib.DeviceArray((3, p.n)), _lib.DeviceArray((9, p.n))
    dv.zero(); dg.zero()
    s, t = _lib.Points(), _lib.Points()
    s.n = t.n = p.n
    for d in range(3):
        s.x[d] = t.x[d] = dp.row(d)
        s.s[d] = ds.row(d)
        t.u[d] = dv.row(d)
    s.r = t.r = dr.ptr
    for k in range(9):
        t.ug[k] = dg.row(k)
    o = _lib.make_opts("exp", True, "comp", method="factored")
    _lib.check(_lib.lib.o3d_points_affect_points_dev(C.byref(s), C.byref(t), C.byref(o), None))
    _lib.synchronize()
    # one collection on the device (sorted once) vs two host copies (sorted twice):
    # the same permutation, so the same bits
    np.testing.assert_array_equal(dv.to_host(), a[0])
    np.testing.assert_array_equal(dg.to_host(), a[1])


def test_factored_rejects_unsupported(infl):
    from omega3d_amd import _lib
    p = scenes.ring(500)
    for kw in ({"core": "wl"}, {"core": "v2"}, {"precision": "fp64"}, {"tile": 512}, {"grads": False}):
        args = dict(core="rm", precision="comp", tile=0, grads=True)
        args.update(kw)
        with pytest.raises(_lib.O3DError) as ei:
            infl.p2p(args["core"], p.pos, p.str, p.rad, p.pos, p.rad, args["grads"], args["precision"],
                     tile=args["tile"], method="factored")
        assert ei.value.code == 1, kw


def _cloud(kind, n, seed):
    """Random particle clouds other than rings: a uniform unit cube (sigma 0.02, unit
    strengths), or two Gaussian blobs of different widths and core radii whose
    strength magnitudes are log-uniform over 1e-3 .. 1e3."""
    rng = np.random.default_rng(seed)
    if kind == "cube":
        pos = rng.uniform(0.0, 1.0, (3, n))
        st = rng.normal(size=(3, n)) / n
        rad = np.full(n, 0.02)
    else:
        h = n // 2
        pos = np.concatenate([rng.normal(0.0, 0.15, (3, h)), rng.normal(0.0, 0.05, (3, n - h)) + 0.6], 1)
        rad = np.concatenate([np.full(h, 0.03), np.full(n - h, 0.01)])
        d = rng.normal(size=(3, n))
        d /= np.linalg.norm(d, axis=0)
        st = d * 10.0 ** rng.uniform(-3.0, 3.0, n) / n
    return (pos.astype(np.float32), st.astype(np.float32), rad.astype(np.float32))


@pytest.mark.parametrize("core", ["rm", "exp"])
@pytest.mark.parametrize("kind,n", [("cube", 70000), ("blobs", 131072)])
def test_factored_random_clouds(infl, core, kind, n):
    """The factored method (AUTO's choice at these sizes) on clouds where the far test,
    the per-tile power-of-two scales and the split FP16 weights meet other
    geometry than rings: compensated within 2e-6 of the FP64 oracle on 1,024
    targets, plain FP32 within twice the direct kernel's own plain error + 1e-6."""
    pos, st, rad = _cloud(kind, n, 11)
    print(f"case: {core} {kind} N={n}", flush=True)
    sel = _sel(n, 1024)
    ov, og = oracle.p2p(core, pos, st, rad, pos[:, sel], rad[sel], True, "f64")
    v, g = infl.p2p(core, pos, st, rad, pos, rad, True, "comp")
    ev, eg = rel_errors(v[:, sel], ov), rel_errors(g[:, sel], og)
    print(f"factored comp vs fp64: vel {ev} grad {eg}", flush=True)
    assert ev[0] <= 2e-6 and eg[0] <= 2e-6
    vf, gf = infl.p2p(core, pos, st, rad, pos, rad, True, "fp32")
    vd, gd = infl.p2p(core, pos, st, rad, pos, rad, True, "fp32", method="direct", tile=512, tpt=1)
    efv, efg = rel_errors(vf[:, sel], ov), rel_errors(gf[:, sel], og)
    edv, edg = rel_errors(vd[:, sel], ov), rel_errors(gd[:, sel], og)
    print(f"plain: factored vel {efv} grad {efg}; direct vel {edv} grad {edg}", flush=True)
    assert efv[0] <= 2 * edv[0] + 1e-6 and efg[0] <= 2 * edg[0] + 1e-6
    assert not np.array_equal(g, infl.p2p(core, pos, st, rad, pos, rad, True, "comp", method="direct")[1])


@pytest.mark.parametrize("core", ["rm", "exp"])
@pytest.mark.parametrize("n", [2049, 30011])
def test_factored_negation_and_zero_strengths(infl, core, n):
    """Negating every strength negates every result exactly (the far field takes all
    strengths times the sign of the first nonzero one), and whole tiles of particles with
    no strength, in sorted order, add nothing: compensated within 2e-6 of the oracle."""
    p = scenes.colliding_rings(n_each=(n + 1) // 2, sigma=0.03, seed=n)
    st = p.str * (p.pos[2] > -1.02)      # the lower part of one ring: no strength
    print(f"case: {core} N={p.n}", flush=True)
    call = lambda s: infl.p2p(core, p.pos, s, p.rad, p.pos, p.rad, True, "comp", method="factored")
    v, g = call(st)
    vn, gn = call(-st)
    assert np.array_equal(vn, -v) and np.array_equal(gn, -g)
    sel = _sel(p.n, 512)
    ov, og = oracle.p2p(core, p.pos, st, p.rad, p.pos[:, sel], p.rad[sel], True, "f64")
    assert rel_errors(v[:, sel], ov)[0] <= 2e-6 and rel_errors(g[:, sel], og)[0] <= 2e-6


@pytest.mark.parametrize("core,grads", [("wl", True), ("v2", True), ("rm", False), ("wl", False), ("exp", False),
                                        ("v2", False)])
@pytest.mark.parametrize("ns,nt", [(65536, 65536), (66001, 70017)])
def test_auto_takes_far_tiles_of_other_cores_and_velocities(infl, core, grads, ns, nt):
    """AUTO at 65,536 and more, compensated: the two-weight form (WL, V2 with gradient) and
    the velocity form, on one collection with varied core radii and on point targets of
    another: within 2e-6 of the oracle and of the direct method, other bits than the
    direct method's, and the self pair left out where asked."""
    same = ns == nt
    c = scenes.colliding_rings(n_each=(ns + 1) // 2, sigma=0.03)
    rad = (c.rad * np.linspace(0.7, 1.3, c.n)[np.random.default_rng(2).permutation(c.n)]).astype(np.float32)[:ns]
    pos, st = c.pos[:, :ns], c.str[:, :ns]
    tp = pos if same else scenes.ring(nt, R=1.2, a=0.4, seed=9).pos
    tr = rad if same else None
    print(f"case: {core} grads={grads} ns={ns} nt={nt}", flush=True)
    args = (core, pos, st, rad, tp, tr, grads, "comp")
    v, g = infl.p2p(*args, self_term=int(same))
    vd, gd = infl.p2p(*args, self_term=int(same), method="direct")
    sel = _sel(tp.shape[1], 512)
    ov, og = oracle.p2p(core, pos, st, rad, tp[:, sel], None if tr is None else tr[sel], grads, "f64")
    assert rel_errors(v[:, sel], ov)[0] <= 2e-6 and rel_errors(v, vd)[0] <= 2e-6
    assert not np.array_equal(v, vd)
    if grads:
        if same:
            og = og - self_term_gradient(core, st[:, sel], rad[sel])
        assert rel_errors(g[:, sel], og)[0] <= 2e-6 and rel_errors(g, gd)[0] <= 2e-6
