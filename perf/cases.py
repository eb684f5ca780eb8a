"""The work that a user of the library has it do, as measurable cases.

Six kinds of call, each through the library's public entry points on arrays that a
program would hold (torch tensors on the GPU, numpy arrays for the host calls):

  points      o3d_points_affect_points_dev, or external_vel_solver_f_ on host arrays:
              a particle collection acting on itself (vortex rings, ring pairs) or on
              inert field points
  panels      o3d_panels_affect_points_dev: a sphere's vortex (and source) sheets
              acting on points around it, recursive or 7-point rule
  bem_rhs     o3d_bem_rhs_dev: the right-hand side of a sphere's boundary elements from
              the particles around it
  bem_matrix  o3d_bem_matrix_dev: the sphere's influence matrix on itself
  batch       o3d_batch_run: independent rings evaluated together
  server      one RK2 step of every session of a server, and their states read back

Inputs are made from the seed alone.  exact() gives the sums in 64 bits from plain
torch, with the tree decisions of the panel rules taken in float as they are defined.
"""
import ctypes as C
import math

import numpy as np
import torch

from omega3d_amd import _lib, batch as _batch, influence, serve
from omega3d_amd.scenes import Particles

lib, check = _lib.lib, _lib.check
DEV = "cuda"
F64 = torch.float64
CORES = ("rm", "wl", "exp", "v2")
EXACT_PAIRS = 1.2e11   # exact() gives nothing beyond this many point pairs (about 20 s)


def listed():
    return [
        # the smallest session: one ring, every call waits for its launches
        {"name": "ring_rm_1024", "kind": "points", "core": "rm", "rings": 1, "ns": 1024, "nt": 0, "grad": True,
         "precision": "comp", "self_term": 0, "varied": False, "host": False},
        # the single ring of 8,192 particles, plain FP32, self term excluded
        {"name": "ring_rm_8192_fp32", "kind": "points", "core": "rm", "rings": 1, "ns": 8192, "nt": 0, "grad": True,
         "precision": "fp32", "self_term": 1, "varied": False, "host": False},
        # the default core and options on a simulation of ordinary size, radii as they vary in a run, ragged count
        {"name": "rings_wl_131071", "kind": "points", "core": "wl", "rings": 2, "ns": 131071, "nt": 0, "grad": True,
         "precision": "comp", "self_term": 0, "varied": True, "host": False},
        # the two colliding rings of 1,048,576 particles, the largest collection
        {"name": "rings_exp_1048576", "kind": "points", "core": "exp", "rings": 2, "ns": 1048576, "nt": 0, "grad": True,
         "precision": "comp", "self_term": 0, "varied": False, "host": False},
        # an existing program that links the external-solver symbol: host arrays in and out
        {"name": "plugin_wl_30000", "kind": "points", "core": "wl", "rings": 2, "ns": 30000, "nt": 30000, "grad": True,
         "precision": "comp", "self_term": 0, "varied": False, "host": True},
        # tracers and measurement points: velocity only at inert points
        {"name": "tracers_rm_100003", "kind": "points", "core": "rm", "rings": 2, "ns": 100003, "nt": 65537,
         "grad": False, "precision": "comp", "self_term": 0, "varied": False, "host": False},
        # the 20,480-panel sphere acting on 524,288 points around it
        {"name": "sphere_points", "kind": "panels", "rule": "auto", "np": 20480, "nt": 524288, "grad": True,
         "precision": "comp", "sources": False},
        # the 7-point rule, vortex and source sheets, a smaller sphere and a ragged count
        {"name": "sphere_gauss7", "kind": "panels", "rule": "gauss7", "np": 5120, "nt": 200003, "grad": True,
         "precision": "comp", "sources": True},
        # the right-hand side of the sphere's boundary elements from 524,288 particles
        {"name": "sphere_bem_rhs", "kind": "bem_rhs", "np": 20480, "ns": 524288, "nunk": 3, "precision": "comp"},
        # a sphere's influence matrix, 15,360 x 15,360
        {"name": "sphere_bem_matrix", "kind": "bem_matrix", "np": 5120, "nunk": 3},
        # an ensemble of independent rings
        {"name": "batch_48_rings", "kind": "batch", "core": "rm", "count": 48, "lo": 2048, "hi": 81920,
         "precision": "comp"},
        # a server's sessions stepped together
        {"name": "server_8_sessions", "kind": "server", "count": 8, "lo": 1024, "hi": 100000},
    ]


def _between(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))


def draw(rng):
    kind = rng.choice(["points"] * 5 + ["panels"] * 2 + ["bem_rhs", "bem_matrix", "batch", "server"])
    if kind == "points":
        core = rng.choice(CORES)
        ns = _between(rng, 1024, 524288 if core in ("rm", "exp") else 300000)
        field = rng.random() < 0.35
        nt = min(_between(rng, 257, 262144), int(1e11 / ns)) if field else 0
        host = not field and ns < 60000 and rng.random() < 0.3
        small = ns <= 32768 and not field
        return {"kind": kind, "core": "wl" if host else core, "rings": rng.choice([1, 2]), "ns": ns,
                "nt": ns if host else nt, "grad": host or not field or rng.random() < 0.4,
                # plain FP32 sums are for previews of small collections
                "precision": "fp32" if small and not host and rng.random() < 0.4 else "comp",
                "self_term": 0 if field or host else rng.choice([0, 1]), "varied": rng.random() < 0.5, "host": host}
    if kind == "panels":
        rule = rng.choice(["auto", "gauss7"])
        np_ = _between(rng, 300, 20480 if rule == "auto" else 8000)
        return {"kind": kind, "rule": rule, "np": np_, "nt": _between(rng, 1000, 524288 if rule == "auto" else 262144),
                "grad": rng.random() < 0.8, "precision": "fp32" if np_ < 4096 and rng.random() < 0.4 else "comp",
                "sources": rng.random() < 0.4}
    if kind == "bem_rhs":
        return {"kind": kind, "np": _between(rng, 300, 20480), "ns": _between(rng, 2000, 524288),
                "nunk": rng.choice([1, 2, 3]), "precision": "comp"}
    if kind == "bem_matrix":
        return {"kind": kind, "np": _between(rng, 300, 8000), "nunk": rng.choice([2, 3])}
    if kind == "batch":
        lo = _between(rng, 1024, 8192)
        return {"kind": kind, "core": rng.choice(["rm", "wl", "exp"]), "count": _between(rng, 8, 64), "lo": lo,
                "hi": _between(rng, 2 * lo, 98304), "precision": "comp"}
    return {"kind": kind, "count": _between(rng, 2, 12), "lo": _between(rng, 1024, 4096),
            "hi": _between(rng, 8192, 131072)}


# ---- inputs ---------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=F64)


def _torus(g, n, R, a):
    """n points uniform in a torus around the z axis, and the unit tangents there"""
    got, have = [], 0
    while have < n:
        m = int((n - have) * 1.2) + 64
        r, ph, th = a * _uniform(g, m).sqrt(), 2 * math.pi * _uniform(g, m), 2 * math.pi * _uniform(g, m)
        rho = R + r * torch.cos(ph)
        keep = _uniform(g, m) * (R + a) < rho
        got.append(torch.stack([rho * torch.cos(th), rho * torch.sin(th), r * torch.sin(ph), -torch.sin(th),
                                torch.cos(th)])[:, keep])
        have += got[-1].shape[1]
    v = torch.cat(got, 1)[:, :n]
    return v[:3], torch.cat([v[3:5], torch.zeros_like(v[:1])])


def _rings(g, rings, n, sigma, R=1.0, varied=False):
    """one ring, or two of opposite circulation at z = 1 and z = -1 with the second tilted
    by 15 degrees: position (3, n), strength (3, n) and core radius (n,) in float"""
    parts = []
    for k in range(rings):
        nk = n // rings + (n % rings if k == 0 else 0)
        pos, tan = _torus(g, nk, R, 0.1)
        s = tan * ((1.0 + 0.05 * (2 * _uniform(g, nk) - 1)) / nk)
        if rings == 2:
            if k == 1:
                c, w = math.cos(math.radians(15)), math.sin(math.radians(15))
                tilt = torch.tensor([[1, 0, 0], [0, c, -w], [0, w, c]], dtype=F64, device=DEV)
                pos, s = tilt @ pos, -(tilt @ s)
            pos[2] += 1.0 - 2.0 * k
        parts.append((pos, s))
    rad = torch.full((n,), sigma, dtype=F64, device=DEV)
    if varied:
        rad = rad * (0.7 + 0.6 * _uniform(g, n))
    return [torch.cat(x, 1).float().contiguous() for x in zip(*parts)] + [rad.float()]


def _shell(g, n):
    """n points uniform in the shell 1.02 < r < 1.5"""
    r = (1.02 ** 3 + _uniform(g, n) * (1.5 ** 3 - 1.02 ** 3)) ** (1.0 / 3.0)
    z, ph = 2 * _uniform(g, n) - 1, 2 * math.pi * _uniform(g, n)
    s = (1 - z * z).clamp_min(0).sqrt()
    return torch.stack([r * s * torch.cos(ph), r * s * torch.sin(ph), r * z]).float().contiguous()


def _sphere(panels):
    """the first `panels` panels of the coarsest icosphere that has as many: nodes (3, nn)
    in float64 and node indices (panels, 3), outward"""
    t = (1 + math.sqrt(5)) / 2
    v = np.array([(-1, t, 0), (1, t, 0), (-1, -t, 0), (1, -t, 0), (0, -1, t), (0, 1, t), (0, -1, -t), (0, 1, -t),
                  (t, 0, -1), (t, 0, 1), (-t, 0, -1), (-t, 0, 1)], float) / math.sqrt(1 + t * t)
    f = np.array([(0, 11, 5), (0, 5, 1), (0, 1, 7), (0, 7, 10), (0, 10, 11), (1, 5, 9), (5, 11, 4), (11, 10, 2),
                  (10, 7, 6), (7, 1, 8), (3, 9, 4), (3, 4, 2), (3, 2, 6), (3, 6, 8), (3, 8, 9), (4, 9, 5), (2, 4, 11),
                  (6, 2, 10), (8, 6, 7), (9, 8, 1)])
    while len(f) < panels:
        e = np.sort(np.concatenate([f[:, [0, 1]], f[:, [1, 2]], f[:, [2, 0]]]), 1)
        u, inv = np.unique(e[:, 0] * len(v) + e[:, 1], return_inverse=True)
        m = v[u // len(v)] + v[u % len(v)]
        ab, bc, ca = (inv + len(v)).reshape(3, -1)
        v = np.concatenate([v, m / np.linalg.norm(m, axis=1)[:, None]])
        a, b, c = f.T
        f = np.stack([np.stack(x, 1) for x in ((a, ab, ca), (b, bc, ab), (c, ca, bc), (ab, bc, ca))], 1).reshape(-1, 3)
    return v.T, f[:panels]


def _surface(panels):
    """nodes, node indices, areas and the in-plane basis x1, x2, normal of each panel, on the GPU"""
    v, f = _sphere(panels)
    nodes = torch.tensor(v, device=DEV).float().contiguous()
    idx = torch.tensor(f, device=DEV)
    p = nodes.double().T[idx]
    e1, e2 = p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
    b = e1.norm(dim=1, keepdim=True)
    x1 = e1 / b
    e2 = e2 - (e2 * x1).sum(1, keepdim=True) * x1
    h = e2.norm(dim=1, keepdim=True)
    x2 = e2 / h
    return {"nodes": nodes, "idx": idx, "idx32": idx.int().contiguous(), "area": (0.5 * b * h)[:, 0].float().contiguous(),
            "x1": x1, "x2": x2, "nm": torch.linalg.cross(x1, x2)}


def _sheets(g, s, sources):
    """absolute vortex strength (3, n) of a random in-plane sheet and a source sheet (n,) or None"""
    n = len(s["area"])
    gam = torch.randn(n, 3, generator=g, device=DEV, dtype=F64)
    gam = gam - (gam * s["nm"]).sum(1, keepdim=True) * s["nm"]
    ts = (gam * s["area"].double()[:, None]).T.float().contiguous()
    return ts, torch.randn(n, generator=g, device=DEV) if sources else None


def _point_inputs(case, seed):
    g = _generator(seed)
    pos, s, r = _rings(g, case["rings"], case["ns"], 0.02 if case["core"] == "exp" else 0.05, varied=case["varied"])
    if not case["nt"]:
        return pos, s, r, pos, r
    if case["host"]:
        return pos, s, r, pos, None
    box = torch.tensor([[1.5], [1.5], [1.5]], dtype=F64, device=DEV)
    return pos, s, r, ((2 * _uniform(g, 3, case["nt"]) - 1) * box).float().contiguous(), None


def _panel_inputs(case, seed):
    g = _generator(seed)
    s = _surface(case["np"])
    return (s,) + _sheets(g, s, case["sources"]) + (_shell(g, case["nt"]),)


def _rhs_inputs(case, seed):
    g = _generator(seed)
    pos = _shell(g, case["ns"])
    return _surface(case["np"]), pos, ((2 * _uniform(g, 3, case["ns"]) - 1) / case["ns"]).float().contiguous()


def _matrix_inputs(case, seed):
    """the sphere stretched to a body of its own for each seed"""
    v, f = _sphere(case["np"])
    scale = 0.8 + 0.4 * _uniform(_generator(seed), 3)
    s = _surface(case["np"])
    nodes = (torch.tensor(v, device=DEV) * scale[:, None]).float().contiguous()
    p = nodes.double().T[s["idx"]]
    s["nodes"] = nodes
    s["area"] = (0.5 * torch.linalg.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]).norm(dim=1)).float().contiguous()
    e1, e2 = p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
    s["x1"] = e1 / e1.norm(dim=1, keepdim=True)
    e2 = e2 - (e2 * s["x1"]).sum(1, keepdim=True) * s["x1"]
    s["x2"] = e2 / e2.norm(dim=1, keepdim=True)
    s["nm"] = torch.linalg.cross(s["x1"], s["x2"])
    return s


def _counts(case):
    """log-spread counts between lo and hi, the same for every seed"""
    r = math.log(case["hi"] / case["lo"])
    return [int(case["lo"] * math.exp(r * ((0.5 + 0.6180339887498949 * i) % 1.0))) for i in range(case["count"])]


def _batch_inputs(case, seed):
    g = _generator(seed)
    out = []
    for n in _counts(case):
        R, sigma = (_uniform(g, 2) * torch.tensor([1.5, 0.04], dtype=F64, device=DEV)).tolist()
        out.append(_rings(g, 1, n, 0.01 + sigma, R=0.5 + R))
    return out


def _session_inputs(case, seed):
    """ring pairs (EXP) and single rings (RM, and the default core WL for small ones) in turn"""
    g = _generator(seed)
    out = []
    for i, n in enumerate(_counts(case)):
        core = "exp" if i % 2 else "wl" if n < 16384 and i % 4 == 0 else "rm"
        out.append((core,) + tuple(_rings(g, 2 if core == "exp" else 1, n, 0.02 if core == "exp" else 0.05)))
    return out


# ---- the calls ------------------------------------------------------------------


class _Batch:
    """a batch handle, released with the state that holds it"""

    def __init__(self, counts, opts):
        n = np.array(counts, np.int64)
        off = np.concatenate([[0], np.cumsum(n)[:-1]]).astype(np.int64)
        h = C.c_void_p()
        check(lib.o3d_batch_create(C.byref(h), len(n), off.ctypes.data, n.ctypes.data, None, None, None, C.byref(opts)))
        self.h = h.value

    def __del__(self):
        _batch.lib.o3d_batch_destroy(self.h)


def _points(pos, s=None, r=None, vel=None, grad=None):
    p = _lib.Points()
    p.n = pos.shape[1]
    for d in range(3):
        p.x[d] = pos[d].data_ptr()
        if s is not None:
            p.s[d] = s[d].data_ptr()
        if vel is not None:
            p.u[d] = vel[d].data_ptr()
    p.r = None if r is None else r.data_ptr()
    if grad is not None:
        for k in range(9):
            p.ug[k] = grad[k].data_ptr()
    return p


def _panels(s, ts=None, ss=None):
    p = _lib.Panels()
    p.np, p.nn = len(s["area"]), s["nodes"].shape[1]
    for d in range(3):
        p.x[d] = s["nodes"][d].data_ptr()
        if ts is not None:
            p.ts[d] = ts[d].data_ptr()
    p.idx, p.area, p.ss = s["idx32"].data_ptr(), s["area"].data_ptr(), None if ss is None else ss.data_ptr()
    return p


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind, "case": case}
    if kind == "points":
        pos, s, r, tpos, tr = _point_inputs(case, seed)
        st["grad"] = case["grad"]
        if case["host"]:
            st["host"] = [x.cpu().numpy() for x in (pos, s, r, tpos)]
            st["vel"], st["dvel"] = np.zeros((3, case["nt"]), np.float32), np.zeros((9, case["nt"]), np.float32)
            return st
        st["out"] = torch.zeros(12 if case["grad"] else 3, tpos.shape[1], device=DEV)
        st["src"] = _points(pos, s, r)
        st["targ"] = _points(tpos, None, tr, st["out"], st["out"][3:] if case["grad"] else None)
        st["opts"] = _lib.make_opts(case["core"], case["grad"], case["precision"], self_term=case["self_term"])
        st["keep"] = (pos, s, r, tpos, tr)
    elif kind == "panels":
        s, ts, ss, tpos = _panel_inputs(case, seed)
        st["out"] = torch.zeros(12 if case["grad"] else 3, case["nt"], device=DEV)
        st["src"] = _panels(s, ts, ss)
        st["targ"] = _points(tpos, None, None, st["out"], st["out"][3:] if case["grad"] else None)
        st["opts"] = _lib.make_opts("rm", case["grad"], case["precision"], method=case["rule"])
        st["keep"] = (s, ts, ss, tpos)
    elif kind == "bem_rhs":
        s, pos, a = _rhs_inputs(case, seed)
        st["pu"] = torch.zeros(3, case["np"], device=DEV)
        st["rhs"] = torch.zeros(case["nunk"] * case["np"], device=DEV)
        st["src"], st["targ"] = (_lib.Points * 1)(_points(pos, a)), _panels(s)
        st["vel"] = (C.c_void_p * 3)(*[st["pu"][d].data_ptr() for d in range(3)])
        st["opts"], st["bem"] = _lib.make_opts("rm", False, case["precision"]), influence.bem_opts((1.0, 0.0, 0.0),
                                                                                                   nunk=case["nunk"])
        st["keep"] = (s, pos, a)
    elif kind == "bem_matrix":
        s = _matrix_inputs(case, seed)
        rows = case["nunk"] * case["np"]
        st["out"] = torch.zeros(rows, rows, device=DEV)
        st["src"], st["keep"] = _panels(s), s
    elif kind == "batch":
        parts = _batch_inputs(case, seed)
        pos, s, r = (torch.cat(x, -1).contiguous() for x in zip(*parts))
        st["out"] = torch.zeros(12, pos.shape[1], device=DEV)
        st["src"] = _points(pos, s, r, st["out"], st["out"][3:])
        st["batch"] = _Batch([p[2].shape[0] for p in parts], _lib.make_opts(case["core"], True, case["precision"]))
        st["keep"] = (pos, s, r)
    else:
        st["server"] = serve.Server(hbm_budget=2 << 30)
        st["ids"] = [st["server"].open_session(Particles(*[x.cpu().numpy() for x in p[1:]]), p[0])
                     for p in _session_inputs(case, seed)]
    return st


def run(st):
    kind = st["kind"]
    if kind == "points":
        if "host" in st:
            pos, s, r, tpos = st["host"]
            st["vel"][:] = 0
            st["dvel"][:] = 0
            if influence.external_vel_solver_f(pos, s, r, tpos, st["vel"], st["dvel"]) < 0:
                raise RuntimeError(_lib.last_error())
            return st["vel"], st["dvel"]
        st["out"].zero_()
        check(lib.o3d_points_affect_points_dev(C.byref(st["src"]), C.byref(st["targ"]), C.byref(st["opts"]), None))
        return (st["out"][:3], st["out"][3:]) if st["grad"] else st["out"]
    if kind == "panels":
        st["out"].zero_()
        check(lib.o3d_panels_affect_points_dev(C.byref(st["src"]), C.byref(st["targ"]), C.byref(st["opts"]), None))
        return (st["out"][:3], st["out"][3:]) if st["case"]["grad"] else st["out"]
    if kind == "bem_rhs":
        check(lib.o3d_bem_rhs_dev(st["src"], 1, C.byref(st["targ"]), C.byref(st["bem"]), C.byref(st["opts"]), st["vel"],
                                  C.c_void_p(st["rhs"].data_ptr())))
        return st["pu"], st["rhs"]
    if kind == "bem_matrix":
        check(lib.o3d_bem_matrix_dev(C.byref(st["src"]), C.byref(st["src"]), st["case"]["nunk"], 1, -1,
                                     C.c_void_p(st["out"].data_ptr()), None))
        return st["out"]
    if kind == "batch":
        check(_batch.lib.o3d_batch_run(st["batch"].h, C.byref(st["src"]), None))
        return st["out"][:3], st["out"][3:]
    srv = st["server"]
    for rid in [srv.submit(i, 1e-3) for i in st["ids"]]:
        if srv.wait(rid)["state"] != "done":
            raise RuntimeError(_lib.last_error())
    return [srv.read_session(i) for i in st["ids"]]


def work(case):
    """bytes: every input read and every output written once; flops: the count that the
    library reports for a pair (o3d_flops_per_interaction), twice for the two stages of a step"""
    kind = case["kind"]
    thick = {"rm": 63, "wl": 70, "exp": 68, "v2": 67}
    if kind == "points":
        nt, rows = case["nt"] or case["ns"], 12 if case["grad"] else 3
        f = {"rm": 61, "wl": 68, "exp": 65, "v2": 64}[case["core"]] if case["nt"] else thick[case["core"]]
        f = f if case["grad"] else {"rm": 28, "wl": 31, "exp": 32, "v2": 31}[case["core"]]
        return {"bytes": 28.0 * case["ns"] + (16.0 + 4 * rows) * nt, "flops": nt * (rows + float(f) * case["ns"])}
    if kind == "panels":
        f = (86 if case["grad"] else 34) * (7 if case["rule"] == "gauss7" else 1)
        return {"bytes": 36.0 * case["np"] + (12.0 + (48 if case["grad"] else 12)) * case["nt"],
                "flops": float(f) * case["np"] * case["nt"]}
    if kind == "bem_rhs":
        return {"bytes": 24.0 * case["ns"] + (20.0 + 12 + 4 * case["nunk"]) * case["np"],
                "flops": 34.0 * case["np"] * case["ns"]}
    if kind == "bem_matrix":
        # per pair: the separation and 1/r^3 (14), a vector per unknown (9) and its projections (5 each)
        u = case["nunk"]
        return {"bytes": 4.0 * (u * case["np"]) ** 2, "flops": case["np"] ** 2 * (14.0 + 9 * u + 5 * u * u)}
    n = np.array(_counts(case), float)
    if kind == "batch":
        return {"bytes": float(76 * n.sum()), "flops": float((n * (12 + thick[case["core"]] * n)).sum())}
    f = np.array([68 if i % 2 else 70 if m < 16384 and i % 4 == 0 else 63 for i, m in enumerate(n)])
    return {"bytes": float(60 * n.sum()), "flops": float((2 * n * (12 + f * n)).sum())}


# ---- the same in 64 bits --------------------------------------------------------

CHUNK = 1 << 26   # pairs evaluated at once


def _core64(core, d2, a, b, grad):
    """K and B of the pairs with squared distance d2, source radii a (1, n) and target radii b (n, 1) or 0"""
    if core in ("rm", "wl"):
        r2 = a * a + b * b
        dd = d2 + r2
        if core == "rm":
            K = 1.0 / (dd * dd.sqrt())
            return K, -3.0 * K / dd if grad else None
        top, n5 = d2 + 2.5 * r2, 1.0 / (dd * dd * dd.sqrt())
        return top * n5, 2.0 * n5 - 5.0 * top * n5 / dd if grad else None
    if core == "v2":
        q = (d2 * d2 + a ** 4 + b ** 4).sqrt()
        K = 1.0 / (q * q.sqrt())
        return K, -3.0 * K / q if grad else None
    dist = d2.sqrt()
    c = 1.0 / (a ** 3 + b ** 3)
    q = d2 * dist * c
    o3 = 1.0 / (d2 * dist)
    e = torch.exp(-q)
    near = q < float(np.float32(0.001))
    K = torch.where(q > 16.0, o3, torch.where(near, c, -o3 * torch.expm1(-q)))
    if not grad:
        return K, None
    return K, torch.where(q > 16.0, -3.0 * K / d2, torch.where(near, -1.5 * dist * K * K, 3.0 * (c * e - K) / d2))


def _moments(x, a, gs=None):
    """per source: the columns that K multiplies and those that B multiplies"""
    m = torch.linalg.cross(a, x)
    k = [a, m]
    b = [a, m] + [x[:, j:j + 1] * a for j in range(3)] + [x[:, j:j + 1] * m for j in range(3)]
    if gs is not None:
        g = gs[:, None]
        k += [g, g * x]
        b += [g, g * x] + [g * x[:, j:j + 1] * x for j in range(3)]
    return torch.cat(k, 1), torch.cat(b, 1)


def _from_moments(t, k, b, sheet, drop=None):
    """velocity (3, n) and gradient (9, n) or None from the sums over the sources of K and B times
    their columns; drop: a part of sum K a to leave out of the gradient"""
    W, M = k[:, :3], k[:, 3:6]
    u = torch.linalg.cross(W, t) - M
    if sheet:
        u = u + t * k[:, 6:7] - k[:, 7:10]
    if b is None:
        return u.T, None
    W = W if drop is None else W - drop
    g = torch.zeros(t.shape[0], 3, 3, dtype=F64, device=DEV)
    P, Q = b[:, :3], b[:, 3:6]
    pt = torch.linalg.cross(P, t)
    for j in range(3):
        R, S = b[:, 6 + 3 * j:9 + 3 * j], b[:, 15 + 3 * j:18 + 3 * j]
        g[:, j] = t[:, j:j + 1] * (pt - Q) - torch.linalg.cross(R, t) + S
        if sheet:
            G, X, XX = b[:, 24:25], b[:, 25:28], b[:, 28 + 3 * j:31 + 3 * j]
            g[:, j] += t[:, j:j + 1] * t * G - t[:, j:j + 1] * X - t * X[:, j:j + 1] + XX
            g[:, j, j] += k[:, 6]
    for j, i, c, sign in ((0, 1, 2, 1), (0, 2, 1, -1), (1, 0, 2, -1), (1, 2, 0, 1), (2, 0, 1, 1), (2, 1, 0, -1)):
        g[:, j, i] += sign * W[:, c]
    return u.T, g.reshape(-1, 9).T


def _point_sums(core, pos, s, r, tpos, tr, grad, self_excl):
    x, a, sr, t = pos.double().T, s.double().T, r.double(), tpos.double().T
    kc, bc = _moments(x, a)
    us, gs = [], []
    step = max(1, CHUNK // x.shape[0])
    for i in range(0, t.shape[0], step):
        ti = t[i:i + step]
        d2 = sum((ti[:, d:d + 1] - x[None, :, d]) ** 2 for d in range(3))
        b = 0.0 if tr is None else tr[i:i + step].double()[:, None]
        K, B = _core64(core, d2, sr[None, :], b, grad)
        drop = None
        if self_excl and grad:
            sri = sr[i:i + step]
            K0 = _core64(core, torch.zeros_like(sri), sri, 0.0 if tr is None else tr[i:i + step].double(), False)[0]
            drop = K0[:, None] * a[i:i + step]
        u, g = _from_moments(ti, K @ kc, B @ bc if grad else None, False, drop)
        us.append(u)
        gs.append(g)
    return torch.cat(us, 1), torch.cat(gs, 1) if grad else None


def _dist32(t, c):
    e = t - c
    return (e[..., 0] * e[..., 0] + e[..., 1] * e[..., 1] + e[..., 2] * e[..., 2]).sqrt()


CHILD = ((0, 1, 3), (1, 2, 4), (1, 4, 3), (3, 4, 5))


def _children(v):
    """the four child triangles (n, 4, 3, 3) of triangles v (n, 3, 3), in v's own type"""
    n = torch.stack([v[:, 0], 0.5 * (v[:, 0] + v[:, 1]), v[:, 1], 0.5 * (v[:, 0] + v[:, 2]), 0.5 * (v[:, 1] + v[:, 2]),
                     v[:, 2]], 1)
    return n[:, torch.tensor(CHILD, device=DEV)]


def _centroid(v):
    return (v[..., 0, :] + v[..., 1, :] + v[..., 2, :]) / 3


def _scatter_pairs(u, g, at, d, ga, gs):
    """adds the singular leaves with separation d (n, 3) and strengths ga (n, 3), gs (n,) to u (n, 3) and g (n, 9)"""
    d2 = (d * d).sum(1)
    K = 1.0 / (d2 * d2.sqrt())
    c = torch.linalg.cross(ga, d) + gs[:, None] * d
    u.index_add_(0, at, K[:, None] * c)
    if g is None:
        return
    m = (-3.0 * K / d2)[:, None, None] * d[:, :, None] * c[:, None, :]
    for j, i, k, sign in ((0, 1, 2, 1), (0, 2, 1, -1), (1, 0, 2, -1), (1, 2, 0, 1), (2, 0, 1, 1), (2, 1, 0, -1)):
        m[:, j, i] += sign * K * ga[:, k]
    for j in range(3):
        m[:, j, j] += K * gs
    g.index_add_(0, at, m.reshape(-1, 9))


def _tree_sums(s, ts, ss, tpos, grad, flip=False):
    """the recursive centroid rule, depth 3: panels on points, or with flip the points' strengths ts
    (3, points) on the panels: velocity (3, n) and gradient (9, n) or None"""
    v32 = s["nodes"].T[s["idx"]]
    v = v32.double()
    c32, c, area = _centroid(v32), _centroid(v), s["area"]
    lim = area.sqrt() * 4
    t32, t, a = tpos.T.contiguous(), tpos.double().T.contiguous(), ts.double().T
    sheet = ss is not None
    gs = ss.double() * area.double() if sheet else torch.zeros(len(area), dtype=F64, device=DEV)
    if not flip:
        kc, bc = _moments(c, a, gs if sheet else None)
    n = len(area) if flip else t.shape[0]
    u, g = torch.zeros(n, 3, dtype=F64, device=DEV), torch.zeros(n, 9, dtype=F64, device=DEV) if grad else None
    step = max(1, CHUNK // len(area))
    for i in range(0, t.shape[0], step):
        ti, ti32 = t[i:i + step], t32[i:i + step]
        e = [ti32[:, d:d + 1] - c32[None, :, d] for d in range(3)]
        near = ~((e[0] * e[0] + e[1] * e[1] + e[2] * e[2]).sqrt() > lim[None, :])
        d2 = sum((ti[:, d:d + 1] - c[None, :, d]) ** 2 for d in range(3))
        K = (1.0 / (d2 * d2.sqrt())).masked_fill_(near, 0.0)
        if flip:
            # sum over the particles of K (a x (x - c))
            x, ai = ti, a[i:i + step]
            u += K.T @ torch.linalg.cross(ai, x) - torch.linalg.cross(K.T @ ai, c)
        else:
            ui, gi = _from_moments(ti, K @ kc, (-3.0 * K / d2).masked_fill_(near, 0.0) @ bc if grad else None, sheet)
            u[i:i + step] += ui.T
            if grad:
                g[i:i + step] += gi.T
        at, pj = near.nonzero(as_tuple=True)
        at = at + i
        w32, w = v32[pj], v[pj]
        for lev in range(1, 4):
            at, pj = at.repeat_interleave(4), pj.repeat_interleave(4)
            w32, w = _children(w32).reshape(-1, 3, 3), _children(w).reshape(-1, 3, 3)
            share = 0.25 ** lev
            leaf = _dist32(t32[at], _centroid(w32)) > (area[pj] * share).sqrt() * 4
            leaf = leaf | (lev == 3)
            k = leaf.nonzero()[:, 0]
            d = t[at[k]] - _centroid(w[k])
            ga = (a[at[k]] if flip else a[pj[k]]) * share
            _scatter_pairs(u, g, pj[k] if flip else at[k], d, ga, gs[pj[k]] * share)
            k = (~leaf).nonzero()[:, 0]
            at, pj, w32, w = at[k], pj[k], w32[k], w[k]
    return u.T, g.T if grad else None


def _triangle_integrals(v, x):
    """I = int (x - y)/|x - y|^3 over the triangles v (n, 3, 3), and dI[:, j] = dI/dx_j"""
    n = torch.linalg.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0])
    n = n / n.norm(dim=1, keepdim=True)
    R = v - x[:, None]
    r = R.norm(dim=2)
    dot = lambda a, b: (a * b).sum(1)   # noqa: E731
    num = dot(R[:, 0], torch.linalg.cross(R[:, 1], R[:, 2]))
    den = r.prod(1) + dot(R[:, 0], R[:, 1]) * r[:, 2] + dot(R[:, 0], R[:, 2]) * r[:, 1] + dot(R[:, 1], R[:, 2]) * r[:, 0]
    I = -2.0 * torch.atan2(num, den)[:, None] * n
    dI = torch.zeros(len(v), 3, 3, dtype=F64, device=DEV)
    for k in range(3):
        a, b = v[:, k], v[:, (k + 1) % 3]
        length = (b - a).norm(dim=1, keepdim=True)
        t = (b - a) / length
        m = torch.linalg.cross(t, n)
        s = dot(x - a, t)
        um, up = -s, length[:, 0] - s
        q = (x - a) - s[:, None] * t
        q2, rm, rp = dot(q, q), r[:, k], r[:, (k + 1) % 3]
        f = torch.where(um >= 0, torch.log((rp + up) / (rm + um)),
                        torch.where(up <= 0, torch.log((rm - um) / (rp - up)), torch.log((rp + up) * (rm - um) / q2)))
        I = I + m * f[:, None]
        c = torch.where(um * up > 0, (up * up - um * um) / (rp * rm * (up * rm + um * rp)), (up / rp - um / rm) / q2)
        df = -(q * c[:, None] + t * (1.0 / rp - 1.0 / rm)[:, None])
        dI = dI + df[:, :, None] * m[:, None, :] - (torch.linalg.cross(t, q) * c[:, None])[:, :, None] * n[:, None, :]
    return I, dI


def _gauss7_sums(s, ts, ss, tpos, grad):
    r = math.sqrt(15.0)
    a1, a2, w1, w2 = (6 - r) / 21, (6 + r) / 21, (155 - r) / 1200, (155 + r) / 1200
    rule = [((1 / 3, 1 / 3, 1 / 3), 0.225)]
    for a, w in ((a1, w1), (a2, w2)):
        rule += [(tuple(1 - 2 * a if k == q else a for k in range(3)), w) for q in range(3)]
    v32 = s["nodes"].T[s["idx"]]
    v, area, a = v32.double(), s["area"].double(), ts.double().T
    e = [v32[:, (k + 1) % 3] - v32[:, k] for k in range(3)]
    lim = 4 * torch.stack([x[:, 0] * x[:, 0] + x[:, 1] * x[:, 1] + x[:, 2] * x[:, 2] for x in e]).amax(0)
    c32 = _centroid(v32)
    sheet = ss is not None
    sg = ss.double() if sheet else torch.zeros(len(area), dtype=F64, device=DEV)
    t32, t = tpos.T, tpos.double().T.contiguous()
    points = [(sum(b * v[:, k] for k, b in enumerate(bary)), w) for bary, w in rule]
    cols = [_moments(y, w * a, w * sg * area if sheet else None) for y, w in points]
    us, gr = [], []
    step = max(1, CHUNK // len(area))
    for i in range(0, t.shape[0], step):
        ti = t[i:i + step]
        d = [t32[i:i + step, k:k + 1] - c32[None, :, k] for k in range(3)]
        near = d[0] * d[0] + d[1] * d[1] + d[2] * d[2] < lim[None, :]
        ks = bs = 0.0
        for (y, _), (kc, bc) in zip(points, cols):
            d2 = sum((ti[:, k:k + 1] - y[None, :, k]) ** 2 for k in range(3))
            K = (1.0 / (d2 * d2.sqrt())).masked_fill_(near, 0.0)
            ks = ks + K @ kc
            if grad:
                bs = bs + (K * -3.0 / d2) @ bc
        u, g = _from_moments(ti, ks, bs if grad else None, sheet)
        at, pj = near.nonzero(as_tuple=True)
        I, dI = _triangle_integrals(v[pj], ti[at])
        gam = a[pj] / area[pj][:, None]
        u = u.T.contiguous().index_add_(0, at, torch.linalg.cross(gam, I) + sg[pj][:, None] * I)
        us.append(u.T)
        if grad:
            m = torch.linalg.cross(gam[:, None].expand(-1, 3, -1), dI) + sg[pj][:, None, None] * dI
            gr.append(g.T.contiguous().index_add_(0, at, m.reshape(-1, 9)).T)
    return torch.cat(us, 1), torch.cat(gr, 1) if grad else None


def _rhs64(case, seed):
    s, pos, a = _rhs_inputs(case, seed)
    u, _ = _tree_sums(s, a, None, pos, False, flip=True)
    u = -u / (4 * math.pi)
    u[0] += 1.0
    bases = {1: ["nm"], 2: ["x1", "x2"], 3: ["x1", "x2", "nm"]}[case["nunk"]]
    return u, torch.stack([-(u.T * s[b]).sum(1) for b in bases], 1).reshape(-1)


def _matrix64(case, seed):
    s = _matrix_inputs(case, seed)
    n, u = case["np"], case["nunk"]
    v32 = s["nodes"].T[s["idx"]]
    v, sq, area = v32.double(), s["area"].sqrt(), s["area"].double()
    c32, c = _centroid(v32), _centroid(v)
    out = torch.zeros(n, u, n, u, dtype=F64, device=DEV)   # source, unknown, target, component
    basis = [s["x1"], s["x2"], s["nm"]]
    step = max(1, (1 << 22) // n)
    for j0 in range(0, n, step):
        j = torch.arange(j0, min(n, j0 + step), device=DEV)
        e = c32[None] - c32[j][:, None]
        dist = (e[..., 0] * e[..., 0] + e[..., 1] * e[..., 1] + e[..., 2] * e[..., 2]).sqrt()
        leaf = dist > (sq[j][:, None] + sq[None]) * 4
        d = c[None] - c[j][:, None]
        d2 = (d * d).sum(2)
        G = torch.where(leaf[..., None], d / (d2 * d2.sqrt()).clamp_min(1e-300)[..., None], torch.zeros_like(d))
        pj, pi = (~leaf).nonzero(as_tuple=True)
        for q in range(0, len(pj), 1 << 15):
            a, b = pj[q:q + (1 << 15)], pi[q:q + (1 << 15)]
            off = a + j0 != b
            a, b = a[off], b[off]
            sub = torch.zeros(len(a), 3, dtype=F64, device=DEV)
            of = torch.arange(len(a), device=DEV)
            tr = (v32[a + j0], v[a + j0], v32[b], v[b])
            for lev in range(1, 4):
                of = of.repeat_interleave(16)
                kids = [_children(x) for x in tr]
                tr = [x[:, :, None].expand(-1, 4, 4, 3, 3).reshape(-1, 3, 3) for x in kids[:2]] + \
                     [x[:, None].expand(-1, 4, 4, 3, 3).reshape(-1, 3, 3) for x in kids[2:]]
                t4 = (sq[a + j0] + sq[b])[of] * (4 * 0.5 ** lev)
                end = (_dist32(_centroid(tr[2]), _centroid(tr[0])) > t4) | (lev == 3)
                k = end.nonzero()[:, 0]
                dd = _centroid(tr[3][k]) - _centroid(tr[1][k])
                r2 = (dd * dd).sum(1)
                sub.index_add_(0, of[k], dd / (r2 * r2.sqrt())[:, None] * 0.0625 ** lev)
                k = (~end).nonzero()[:, 0]
                of, tr = of[k], [x[k] for x in tr]
            G[a, b] = sub
        G = G * (area[j] / (4 * math.pi))[:, None, None]
        for k in range(u):
            w = torch.linalg.cross(basis[k][j][:, None].expand(-1, n, -1), G) if k < 2 else G
            for m in range(u):
                out[j, k, :, m] = (w * basis[m][None]).sum(2)
    i = torch.arange(n, device=DEV)
    out[i, :, i, :] = 0.0
    out[i, 0, i, 1] = 0.5
    out[i, 1, i, 0] = -0.5
    if u == 3:
        out[i, 2, i, 2] = 0.5
    return out.reshape(n * u, n * u)


def _step64(core, pos, s, r):
    """one Ralston step of 1e-3 with stretching: position, strength and elongation"""
    x0, s0, dt = pos.double(), s.double(), 1e-3
    f = 0.25 / math.pi
    stretch = lambda g: torch.stack([sum(s0[j] * g[3 * j + i] for j in range(3)) for i in range(3)])   # noqa: E731
    u1, g1 = (f * y for y in _point_sums(core, x0, s0, r, x0, r, True, False))
    w1 = stretch(g1)
    x1, s1 = x0 + dt * 2 / 3 * u1, s0 + dt * 2 / 3 * w1
    u2, g2 = (f * y for y in _point_sums(core, x1, s1, r, x1, r, True, False))
    w = 0.25 * w1 + 0.75 * stretch(g2)
    return x0 + dt * (0.25 * u1 + 0.75 * u2), s0 + dt * w, 1.0 + dt * (s0 * w).sum(0) / (s0 * s0).sum(0)


def exact(case, seed):
    kind = case["kind"]
    if kind == "points":
        if float(case["ns"]) * (case["nt"] or case["ns"]) > EXACT_PAIRS:
            return None
        u, g = _point_sums(case["core"], *_point_inputs(case, seed), case["grad"], case["self_term"] == 1)
        return (u, g) if case["grad"] else u
    if kind == "panels":
        s, ts, ss, tpos = _panel_inputs(case, seed)
        u, g = (_tree_sums if case["rule"] == "auto" else _gauss7_sums)(s, ts, ss, tpos, case["grad"])
        return (u, g) if case["grad"] else u
    if kind == "bem_rhs":
        return _rhs64(case, seed)
    if kind == "bem_matrix":
        return _matrix64(case, seed)
    if kind == "batch":
        parts = [_point_sums(case["core"], *p, p[0], p[2], True, False) for p in _batch_inputs(case, seed)]
        return tuple(torch.cat(x, 1) for x in zip(*parts))
    return [_step64(*p) for p in _session_inputs(case, seed)]
