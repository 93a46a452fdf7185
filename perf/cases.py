"""Performance cases of the pair-histogram library: what its users have it compute, through its
public entry points.

A case is one call (or one execution of a kept plan) on synthetic drifter-like points in a
multi-scale velocity field.  Its keys:

    form    call            one operator, 1D (nv = 0) or joint (nv value bins)
            single_pass     the six invariants in one pass, 1D
            single_pass_2d  the six invariants, each binned by distance and by its own values
            fused           several operators and one joint histogram from one evaluation per pair
            plan            a ragged batch of 2D slices, fused outputs, a kept plan replayed as a graph
            aux             one field with an auxiliary axis (b velocity fields on shared positions)
    entry   host (numpy in, numpy out, the mirror of the reference's functions) or device (fields
            and outputs stay in device memory)
    geom    flat2, flat3 (Euclidean) or sphere (lon, lat in degrees, unit radius)
    n       points; op: operator; bins / nd: distance axis; nv: value bins; prec: backend precision
    reach   largest distance edge as a share of the domain's (1: every pair is binned)
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "structurefunctions.jl_amd"))
import sfamd  # noqa: E402
from sfamd import _native  # noqa: E402

OPS = {"L1": sfamd.L1SF, "T1": sfamd.T1SF, "L2": sfamd.L2SF, "T2": sfamd.T2SF, "L3": sfamd.L3SF,
       "T3": sfamd.T3SF, "S2": sfamd.S2SF, "S3": sfamd.S3SF}
FUSED = {"spectrum": ["L2", "T2", "L3", "T3"], "energy": ["L2", "T2"]}
PREC = {"fp64": _native.PREC_FP64, "mixed": _native.PREC_MIXED, "mixed_fixed": _native.PREC_MIXED_FIXED}


def listed():
    call = {"form": "call", "entry": "device", "reach": 1.0}
    return [
        # the smallest ordinary call: a notebook user's few hundred drifters, defaults throughout
        dict(call, name="host_flat2_small", entry="host", geom="flat2", n=777, op="L2", bins="log", nd=32, nv=0,
             prec="fp64"),
        # the reference's own CPU benchmark size, called with arrays of the host
        dict(call, name="host_flat2_4096", entry="host", geom="flat2", n=4096, op="L2", bins="log", nd=32, nv=0,
             prec="mixed"),
        # second-order moments of one 2D snapshot
        dict(call, name="flat2_L2_mixed", geom="flat2", n=65536, op="L2", bins="log", nd=64, nv=0, prec="mixed"),
        # the default precision on a linear axis (a Julia range), odd point count, third order
        dict(call, name="flat2_L3_fp64_linear", geom="flat2", n=30011, op="L3", bins="linear", nd=100, nv=0,
             prec="fp64"),
        # increment distribution of a 3D field
        dict(call, name="flat3_joint_fixed", geom="flat3", n=131072, op="L1", bins="log", nd=48, nv=128,
             prec="mixed_fixed"),
        # the headline workload: increment distribution over the globe
        dict(call, name="sphere_joint_fixed", geom="sphere", n=262144, op="L1", bins="log", nd=64, nv=96,
             prec="mixed_fixed"),
        # the same at the default precision, odd point count
        dict(call, name="sphere_joint_fp64", geom="sphere", n=100003, op="L1", bins="log", nd=64, nv=96,
             prec="fp64"),
        # local statistics: the largest edge is small against the domain
        dict(call, name="sphere_local_joint", geom="sphere", n=262144, op="L1", bins="log", nd=64, nv=96,
             prec="mixed_fixed", reach=0.05 / math.pi),
        # all six invariants of a global field at once
        {"name": "sphere_single_pass", "form": "single_pass", "entry": "device", "geom": "sphere", "n": 98304,
         "bins": "log", "nd": 64, "nv": 0, "prec": "mixed", "reach": 1.0},
        # every output of the global workload from one evaluation of each pair
        {"name": "sphere_fused", "form": "fused", "entry": "device", "geom": "sphere", "n": 131072, "ops": "spectrum",
         "bins": "log", "nd": 64, "nv": 96, "prec": "mixed_fixed", "reach": 1.0},
        # a time series of ragged 2D snapshots, replayed from a plan
        {"name": "plan_ragged_2d", "form": "plan", "entry": "device", "geom": "flat2", "n": 16000, "nmin": 2000,
         "slices": 64, "ops": "one", "bins": "log", "nd": 48, "nv": 64, "prec": "mixed_fixed", "reach": 1.0},
        # an ensemble: velocity fields on shared 3D positions, defaults throughout
        {"name": "host_aux_flat3", "form": "aux", "entry": "host", "geom": "flat3", "n": 5003, "b": 8, "op": "L2",
         "bins": "log", "nd": 40, "nv": 0, "prec": "fp64", "reach": 1.0},
    ]


def _n(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi], odd ones among them."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return n if rng.random() < 0.7 else max(lo, n // 64 * 64)


def draw(rng):
    kind = rng.choice(["small", "1d", "1d", "joint", "joint", "sphere64", "local", "single", "single2d", "fused", "plan",
                       "aux"])
    bins = rng.choice(["log", "log", "linear"])
    nd = rng.randint(20, 100)
    c = {"form": "call", "entry": "device", "bins": bins, "nd": nd, "nv": 0, "reach": 1.0}
    if kind == "small":
        return dict(c, entry="host", geom=rng.choice(["flat2", "flat3", "sphere"]), n=_n(rng, 300, 8192),
                    op=rng.choice(["L2", "T2", "S2"]), prec=rng.choice(["fp64", "mixed"]))
    if kind == "1d":
        prec = rng.choice(["fp64", "mixed", "mixed"])
        return dict(c, geom=rng.choice(["flat2", "flat3", "sphere"]), n=_n(rng, 16384, 131072 if prec == "mixed" else 65536),
                    op=rng.choice(["L2", "T2", "S2", "L3", "S3"]), prec=prec)
    if kind == "joint":
        return dict(c, geom=rng.choice(["flat2", "flat3", "sphere"]), n=_n(rng, 16384, 196608), op="L1",
                    nd=rng.randint(20, 64), nv=rng.randint(32, 96), prec=rng.choice(["mixed", "mixed_fixed"]))
    if kind == "sphere64":
        return dict(c, geom=rng.choice(["flat3", "sphere"]), n=_n(rng, 16384, 100003), op=rng.choice(["L1", "L2"]),
                    nd=rng.randint(20, 64), nv=rng.choice([0, rng.randint(32, 96)]), prec="fp64")
    if kind == "local":
        return dict(c, bins="log", geom=rng.choice(["flat2", "sphere"]), n=_n(rng, 65536, 262144), op="L1",
                    nd=rng.randint(20, 64), nv=rng.randint(32, 96), prec="mixed_fixed", reach=rng.choice([0.01, 0.02]))
    if kind == "single":
        return dict(c, form="single_pass", geom=rng.choice(["flat2", "sphere"]), n=_n(rng, 16384, 98304),
                    prec="mixed")
    if kind == "single2d":
        return dict(c, form="single_pass_2d", bins="log", geom=rng.choice(["flat2", "sphere"]), n=_n(rng, 8192, 32768),
                    nd=rng.randint(20, 64), nv=rng.randint(24, 48), prec="mixed")
    if kind == "fused":
        return dict(c, form="fused", geom=rng.choice(["flat2", "sphere"]), n=_n(rng, 16384, 131072),
                    ops=rng.choice(["spectrum", "energy"]), nd=rng.randint(20, 64), nv=rng.randint(32, 96),
                    prec="mixed_fixed")
    if kind == "plan":
        return dict(c, form="plan", geom="flat2", n=_n(rng, 6000, 24000), nmin=1000, slices=rng.randint(8, 48),
                    ops="one", nd=rng.randint(20, 48), nv=rng.randint(32, 64), prec="mixed_fixed")
    return dict(c, form="aux", entry="host", geom=rng.choice(["flat2", "flat3"]), n=_n(rng, 1000, 8192),
                b=rng.randint(2, 8), op=rng.choice(["L2", "S2"]), prec=rng.choice(["fp64", "mixed"]))


# ---- inputs ------------------------------------------------------------------------------------

def _modes(g, dim, m, kmin, kmax, power):
    """Solenoidal Fourier modes: wave vectors (dim, m), amplitude vectors (dim, m), phases (m, 1)."""
    r = lambda *s: torch.rand(*s, generator=g, device="cuda", dtype=torch.float64)  # noqa: E731
    z = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=torch.float64)  # noqa: E731
    k = kmin * (kmax / kmin) ** r(m)
    kh = z(dim, m)
    kh = kh / kh.norm(dim=0)
    e = z(dim, m)
    e = e - kh * (e * kh).sum(0)
    e = e / e.norm(dim=0)
    return kh * k, e * k ** power, 2 * math.pi * r(m, 1)


def _eval(modes, p):
    k, a, ph = modes
    return a @ torch.cos(k.T @ p + ph)


def _flat(g, dim, n, fields=1):
    """Drifters in a box: a multi-scale solenoidal field about a rotating mean flow, the positions
    carried along by it for a short time (which skews the increments, as a turbulent flow's are)."""
    x = torch.rand(dim, n, generator=g, device="cuda", dtype=torch.float64)
    us = []
    for f in range(fields):
        m = _modes(g, dim, 48, 2 * math.pi, 2 * math.pi * 48, -5 / 6)
        u = _eval(m, x)
        u = u / u.square().mean().sqrt()
        u[0] += 1.2 * (0.5 - x[1])
        u[1] += 1.2 * (x[0] - 0.5)
        if f == 0:
            moved = x + 0.02 * u
        us.append(u)
    return moved, us


def _sphere(g, n):
    """Points on the unit sphere, half uniform, half on great-circle tracks of 256 points, carried
    along by a multi-scale field about a rotating mean flow; (lon, lat) degrees and (east, north)."""
    z = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=torch.float64)  # noqa: E731
    nt = (n // 2 + 255) // 256
    v = z(3, n - n // 2)
    a, b = z(3, nt, 1), z(3, nt, 1)
    a = a / a.norm(dim=0)
    b = b - a * (a * b).sum(0)
    b = b / b.norm(dim=0)
    t = 2 * math.pi * torch.rand(nt, 1, generator=g, device="cuda", dtype=torch.float64)
    t = t + 1e-3 * torch.arange(256, device="cuda", dtype=torch.float64)
    tr = (a * torch.cos(t) + b * torch.sin(t) + 1e-4 * z(3, nt, 256)).reshape(3, -1)[:, : n // 2]
    p = torch.cat([v, tr], dim=1)
    p = p / p.norm(dim=0)

    def frame(p):
        lon, lat = torch.atan2(p[1], p[0]), torch.asin(p[2].clamp(-1, 1))
        e = torch.stack([-torch.sin(lon), torch.cos(lon), torch.zeros_like(lon)])
        nn = torch.stack([-torch.sin(lat) * torch.cos(lon), -torch.sin(lat) * torch.sin(lon), torch.cos(lat)])
        return lon, lat, e, nn

    f = _eval(_modes(g, 3, 48, 1.0, 128.0, -5 / 6), p)
    lon, lat, e, nn = frame(p)
    uv = torch.stack([(f * e).sum(0), (f * nn).sum(0)])
    uv = uv / uv.square().mean().sqrt()
    uv[0] += 1.2 * torch.cos(lat)
    q = p + 0.02 * (uv[0] * e + uv[1] * nn)
    lon, lat, _, _ = frame(q / q.norm(dim=0))
    return torch.stack([torch.rad2deg(lon), torch.rad2deg(lat)]), uv


def _domain(geom):
    return {"flat2": (2.0 ** 0.5, 1e-4), "flat3": (3.0 ** 0.5, 1e-3), "sphere": (math.pi, 1e-5)}[geom]


def _dist_axis(c):
    top, low = _domain(c["geom"])
    top = top * c["reach"]
    if c["bins"] == "linear":
        return sfamd.LinearBinEdges(0.0, top, c["nd"] + 1)
    return np.geomspace(low if c["geom"] != "flat3" else max(low, top * 1e-3), top, c["nd"] + 1)


def _value_axis(u, nv):
    s = float(u.square().mean().sqrt()) * math.sqrt(2.0)
    return np.linspace(-4 * s, 4 * s, nv + 1)


def _value_axes_2d(u, nv):
    """|du|^2, du_L^2, du_T^2 on log edges; du_L |du|^2, du_L^3, du_L du_T^2 on linear edges."""
    m = 2 * float(u.square().mean())
    pos = np.concatenate([[0.0], np.geomspace(1e-3 * m, 60 * m, nv)])
    sgn = np.linspace(-20 * m ** 1.5, 20 * m ** 1.5, nv + 1)
    return [pos, pos, pos, sgn, sgn, sgn]


_CTX = {}


def _ctx():
    if "c" not in _CTX:
        _CTX["c"] = sfamd.MI355XBackend().context()
    return _CTX["c"]


def _inputs(c, seed):
    """Fields of the case as device tensors: list of (x (W, n), [u (D, n), ...])."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    if c["form"] == "plan":
        # sizes from the seed, the total kept near the same for every seed
        r = np.random.default_rng(int(seed))
        f = (np.arange(c["slices"]) + r.uniform(size=c["slices"])) / c["slices"]
        ns = np.round(c["nmin"] * (c["n"] / c["nmin"]) ** f).astype(int)
        r.shuffle(ns)
        return [_flat(g, 2, int(n)) for n in ns]
    if c["geom"] == "sphere":
        x, u = _sphere(g, c["n"])
        return [(x, [u])]
    return [_flat(g, 2 if c["geom"] == "flat2" else 3, c["n"], c.get("b", 1))]


def _problem(c, x, u, de, ve, keep, op=(0, 1, 0)):
    """sf_problem of device-resident points: x and u as (n, W) / (n, D) row-major tensors."""
    e = sfamd.as_edges(de)
    p = _native.SfProblem()
    p.D, p.W, p.N = u.shape[1], x.shape[1], x.shape[0]
    p.x, p.u = x.data_ptr(), u.data_ptr()
    p.geometry, p.radius = (1, 1.0) if c["geom"] == "sphere" else (0, 1.0)
    p.op, p.nl, p.nt = op
    p.n_dist, p.dist_edges = len(e) - 1, e.ctypes.data
    keep += [x, u, e]
    if isinstance(de, sfamd.LinearBinEdges):
        r = _native.make_rule(de.rule())
        keep.append(r)
        p.dist_rule = ctypes.addressof(r)
    if ve is not None:
        v = np.concatenate(ve) if isinstance(ve, list) else np.ascontiguousarray(ve)
        keep.append(v)
        p.n_val, p.val_edges = c["nv"], v.ctypes.data
    p.precision, p.count_bits = PREC[c["prec"]], 64
    return p


def _fused_outputs(c):
    """(operator, joint) of every output of a fused case."""
    names = ["L2"] if c["ops"] == "one" else FUSED[c["ops"]]
    return [(k, False) for k in names] + [("L1", True)]


def prepare(case, seed):
    c = case
    fields = _inputs(c, seed)
    de = _dist_axis(c)
    s = {"case": c, "de": de, "keep": []}
    if c["entry"] == "host":
        x, us = fields[0]
        s["x"] = x.cpu().numpy()
        s["u"] = us[0].cpu().numpy() if c["form"] != "aux" else torch.stack(us, dim=2).cpu().numpy()
        s["backend"] = sfamd.MI355XBackend(0, c["prec"])
        s["metric"] = sfamd.Haversine(1.0) if c["geom"] == "sphere" else sfamd.Euclidean()
        return s
    probs = []
    for x, us in fields:
        xt, ut = x.T.contiguous(), us[0].T.contiguous()
        ve, op = None, (0, 1, 0)
        if c["form"] == "single_pass_2d":
            ve, op = _value_axes_2d(us[0], c["nv"]), (_native.OP_SINGLE_PASS, 0, 0)
        elif c["form"] == "single_pass":
            op = (_native.OP_SINGLE_PASS, 0, 0)
        else:
            if c["nv"]:
                ve = _value_axis(us[0], c["nv"])
            if c["form"] == "call":
                op = OPS[c["op"]].code
        probs.append(_problem(c, xt, ut, de, ve, s["keep"], op))
    s["problems"] = probs
    nd, nv, n = c["nd"], max(c["nv"], 1), len(probs)
    new = lambda *shape: (torch.zeros(*shape, device="cuda", dtype=torch.float64),  # noqa: E731
                          torch.zeros(*shape, device="cuda", dtype=torch.int64))
    if c["form"] in ("fused", "plan"):
        outs = []
        s["out"] = []
        for k, joint in _fused_outputs(c):
            o = _native.SfOutput()
            o.op, o.nl, o.nt = OPS[k].code
            o.n_val = c["nv"] if joint else 0
            outs.append(o)
            s["out"].append(new(n, nv, nd) if joint else new(n, nd))
        s["outputs"] = outs
    else:
        rows = 6 if c["form"].startswith("single_pass") else 1
        s["out"] = [new(nv, nd, rows)]
    s["ctx"] = _ctx()
    if c["form"] == "plan":
        s["plan"] = _native.Plan(s["ctx"], probs, s["outputs"])
    torch.cuda.synchronize()
    return s


def run(state):
    s, c = state, state["case"]
    if c["entry"] == "host":
        r = sfamd.calculate_structure_function(OPS[c["op"]], s["x"], s["u"], s["de"], np.uint64, backend=s["backend"],
                                               output_type=sfamd.StructureFunctionSumsAndCounts,
                                               distance_metric=s["metric"])
        return {"sums": r.sums, "counts": r.counts.astype(np.int64)}
    for a, b in s["out"]:  # the entry points accumulate
        a.zero_()
        b.zero_()
    ps, pc = [a.data_ptr() for a, _ in s["out"]], [b.data_ptr() for _, b in s["out"]]
    if c["form"] == "plan":
        s["plan"].execute_multi(ps, pc, 0, graph=True)
        s["plan"].sync()  # results are read after every snapshot
    elif c["form"] == "fused":
        s["ctx"].hist_multi_device(s["problems"], s["outputs"], ps, pc, 0)
    else:
        s["ctx"].hist_device(s["problems"], ps[0], pc[0], 0)
    return {"sums": [a for a, _ in s["out"]], "counts": [b for _, b in s["out"]]}


# ---- the same sums in plain 64-bit torch --------------------------------------------------------

def _pairs(c, fields):
    return sum(x.shape[1] * (x.shape[1] - 1) // 2 for x, _ in fields) * c.get("b", 1)


def _hist(geom, x, u, de, wanted):
    """Sums over all pairs i < j.  wanted: list of (values(L, T, n2), value edges or None)."""
    n = x.shape[1]
    nd = len(de) - 1
    e = torch.as_tensor(de, device="cuda")
    if geom == "sphere":
        lon, lat = torch.deg2rad(x[0]), torch.deg2rad(x[1])
        p = torch.stack([torch.cos(lat) * torch.cos(lon), torch.cos(lat) * torch.sin(lon), torch.sin(lat)])
        ea = torch.stack([-torch.sin(lon), torch.cos(lon), torch.zeros_like(lon)])
        no = torch.stack([-torch.sin(lat) * torch.cos(lon), -torch.sin(lat) * torch.sin(lon), torch.cos(lat)])
        w = u[0] * ea + u[1] * no
        half = torch.sin(0.5 * e.clamp(max=math.pi))
        edges = (2 * half).square()
    else:
        p, w = x, u
        edges = e.square()
    outs = [torch.zeros(nd + 2 if v is None else (nd + 2) * (len(v) + 1), device="cuda", dtype=torch.float64)
            for _, v in wanted]
    ved = [None if v is None else torch.as_tensor(v, device="cuda") for _, v in wanted]
    rows = max(1, (1 << 25) // n)
    col = torch.arange(n, device="cuda")
    for i0 in range(0, n - 1, rows):
        i1 = min(n, i0 + rows)
        d = [p[k][None, i0:] - p[k][i0:i1, None] for k in range(p.shape[0])]
        du = [w[k][None, i0:] - w[k][i0:i1, None] for k in range(p.shape[0])]
        key = sum(q * q for q in d)
        dot = sum(a * b for a, b in zip(d, du))
        if geom == "sphere":
            pr = [p[k][i0:i1, None] for k in range(3)]
            cr = [pr[1] * d[2] - pr[2] * d[1], pr[2] * d[0] - pr[0] * d[2], pr[0] * d[1] - pr[1] * d[0]]
            inv = 1 / sum(q * q for q in cr).sqrt()
            L = dot * inv
            T = sum(a * b for a, b in zip(cr, du)) * inv
            n2 = L * L + T * T
        else:
            r = key.sqrt()
            L = dot / r
            n2 = sum(q * q for q in du)
            T = (du[1] * d[0] - du[0] * d[1]) / (r if len(d) == 2 else (d[0] * d[0] + d[1] * d[1]).sqrt())
        up = col[None, i0:] > col[i0:i1, None]
        b = torch.bucketize(key, edges)
        for k, (fn, v) in enumerate(wanted):
            val = fn(L, T, n2)
            idx = b
            if v is not None:
                idx = b * (len(v) + 1) + torch.bucketize(val, ved[k])
            outs[k] += torch.bincount(idx[up], weights=val[up], minlength=outs[k].numel())
    res = []
    for (fn, v), o in zip(wanted, outs):
        if v is None:
            res.append(o[1:nd + 1])
        else:
            res.append(o.reshape(nd + 2, len(v) + 1)[1:nd + 1, 1:len(v)].T.contiguous())
    return res


VALUES = {"L1": lambda L, T, n2: L, "T1": lambda L, T, n2: T, "L2": lambda L, T, n2: L * L,
          "T2": lambda L, T, n2: n2 - L * L, "L3": lambda L, T, n2: L * L * L, "T3": lambda L, T, n2: T * T * T,
          "S2": lambda L, T, n2: n2, "S3": lambda L, T, n2: L * n2, "L1T2": lambda L, T, n2: L * (n2 - L * L)}
SIX = ["S2", "L2", "T2", "S3", "L3", "L1T2"]


def exact(case, seed):
    c = case
    fields = _inputs(c, seed)
    if _pairs(c, fields) > 4.0e9:
        return None  # more than about 20 seconds
    de = sfamd.as_edges(_dist_axis(c))
    if c["form"] == "aux":
        x, us = fields[0]
        return {"sums": torch.stack([_hist(c["geom"], x, u, de, [(VALUES[c["op"]], None)])[0] for u in us], dim=1),
                "counts": None}
    if c["form"] in ("fused", "plan"):
        got = []
        for x, us in fields:
            ve = _value_axis(us[0], c["nv"])
            got.append(_hist(c["geom"], x, us[0], de,
                             [(VALUES[k], ve if joint else None) for k, joint in _fused_outputs(c)]))
        return {"sums": [torch.stack(o) for o in zip(*got)], "counts": None}
    x, us = fields[0]
    if c["form"] == "single_pass":
        r = _hist(c["geom"], x, us[0], de, [(VALUES[k], None) for k in SIX])
        return {"sums": [torch.stack(r, dim=1)[None]], "counts": None}
    if c["form"] == "single_pass_2d":
        r = _hist(c["geom"], x, us[0], de, [(VALUES[k], v) for k, v in zip(SIX, _value_axes_2d(us[0], c["nv"]))])
        return {"sums": [torch.stack(r, dim=2)], "counts": None}
    ve = _value_axis(us[0], c["nv"]) if c["nv"] else None
    r = _hist(c["geom"], x, us[0], de, [(VALUES[c["op"]], ve)])[0]
    if c["entry"] == "host":
        return {"sums": r, "counts": None}
    return {"sums": [(r if ve is not None else r[None])[:, :, None]], "counts": None}


# floating operations of one pair: separation and key, the pair's frame, increments and operator
# value, the bins and the accumulation (an fma counts two, a square root or reciprocal four)
_FLOPS = {("flat2", 0): 28, ("flat3", 0): 33, ("sphere", 0): 53, ("flat2", 1): 36, ("flat3", 1): 41, ("sphere", 1): 60}


def work(case):
    c = case
    if c["form"] == "plan":
        f = (np.arange(c["slices"]) + 0.5) / c["slices"]
        ns = np.round(c["nmin"] * (c["n"] / c["nmin"]) ** f)
    else:
        ns = np.array([float(c["n"])])
    b = c.get("b", 1)
    pairs = float(np.sum(ns * (ns - 1) / 2)) * b
    if c["reach"] < 0.5:  # only pairs within the largest edge need evaluating
        top = _domain(c["geom"])[0] * c["reach"]
        pairs *= {"flat2": math.pi * top ** 2, "flat3": 4 / 3 * math.pi * top ** 3,
                  "sphere": math.sin(top / 2) ** 2}[c["geom"]]
    joint = 1 if c["nv"] else 0
    per = _FLOPS[(c["geom"], joint)]
    outs = 1
    if c["form"] == "single_pass":
        per, outs = per + 16, 6
    elif c["form"] == "single_pass_2d":
        per, outs = per + 64, 6
    elif c["form"] in ("fused", "plan"):
        per += 4 * (len(_fused_outputs(c)) - 1)
    cells = len(ns) * b * c["nd"] * max(c["nv"], 1) * outs
    dims = 6 if c["geom"] == "flat3" else 4
    points = float(np.sum(ns)) * (dims if c["form"] != "aux" else dims / 2 * (1 + b))
    return {"bytes": points * 8 + cells * 16, "flops": pairs * per}
