"""The work whose speed is followed: calls through the public entry points, over the sizes in use.

Every case names its path and its sizes. The particle sets are the five benchmark
configurations' distributions (omega2d_amd/workloads.py) at other sizes and seeds:

  disc    particles in a disc of radius 0.5 with a Gaussian vorticity profile, uniform radius
  blobs   64 Lamb-Oseen blobs stored blob by blob, tracers over a wider square, Gaussian core
  wake    the downstream half-annulus behind a unit circle of panels
  square  particles over a square with radii U[0.005, 0.02], probes on a circle around it

Paths:
  host    points_on_points on float32 host arrays, the form the reference application calls
  step    whole Ralston steps on the device, with or without a body
  pairs   points_on_points on device tensors (any core, precision and result type)
  tree    points_on_points_tree on device tensors
  panels  both panel sums of one solver stage: particles on panels, panels on particles
  bem     one body's system: assembly, factorisation, two solves
  probe   probe_velocity with its backward pass
  wall    the clearing pass and the nearest distances after a move
  vort    the Gaussian vorticity of the particles on themselves
"""
import math

import numpy as np
import torch

import omega2d_amd as o2d
from omega2d_amd import autograd, device as dv
from omega2d_amd.device_step import CLEAR_CUTOFF, Body, Stepper

CORES = ("rm", "gauss", "wl", "v2", "v3")


def listed():
    return [
        # the drop-in call of a small run: float32 host arrays, the reference's default core;
        # copies and launches dominate
        dict(name="host-1.5k", path="host", ns=1531, nt=977, core="v2", precision="split",
             targets="other"),
        # the smallest benchmark configuration: one RK2 step of 10,000 particles
        dict(name="disc-10k-rk2", path="step", ns=10000, npan=0, nunk=1, core="rm",
             precision="split", order=2),
        # the headline: one velocity evaluation of 1M particles and 64k tracers
        dict(name="blobs-1M-split", path="pairs", set="blobs", ns=1 << 20, nt=1 << 16,
             core="gauss", precision="split", results="vel", targets="self+tracers"),
        # the same evaluation in the accurate form, at an odd size of a production run
        dict(name="blobs-262k-fp64", path="pairs", set="blobs", ns=262147, nt=9973,
             core="gauss", precision="fp64", results="vel", targets="self+tracers"),
        # the fast summation at the headline's size
        dict(name="blobs-1M-tree", path="tree", ns=1 << 20, nt=1 << 16, core="gauss"),
        # velocity with the shear rate, as output steps and adaptive schemes ask for it
        dict(name="wake-100k-shear", path="pairs", set="wake", ns=100003, nt=0, core="v2",
             precision="fp64", results="shear", targets="self"),
        # a whole RK2 step around a body, everything on the device
        dict(name="wake-200k-rk2", path="step", ns=200000, npan=2048, nunk=1, core="v2",
             precision="split", order=2),
        # the panel sums of one stage: right-hand side and panels on the wake
        dict(name="panels-2048", path="panels", ns=200000, npan=2048, nunk=2),
        # the body's system, solved from scratch (the setup of a run; every step of a moving body)
        dict(name="bem-2049", path="bem", npan=2048, nunk=1),
        # gradient of a probe objective, forward and backward
        dict(name="probe-250k", path="probe", ns=250000, nt=4096, core="gauss"),
        # what follows every move: particles pushed out of the body's layer, distances
        dict(name="wall-200k", path="wall", ns=200000, npan=2048),
        # vorticity output of the wake
        dict(name="vort-200k", path="vort", ns=200000),
    ]


def _size(rng, lo, hi):
    """A size spread over its logarithm, mostly odd."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return n if rng.random() < 0.25 else n | 1


def draw(rng):
    path = rng.choice(["host", "step", "body", "pairs", "pairs", "gauss", "tree", "panels",
                       "bem", "probe", "wall", "vort"])
    if path == "host":
        return dict(path="host", ns=_size(rng, 100, 30000), nt=_size(rng, 100, 30000),
                    core=rng.choice(CORES), precision=rng.choice(["fp64", "split"]),
                    targets=rng.choice(["self", "other", "inert"]))
    if path == "step":
        return dict(path="step", ns=_size(rng, 500, 100000), npan=0, nunk=1,
                    core=rng.choice(CORES), precision=rng.choice(["fp64", "split"]),
                    order=rng.choice([1, 2, 3]))
    if path == "body":
        return dict(path="step", ns=_size(rng, 2000, 200000), npan=_size(rng, 100, 2048),
                    nunk=rng.choice([1, 2]), core=rng.choice(["v2", "rm", "gauss"]),
                    precision="split", order=rng.choice([1, 2]))
    if path == "pairs":
        results = rng.choice(["vel", "vel", "vort", "shear"])
        return dict(path="pairs", set=rng.choice(["disc", "wake"]), ns=_size(rng, 300, 150000),
                    nt=_size(rng, 100, 30000), core=rng.choice(CORES),
                    precision=rng.choice(["fp64", "split"]), results=results,
                    targets=rng.choice(["self", "other", "self+tracers"]))
    if path == "gauss":
        return dict(path="pairs", set="blobs", ns=_size(rng, 2000, 400000),
                    nt=_size(rng, 500, 60000), core="gauss",
                    precision=rng.choice(["fp64", "split"]), results="vel",
                    targets="self+tracers")
    if path == "tree":
        return dict(path="tree", ns=_size(rng, 5000, 1000000), nt=_size(rng, 500, 60000),
                    core=rng.choice(["gauss", "gauss", "v2"]))
    if path == "panels":
        return dict(path="panels", ns=_size(rng, 500, 200000), npan=_size(rng, 50, 3000),
                    nunk=rng.choice([1, 2]))
    if path == "bem":
        nunk = rng.choice([1, 2])
        return dict(path="bem", npan=_size(rng, 50, 3000 // nunk), nunk=nunk)
    if path == "probe":
        return dict(path="probe", ns=_size(rng, 1000, 300000), nt=_size(rng, 50, 5000),
                    core=rng.choice(["gauss", "gauss", "rm"]))
    if path == "wall":
        return dict(path="wall", ns=_size(rng, 1000, 300000), npan=_size(rng, 50, 3000))
    return dict(path="vort", ns=_size(rng, 500, 300000))


# ---- inputs --------------------------------------------------------------------------------

def _disc(rng, n):
    r = 0.5 * np.sqrt(rng.uniform(size=n))
    th = 2.0 * np.pi * rng.uniform(size=n)
    g = np.exp(-r * r / 0.05)
    return r * np.cos(th), r * np.sin(th), g / g.sum(), np.full(n, 0.02)


def _blobs(rng, n, nblob=64):
    cx, cy = rng.uniform(-4, 4, nblob), rng.uniform(-4, 4, nblob)
    rb, gb = rng.uniform(0.1, 0.5, nblob), rng.uniform(-1, 1, nblob)
    b = np.arange(n) * nblob // n
    x = cx[b] + rb[b] / np.sqrt(2.0) * rng.normal(size=n)
    y = cy[b] + rb[b] / np.sqrt(2.0) * rng.normal(size=n)
    s = gb[b] * (nblob / n) + rng.normal(0.0, 1e-4, n)
    return x, y, s, np.full(n, 0.01 * np.sqrt(64.0 / n))


def _wake(rng, n):
    r = np.sqrt(rng.uniform(0.52 ** 2, 3.0 ** 2, n))
    t = rng.uniform(-np.pi / 2, np.pi / 2, n)
    return r * np.cos(t), r * np.sin(t), rng.normal(0, 2e-4, n), np.full(n, 0.005)


def _square(rng, n):
    return (rng.uniform(-1, 1, n), rng.uniform(-1, 1, n), rng.normal(0, 1e-3, n),
            rng.uniform(0.005, 0.02, n))


_SETS = {"disc": _disc, "blobs": _blobs, "wake": _wake, "square": _square}
_TRACERS = {"disc": 1.0, "blobs": 5.0, "wake": 3.0}


def _circle(npan):
    """The unit-diameter circle, clockwise, its nodes stored as float."""
    th = 2.0 * np.pi * np.arange(npan) / npan
    nx = (0.5 * np.cos(th)).astype(np.float32).astype(np.float64)
    ny = (-0.5 * np.sin(th)).astype(np.float32).astype(np.float64)
    idx = np.stack([np.arange(npan), (np.arange(npan) + 1) % npan], 1).astype(np.int32)
    return nx, ny, idx.ravel()


def _rotation(nx, ny, idx):
    """Velocity of the unit rotation about the origin just outside each panel's centre."""
    a, b = idx[0::2], idx[1::2]
    return -0.5 * (ny[a] + ny[b]), 0.5 * (nx[a] + nx[b])


def _arrays(case, seed):
    """The case's inputs as numpy arrays by name."""
    rng = np.random.default_rng(seed)
    p, a = case["path"], {}
    if p == "host":
        x, y, s, r = _wake(rng, case["ns"])
        f = [v.astype(np.float32) for v in (x, y, s, r)]
        a.update(zip(("x", "y", "s", "r"), f))
        if case["targets"] == "self":
            a.update(tx=a["x"], ty=a["y"], tr=a["r"])
        else:
            tx, ty, _, tr = _wake(rng, case["nt"])
            a.update(tx=tx.astype(np.float32), ty=ty.astype(np.float32))
            if case["targets"] == "other":
                a.update(tr=tr.astype(np.float32))
        return a
    kind = {"pairs": case.get("set"), "tree": "blobs", "probe": "square",
            "step": "wake" if case.get("npan") else "disc"}.get(p, "wake")
    if "ns" in case:
        a.update(zip(("x", "y", "s", "r"), _SETS[kind](rng, case["ns"])))
    if p in ("pairs", "tree") and case["nt"]:
        half = _TRACERS[kind]
        a.update(tx=rng.uniform(-half, half, case["nt"]), ty=rng.uniform(-half, half, case["nt"]))
        a.update(tr=np.full(case["nt"], a["r"][0]))
    if p == "probe":
        k = 2.0 * np.pi * np.arange(case["nt"]) / case["nt"]
        a.update(tx=1.5 * np.cos(k), ty=1.5 * np.sin(k))
        # upstream gradients of the two velocity components
        a.update(gu=rng.normal(size=case["nt"]), gv=rng.normal(size=case["nt"]))
    if p in ("panels", "bem", "wall") or (p == "step" and case["npan"]):
        a.update(zip(("nx", "ny", "idx"), _circle(case["npan"])))
    if p == "panels":
        a["vs"] = rng.normal(0, 1.0, case["npan"])
        if case["nunk"] == 2:
            a["ss"] = rng.normal(0, 1.0, case["npan"])
    if p == "bem":
        a.update(zip(("uu", "uv"), _rotation(a["nx"], a["ny"], a["idx"])))
        n = case["npan"] * case["nunk"] + 1
        a["b0"], a["b1"] = rng.normal(size=n), rng.normal(size=n)
    if p == "wall":
        # a move of up to a few layer thicknesses takes some particles into the body's layer
        near = rng.integers(0, case["ns"], case["ns"] // 50 + 1)
        th, h = rng.uniform(-np.pi, np.pi, len(near)), rng.uniform(-0.002, 0.004, len(near))
        a["x"][near], a["y"][near] = (0.5 + h) * np.cos(th), (0.5 + h) * np.sin(th)
        i, j = a["idx"][0::2], a["idx"][1::2]
        ex, ey = a["nx"][j] - a["nx"][i], a["ny"][j] - a["ny"][i]
        ln = np.sqrt(ex * ex + ey * ey)
        a["pnx"], a["pny"] = -ey / ln, ex / ln
    return a


_VOL = 0.25 * math.pi  # the disc's area, for the system's corner entry


def prepare(case, seed):
    a = _arrays(case, seed)
    if case["path"] == "host":
        return dict(case=case, a=a)
    t = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in a.items()}
    st = dict(case=case, t=t)
    if case["path"] == "step":
        st["body"] = (Body(a["nx"], a["ny"], a["idx"].astype(np.uint32), case["nunk"])
                      if case["npan"] else None)
    if case["path"] == "bem":
        n = case["npan"] * case["nunk"] + 1
        st["A"] = torch.empty((n, n), dtype=torch.float64, device="cuda")
    if case["path"] == "probe":
        for k in ("x", "y", "s", "r"):
            t[k].requires_grad_(True)
    return st


# ---- one pass ------------------------------------------------------------------------------

def run(state):
    return _RUN[state["case"]["path"]](state["case"], state)


def _run_host(case, st):
    a = st["a"]
    return o2d.points_on_points(a["x"], a["y"], a["s"], a["r"], a["tx"], a["ty"], a.get("tr"),
                                core=case["core"], precision=case["precision"])


def _run_step(case, st):
    t, body = st["t"], st["body"]
    if body is not None:  # each pass is a first step
        body.omega_error = torch.zeros_like(body.omega_error)
        body.reabsorbed = torch.zeros_like(body.reabsorbed)
    sim = Stepper(t["x"].clone(), t["y"].clone(), t["s"], t["r"], core=case["core"],
                  precision=case["precision"], fs=(1.0, 0.0) if body else (0.0, 0.0), body=body,
                  ips=0.005)
    u, v = sim.step(0.01, case["order"])
    out = dict(x=sim.x, y=sim.y, u=u, v=v)
    if body is not None:
        out.update(vs=body.vs, ss=body.ss)
    return out


def _run_pairs(case, st):
    t, out = st["t"], {}
    kw = dict(core=case["core"], precision=case["precision"], results=case["results"])
    if case["targets"] != "other":
        out["self"] = dv.points_on_points(t["x"], t["y"], t["s"], t["r"], t["x"], t["y"], t["r"],
                                          **kw)
    if case["targets"] == "other":
        out["other"] = dv.points_on_points(t["x"], t["y"], t["s"], t["r"], t["tx"], t["ty"],
                                           t["tr"], **kw)
    if case["targets"] == "self+tracers":
        out["tracers"] = dv.points_on_points(t["x"], t["y"], t["s"], t["r"], t["tx"], t["ty"],
                                             **kw)
    return out


def _run_tree(case, st):
    t = st["t"]
    return dict(self=dv.points_on_points_tree(t["x"], t["y"], t["s"], t["r"], t["x"], t["y"],
                                              t["r"], core=case["core"]),
                tracers=dv.points_on_points_tree(t["x"], t["y"], t["s"], t["r"], t["tx"],
                                                 t["ty"], core=case["core"]))


def _run_panels(case, st):
    t = st["t"]
    return dict(rhs=dv.points_on_panels(t["x"], t["y"], t["s"], t["nx"], t["ny"], t["idx"]),
                vel=dv.panels_on_points(t["nx"], t["ny"], t["idx"], t["vs"], t.get("ss"), t["x"],
                                        t["y"]))


def _run_bem(case, st):
    t, A = st["t"], st["A"]
    dv.bem_assemble(t["nx"], t["ny"], t["idx"], case["nunk"], True, t["uu"], t["uv"], _VOL, out=A)
    dv.bem_factor(A)
    return dict(A=A, x0=dv.bem_solve(t["b0"]), x1=dv.bem_solve(t["b1"]))


def _run_probe(case, st):
    t = st["t"]
    src = [t["x"], t["y"], t["s"], t["r"]]
    u, v = autograd.probe_velocity(*src, t["tx"], t["ty"], core=case["core"])
    g = torch.autograd.grad([u, v], src, [t["gu"], t["gv"]])
    return dict(u=u.detach(), v=v.detach(), grad=g)


def _run_wall(case, st):
    t = st["t"]
    x, y = t["x"].clone(), t["y"].clone()
    circ, counts = dv.clear_inner(1, t["nx"], t["ny"], t["idx"], t["pnx"], t["pny"], CLEAR_CUTOFF,
                                  0.005, x, y, t["s"], t["r"])
    return dict(x=x, y=y, circ=circ, counts=counts,
                dist=dv.nearest_distances(t["nx"], t["ny"], t["idx"], t["x"], t["y"]))


def _run_vort(case, st):
    t = st["t"]
    return dv.points_vorticity(t["x"], t["y"], t["s"], t["r"], t["x"], t["y"])


_RUN = dict(host=_run_host, step=_run_step, pairs=_run_pairs, tree=_run_tree, panels=_run_panels,
            bem=_run_bem, probe=_run_probe, wall=_run_wall, vort=_run_vort)


# ---- what a pass cannot do without ---------------------------------------------------------

def _pair_work(ns, nt, core, point, results="vel", item=8):
    outs = 2 if results == "vel" else 3
    return dict(bytes=item * (4 * ns + (2 if point else 3) * nt + outs * nt),
                flops=o2d.flops_per_pair(core, point) * ns * nt)


def _add(*ws):
    return dict(bytes=sum(w["bytes"] for w in ws), flops=sum(w["flops"] for w in ws))


def work(case):
    p, ns, nt, npan = case["path"], case.get("ns", 0), case.get("nt", 0), case.get("npan", 0)
    if p == "host":
        n = ns if case["targets"] == "self" else nt
        return _pair_work(ns, n, case["core"], case["targets"] == "inert", item=4)
    if p == "step":
        one = _pair_work(ns, ns, case["core"], False)
        ws = [dict(bytes=one["bytes"] * case["order"], flops=one["flops"] * case["order"]),
              dict(bytes=8 * ns * (4 + 2 * case["order"]), flops=8 * ns * case["order"])]
        if npan:
            n = npan * case["nunk"] + 1
            ws.append(dict(bytes=case["order"] * 8 * n * n, flops=case["order"] * 2 * n * n))
        return _add(*ws)
    if p == "pairs":
        ws = []
        if case["targets"] != "other":
            ws.append(_pair_work(ns, ns, case["core"], False, case["results"]))
        if case["targets"] != "self":
            ws.append(_pair_work(ns, nt, case["core"], case["targets"] != "other",
                                 case["results"]))
        return _add(*ws)
    if p == "tree":  # one expansion per source and one per target, of the default order
        return dict(bytes=8 * (2 * 4 * ns + 5 * ns + 4 * nt), flops=8 * 28 * (3 * ns + nt))
    if p == "panels":  # one panel per particle in each sum, the other panels through expansions
        return dict(bytes=8 * (3 * ns + 4 * ns + 10 * npan), flops=(39 + 47) * ns)
    if p == "bem":
        n = npan * case["nunk"] + 1
        return dict(bytes=8 * n * n + 32 * n,
                    flops=2 * n ** 3 / 3 + 4 * n * n + (92 if case["nunk"] == 1 else 122)
                    * npan * npan)
    if p == "probe":
        w = _pair_work(ns, nt, case["core"], True)
        return dict(bytes=2 * w["bytes"], flops=3 * w["flops"])
    if p == "wall":  # one panel per target and scan
        return dict(bytes=8 * (4 * ns + 3 * ns + 16 * npan), flops=2 * 27 * ns)
    # vort: the pairs within the distance where the exponential underflows
    share = min(1.0, math.pi * 746.0 * 0.005 ** 2 / (0.5 * math.pi * (9.0 - 0.52 ** 2)))
    return dict(bytes=8 * 7 * ns, flops=13 * ns * max(1.0, share * ns))


# ---- the same in 64 bits, without this package's kernels -----------------------------------

_MOST_PAIRS = 9e10  # sums beyond this take too long to repeat pair by pair


def _core(core, d2, w):
    """K and bbb = 2 dK/d(d^2) of src/CoreFunc.h."""
    if core == "rm":
        k = 1.0 / (d2 + w)
        return k, -2.0 * k * k
    if core == "gauss":
        near, x = float(np.float32(0.001)), d2 / w
        e = torch.exp(-x)
        k = torch.where(x > 16.0, 1.0 / d2, torch.where(x < near, 1.0 / w + 0 * d2,
                                                        -torch.expm1(-x) / d2))
        bbb = torch.where(d2 == 0, torch.zeros_like(d2), -2.0 * (k - e / w) / d2)
        return k, bbb
    if core == "wl":
        dd = d2 + w
        return (dd + w) / dd ** 2, (2.0 - 4.0 * (dd + w) / dd) / dd ** 2
    if core == "v2":
        k = (d2 * d2 + w) ** -0.5
        return k, -2.0 * k ** 3 * d2
    v = d2 ** 3 + w
    k = v ** (-1.0 / 3.0)
    return k, -2.0 * d2 * d2 * k / v


_POWER = {"rm": 2, "gauss": 2, "wl": 2, "v2": 4, "v3": 6}


def _exact_pairs(core, x, y, s, r, tx, ty, tr, results="vel"):
    if len(x) * len(tx) > _MOST_PAIRS:
        return (None,) * (2 if results == "vel" else 3)
    p = _POWER[core]
    sw = r ** p
    outs = [torch.zeros_like(tx) for _ in range(2 if results == "vel" else 3)]
    rows = max(1, int(6e7 // len(x)))
    for i in range(0, len(tx), rows):
        j = slice(i, i + rows)
        dx, dy = tx[j, None] - x, ty[j, None] - y
        d2 = dx * dx + dy * dy
        w = sw + (tr[j, None] ** p if tr is not None else 0.0)
        if results == "vel" and core == "gauss":
            k = torch.where(d2 > 16.0 * w, 1.0 / d2, _core(core, d2, w)[0])
        elif results == "vel":
            k = _core(core, d2, w)[0]
        else:
            k, bbb = _core(core, d2, w)
            if results == "vort":
                outs[2][j] = (s * (bbb * d2 + 2.0 * k)).sum(1)
            else:
                outs[2][j] = (0.5 * (s * bbb).abs() * d2).sum(1)
        k = s * k
        outs[0][j] = -(k * dy).sum(1)
        outs[1][j] = (k * dx).sum(1)
    return tuple(outs)


def _panel_log(x0, y0, x1, y1, tx, ty):
    """log((z - z0)/(z - z1)) as (real, imaginary), without cancellation far away."""
    ax, ay, bx, by = tx - x0, ty - y0, tx - x1, ty - y1
    rb = bx * bx + by * by
    diff = (x1 - x0) * (ax + bx) + (y1 - y0) * (ay + by)
    return (0.5 * torch.log1p(diff / rb),
            torch.atan2((y1 - y0) * ax - (x1 - x0) * ay, ax * bx + ay * by))


def _ends(t):
    i, j = t["idx"][0::2].long(), t["idx"][1::2].long()
    x0, y0, x1, y1 = t["nx"][i], t["ny"][i], t["nx"][j], t["ny"][j]
    ln = torch.sqrt((x1 - x0) ** 2 + (y1 - y0) ** 2)
    return x0, y0, x1, y1, (x1 - x0) / ln, (y1 - y0) / ln, ln


def _exact_panels(t):
    x0, y0, x1, y1, ex, ey, ln = _ends(t)
    npan = len(ln)
    pu, pv = torch.zeros_like(ln), torch.zeros_like(ln)
    u, v = torch.zeros_like(t["x"]), torch.zeros_like(t["x"])
    ss = t["ss"] if "ss" in t else torch.zeros_like(ln)
    rows = max(1, int(2e7 // npan))
    for i in range(0, len(u), rows):
        j = slice(i, i + rows)
        lr, li = _panel_log(x0, y0, x1, y1, t["x"][j, None], t["y"][j, None])
        a, b = li * ex - lr * ey, li * ey + lr * ex
        u[j] = (t["vs"] * a + ss * b).sum(1)
        v[j] = (t["vs"] * b - ss * a).sum(1)
        s = t["s"][j, None]
        pu -= (s * a).sum(0) / ln
        pv -= (s * b).sum(0) / ln
    return dict(rhs=(pu, pv), vel=(u, v))


def _exact_bem(case, t):
    x0, y0, x1, y1, ex, ey, ln = _ends(t)
    npan, nunk = case["npan"], case["nunk"]
    mx, my = 0.5 * (x0 + x1), 0.5 * (y0 + y1)
    # [j, i]: panel j on the centre of panel i, and the reverse
    lr, li = _panel_log(x0[:, None], y0[:, None], x1[:, None], y1[:, None], mx, my)
    a1, b1 = li * ex[:, None] - lr * ey[:, None], li * ey[:, None] + lr * ex[:, None]
    a2, b2 = li.T * ex - lr.T * ey, li.T * ey + lr.T * ex
    f = ln[:, None] / ln
    eye = torch.eye(npan, dtype=torch.float64, device=ln.device)

    def entry(p1, q1, p2, q2, nx, ny, diag):
        c = 0.5 * ((p1 * nx + q1 * ny) - f * (p2 * nx + q2 * ny))
        return (torch.where(eye > 0, torch.full_like(c, diag), c)) / (2.0 * math.pi)

    A = torch.zeros((npan * nunk + 1, npan * nunk + 1), dtype=torch.float64, device=ln.device)
    A[:-1:nunk, :-1:nunk] = entry(a1, b1, a2, b2, ex, ey, math.pi)
    A[-1, :-1:nunk] = t["uu"] * ex + t["uv"] * ey
    A[:-1:nunk, -1] = ln
    A[-1, -1] = 2.0 * _VOL
    if nunk == 2:
        A[:-1:2, 1:-1:2] = entry(a1, b1, a2, b2, -ey, ex, 0.0)
        A[1:-1:2, :-1:2] = entry(b1, -a1, b2, -a2, ex, ey, 0.0)
        A[1:-1:2, 1:-1:2] = entry(b1, -a1, b2, -a2, -ey, ex, math.pi)
        A[-1, 1:-1:2] = t["uv"] * ex - t["uu"] * ey
    # A holds the columns as rows
    x = torch.linalg.solve(A.T.contiguous().cpu(), torch.stack([t["b0"], t["b1"]], 1).cpu())
    return dict(A=A, x0=x[:, 0].contiguous(), x1=x[:, 1].contiguous())


def _exact_probe(case, t):
    x, y, s, r = (t[k].detach() for k in ("x", "y", "s", "r"))
    c = 0.5 / math.pi
    u, v = _exact_pairs(case["core"], x, y, s, r, t["tx"], t["ty"], None)
    g = [torch.zeros_like(x) for _ in range(4)]
    gu, gv = c * t["gu"], c * t["gv"]
    cols = max(1, int(6e7 // len(gu)))
    for i in range(0, len(x), cols):
        j = slice(i, i + cols)
        dx, dy = t["tx"] - x[j, None], t["ty"] - y[j, None]
        d2, w = dx * dx + dy * dy, (r[j] ** 2)[:, None]
        k, bbb = _core(case["core"], d2, w)
        if case["core"] == "gauss":
            xx = d2 / w
            far = xx > 16.0
            low = xx < float(np.float32(0.001))
            bbb = torch.where(far, -2.0 / d2 ** 2, torch.where(low, torch.zeros_like(d2), bbb))
            dks = torch.where(far, torch.zeros_like(d2),
                              torch.where(low, -2.0 / (w * r[j, None]) + 0 * d2,
                                          -2.0 * torch.exp(-xx) / (w * r[j, None])))
        else:
            dks = -2.0 * r[j, None] * k * k
        cross = gv * dx - gu * dy
        g[0][j] = s[j] * (gu * bbb * dx * dy - gv * (k + bbb * dx * dx)).sum(1)
        g[1][j] = s[j] * (gu * (k + bbb * dy * dy) - gv * bbb * dx * dy).sum(1)
        g[2][j] = (k * cross).sum(1)
        g[3][j] = s[j] * (dks * cross).sum(1)
    return dict(u=c * u, v=c * v, grad=tuple(g))


def _exact_wall(t):
    x0, y0, x1, y1, ex, ey, ln = _ends(t)
    d = torch.empty_like(t["x"])
    rows = max(1, int(6e7 // len(ln)))
    for i in range(0, len(d), rows):
        j = slice(i, i + rows)
        ax, ay = t["x"][j, None] - x0, t["y"][j, None] - y0
        f = ((ax * ex + ay * ey) / ln).clamp(0.0, 1.0)
        qx, qy = ax - f * (x1 - x0), ay - f * (y1 - y0)
        d[j] = torch.sqrt((qx * qx + qy * qy).amin(1))
    return dict(x=None, y=None, circ=None, counts=None, dist=d)


def _exact_vort(t):
    out = torch.zeros_like(t["x"])
    rr = 1.0 / t["r"] ** 2
    c = 2.0 * t["s"] * rr
    rows = max(1, int(6e7 // len(out)))
    for i in range(0, len(out), rows):
        j = slice(i, i + rows)
        dx, dy = t["x"][j, None] - t["x"], t["y"][j, None] - t["y"]
        out[j] = (c * torch.exp(-(dx * dx + dy * dy) * rr)).sum(1)
    return out


def exact(case, seed):
    p = case["path"]
    a = _arrays(case, seed)
    t = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in a.items()}
    if p == "host":
        d = {k: v.double() for k, v in t.items()}
        return _exact_pairs(case["core"], d["x"], d["y"], d["s"], d["r"], d["tx"], d["ty"],
                            d.get("tr"))
    if p in ("pairs", "tree"):
        src, res, out = [t[k] for k in ("x", "y", "s", "r")], case.get("results", "vel"), {}
        targets = case.get("targets", "self+tracers")
        if targets != "other":
            out["self"] = _exact_pairs(case["core"], *src, t["x"], t["y"], t["r"], res)
        if targets == "other":
            out["other"] = _exact_pairs(case["core"], *src, t["tx"], t["ty"], t["tr"], res)
        if targets == "self+tracers":
            out["tracers"] = _exact_pairs(case["core"], *src, t["tx"], t["ty"], None, res)
        return out
    if p == "panels":
        return _exact_panels(t)
    if p == "bem":
        return _exact_bem(case, t)
    if p == "probe":
        return _exact_probe(case, t)
    if p == "wall":
        return _exact_wall(t)
    if p == "vort":
        return _exact_vort(t)
    if not case["npan"]:  # a step without a body
        x, y, s, r = (t[k] for k in ("x", "y", "s", "r"))
        if case["order"] * len(x) ** 2 > _MOST_PAIRS:
            return None
        vel = lambda px, py: [0.5 / math.pi * v for v in  # noqa: E731
                              _exact_pairs(case["core"], px, py, s, r, px, py, r)]
        c, w = {1: ([], [1.0]), 2: ([2.0 / 3.0], [0.25, 0.75]),
                3: ([0.5, 0.75], [2.0 / 9.0, 3.0 / 9.0, 4.0 / 9.0])}[case["order"]]
        k = [vel(x, y)]
        for ci in c:
            k.append(vel(x + ci * 0.01 * k[-1][0], y + ci * 0.01 * k[-1][1]))
        u = sum(wi * ki[0] for wi, ki in zip(w, k))
        v = sum(wi * ki[1] for wi, ki in zip(w, k))
        return dict(x=x + 0.01 * u, y=y + 0.01 * v, u=u, v=v)
    return None
