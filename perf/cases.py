"""What a user of this framework has it do, as cases that can be timed and checked.

A case is a dict of plain values. `listed()` gives the fixed ones, `draw(rng)` one more of
the same ranges, `prepare(case, seed)` the inputs and handles a program holds before the
call, `run(state)` one pass through the public entry points, `work(case)` the bytes and
operations that pass cannot do without, and `exact(case, seed)` the same outputs from plain
torch in 64 bits.

Kinds of case:
  quote      host options -> host prices, kwgpu_fd1d_price: a desk or a unit test that
             prices a handful of contracts, or a book in which options that differ only in
             spot share one PDE
  control    host options -> host prices of the FD1D-BS control variate
  greeks     host options -> price and five Greeks by central bumps
  batch      device options -> device prices, one grid for all (FP64 or FP32-mixed)
  uneven     device options -> device prices, a grid size per option
  european   device options -> closed-form device prices
  serving    surrogate-first pricing of a device batch through the gate by class
  training   passes of Adam over labelled rows on the device, and the weights they give
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "kwinto-cuda_amd"))

import kwgpu  # noqa: E402
from kwgpu.workloads import OPTION_DTYPE  # noqa: E402

DENSITY, SCALE = 0.25, 50.0
BUMP = 0.01
# training box and gate classes as the serving pipeline uses them
BOX = {"k": (40.0, 200.0), "t": (1.0 / 52.0, 5.0), "z": (0.1, 0.6)}
PLAIN = {"k": (50.0, 150.0), "t": (1.0 / 12.0, 3.0), "z": (0.1, 0.6)}
WIDE = {"k": (50.0, 150.0), "t": (1.0 / 12.0, 3.0), "z": (0.05, 0.8)}
T_EDGES, M_EDGES = (0.5, 2.0), (0.0,)
SPREAD_MAX, SCALE_MAX = 2e-5, 0.1
# point-steps of the largest listed case: no drawn case costs more
MOST = 32768 * 1024 * 1023


def listed():
    return [
        # twelve contracts, the reference's unit test: latency and launches, not throughput
        {"name": "quote_12", "kind": "quote", "pdes": 12, "spots": 1, "x": 512, "t": 512},
        # a put portfolio of 600 PDEs with ten spots each, the reference's own fixture
        {"name": "book_6000", "kind": "quote", "pdes": 600, "spots": 10, "x": 512, "t": 512},
        # the control variate on an overnight book: American and European legs
        {"name": "control_500", "kind": "control", "n": 500, "x": 512, "t": 512},
        # risk of a book: seven PDEs per option
        {"name": "greeks_300", "kind": "greeks", "n": 300, "x": 512, "t": 512},
        # the smallest published device batch at the default grid
        {"name": "batch_128x512", "kind": "batch", "n": 128, "x": 512, "t": 512, "mixed": False,
         "american": True},
        # an ordinary batch of odd sizes, European and not
        {"name": "batch_3001x777", "kind": "batch", "n": 3001, "x": 777, "t": 301, "mixed": False,
         "american": False},
        # the headline workload
        {"name": "batch_32768x1024", "kind": "batch", "n": 32768, "x": 1024, "t": 1024,
         "mixed": False, "american": True},
        # the FP32-mixed march
        {"name": "mixed_4096x1024", "kind": "batch", "n": 4096, "x": 1024, "t": 1024,
         "mixed": True, "american": True},
        # grid sizes per option: 256 to 2048 x-points, a step per day
        {"name": "uneven_16384", "kind": "uneven", "n": 16384},
        # closed-form prices of a million European options
        {"name": "european_1m", "kind": "european", "n": 1 << 20},
        # surrogate-first serving in front of FP64 FD
        {"name": "serving_32768", "kind": "serving", "n": 32768, "x": 1024, "t": 1024},
        # two epochs of ensemble training at the default batch size
        {"name": "training_32768", "kind": "training", "n": 16384, "epochs": 2, "batch": 8192},
    ]


def _size(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi], odd ones among them."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["quote", "control", "greeks", "batch", "batch", "batch", "uneven", "european",
                       "serving", "training"])
    if kind == "european":
        return {"kind": kind, "n": _size(rng, 1 << 17, 1 << 20)}
    if kind == "uneven":
        return {"kind": kind, "n": _size(rng, 256, 32768)}
    if kind == "training":
        batch = _size(rng, 1024, 8192)
        return {"kind": kind, "n": _size(rng, batch, 24576), "epochs": rng.randint(1, 2), "batch": batch}
    if kind == "serving":
        return {"kind": kind, "n": _size(rng, 2048, 32768), "x": 1024, "t": 1024}
    x = rng.choice([128, 256, 512, 1024, _size(rng, 64, 2048), _size(rng, 64, 2048)])
    t = rng.choice([256, 512, 1024, _size(rng, 32, 1100), _size(rng, 32, 1100)])
    most = MOST // (x * t)
    if kind == "quote":
        pdes = _size(rng, 1, min(2000, most))
        return {"kind": kind, "pdes": pdes, "spots": rng.choice([1, 1, 3, 10]), "x": x, "t": t}
    if kind in ("control", "greeks"):
        return {"kind": kind, "n": _size(rng, 1, min(600, most // 9)), "x": x, "t": t}
    mixed = rng.random() < 0.25
    return {"kind": kind, "n": _size(rng, 64, min(32768, most // (3 if mixed else 1))), "x": x, "t": t,
            "mixed": mixed, "american": rng.random() < 0.75}


# ---- inputs ----------------------------------------------------------------------------


def _options(n, seed, box, american=True):
    g = np.random.default_rng([20240, int(seed)])
    o = np.zeros(n, OPTION_DTYPE)
    o["k"] = g.uniform(*box["k"], n)
    o["t"] = g.uniform(*box["t"], n)
    o["z"] = g.uniform(*box["z"], n)
    o["r"] = g.uniform(0.0, 0.1, n)
    o["q"] = g.uniform(0.0, 0.08, n)
    o["w"] = np.where(g.random(n) < 0.5, -1, 1)
    o["s"] = 100.0
    o["e"] = 1 if american else g.random(n) < 0.5
    return o, g


def _book(case, seed):
    """pdes contracts, each at `spots` spots around its strike (spots 1: at 100)."""
    o, g = _options(case["pdes"], seed, PLAIN)
    if case["spots"] > 1:
        o["k"] = 100.0
        o = np.repeat(o, case["spots"])
        o["s"] = np.tile(np.linspace(50.0, 175.0, case["spots"]), case["pdes"]) * g.uniform(0.95, 1.05, len(o))
    return o


def _uneven_grids(n, o, g):
    """Grid sizes as the uneven workload takes them, and its 2 % low-vol long-dated slice."""
    x = np.array([256, 512, 1024, 2048], np.int32)[g.integers(0, 4, n)]
    s = np.arange(n) % 50 == 0
    o["z"] = np.where(s, g.uniform(0.05, 0.08, n), o["z"])
    o["t"] = np.where(s, g.uniform(2.5, 3.0, n), o["t"])
    return x, np.maximum(32, np.ceil(365.0 * o["t"])).astype(np.int32)


def _inputs(case, seed):
    """(options, per-option x points or None, per-option t points or None)"""
    kind = case["kind"]
    if kind == "quote":
        return _book(case, seed), None, None
    if kind in ("control", "greeks"):
        return _options(case["n"], seed, PLAIN)[0], None, None
    if kind == "batch":
        return _options(case["n"], seed, PLAIN, case["american"])[0], None, None
    if kind == "uneven":
        o, g = _options(case["n"], seed, WIDE)
        x, t = _uneven_grids(case["n"], o, g)
        return o, x, t
    if kind == "european":
        o = _options(case["n"], seed, PLAIN)[0]
        o["e"] = 0
        return o, None, None
    if kind == "serving":
        # every tenth option outside the training box, as in the serving workload
        o, g = _options(case["n"], seed, BOX)
        out = np.arange(case["n"]) % 10 == 0
        far = g.random(case["n"]) < 0.5
        o["t"] = np.where(out & far, g.uniform(5.0, 6.0, case["n"]), o["t"])
        o["z"] = np.where(out & ~far, g.uniform(0.6, 0.8, case["n"]), o["z"])
        return o, None, None
    return _options(case["n"], seed, BOX)[0], None, None


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.uint8).copy()).cuda()


def _ensemble(ctx, members=4):
    """Four networks whose outputs are as small and as near each other as a fitted
    ensemble's: the initial weights with the output layer scaled down."""
    s = kwgpu.Surrogate(ctx, members, seed=1)
    for m in range(members):
        w = s.get_params(m)
        w[-257:] *= 1e-3  # W5 and b5
        s.set_params(m, w)
    return s


def prepare(case, seed):
    o, x, t = _inputs(case, seed)
    n = len(o)
    s = {"case": case, "n": n, "ctx": kwgpu.Context(0)}
    kind = case["kind"]
    if kind in ("quote", "control", "greeks"):
        s["opts"] = o
        return s
    s["d_opts"] = _dev(o)
    s["prices"] = torch.empty(n, dtype=torch.float64, device="cuda")
    s["status"] = torch.empty(n, dtype=torch.int32, device="cuda")
    if kind == "batch":
        s["p"] = kwgpu.params(case["x"], case["t"],
                              precision=kwgpu.FP32_MIXED if case["mixed"] else kwgpu.FP64)
    elif kind == "uneven":
        s["x"], s["t"] = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
        s["p"] = kwgpu.params(x_dims=s["x"].data_ptr(), t_dims=s["t"].data_ptr())
    elif kind == "serving":
        s["sur"] = _ensemble(s["ctx"])
        s["p"] = kwgpu.params(case["x"], case["t"])
        k = 2 * (len(T_EDGES) + 1) * (len(M_EDGES) + 1)
        s["gate"] = kwgpu.gate(T_EDGES, M_EDGES, [SPREAD_MAX] * k, [SCALE_MAX] * k)
    elif kind == "training":
        # rows at the two mesh nodes around each option's spot, labelled by the FD pricer
        s["sur"] = kwgpu.Surrogate(s["ctx"], 4, seed=2)
        s["nodes"] = torch.empty(2 * n * OPTION_DTYPE.itemsize, dtype=torch.uint8, device="cuda")
        s["premium"] = torch.empty(2 * n, dtype=torch.float64, device="cuda")
        keep = torch.empty(n, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        kwgpu.surrogate_labels(s["ctx"], s["d_opts"].data_ptr(), n, kwgpu.params(1024, 256),
                               s["nodes"].data_ptr(), s["premium"].data_ptr(), keep.data_ptr())
    return s


# ---- one pass --------------------------------------------------------------------------


def run(s):
    case, ctx, n = s["case"], s["ctx"], s["n"]
    kind = case["kind"]
    if kind == "quote":
        prices, status, _, _ = ctx.fd1d_price(s["opts"], case["x"], case["t"])
        return {"prices": prices, "status": status}
    if kind == "control":
        prices, status, _, _ = ctx.fd1d_bs_price(s["opts"], case["x"], case["t"])
        return {"prices": prices, "status": status}
    if kind == "greeks":
        g, status, _, _ = ctx.fd1d_greeks(s["opts"], case["x"], case["t"], bump=BUMP)
        return {**{f: g[f] for f in g.dtype.names}, "status": status}
    if kind in ("batch", "uneven"):
        ctx.fd1d_price_device(s["d_opts"].data_ptr(), n, s["prices"].data_ptr(),
                              s["status"].data_ptr(), s["p"])
        return {"prices": s["prices"], "status": s["status"]}
    if kind == "european":
        ctx.bs_price_device(s["d_opts"].data_ptr(), n, s["prices"].data_ptr())
        return {"prices": s["prices"]}
    if kind == "serving":
        routed = s["sur"].price_gated(s["d_opts"].data_ptr(), n, s["gate"], s["p"],
                                      s["prices"].data_ptr(), s["status"].data_ptr())
        return {"prices": s["prices"], "route": s["status"], "routed": routed}
    loss = s["sur"].train(s["nodes"].data_ptr(), s["premium"].data_ptr(), 2 * n,
                          epochs=case["epochs"], batch=case["batch"])
    return {"loss": loss, "weights": [s["sur"].get_params(m) for m in range(4)]}


def work(case):
    """FD: 10 operations per grid point and step (three-point right-hand side, forward and
    backward substitution), an option's record read and its price and status written.
    European: the closed form's two normal distributions. Network: 2 operations per weight
    and row, three times that for a training step."""
    kind = case["kind"]
    dense = 8 * 256 + 3 * 256 * 256 + 256
    if kind == "european":
        return {"bytes": 64 * case["n"], "flops": 100 * case["n"]}
    if kind == "training":
        rows = (2 * case["n"]) // case["batch"] * case["batch"] * case["epochs"]
        return {"bytes": 64 * 2 * case["n"] + 4 * 4 * 199937 * 4, "flops": 6 * dense * rows * 4}
    if kind == "uneven":
        # mean of x in {256, 512, 1024, 2048}, and of 365 T over the drawn maturities
        return {"bytes": 76 * case["n"], "flops": 10 * 960 * 570 * case["n"]}
    pde = 10 * case["x"] * (case["t"] - 1)
    if kind == "quote":
        return {"bytes": 68 * case["pdes"] * case["spots"], "flops": pde * case["pdes"]}
    if kind == "control":
        return {"bytes": 68 * case["n"], "flops": 2 * pde * case["n"]}
    if kind == "greeks":
        return {"bytes": 108 * case["n"], "flops": 7 * pde * case["n"]}
    if kind == "serving":
        # about a third of the options served by four networks at two nodes each
        return {"bytes": 68 * case["n"], "flops": (0.65 * pde + 0.35 * 8 * 2 * dense) * case["n"]}
    return {"bytes": 68 * case["n"], "flops": pde * case["n"]}


# ---- the same in 64 bits ----------------------------------------------------------------


def _fields(o):
    return {f: torch.from_numpy(o[f].astype(np.float64)).cuda() for f in "tkzrqsew"}


def _fd_group(o, N, tn):
    """Crank-Nicolson prices of options on one x size: N points, tn[i] t-points each. Every
    row is built as the finite-difference scheme states it; each step's tridiagonal system
    is solved by parallel cyclic reduction over the rows, whose coefficients are the same at
    every step."""
    f = _fields(o)
    n = len(o)
    T, z, r, q = f["t"], f["z"], f["r"], f["q"]
    steps = torch.from_numpy(tn.astype(np.int64)).cuda() - 1
    dt = T / steps
    half = SCALE * z * torch.sqrt(T)
    y0, y1 = torch.asinh(-half / DENSITY), torch.asinh(half / DENSITY)
    u = (torch.arange(N, device="cuda", dtype=torch.float64) / (N - 1))[:, None]
    x = DENSITY * torch.sinh(y0 * (1 - u) + y1 * u)  # rows x options
    call = f["w"] > 0
    pay = torch.where(call, torch.exp(x) - 1, 1 - torch.exp(x)).clamp(min=0)
    ax, axx = r - q - z * z / 2, z * z / 2
    lo, di, up = (torch.zeros_like(x) for _ in range(3))  # rows of the operator
    du, dd, dm = x[2:] - x[1:-1], x[1:-1] - x[:-2], x[2:] - x[:-2]
    lo[1:-1] = -ax / dm + 2 * axx / (dd * dm)
    up[1:-1] = ax / dm + 2 * axx / (du * dm)
    di[1:-1] = -r - 2 * axx / (dd * du)
    di[0], up[0] = -r - ax / (x[1] - x[0]), ax / (x[1] - x[0])
    lo[-1], di[-1] = -ax / (x[-1] - x[-2]), -r + ax / (x[-1] - x[-2])
    h = 0.5 * dt
    a, b, c = -h * lo, 1 - h * di, -h * up
    stages, s = [], 1
    while s < N:
        k1, k2 = torch.zeros_like(x), torch.zeros_like(x)
        k1[s:] = -a[s:] / b[:-s]
        k2[:-s] = -c[:-s] / b[s:]
        nb = b.clone()
        nb[s:] += k1[s:] * c[:-s]
        nb[:-s] += k2[:-s] * a[s:]
        na, nc = torch.zeros_like(x), torch.zeros_like(x)
        na[s:] = k1[s:] * a[:-s]
        nc[:-s] = k2[:-s] * c[s:]
        a, b, c = na, nb, nc
        stages.append((s, k1[s:].contiguous(), k2[:-s].contiguous()))
        s *= 2
    inv = 1 / b
    del a, b, c, na, nb, nc
    floor = torch.where((f["e"] > 0), pay, torch.full_like(pay, -math.inf))
    floor[-1] = -math.inf
    v = pay.clone()
    el, ed, eu = h * lo, 1 + h * di, h * up
    del lo, di, up
    most, least = int(steps.max()), int(steps.min())
    d, w = torch.empty_like(v), torch.empty_like(v)
    for k in range(most):
        torch.mul(ed, v, out=d)
        d[1:].addcmul_(el[1:], v[:-1])
        d[:-1].addcmul_(eu[:-1], v[1:])
        for s, k1, k2 in stages:
            w.copy_(d)
            w[s:].addcmul_(k1, d[:-s])
            w[:-s].addcmul_(k2, d[s:])
            d, w = w, d
        d.mul_(inv)
        torch.maximum(d, floor, out=d)
        if k < least:
            d, v = v, d
        else:
            v = torch.where(k < steps, d, v)
    xs = torch.log(f["s"] / f["k"])
    j = (x < xs).sum(0).clamp(1, N - 1)
    i = torch.arange(n, device="cuda")
    x1, x0 = x[j, i], x[j - 1, i]
    return (f["k"] * ((x1 - xs) * v[j - 1, i] + (xs - x0) * v[j, i]) / (x1 - x0)).cpu().numpy()


def _fd(o, x, t):
    out = np.empty(len(o))
    for N in np.unique(x):
        at = np.flatnonzero(x == N)
        at = at[np.argsort(t[at], kind="stable")]
        per = max(1, (1 << 25) // int(N))  # 256 MiB an array
        for k in range(0, len(at), per):
            sel = at[k:k + per]
            out[sel] = _fd_group(o[sel], int(N), t[sel])
    return out


def _bs(o):
    f = _fields(o)
    sd = f["z"] * torch.sqrt(f["t"])
    d1 = (torch.log(f["s"] / f["k"]) + (f["r"] - f["q"] + 0.5 * f["z"] ** 2) * f["t"]) / sd
    w = f["w"]

    def cdf(v):
        return 0.5 * torch.erfc(-v / math.sqrt(2.0))

    p = w * (f["s"] * torch.exp(-f["q"] * f["t"]) * cdf(w * d1)
             - f["k"] * torch.exp(-f["r"] * f["t"]) * cdf(w * (d1 - sd)))
    return p.cpu().numpy()


def _same_grid(o, case):
    return _fd(o, np.full(len(o), case["x"], np.int32), np.full(len(o), case["t"], np.int32))


def exact(case, seed):
    """Prices and Greeks of the finite-difference scheme in 64 bits, also for the FP32-mixed
    march and for surrogate-first serving (whose prices stand for it). None for training,
    whose rows are shuffled by a generator of the framework's own."""
    kind = case["kind"]
    if kind == "training":
        return None
    o, x, t = _inputs(case, seed)
    if kind == "uneven":
        return {"prices": _fd(o, x, t), "status": None}
    if kind == "european":
        return {"prices": _bs(o)}
    if kind == "control":
        e = o.copy()
        e["e"] = 0
        return {"prices": _same_grid(o, case) + _bs(e) - _same_grid(e, case), "status": None}
    if kind == "greeks":
        def at(field, by):
            b = o.copy()
            b[field] = b[field] * by
            return _same_grid(b, case)

        out = {"price": _same_grid(o, case), "status": None}
        for name, field, per in (("vega", "z", 100.0), ("theta", "t", 360.0), ("rho", "r", 100.0)):
            out[name] = (at(field, 1 + BUMP) - at(field, 1 - BUMP)) / (2 * BUMP * o[field]) / per
        up, down = at("s", 1 + BUMP), at("s", 1 - BUMP)
        out["delta"] = (up - down) / (2 * BUMP * o["s"])
        out["gamma"] = (up - 2 * out["price"] + down) / (BUMP * o["s"]) ** 2
        return out
    if kind == "serving":
        return {"prices": _same_grid(o, case), "route": None, "routed": None}
    return {"prices": _same_grid(o, case), "status": None}
