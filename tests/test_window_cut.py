"""The in-the-money cut of the windowed march (csrc/fd1d_plan.h) over the rates at which it can be
put too near the strike: an option whose exercise boundary passes its cut is marched twice.
On the CPU, with the serial marches of tests/cpp/window_test.cpp."""
from __future__ import annotations

import pathlib
import subprocess

import numpy as np
import pytest

from kwgpu.workloads import OPTION_DTYPE

ROOT = pathlib.Path(__file__).resolve().parents[1]
TOL = 1e-11  # as in test_window.py


@pytest.fixture(scope="module")
def cases(tmp_path_factory):
    """cases(options, x_dim, t_dim): per option lo, end, pinned, inside, the price on the window
    as it is and the price on the whole grid."""
    exe = str(tmp_path_factory.mktemp("cases") / "window_cases")
    subprocess.run(["g++", "-O3", "-std=c++17", f"-I{ROOT / 'include'}",
                    str(ROOT / "tests" / "cpp" / "window_cases.cpp"), "-o", exe], check=True)

    def run(o, x_dim, t_dim, *mesh):
        text = "\n".join(" ".join(repr(float(o[c][i])) if c not in "ew" else str(int(o[c][i]))
                                  for c in ("t", "k", "z", "r", "q", "s", "e", "w"))
                         for i in range(len(o)))
        out = subprocess.run([exe, str(x_dim), str(t_dim), *map(str, mesh)], input=text, text=True,
                             capture_output=True, check=True, timeout=300).stdout
        return np.array([[float(v) for v in ln.split()] for ln in out.splitlines()])
    return run


def draw(n, seed, rate, vol):
    """American puts and calls whose early exercise is worth something: `rate` is a put's rate
    and a call's yield, log-uniform."""
    g = np.random.default_rng(seed)
    o = np.zeros(n, OPTION_DTYPE)
    o["t"] = np.exp(g.uniform(np.log(0.01), np.log(10.0), n))
    o["k"] = 100.0
    o["z"] = g.uniform(*vol, n)
    o["s"] = 100 * np.exp(g.uniform(-1.0, 1.0, n) * np.minimum(1.0, 3 * o["z"] * np.sqrt(o["t"])))
    o["e"] = 1
    o["w"] = np.where(g.random(n) < 0.5, -1, 1)
    earns = np.exp(g.uniform(*np.log(rate), n))
    pays = np.select([np.arange(n) % 3 == 0, np.arange(n) % 3 == 1], [0.0, earns * g.random(n)],
                     g.uniform(-0.01, 0.05, n))
    o["r"] = np.where(o["w"] < 0, earns, pays)
    o["q"] = np.where(o["w"] < 0, pays, earns)
    return o


@pytest.mark.parametrize("rate", [(1e-5, 1e-4), (1e-4, 1e-3), (1e-3, 1e-2), (1e-2, 0.25)])
@pytest.mark.parametrize("vol", [(0.03, 0.3), (0.3, 0.8), (0.8, 1.6)])
@pytest.mark.parametrize("x_dim,t_dim,n", [(512, 300, 400), (1024, 66, 400)])
def test_few_boundaries_pass_their_cut(cases, x_dim, t_dim, n, rate, vol):
    c = cases(draw(n, x_dim + int(1e6 * rate[0]), rate, vol), x_dim, t_dim)
    cut = c[:, 0] > 0
    assert cut.sum() > 0.1 * n
    assert np.sum(cut & (c[:, 2] == 0)) <= 0.02 * cut.sum()
    ok = (c[:, 2] == 1) & (c[:, 3] == 1)
    assert np.max(np.abs(c[ok, 4] - c[ok, 5]) / np.maximum(100.0, c[ok, 5])) <= TOL


@pytest.mark.parametrize("x_dim,t_dim", [(256, 66), (400, 90), (512, 130), (777, 70), (1024, 66)])
def test_calls_of_long_maturity_and_low_yield(cases, x_dim, t_dim):
    """Far in the money a call's payoff grows with the spot, and so does what the differences are
    off by there: past some row the scheme never exercises, and a cut must not take those rows for
    pinned. Spots deep in the money, near the boundary, and at the strike."""
    g = np.random.default_rng(x_dim)
    n = 600
    o = np.zeros(n, OPTION_DTYPE)
    s = g.uniform(0.8, 1.8, n)
    o["z"] = g.uniform(0.25, 0.7, n)
    o["t"] = (s / o["z"]) ** 2
    o["k"], o["e"], o["w"] = 100.0, 1, 1
    o["r"] = g.uniform(1.0, 3.5, n) / o["t"]
    o["q"] = o["r"] * np.exp(-g.uniform(2.0, 4.4, n) * s)
    o["s"] = 100 * np.where(np.arange(n) % 4 == 0, 1.0, np.exp(g.uniform(3.0, 4.9, n) * s))
    c = cases(o, x_dim, t_dim)
    cut = c[:, 0] > 0
    assert np.sum(cut & (c[:, 2] == 0)) <= 0.02 * n
    ok = (c[:, 2] == 1) & (c[:, 3] == 1)
    assert np.max(np.abs(c[ok, 4] - c[ok, 5]) / np.maximum(100.0, c[ok, 5])) <= TOL


def extreme(n, seed):
    """Maturities and rates at which the march on a whole grid can overflow, the drift small: cost
    of carry near half the variance. Sizes too: x points and t points."""
    g = np.random.default_rng(seed)
    o = np.zeros(n, OPTION_DTYPE)
    s = 3.0 * np.exp(g.uniform(np.log(1e-3), 0.0, n))
    o["t"] = np.exp(g.uniform(np.log(100.0), np.log(1000.0), n))
    o["k"] = o["s"] = 100.0
    o["z"] = s / np.sqrt(o["t"])
    o["r"] = g.uniform(-0.99, -0.2, n)
    o["q"] = o["r"] - 0.5 * o["z"] ** 2 - 2.9 * s / o["t"] * g.uniform(-1, 1, n)
    o["e"] = np.arange(n) % 4 != 0
    o["w"] = np.where(g.random(n) < 0.5, -1, 1)
    return o, g.integers(129, 1024, n), g.integers(66, 500, n)


def test_no_window_where_the_whole_grid_overflows(cases):
    o, xd, td = extreme(400, 1)
    over = 0
    for i in range(len(o)):
        lo, end, _, _, _, whole = cases(o[i:i + 1], xd[i], td[i])[0]
        if not np.isfinite(whole):
            over += 1
            assert (lo, end) == (0, xd[i]), (o[i], xd[i], td[i])
    assert over >= 40


@pytest.mark.gpu
def test_overflow_is_reported(ctx, tmp_path):
    """A march that overflows reports it, whichever launch form its batch takes: the statuses are
    those of the whole-grid kernels (the oracle eliminates serially, and overflows for nearly
    the same options)."""
    import torch

    import kwgpu
    import oracle
    print("overflow", flush=True)
    o, xd, td = extreme(1200, 2)
    whole = kwgpu.Context(0)
    (tmp_path / "tune").write_text("256 0 2 0\n512 0 5 0\n1024 0 8 0\n2048 0 9 0\n")
    whole.tune_load(str(tmp_path / "tune"))
    for cap in (1024, 512):  # a wave an option; with one grid of over 1024 points among them
        m = 1200 if cap == 1024 else 500
        x = np.minimum(xd[:m], cap).astype(np.int32)
        if cap == 512:
            x[0] = 1500
        t = td[:m].astype(np.int32)
        d_o = torch.from_numpy(o[:m].view(np.uint8).copy()).cuda()
        d_x, d_t = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
        prm = kwgpu.params(x_dims=d_x.data_ptr(), t_dims=d_t.data_ptr())
        st = []
        for c in (ctx, whole):
            d_p = torch.zeros(m, dtype=torch.float64, device="cuda")
            d_s = torch.full((m,), -1, dtype=torch.int32, device="cuda")
            torch.cuda.synchronize()
            c.fd1d_price_device(d_o.data_ptr(), m, d_p.data_ptr(), d_s.data_ptr(), prm)
            c.synchronize()
            st.append(d_s.cpu().numpy())
        assert np.array_equal(st[0], st[1])
        bad = ~np.isfinite(oracle.fd1d_price_uneven(o[:m], x, t)[0])
        assert bad.sum() > 50 and np.mean(st[0][bad] == kwgpu.STATUS_NONFINITE) > 0.95
    whole.close()
