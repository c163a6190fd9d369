"""The second solve of the windowed march (csrc/fd1d_window.h): an option whose exercise boundary
passes its window's cut, or whose price is asked for at a call's unprojected edge row, is solved
again on its whole grid. Each place that does so, with options that the first solve prices wrongly.

The rule places a cut in FP32, which at sigma sqrt(T) of 1e-4 to 4e-4 and rates next to the yield is
off by up to 0.4 sigma sqrt(T): nearly every boundary of such options passes its cut, on meshes laid
as close to the strike. Their spots are put just inside the cut, where the price of the first
solve is off by over 1e-6 (asserted on the CPU with the serial marches of
tests/cpp/window_test.cpp). The oracle's price is met to 1e-8: 512 steps round by 8e-12 of
max(strike, price) at most, as derived in test_window.py."""
from __future__ import annotations

import numpy as np
import pytest

from kwgpu.workloads import OPTION_DTYPE
from test_window_cut import cases  # noqa: F401

EPS = 1e-8
# density, x points, t points: windows of 16 lanes, 16 and 32, 32, 64, 64; then of grids of over 1024
# points in 64 lanes, 64 lanes, two waves
GRIDS = [(5e-4, 512, 130), (5e-4, 1024, 257), (2e-4, 1000, 66), (2e-5, 1024, 257), (2e-7, 1024, 257)]
BIG = [(5e-4, 2048, 257), (2e-5, 1500, 90), (2e-6, 1500, 90), (2e-5, 2048, 257)]


def mesh(o, x_dim, density):
    y = np.arcsinh(50 * o["z"] * np.sqrt(o["t"]) / density)
    return density * np.sinh(-y + 2 * y * np.arange(x_dim) / (x_dim - 1))


def passers(cases, n, seed, density, x_dim, t_dim):
    """n options that pass their cut, the price of the first solve off by over 1e-6."""
    m = 16 * n
    g = np.random.default_rng(seed)
    o = np.zeros(m, OPTION_DTYPE)
    o["t"] = np.exp(g.uniform(np.log(0.0012), np.log(0.004), m))
    o["z"] = np.exp(g.uniform(np.log(0.003), np.log(0.006), m))
    o["k"] = o["s"] = 100.0
    o["e"] = 1
    o["w"] = np.where(g.random(m) < 0.5, -1, 1)
    o["r"] = g.uniform(0.3, 0.9, m)
    o["q"] = o["r"] * (1 + g.uniform(-3e-6, 3e-6, m))
    c = cases(o, x_dim, t_dim, density, 50)
    for i in np.nonzero(c[:, 0] > 0)[0]:
        x = mesh(o[i], x_dim, density)[int(c[i, 0]):][:2].mean()
        o["s"][i] = 100 * np.exp(x if o["w"][i] < 0 else -x)
    c = cases(o, x_dim, t_dim, density, 50)
    hit = (c[:, 0] > 0) & (c[:, 2] == 0) & (np.abs(c[:, 4] - c[:, 5]) > 1e-6)
    assert hit.sum() >= n, (density, x_dim, t_dim, hit.sum())
    return o[hit][:n]


def batch(cases, n, seed, density, x_dim, t_dim):
    """Passers and, every third, their European twins, which have no cut (options of ordinary sigma
    sqrt(T) round by up to 1e-5 on such meshes, in any march); every ninth a call priced in its
    mesh's last cell."""
    p = passers(cases, 12, seed, density, x_dim, t_dim)
    i = np.arange(n)
    o = p[i % len(p)].copy()
    o["e"] = i % 3 != 1
    for k in np.nonzero(i % 9 == 5)[0]:
        o["w"][k] = 1
        o["s"][k] = 100 * np.exp(mesh(o[k], x_dim, density)[-2:].mean())
    return o


@pytest.mark.parametrize("density,x_dim,t_dim", GRIDS + BIG)
def test_the_first_solve_is_not_enough(cases, density, x_dim, t_dim):
    assert len(passers(cases, 12, x_dim, density, x_dim, t_dim)) == 12


@pytest.mark.gpu
@pytest.mark.parametrize("form,density,x_dim,t_dim",
                         [(f, *g) for f in ("lone", "listed") for g in GRIDS] +
                         [(f, *g) for f in ("lone_big", "listed_big") for g in GRIDS[::2] + BIG])
def test_solved_again(ctx, cases, form, density, x_dim, t_dim):
    """lone: an option a wave, up to 2048; lone_big: up to 1024 with grids of over 1024 points;
    listed by class beyond. Per-option grids take the windowed march whatever the sizes."""
    import torch

    import kwgpu
    import oracle
    print("solved again", form, density, x_dim, t_dim, flush=True)
    n = {"lone": 64, "listed": 2400, "lone_big": 64, "listed_big": 1400}[form]
    o = batch(cases, n, x_dim, density, x_dim, t_dim)
    xd = np.full(n, x_dim, np.int32)
    if form.endswith("big"):
        xd[1::30] = 1100
    td = np.full(n, t_dim, np.int32)
    d_o = torch.from_numpy(o.view(np.uint8).copy()).cuda()
    d_x, d_t = torch.from_numpy(xd).cuda(), torch.from_numpy(td).cuda()
    d_p = torch.full((n,), np.nan, dtype=torch.float64, device="cuda")
    d_s = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    ctx.fd1d_price_device(d_o.data_ptr(), n, d_p.data_ptr(), d_s.data_ptr(),
                          kwgpu.params(density=density, x_dims=d_x.data_ptr(), t_dims=d_t.data_ptr()))
    ctx.synchronize()
    p, st = d_p.cpu().numpy(), d_s.cpu().numpy()
    assert np.all(st == kwgpu.STATUS_OK), np.unique(st, return_counts=True)
    idx = np.arange(n) if n == 64 else np.concatenate([np.arange(32), np.arange(32, n, 41)])
    ref, rst = oracle.fd1d_price_uneven(o[idx], xd[idx], td[idx], density=density)
    assert np.all(rst == 0)
    d = np.abs(p[idx] - ref) / np.maximum(1.0, ref)
    print("  max", d.max(), flush=True)
    assert d.max() <= EPS
