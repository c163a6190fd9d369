"""The windowed FP64 march (each option on its window of rows, csrc/fd1d_plan.h and
csrc/fd1d_window.h) against the march on the whole grid.

On the CPU: the window rule over random options of a wide domain, windowed march against
whole-grid march, both serial (tests/cpp/window_test.cpp). The tolerance is relative to
max(strike, price): the truncation is bounded by e^-36 = 2e-16, and each of up to 700 steps
rounds a solve whose rows sum terms up to a few hundred times their result, 1.1e-16 x 100 x
700 = 8e-12 at most.

On the GPU, against the oracle to 1e-8: grids around the row counts that the march is built
for, in both launch forms (one option to a wave; listed by class, with several to a wave),
with options whose exercise boundary goes past their window's cut and are solved again."""
from __future__ import annotations

import os
import pathlib
import subprocess

import numpy as np
import pytest

from kwgpu import workloads as W

ROOT = pathlib.Path(__file__).resolve().parents[1]
TOL_CPU = 1e-11
EPS = 1e-8


@pytest.fixture(scope="module")
def window_test(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("window") / "window_test")
    subprocess.run(["g++", "-O3", "-std=c++17", f"-I{ROOT / 'include'}",
                    str(ROOT / "tests" / "cpp" / "window_test.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("x_dim,t_dim,n", [(128, 65, 1500), (150, 300, 1500), (256, 65, 1000),
                                           (512, 128, 800), (777, 301, 400), (1024, 700, 250),
                                           (2048, 65, 500), (2048, 366, 150)])
def test_windowed_march_on_the_cpu(window_test, x_dim, t_dim, n):
    out = subprocess.run([window_test, str(x_dim), str(t_dim), str(n), "11"], check=True,
                         capture_output=True, text=True, timeout=300).stdout.split()
    windowed, past, outside = map(int, out[:3])
    assert windowed > 0.3 * n          # the rule takes most of the domain
    assert past <= 0.02 * windowed and outside <= 0.02 * windowed
    assert float(out[4]) <= TOL_CPU


# (t, z, r, q, s, w) at strike 100: high volatility and rates near 0, where the approximate
# critical spot is poor and the boundary goes past the cut
PAST_THE_CUT = [
    (0.16324529476271932, 1.1542074201706187, 0.0058532783598809757, -0.02541368762541274, 130.23249887264421, -1),
    (0.0051357653926332762, 1.7302695450043479, 0.032854297777824393, 0.030261211159688689, 52.660916618737311, -1),
    (0.40011942746773849, 1.2247535921312318, 0.00060780990208615313, 0.030878765156926974, 91.590938721047195, 1),
    (0.45726650904244898, 1.1193627107587862, 0.0059062115703023971, -0.0095859986075119592, 399.32953389611703, -1),
    (0.0098166752908992912, 1.79819431433504, 0.021044491937817066, 0.00092198608223913181, 351.64132213923847, -1),
    (0.19437431151915938, 1.8509791712616819, -0.0047107115412769809, 0.021808429681765919, 122.9902156248653, 1),
]


def _options(n, seed):
    """Plain options, every fifth European, spots from deep in to far out of the money, rates
    and yields of 0 and below, and the ones above."""
    o = W.plain(n, seed)
    i = np.arange(n)
    o["e"] = i % 5 != 0
    o["s"] = o["k"] * np.exp(np.linspace(-0.9, 0.9, 31)[i % 31] * np.minimum(1.0, 3 * o["z"] * np.sqrt(o["t"])))
    o["r"] = np.where(i % 11 == 3, -0.01, np.where(i % 11 == 7, 0.0, o["r"]))
    o["q"] = np.where(i % 13 == 5, 0.0, o["q"])
    for k, (t, z, r, q, s, w) in enumerate(PAST_THE_CUT):
        o[7 * k + 1] = (t, 100.0, z, r, q, s, 1, w)
    return o


@pytest.mark.gpu
@pytest.mark.parametrize("x_dim,t_dim", [(129, 65), (192, 80), (256, 66), (257, 90), (400, 65), (512, 130),
                                         (640, 70), (777, 100), (1000, 65), (1024, 256), (1025, 70),
                                         (1500, 90), (2048, 257)])
@pytest.mark.parametrize("n", [64, 2400])
def test_windowed_march_against_the_oracle(ctx, x_dim, t_dim, n):
    import torch

    import kwgpu
    import oracle
    print("windowed march", x_dim, t_dim, n, flush=True)
    o = _options(n, 100 + x_dim)
    d_o = torch.from_numpy(o.view(np.uint8).copy()).cuda()
    d_p = torch.full((n,), np.nan, dtype=torch.float64, device="cuda")
    d_s = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    ctx.fd1d_price_device(d_o.data_ptr(), n, d_p.data_ptr(), d_s.data_ptr(), kwgpu.params(x_dim, t_dim))
    ctx.synchronize()
    p, st = d_p.cpu().numpy(), d_s.cpu().numpy()
    assert np.all(st == kwgpu.STATUS_OK)
    idx = np.arange(64) if n == 64 else np.concatenate([np.arange(48), np.arange(48, n, 147)])
    ref, err = oracle.fd1d_price(o[idx], x_dim, t_dim)
    assert not err
    d = np.abs(p[idx] - ref) / np.maximum(1.0, ref)
    print("  max", d.max(), flush=True)
    assert d.max() <= EPS
