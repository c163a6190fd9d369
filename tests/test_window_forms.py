"""Every launch form of the windowed march over the row counts that it is built for. Per-option grid
sizes always take the windowed march (test_window.py's uniform batches mostly do not: those of
few point-steps take the whole-grid kernels, which test_routes.py and the last test here hold);
the oracle is met to 1e-8, as there. (Its PAST_THE_CUT boundaries stay within the cuts as they are
placed now; test_window_again.py has options that pass theirs.) And the windowed bucket of an uneven batch beside others."""
from __future__ import annotations

import numpy as np
import pytest

import kwgpu
import oracle
from kwgpu import workloads as W
from test_window import EPS, _options

pytestmark = pytest.mark.gpu


def price(ctx, o, xd, td, **kw):
    import torch
    n = len(o)
    d_o = torch.from_numpy(o.view(np.uint8).copy()).cuda()
    d_x, d_t = torch.from_numpy(xd.astype(np.int32)).cuda(), torch.from_numpy(td.astype(np.int32)).cuda()
    d_p = torch.full((n,), np.nan, dtype=torch.float64, device="cuda")
    d_s = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    for _ in range(2):  # the second replays the first one's graph
        ctx.fd1d_price_device(d_o.data_ptr(), n, d_p.data_ptr(), d_s.data_ptr(),
                              kwgpu.params(x_dims=d_x.data_ptr(), t_dims=d_t.data_ptr(), **kw))
        ctx.synchronize()
    assert np.all(d_s.cpu().numpy() == kwgpu.STATUS_OK)
    return d_p.cpu().numpy()


def against_oracle(p, o, xd, td):
    n = len(o)
    idx = np.arange(n) if n <= 64 else np.concatenate([np.arange(48), np.arange(48, n, 147)])
    ref, st = oracle.fd1d_price_uneven(o[idx], xd[idx], td[idx])
    assert np.all(st == 0)
    d = np.abs(p[idx] - ref) / np.maximum(1.0, ref)
    print("  max", d.max(), flush=True)
    assert d.max() <= EPS


@pytest.mark.parametrize("x_dim,t_dim", [(129, 65), (192, 80), (256, 66), (257, 90), (400, 65), (512, 130),
                                         (640, 70), (777, 100), (1000, 65), (1024, 256), (1025, 70),
                                         (1500, 90), (2048, 257)])
@pytest.mark.parametrize("n", [64, 2400])
def test_forms_against_the_oracle(ctx, x_dim, t_dim, n):
    """64 options: one to a wave; 2400: listed by class. Above 1024 points the kernels of both forms
    that take two waves, a few smaller grids among them."""
    print("forms", x_dim, t_dim, n, flush=True)
    o = _options(n, 100 + x_dim)
    xd = np.full(n, x_dim, np.int32)
    if x_dim > 1024:
        xd[2::5] = 700
    against_oracle(price(ctx, o, xd, np.full(n, t_dim, np.int32)), o, xd, np.full(n, t_dim, np.int32))


def test_windowed_bucket_beside_others(tmp_path):
    """Grids of up to 128 points, windowed ones and ones tuned to a whole-grid variant: several
    buckets, launched one after another and side by side, bitwise the same."""
    print("buckets beside each other", flush=True)
    o, xd, td = W.uneven(3000, 79)
    td = np.clip(td, 65, 130).astype(np.int32)
    xd = xd.copy()
    xd[::6], xd[3::6] = 100, 60
    out = []
    for serial in (0, 1):
        path = tmp_path / f"tune{serial}"
        path.write_text(f"512 0 7 1\n-1 {kwgpu.FP64} {serial} 0\n")
        c = kwgpu.Context(0)
        c.tune_load(str(path))
        out.append(price(c, o, xd, td))
        c.close()
    assert np.array_equal(out[0], out[1])
    against_oracle(out[0], o, xd, td)


@pytest.mark.parametrize("n,x_dim,t_dim", [(1024, 896, 65), (1024, 897, 65), (1025, 256, 65), (1025, 257, 65),
                                           (2048, 256, 99), (2048, 256, 100), (2049, 512, 256),
                                           (2049, 512, 257), (512, 1100, 65), (1025, 1025, 65)])
def test_either_side_of_the_rule(ctx, n, x_dim, t_dim):
    """Uniform batches at the lines between the windowed march and the whole-grid kernels."""
    import torch
    print("rule", n, x_dim, t_dim, flush=True)
    o = _options(n, n + x_dim)
    d_o = torch.from_numpy(o.view(np.uint8).copy()).cuda()
    d_p = torch.full((n,), np.nan, dtype=torch.float64, device="cuda")
    d_s = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    ctx.fd1d_price_device(d_o.data_ptr(), n, d_p.data_ptr(), d_s.data_ptr(), kwgpu.params(x_dim, t_dim))
    ctx.synchronize()
    assert np.all(d_s.cpu().numpy() == kwgpu.STATUS_OK)
    against_oracle(d_p.cpu().numpy(), o, np.full(n, x_dim, np.int32), np.full(n, t_dim, np.int32))
