"""The tuner's last step: every bucket windowed that can be, in one launch, against the buckets' own
choices. Whatever it keeps is what its report says, holds the prices, and survives a tune file."""
from __future__ import annotations

import numpy as np
import pytest

import kwgpu
from kwgpu import workloads as W

pytestmark = pytest.mark.gpu


def test_windows_together(tmp_path):
    import torch
    print("tuner, windows together", flush=True)
    o, xd, td = W.uneven(6000, 78)
    td = np.clip(td, 65, 200).astype(np.int32)
    n = len(o)
    d_o = torch.from_numpy(o.view(np.uint8).copy()).cuda()
    d_x, d_t = torch.from_numpy(xd).cuda(), torch.from_numpy(td).cuda()
    d_p = torch.empty(n, dtype=torch.float64, device="cuda")
    d_s = torch.empty(n, dtype=torch.int32, device="cuda")
    prm = kwgpu.params(x_dims=d_x.data_ptr(), t_dims=d_t.data_ptr())
    torch.cuda.synchronize()

    def price(c):
        d_p.fill_(np.nan)
        torch.cuda.synchronize()
        c.fd1d_price_device(d_o.data_ptr(), n, d_p.data_ptr(), d_s.data_ptr(), prm)
        c.synchronize()
        assert np.all(d_s.cpu().numpy() == 0)
        return d_p.cpu().numpy()

    c = kwgpu.Context(0)
    before = price(c)
    rep = c.autotune(d_o.data_ptr(), n, d_p.data_ptr(), d_s.data_ptr(), prm)
    windowed = [b["candidates"][b["chosen"]].get("windowed", False) for b in rep["buckets"]]
    together, apart = rep.get("windowed_together"), rep["schedule"]
    assert (together is None) == all(windowed)
    if together:
        fastest = min(apart["concurrent_ms"], apart["serial_ms"])
        # (printed to 1e-4 ms)
        assert together["chosen"] == (together["ms"] < 0.98 * fastest) or \
            abs(together["ms"] - 0.98 * fastest) < 2e-4
    after = price(c)
    assert np.max(np.abs(after - before) / np.maximum(o["k"], before)) <= 1e-10
    path = str(tmp_path / "tune")
    c.tune_save(path)
    d = kwgpu.Context(0)
    d.tune_load(path)
    assert np.array_equal(price(d), after)
    c.close()
    d.close()
