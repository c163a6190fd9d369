"""Uniform batches recorded into a HIP graph by the caller: replays between other work of the
same context give the eager prices (to the rounding of the march: a captured batch that
would need scratch marches on whole grids, 1e-9 of max(strike, price) at most) and are
bitwise the same."""
from __future__ import annotations

import numpy as np
import pytest

import kwgpu
from kwgpu import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("entry", ["device", "noalloc"])
@pytest.mark.parametrize("n,x_dim,t_dim", [(64, 512, 130), (2400, 1024, 256), (1100, 1025, 90)])
def test_replays_of_a_captured_batch(n, x_dim, t_dim, entry):
    import torch
    print("capture", entry, n, x_dim, t_dim, flush=True)
    s = torch.cuda.Stream()
    ctx = kwgpu.Context(0)
    price = ctx.fd1d_price_device if entry == "device" else ctx.fd1d_price_device_noalloc

    def batch(m, seed):
        o = W.plain(m, seed)
        return (o, torch.from_numpy(o.view(np.uint8).copy()).cuda(),
                torch.full((m,), np.nan, dtype=torch.float64, device="cuda"),
                torch.full((m,), -1, dtype=torch.int32, device="cuda"))

    def run(b, x, t):
        price(b[1].data_ptr(), len(b[0]), b[2].data_ptr(), b[3].data_ptr(), kwgpu.params(x, t),
              stream=s.cuda_stream)

    b, other = batch(n, 5), batch(5000, 6)
    torch.cuda.synchronize()
    run(b, x_dim, t_dim)
    torch.cuda.synchronize()
    eager = b[2].cpu().numpy()
    assert np.all(b[3].cpu().numpy() == 0)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        run(b, x_dim, t_dim)
    replays = []
    for _ in range(3):
        with torch.cuda.stream(s):
            b[2].fill_(np.nan)
            b[3].fill_(-1)
            run(other, 512, 400)  # a larger batch, which uses the scratch
            g.replay()
        torch.cuda.synchronize()
        assert np.all(b[3].cpu().numpy() == 0) and np.all(other[3].cpu().numpy() == 0)
        replays.append(b[2].cpu().numpy())
    assert np.array_equal(replays[0], replays[1]) and np.array_equal(replays[0], replays[2])
    assert np.max(np.abs(replays[0] - eager) / np.maximum(b[0]["k"], eager)) <= 1e-9
    ctx.close()
