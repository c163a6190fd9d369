"""The training step's kernels (csrc/surrogate_step.h) at the edges of their tiles: blocks of
fewer rows than a tile, a block's seventeenth row (five 16-row tiles), several passes over a
block, ragged last splits of the weight gradients; and the BF16 weights that an Adam step
leaves, as they are and transposed, for every member.

Against the FP64 oracle with the kernels' BF16 roundings. An FP32 pre-activation next to a
rounding edge may round the other way: one activation in about 2^24 / 2^9 x 100 by 2^-8 of
itself, so a gradient slice's relative error stays under 2^-8 = 4e-3 at any number of rows."""
from __future__ import annotations

import numpy as np
import pytest

from test_surrogate_gpu import F, H, SLICES, kB1, kB2, kB3, kB4, kB5, kW5, oracle_loss_grad

kwgpu = pytest.importorskip("kwgpu")
pytestmark = pytest.mark.gpu
TOL = 4e-3


def _check(sur, member, n, seed):
    rng = np.random.default_rng(seed)
    x = rng.uniform(-1, 1, (n, F)).astype(np.float32)
    t = rng.normal(0, 0.5, n).astype(np.float32)
    loss, g = sur.loss_grad(member, x, t)
    rl, rg = oracle_loss_grad(sur.get_params(member), x, t)
    assert abs(loss - rl) <= 1e-4 * abs(rl)
    for name, (a, b) in SLICES.items():
        err = np.linalg.norm(g[a:b] - rg[a:b]) / max(np.linalg.norm(rg[a:b]), 1e-30)
        assert err < TOL, (n, name, err)


@pytest.mark.parametrize("n", [1, 3, 63, 65, 127, 129, 1025, 1087, 4100, 8192, 8193, 16400, 40000])
def test_gradient_at_tile_edges(ctx, n):
    print("rows", n, flush=True)
    sur = kwgpu.Surrogate(ctx, members=2, seed=17)
    w = sur.get_params(1)
    rng = np.random.default_rng(n)
    w[kW5:kB5] = rng.uniform(-0.3, 0.3, H).astype(np.float32)
    for b in (kB1, kB2, kB3, kB4):
        w[b:b + H] = rng.uniform(-0.1, 0.1, H).astype(np.float32)
    sur.set_params(1, w)
    _check(sur, 1, n, n)
    sur.close()


@pytest.mark.parametrize("members,batch", [(1, 64), (3, 333), (5, 1025)])
def test_weights_after_adam_steps(ctx, members, batch):
    torch = pytest.importorskip("torch")
    from kwgpu import workloads as W
    n = 2 * batch + 7
    rng = np.random.default_rng(members)
    d = torch.from_numpy(W.plain(n, 5).view(np.uint8).copy()).cuda()
    prem = torch.from_numpy(np.abs(rng.normal(size=n)) * 0.3).cuda()
    torch.cuda.synchronize()
    sur = kwgpu.Surrogate(ctx, members, seed=23)
    before = [sur.get_params(m) for m in range(members)]
    sur.train(d.data_ptr(), prem.data_ptr(), n, epochs=2, batch=batch)
    for m in range(members):
        w = sur.get_params(m)
        assert np.isfinite(w).all()
        for name, (a, b) in SLICES.items():
            # four Adam steps of at most 2e-3 a weight, and no slice left out
            step = np.abs(w[a:b] - before[m][a:b])
            assert 0 < step.max() < 9e-3, (m, name)
        _check(sur, m, 200, m)
    sur.close()
