"""The control variate (FD as given + closed form - FD of the European twin) rounds as the two legs'
difference: both march the same rows in the same lanes, so what their hundreds of steps round
cancels. Windows keep that: against the oracle's difference the windowed legs are as far off as
the whole-grid kernels' (which a tune file selects), give or take half as much and the 1e-14 that
forming the price takes; legs on windows of their own were 4 to 12 times as far."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from kwgpu import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def whole(tmp_path_factory):
    import kwgpu
    f = tmp_path_factory.mktemp("whole") / "tune"
    f.write_text("256 0 2 0\n512 0 5 0\n1024 0 8 0\n2048 0 9 0\n")
    c = kwgpu.Context(0)
    c.tune_load(str(f))
    yield c
    c.close()


def book(n, seed, per=1):
    """n options, `per` spots of each set of parameters, every tenth European: sharing a PDE with
    its neighbours' European legs, and further out of the money."""
    o = W.plain(n, seed)
    for c in ("t", "z", "r", "q", "w"):
        o[c] = np.repeat(o[c][::per], per)[:n]
    if per > 1:
        e = np.arange(n) % 10 == 9
        o["e"][e] = 0
        o["s"][e] = o["k"][e] * np.exp(-1.5 * o["w"][e] * o["z"][e] * np.sqrt(o["t"][e]))
    return o


def check(contexts, o, ref, *sizes, **grids):
    err = []
    for c in contexts:
        p, st, rc, msg = c.fd1d_bs_price(o, *sizes, **grids)
        assert rc == 0 and np.all(st == 0), msg
        err.append(np.linalg.norm(p - ref) / np.linalg.norm(ref))
    print("  windowed, whole grids:", *err, flush=True)
    assert err[0] <= 1.5 * err[1] + 1e-14


@pytest.mark.parametrize("n,per,x_dim,t_dim", [(12, 1, 512, 512), (500, 1, 512, 512), (900, 5, 777, 301),
                                               (3000, 1, 256, 300), (3000, 5, 1000, 260),
                                               (700, 1, 1500, 257), (300, 1, 2048, 130)])
def test_legs_round_alike(ctx, whole, n, per, x_dim, t_dim):
    print("control variate", n, per, x_dim, t_dim, flush=True)
    o = book(n, n + per, per)
    ref, e = oracle.fd1d_bs_price(o, x_dim, t_dim)
    assert not e
    check((ctx, whole), o, ref, x_dim, t_dim)


def test_legs_round_alike_on_per_option_grids(ctx, whole):
    print("control variate, per-option grids", flush=True)
    o, xd, td = W.uneven(400, 31)
    td = np.clip(td, 65, 300).astype(np.int32)
    eu = o.copy()
    eu["e"] = 0
    ref = (oracle.fd1d_price_uneven(o, xd, td)[0] + oracle.bs_price(eu) -
           oracle.fd1d_price_uneven(eu, xd, td)[0])
    check((ctx, whole), o, ref, x_dims=xd, t_dims=td)
