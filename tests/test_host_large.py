"""Host calls whose inputs and results are over what is kept in pinned memory (16 MiB) go over part by
part: the prices of their first and last options are bitwise those of small calls."""
from __future__ import annotations

import numpy as np
import pytest

from kwgpu import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("call,n", [("fd1d_price", 200000), ("fd1d_price", 183000), ("fd1d_bs_price", 100000)])
@pytest.mark.parametrize("uneven", [False, True])
def test_large_calls(ctx, call, n, uneven):
    print("large host call", call, n, uneven, flush=True)
    o = W.plain(n, 3)
    o["e"] = np.arange(n) % 7 != 0
    o["s"][5] = 1e9  # outside its grid
    xd, td = 64 + np.arange(n, dtype=np.int32) % 3 * 30, 5 + np.arange(n, dtype=np.int32) % 4

    def price(idx):
        f = getattr(ctx, call)
        if uneven:
            return f(o[idx], x_dims=np.ascontiguousarray(xd[idx]), t_dims=np.ascontiguousarray(td[idx]))
        return f(o[idx], 100, 6)

    p, st, rc, err = price(np.arange(n))
    ends = np.concatenate([np.arange(400), np.arange(n - 400, n)])
    q, sq, rcq, errq = price(ends)
    assert np.array_equal(st[ends], sq) and rc == rcq and err == errq
    assert np.array_equal(p[ends], q, equal_nan=True)
    assert st[5] != 0 and np.all(np.delete(st, 5) == 0)
