"""The mixed cache policy of solvedim-0 solves between 256 and 384 MiB: taken
where a wave's loads take whole cache lines (staged spans, one 16-byte vector
per chunk), not where lanes walk their chunks row by row or vector by vector."""
from __future__ import annotations

import pytest

import tridsolver_amd as ta
from tridsolver_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,pad,off,policy", [
    ("float64", 0, 0, "mixed"), ("float32", 0, 0, "mixed"), ("float32", 4, 0, "mixed"),
    ("float64", 8, 0, "cached"), ("float64", 8, 1, "cached"), ("float32", 4, 1, "cached")])
def test_policy(dtype, pad, off, policy):
    import torch
    dt = getattr(torch, dtype)
    n, p = 200, 200 + pad
    k = (300 << 20) // (4 * p * dt.itemsize)  # 4 arrays of 75 MiB
    # tridiag(-1, 4, -1) x = 1: every line's solution is symmetric, in (1/4, 1/2]
    bufs = [torch.full((k * p + 1,), v, dtype=dt, device="cuda") for v in (-1.0, 4.0, -1.0, 1.0)]
    ptr = [t.data_ptr() + off * dt.itemsize for t in bufs]
    fn = api.tridDmtsvStridedBatchPadded if dtype == "float64" else api.tridSmtsvStridedBatchPadded
    pads = [p, k]
    assert fn(ptr[0], pads, ptr[1], pads, ptr[2], pads, ptr[3], pads, None, pads, 2, 0, [n, k],
              None, 1) == 0, ta.last_error()
    cfg = ta.last_config()
    assert f",{policy}" in cfg, cfg
    x = bufs[3][off:off + k * p].view(k, p)[:, :n]
    tol = 1e-14 if dtype == "float64" else 1e-6
    assert float((x - x.flip(1)).abs().max()) <= tol and (x == x[:1]).all()
    assert float(x.min()) > 0.25 and float(x.max()) <= 0.5 + tol
    if pad:
        assert (bufs[3][off:off + k * p].view(k, p)[:, n:] == 1).all()
