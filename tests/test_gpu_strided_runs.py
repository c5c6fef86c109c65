"""Layouts of strided batches whose row runs are whole cache lines, and of
batches past the last-level cache: chunk counts, systems side by side and
orders other than those of small batches off the line.  Solutions against the
oracle as in test_gpu_scalar; the configuration names the layout."""
from __future__ import annotations

import numpy as np
import pytest

import tridsolver_amd as ta
from tests.test_gpu_scalar import run_case

pytestmark = pytest.mark.gpu

F64, F32 = np.float64, np.float32


@pytest.mark.parametrize("dtype,sd,dims,cfg,cfg_inc", [
    # whole lines, rows less than a page apart
    (F64, 1, [144, 64, 30], "R8,cps8,spb64>", None),
    (F64, 1, [208, 150, 6], "R16,cps16,spb16>", "R8,cps32,spb16>"),
    (F64, 1, [208, 257, 4], "R16,cps32,spb8,xcd>", None),
    (F64, 1, [208, 513, 4], "R8,cps72,spb8,xcd>", None),
    # rows a page and more apart, 32 KiB apart
    (F64, 2, [16, 150, 100], "R8,cps16,spb32>", None),
    (F64, 2, [100, 48, 150], "R16,cps16,spb16,xcd>", "R8,cps32,spb16,xcd>"),
    (F64, 1, [512, 200, 3], "R8,cps32,spb16,xcd>", None),
    (F64, 2, [64, 64, 200], "R8,cps32,spb16,xcd>", None),
    (F64, 2, [64, 64, 384], "R16,cps32,spb8,xcd>", None),
    (F64, 2, [64, 64, 385], "R16,cps32,spb16>", None),
    (F32, 1, [4128, 64, 1], "R8,cps8,spb64>", None),
    (F32, 1, [4128, 65, 1], "R16,cps8,spb64,xcd>", None),
    (F32, 1, [8192, 65, 1], "R8,cps16,spb64>", None),
    (F32, 2, [96, 22, 180], "R8,cps32,spb32,xcd>", "R8,cps24,spb32,xcd>"),
    (F32, 1, [352, 300, 6], "R16,cps20,spb32,xcd>", None),
    (F32, 1, [352, 448, 4], "R16,cps32,spb16,xcd>", None),
    (F32, 1, [352, 449, 6], "R16,cps32,spb32,xcd>", "R16,cps32,spb16,xcd>"),
    # off the line
    (F32, 1, [333, 144, 7], "R8,cps18,spb32,xcd>", None),
    (F32, 1, [333, 145, 7], "R8,cps32,spb32,xcd>", "R8,cps20,spb32,xcd>"),
    (F64, 1, [333, 192, 18], "R16,cps16,spb16,xcd>", "R8,cps32,spb16,xcd>"),
    (F64, 1, [333, 193, 18], "R8,cps32,spb16,xcd>", None)])
def test_cached(dtype, sd, dims, cfg, cfg_inc):
    for inc in (False, True):
        run_case(dims, sd, dtype, inc, seed=sum(dims))
        want = cfg_inc if inc and cfg_inc else cfg
        assert ta.last_config().replace(",cached", "").endswith(want), ta.last_config()


@pytest.mark.parametrize("dtype,N,w,inc,cfg", [
    (F64, 100, 400, 0, "R8,cps16,spb32>"), (F64, 100, 333, 0, "R8,cps16,spb32,xcd>"),
    (F64, 150, 333, 0, "R8,cps20,spb32,xcd>"), (F64, 150, 333, 1, "R8,cps32,spb16,xcd>"),
    (F64, 300, 400, 0, "R16,cps32,spb16>"), (F64, 300, 333, 0, "R16,cps32,spb16,xcd>"),
    (F64, 512, 333, 0, "R16,cps32,spb16,xcd>"), (F64, 512, 333, 1, "R8,cps64,spb16,xcd>"),
    (F64, 700, 333, 0, "R16,cps64,spb8,xcd>"), (F64, 700, 333, 1, "R8,cps88,spb8,xcd>"),
    (F32, 100, 333, 0, "R16,cps8,spb64,xcd>"), (F32, 150, 333, 0, "R8,cps32,spb32,xcd>"),
    (F32, 300, 333, 0, "R16,cps32,spb32,xcd>"), (F32, 300, 333, 1, "R16,cps20,spb32,xcd>"),
    (F32, 300, 512, 0, "R16,cps20,spb32,xcd>"), (F32, 400, 333, 0, "R16,cps32,spb32,xcd>"),
    (F32, 400, 333, 1, "R16,cps32,spb32,xcd>"), (F32, 700, 333, 0, "R16,cps64,spb16,xcd>"),
    (F32, 700, 333, 1, "R16,cps44,spb16,xcd>")])
def test_past_the_cache(dtype, N, w, inc, cfg):
    """More than 400 MiB of arrays: tridiag(-1, 4, -1) x = d with a d of the
    plane's number, every system against the 64-bit solution of one."""
    import torch

    from tridsolver_amd import api
    dt = torch.float64 if dtype == F64 else torch.float32
    k = (400 << 20) // ((4 + inc) * w * N * dt.itemsize) + 1
    a, b, c = (torch.full((k, N, w), v, dtype=dt, device="cuda") for v in (-1.0, 4.0, -1.0))
    plane = torch.arange(1, k + 1, device="cuda", dtype=dt)[:, None, None] / k
    d = plane.expand(k, N, w).contiguous()
    u = plane.neg().expand(k, N, w).contiguous() if inc else None
    fn = getattr(api, f"trid{'D' if dtype == F64 else 'S'}mtsvStridedBatch{'Inc' if inc else ''}")
    assert fn(a, b, c, d, u, 3, 1, [w, N, k], [w, N, k], None, 1) == 0, ta.last_error()
    got = ta.last_config().replace(",mixed", "")
    assert got.endswith(cfg), got
    from scipy.linalg import solve_banded
    band = np.array([[0.0] + [-1.0] * (N - 1), [4.0] * N, [-1.0] * (N - 1) + [0.0]])
    x = torch.from_numpy(solve_banded((1, 1), band, np.ones(N))).cuda()[None, :, None]
    x = (x - 1) * plane.double() if inc else x * plane.double()
    err = ((u if inc else d).double() - x).abs().max().item()
    assert err <= (1e-14 if dtype == F64 else 1e-6), err
