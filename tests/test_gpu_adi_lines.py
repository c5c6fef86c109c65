"""GPU parity of the whole-line right-hand side + x kernel of the ADI step
(lines of any length and alignment) at the edges of its layouts: the shortest
lines, one row more and less than whole chunks of every chunk length, one and
many lines per wave, the longest line it takes and the first one past it,
grids of one or two lines or planes, and arrays off the 16-byte alignment.
Tolerance as the other ADI tests: 1e-12 (FP64) / 1e-5 (FP32) normwise against
the oracle after 3 steps, and replayed steps bitwise equal to eager ones.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle
import tridsolver_amd as ta
from tests.test_gpu_adi import rand_init, ref_init, tol, torch_dt
from tridsolver_amd.adi import AdiPlan

pytestmark = pytest.mark.gpu

SHAPES = [(nx, 6, 5) for nx in (3, 4, 5, 7, 8, 9, 10, 11, 13, 15, 16, 28, 44, 65, 66, 67, 130, 200,
                                201, 250, 321, 322, 323, 449, 450, 451, 577, 578, 579, 834, 835)] + \
    [(40, 1, 7), (40, 7, 1), (9, 2, 3), (5, 3, 3), (4, 3, 70), (128, 33, 21), (256, 9, 8),
     (199, 40, 31), (100, 64, 64)]


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("shape", SHAPES)
def test_adi_lines_vs_oracle(shape, dt, offset):
    import torch
    nx, ny, nz = shape
    for mode in (0, 1):
        u0 = rand_init(nx, ny, nz, dt, seed=nx) if mode == 1 else ref_init(nx, ny, nz, dt)
        exp = u0.ravel().copy()
        assert oracle.adi(exp, nx, ny, nz, 3, 1.0, mode) == 0
        # u and du between guard values, `offset` elements off the alignment
        n = u0.size
        bufs = [torch.full((n + 16,), float("nan"), device="cuda", dtype=torch_dt(dt))
                for _ in range(2)]
        u, du = (b[8 + offset:8 + offset + n].view(nz, ny, nx) for b in bufs)
        plan = AdiPlan(nx, ny, nz, torch_dt(dt), 1.0, mode)
        got = []
        for _ in range(3):  # kernel by kernel, then captured and replayed
            u.copy_(torch.from_numpy(u0))
            plan.step(u, du, 3)
            got.append(u.cpu().numpy().ravel())
        what = f"{shape} mode {mode} [{plan.describe()}]"
        assert oracle.rel_err(exp, got[0]) <= tol(dt), what
        for g in got[1:]:
            np.testing.assert_array_equal(got[0], g, err_msg=what)
        for b in bufs:
            assert torch.isnan(b[:8 + offset]).all() and torch.isnan(b[8 + offset + n:]).all(), what


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_adi_lines_boundary_values_stay_out(dt):
    """NaN on the edges of the grid, which no interior point's stencil reads,
    reaches no other point."""
    import torch
    nx, ny, nz = 37, 11, 9
    u0 = rand_init(nx, ny, nz, dt, seed=3)
    exp = u0.ravel().copy()
    assert oracle.adi(exp, nx, ny, nz, 2, 1.0, 1) == 0
    exp = exp.reshape(u0.shape)
    for sl in ((0, 0), (0, -1), (-1, 0), (-1, -1)):
        u0[sl[0], sl[1], :] = np.nan
        u0[sl[0], :, sl[1]] = np.nan
        u0[:, sl[0], sl[1]] = np.nan
    u = torch.from_numpy(u0).cuda()
    plan = AdiPlan(nx, ny, nz, torch_dt(dt))
    plan.step(u, torch.empty_like(u), 2)
    got = u.cpu().numpy()
    edge = np.isnan(u0)
    assert np.isnan(got[edge]).all()
    assert oracle.rel_err(exp[~edge], got[~edge]) <= tol(dt)


def test_adi_lines_autotuned():
    """The tuner may take either kernel; pinning the fused one keeps it."""
    import torch
    nx, ny, nz = 128, 20, 18
    for dt in (np.float64, np.float32):
        u0 = rand_init(nx, ny, nz, dt, seed=4)
        exp = u0.ravel().copy()
        assert oracle.adi(exp, nx, ny, nz, 3, 1.0, 1) == 0
        ta.set_autotune(1)
        try:
            plan = AdiPlan(nx, ny, nz, torch_dt(dt))
            u = torch.from_numpy(u0.copy()).cuda()
            du = torch.empty_like(u)
            plan.step(u, du, 3)
        finally:
            ta.set_autotune(0)
        assert oracle.rel_err(exp, u.cpu().numpy().ravel()) <= tol(dt), plan.describe()
        plan.set_sweep(0, 8)
        assert "step:" not in plan.describe()


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [(256, 300, 130), (256, 130, 300), (190, 128, 180),
                                   (181, 257, 182), (64, 129, 513)])
def test_adi_default_sweep_layouts(shape, dt):
    """The untuned y and z layouts on both sides of their rules: line lengths
    around 128, 256 and 512 points, batches that fill the work-groups of two
    lines per lane (32768 lines) or not, odd line counts, chunk counts that are
    no power of two."""
    import torch
    nx, ny, nz = shape
    u0 = rand_init(nx, ny, nz, dt, seed=ny)
    exp = u0.ravel().copy()
    assert oracle.adi(exp, nx, ny, nz, 1, 1.0, 1) == 0
    plan = AdiPlan(nx, ny, nz, torch_dt(dt))
    u = torch.from_numpy(u0).cuda()
    plan.step(u, torch.empty_like(u), 1)
    err = oracle.rel_err(exp, u.cpu().numpy().ravel())
    assert err <= tol(dt), f"{err:.2e} [{plan.describe()}]"
