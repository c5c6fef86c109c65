"""Chunk lengths of the untuned FP64 y and z sweeps of lines up to 128 points:
on both sides of the line length and of one work-group per CU, against the
oracle (bar as in test_gpu_adi)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from tests.test_gpu_adi import rand_init, tol, torch_dt
from tridsolver_amd.adi import AdiPlan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,shape,y,z", [
    (np.float64, (149, 96, 110), 8, 8), (np.float64, (149, 97, 110), 16, 8),
    (np.float64, (128, 97, 128), 8, 8), (np.float64, (128, 97, 129), 16, 16),
    (np.float64, (129, 128, 100), 8, 16), (np.float32, (149, 97, 112), 8, 8)])
def test_rows(dt, shape, y, z):
    import torch
    nx, ny, nz = shape
    u0 = rand_init(nx, ny, nz, dt, seed=ny)
    exp = u0.ravel().copy()
    assert oracle.adi(exp, nx, ny, nz, 2, 1.0, 1) == 0
    plan = AdiPlan(nx, ny, nz, torch_dt(dt))
    assert f" y:cc<R{y}," in plan.describe() and f" z:cc<R{z}," in plan.describe(), plan.describe()
    u = torch.from_numpy(u0).cuda()
    plan.step(u, torch.empty_like(u), 2)
    assert oracle.rel_err(exp, u.cpu().numpy().ravel()) <= tol(dt)
