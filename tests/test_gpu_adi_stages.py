"""The ADI stages are the kernels of the steps: stages 4, 2, 3 (where a plan
has stage 4) give bitwise what one step gives, on grids whose steps take the
fused right-hand side + x kernel and on those whose steps take the whole-line
one in its place."""
from __future__ import annotations

import numpy as np
import pytest

from tests.test_gpu_adi import rand_init, torch_dt
from tridsolver_amd.adi import AdiPlan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [(64, 24, 10), (128, 24, 10), (256, 20, 9), (512, 10, 7)])
def test_stages_are_the_steps_kernels(shape, dt):
    import torch
    nx, ny, nz = shape
    u0 = torch.from_numpy(rand_init(nx, ny, nz, dt, seed=nx)).cuda()
    plan = AdiPlan(nx, ny, nz, torch_dt(dt))
    got = []
    for run in (lambda u, du: plan.step(u, du, 1),
                lambda u, du: [plan.stage(u, du, s) for s in (4, 2, 3)]):
        u = u0.clone()
        du = torch.full_like(u, float("nan"))
        run(u, du)
        got.append((u.cpu().numpy(), du.cpu().numpy()))
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b, err_msg=plan.describe())


@pytest.mark.parametrize("n,dtype,kernels", [(20, "f64", ("step",)), (20, "f32", ("step",)),
                                             (64, "f64", ("rhs_x_fused", "sweep_y", "sweep_z_inc")),
                                             (128, "f32", ("rhs_x_fused", "sweep_y", "sweep_z_inc"))])
def test_benchmark_times_the_steps_kernels(n, dtype, kernels):
    """What the benchmark times and checks is bitwise what the steps compute."""
    from types import SimpleNamespace

    import torch

    import bench
    import tridsolver_amd as ta
    from tridsolver_amd import api
    w = bench.adi_workload(SimpleNamespace(n=n, dtype=dtype), torch, np, api, ta)
    assert w["kernels"] == kernels
    u = torch.from_numpy(w["host"][0].copy()).cuda()
    plan = AdiPlan(n, n, n, u.dtype)
    for _ in range(2):
        plan.step(u, torch.empty_like(u), 1)
    np.testing.assert_array_equal(w["result"](2), u.cpu().numpy())
