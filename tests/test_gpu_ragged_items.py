"""Work items of the ragged launches: fewer, exactly as many and more items
than work-groups, and two solves of one plan on different streams at once."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
import tridsolver_amd as ta
from tests.helpers import check_close
from tests.test_gpu_ragged import ragged_inputs, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nsys", [1, 255, 256, 257, 1024, 1025, 2600])
def test_item_counts(dtype, nsys):
    """Systems of 2049..4096 rows: one item each."""
    lengths = np.random.default_rng(nsys).integers(2049, 4097, nsys)
    off, arrs = ragged_inputs(lengths, dtype, seed=nsys)
    (got,), plan = run(off, arrs, dtype)
    exp = arrs[3].copy()
    assert oracle.ragged(arrs[0], arrs[1], arrs[2], exp, None, off) == 0
    check_close(exp, got, dtype, plan.describe())


def test_one_plan_on_two_streams():
    import torch
    from tridsolver_amd.ragged import RaggedPlan
    lengths = np.random.default_rng(5).integers(1, 700, 20000)
    off, arrs = ragged_inputs(lengths, np.float64, seed=6)
    exp = arrs[3].copy()
    assert oracle.ragged(arrs[0], arrs[1], arrs[2], exp, None, off) == 0
    a, b, c = (torch.from_numpy(x).cuda() for x in arrs[:3])
    plan = RaggedPlan(torch.from_numpy(np.asarray(off, dtype=np.int64)).cuda(), torch.float64)
    ds = [torch.from_numpy(arrs[3]).cuda() for _ in range(4)]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    try:
        for i, d in enumerate(ds):
            ta.set_stream(streams[i % 2])
            plan.solve(a, b, c, d, sync=0)
    finally:
        ta.set_stream(None)
        torch.cuda.synchronize()
    for d in ds:
        check_close(exp, d.cpu().numpy(), np.float64, "one plan, two streams")
