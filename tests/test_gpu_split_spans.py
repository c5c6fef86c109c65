"""GPU parity of the split-line solves' default layouts: last segments of every
kind (whole, one row, one row short, one chunk), lines off the 16-byte
alignment, padded batches, reduced systems on both sides of a work-group, and
the cached and 64-bit-offset forms.  Bars as in test_gpu_split.
"""
from __future__ import annotations

import numpy as np
import pytest

import tridsolver_amd as ta
from tests.helpers import check_close, dd_system, oracle_solve
from tests.test_gpu_scalar import run_case

pytestmark = pytest.mark.gpu

SD0 = [([n, 3], None) for n in (8193, 8704, 8705, 9215, 16384, 17408, 17409, 17416)] + \
    [([9001, 5], [9003, 5]), ([10240, 2, 3], [10256, 2, 3])]
SD1 = [([k, n], None) for k, n in ((1, 2048), (3, 2049), (48, 2111), (64, 2112), (65, 2113),
                                   (100, 3000), (5, 70000))] + \
    [([33, 2500, 4], [37, 2503, 4]), ([7, 4100, 9], None)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("sd,dims,pads", [(0, d, p) for d, p in SD0] + [(1, d, p) for d, p in SD1])
def test_split_default_layouts(sd, dims, pads, dtype):
    for policy in (-1, 0, 1):
        ta.force_cache_policy(policy)
        try:
            for inc in (False, True):
                run_case(dims, sd, dtype, inc, pads=pads, seed=dims[0] + 3)
                assert ta.last_config().startswith("split<"), ta.last_config()
        finally:
            ta.force_cache_policy(-1)
    ta.force_wide_index(True)
    try:
        run_case(dims, sd, dtype, False, pads=pads, seed=dims[0] + 4)
    finally:
        ta.force_wide_index(False)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("sd,dims", [(0, [9216, 3]), (0, [8711, 2]), (1, [50, 2500])])
def test_split_unaligned_arrays(sd, dims, dtype):
    """Arrays one element off the 16-byte alignment."""
    import torch

    from tridsolver_amd import api
    host = dd_system(dims, sd, dtype, seed=9)
    dev = []
    for x in host:
        t = torch.full((x.size + 2,), float("nan"), device="cuda",
                       dtype=torch.float64 if dtype == np.float64 else torch.float32)
        t[1:-1] = torch.from_numpy(x)
        dev.append(t)
    fn = api.tridDmtsvStridedBatch if dtype == np.float64 else api.tridSmtsvStridedBatch
    p = [t.data_ptr() + t.element_size() for t in dev]
    assert fn(p[0], p[1], p[2], p[3], None, len(dims), sd, dims, dims, None, 1) == 0
    check_close(oracle_solve(*host, None, dims, sd), dev[3][1:-1].cpu().numpy(), dtype)
    assert torch.isnan(dev[3][[0, -1]]).all()
