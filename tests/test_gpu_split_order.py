"""Strided split-line solves: reduced systems contiguous (few systems) or in the
long systems' order (1024 systems and more, or reduced systems that are split
again), one segment per system, and the block order and cache policy of row
runs that are whole cache lines or not.  Bars as in test_gpu_split."""
from __future__ import annotations

import numpy as np
import pytest

import tridsolver_amd as ta
from tests.test_gpu_scalar import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("dims,sd,tags", [
    ([1, 2048], 1, ",xcd,cached>"), ([1, 4000], 1, ",xcd,cached>"),    # one segment
    ([1023, 2049], 1, ",xcd,cached>"), ([1025, 2049], 1, ",xcd,cached>"),
    ([224, 2050], 1, ",xcd,cached>"), ([1024, 2050], 1, ",cached>"),
    ([32, 32, 2113], 2, ",cached>"), ([31, 34, 2113], 2, ",xcd,cached>")])
def test_orders(dims, sd, tags, dtype):
    for inc in (False, True):
        run_case(dims, sd, dtype, inc, seed=sum(dims))
        assert ta.last_config().startswith("split<") and ta.last_config().endswith(tags)
    ta.force_wide_index(True)
    try:
        run_case(dims, sd, dtype, False, seed=3)
    finally:
        ta.force_wide_index(False)


def test_reduced_systems_split_again():
    """4100 segments per system: reduced systems of 8200 rows."""
    run_case([64, 4100 * 64 - 5], 1, np.float32, False, seed=4)
    assert ta.last_config().startswith("split<"), ta.last_config()


@pytest.mark.parametrize("w,k,tags", [(4096, 2048, ">"), (4064, 2048, ",cached>"),
                                      (4090, 2056, ",xcd,cached>")])
def test_policy_of_whole_lines(w, k, tags):
    """256 MiB of arrays in whole-line runs stream, fewer and others do not."""
    import torch

    from tridsolver_amd import api
    a, b, c, d = (torch.full((k, w), v, dtype=torch.float64, device="cuda")
                  for v in (-1.0, 4.0, -1.0, 1.0))
    assert api.tridDmtsvStridedBatch(a, b, c, d, None, 2, 1, [w, k], [w, k], None, 1) == 0
    assert ta.last_config().endswith("spb64" + tags), ta.last_config()
    from scipy.linalg import solve_banded
    band = np.array([[0.0] + [-1.0] * (k - 1), [4.0] * k, [-1.0] * (k - 1) + [0.0]])
    x = torch.from_numpy(solve_banded((1, 1), band, np.ones(k))).cuda()[:, None]
    assert (d - x).abs().max().item() <= 1e-14


@pytest.mark.parametrize("segments,fits", [(15800, True), (16200, True), (16400, False)])
def test_fixed_scratch_limit(segments, fits):
    """FP64, 64 systems of 64-row segments whose reduced systems are split
    again: in the systems' order the scratch is 4224 bytes per segment (4 arrays
    of 2 rows for each system's segment, and of 2 rows per 32 of them), as
    contiguous systems 4112.  A solve is refused where neither fits 64 MiB."""
    import ctypes as C

    import torch
    w, k = 64, segments * 64
    gen = torch.Generator(device="cuda").manual_seed(segments)
    x, a, c = (torch.rand((k, w), generator=gen, dtype=torch.float64, device="cuda")
               for _ in range(3))
    b = a + c + 1.5
    d = b * x
    d[1:] -= a[1:] * x[:-1]
    d[:-1] -= c[:-1] * x[1:]
    a.neg_(), c.neg_()
    dims = (C.c_int * 2)(w, k)
    got = d.clone()
    st = ta.lib().tridDmtsvStridedBatchNoAlloc(*(t.data_ptr() for t in (a, b, c, got)), None, 2,
                                               1, dims, dims, None, 1)
    assert st == (0 if fits else 3), ta.last_error()
    if fits:  # the allocating form gives the same bits
        other = d.clone()
        assert ta.lib().tridDmtsvStridedBatch(*(t.data_ptr() for t in (a, b, c, other)), None, 2,
                                              1, dims, dims, None, 1) == 0
        assert torch.equal(got, other)
    want = x if fits else d
    assert ((got - want).abs().max() / want.abs().max()).item() <= (1e-12 if fits else 0.0)
