"""GPU parity of the one-pass strided adjoint at the edges of its layouts:
system lengths around one chunk, one wave of chunks and the longest of every
chunk length, several systems per wave, padded arrays, arrays that are not
16-byte aligned, and 64-bit offsets.  The bar is the one of the strided
solves: 1e-12 (FP64) / 1e-5 (FP32) normwise against the FP64 oracle.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from tests.helpers import dd_system, oracle_solve, view

pytestmark = pytest.mark.gpu

CASES = [([n, 37], None, 0) for n in (1, 2, 3, 7, 8, 9, 12, 13, 96, 97)] + \
    [([n, 5], None, 0) for n in (511, 512, 513, 768, 769, 4096, 4097, 6145, 8192)] + \
    [([30, 9], [33, 9], 0), ([1000, 3], [1001, 4], 0), ([33, 40, 6], [36, 41, 6], 1),
     ([7, 2, 5], None, 1), ([3, 700], None, 1), ([5, 3, 1200], None, 2), ([70, 257], None, 1)]


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("dims,pads,sd", CASES)
def test_adjoint_layouts(dims, pads, sd, dtype, offset):
    import torch

    import tridsolver_amd as ta
    from tridsolver_amd.api import _iv
    pads = pads or dims
    a, b, c, d = dd_system(dims, sd, np.float64, seed=5, pads=pads, pad_fill=0.0)
    x = oracle_solve(a, b, c, d, None, dims, sd, pads)
    g = np.random.default_rng(2).uniform(-1, 1, x.shape)
    exp = oracle.adjoint(a, b, c, x, g, len(dims), sd, dims, pads)

    def dev(v):
        # `offset` elements past a 16-byte boundary
        t = torch.full((v.size + offset,), float("nan"), device="cuda",
                       dtype=torch.float64 if dtype == np.float64 else torch.float32)
        t[offset:] = torch.from_numpy(v.astype(dtype))
        return t[offset:]
    # the ends of every system are never read
    va, vc = view(a, dims, pads), view(c, dims, pads)
    ax = len(dims) - 1 - sd
    va[(slice(None),) * ax + (0,)] = np.nan
    vc[(slice(None),) * ax + (-1,)] = np.nan
    t = [dev(v) for v in (a, b, c, x, g)]
    outs = [dev(np.full(x.shape, np.nan)) for _ in range(4)]
    fn = ta.lib().tridDmtsvStridedBatchAdjoint if dtype == np.float64 else \
        ta.lib().tridSmtsvStridedBatchAdjoint
    for wide in (False, True):
        ta.force_wide_index(wide)
        try:
            st = fn(*[v.data_ptr() for v in t], *[o.data_ptr() for o in outs], len(dims), sd,
                    _iv(dims), _iv(pads), 1)
        finally:
            ta.force_wide_index(False)
        assert st == 0, ta.last_error()
        tol = 1e-12 if dtype == np.float64 else 1e-5
        for name, e, o in zip("abcd", exp, outs):
            got = o.cpu().numpy()
            err = oracle.rel_err(view(e, dims, pads), view(got, dims, pads))
            assert err <= tol, f"grad_{name}: {err:.2e}"
            # padding stays untouched
            pad = np.ones(e.shape, bool)
            view(pad, dims, pads)[...] = False
            assert np.isnan(got[pad]).all(), f"grad_{name}: padding written"
