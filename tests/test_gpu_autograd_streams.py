"""trid_solve on torch's default stream and on a side stream: its calls do not
wait for the device where the library launches on the stream torch works on,
and do elsewhere."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
import tridsolver_amd as ta
from tests.helpers import dd_system, oracle_solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side", [False, True])
@pytest.mark.parametrize("sd", [0, 1])
def test_streams(side, sd):
    import torch
    from tridsolver_amd.autograd import _sync, trid_solve
    dims = [301, 257, 5]
    abcd = dd_system(dims, sd, np.float64, seed=3)
    exp = oracle_solve(*abcd, None, dims, sd)
    t = [torch.from_numpy(x).cuda().reshape(5, 257, 301).requires_grad_(True) for x in abcd]
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    assert _sync(t[0]) == 0
    with torch.cuda.stream(s):
        assert _sync(t[0]) == 1
    ta.set_stream(s if side else None)
    try:
        with torch.cuda.stream(s if side else torch.cuda.default_stream()):
            assert _sync(t[0]) == 0
            for _ in range(3):
                x = trid_solve(*t, sd)
                # <A^{-T} 1, d> = <1, x>
                (gd,) = torch.autograd.grad(x.sum(), t[3])
                # the temporaries' memory is reused at once
                torch.full_like(x, float("nan"))
                assert oracle.rel_err(exp, x.detach().cpu().numpy().ravel()) <= 1e-12
                assert (gd * t[3]).sum().item() == pytest.approx(x.sum().item(), rel=1e-9)
    finally:
        torch.cuda.synchronize()
        ta.set_stream(None)
