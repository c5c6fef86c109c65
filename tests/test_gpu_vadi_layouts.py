"""Layouts of the variable-diffusivity sweeps on small grids: on both sides of
their rules (line length, work-groups, whole-line rows), each sweep against a
64-bit Thomas solve of the same operator on the CPU."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
import tridsolver_amd as ta
from tests.test_gpu_vadi_lines import thomas

pytestmark = pytest.mark.gpu


def want(kap, d, axis, lam):
    """A^{-1} d along `axis` (0 = x) of the grid-interior operator."""
    import torch
    dim = 2 - axis
    inner = torch.zeros_like(d)
    inner[1:-1, 1:-1, 1:-1] = 1
    n = d.shape[dim]
    face = 0.5 * lam * (kap.narrow(dim, 0, n - 1) + kap.narrow(dim, 1, n - 1))
    edge = torch.zeros_like(d.narrow(dim, 0, 1))
    a, c = -torch.cat([edge, face], dim) * inner, -torch.cat([face, edge], dim) * inner
    return thomas(a, 1.0 - a - c, c, d, dim)


@pytest.mark.parametrize("grid,axis,cfg", [
    ([33, 33, 33], 1, "R4,cps16,spb8"), ([64, 127, 64], 2, "R4,cps16,spb8"),
    ([64, 128, 64], 2, "R4,cps16,spb8"), ([64, 129, 64], 2, "R8,cps8,spb64"), ([65, 32, 256], 1, "R8,cps4,spb64"),
    ([96, 96, 90], 1, "R8,cps16,spb16"), ([96, 96, 85], 1, "R8,cps16,spb32"),
    ([95, 96, 90], 1, "R8,cps16,spb32"), ([100, 100, 80], 2, "R8,cps16,spb16"),
    ([99, 100, 80], 2, "R8,cps16,spb32"), ([16, 40, 300], 2, "R8,cps64,spb16"),
    ([33, 124, 300], 2, "R8,cps64,spb16"), ([33, 125, 300], 2, "R8,cps64,spb8"),
    ([80, 60, 300], 2, "R8,cps64,spb16"), ([20, 20, 600], 2, "R16,cps64,spb8"),
    ([600, 20, 9], 0, "R4,cps256,spb1")])
def test_sweep_layout(grid, axis, cfg):
    import torch
    nx, ny, nz = grid
    rng = np.random.default_rng(nx + axis)
    kap, d, u = (torch.from_numpy(rng.uniform(lo, hi, (nz, ny, nx)))
                 for lo, hi in ((0.5, 1.5), (-1, 1), (-1, 1)))
    exp = want(kap, d, axis, 0.7)
    for inc in (0, 1):
        kd, dd, ud = kap.cuda(), d.cuda(), u.cuda()
        assert ta.lib().tridVadiSweep(kd.data_ptr(), dd.data_ptr(), ud.data_ptr(), nx, ny, nz,
                                      axis, 0.7, 0, inc) == 0, ta.last_error()
        assert f",{cfg}" in ta.last_config(), ta.last_config()
        got = (ud - u.cuda() if inc else dd).cpu().numpy().ravel()
        assert oracle.rel_err(exp.numpy().ravel(), got) <= 1e-12
