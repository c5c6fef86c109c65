"""Layouts of strided batches that fill the chip (64 work-groups and more):
chunk counts between the powers of two, 8 to 64 systems side by side, the
XCD-contiguous order.  Lengths sit at the edges of the layout rule, batches
at one system more or fewer than whole work-groups."""
from __future__ import annotations

import numpy as np
import pytest

import tridsolver_amd as ta
from tests.test_gpu_scalar import run_case

pytestmark = pytest.mark.gpu


def config():
    return ta.last_config().replace(",cached", "")


@pytest.mark.parametrize("dtype,N,cfg", [
    (np.float64, 9, "R8,cps2,spb64,xcd>"), (np.float64, 64, "R8,cps8,spb64,xcd>"),
    (np.float64, 65, "R8,cps10,spb32,xcd>"), (np.float64, 129, "R8,cps18,spb32,xcd>"),
    (np.float64, 150, "R8,cps20,spb32,xcd>"), (np.float64, 192, "R8,cps24,spb32,xcd>"),
    (np.float64, 193, "R8,cps32,spb16,xcd>"), (np.float64, 257, "R16,cps32,spb8,xcd>"),
    (np.float64, 513, "R8,cps72,spb8,xcd>"), (np.float64, 768, "R8,cps96,spb8,xcd>"),
    (np.float64, 769, "R16,cps64,spb8,xcd>"), (np.float64, 1025, "R16,cps128,spb4,xcd>"),
    (np.float32, 9, "R16,cps1,spb64,xcd>"), (np.float32, 128, "R16,cps8,spb64,xcd>"),
    (np.float32, 129, "R8,cps18,spb32,xcd>"), (np.float32, 193, "R8,cps32,spb32,xcd>"),
    (np.float32, 257, "R16,cps18,spb32,xcd>"), (np.float32, 384, "R16,cps24,spb32,xcd>"),
    (np.float32, 385, "R16,cps32,spb16,xcd>"), (np.float32, 600, "R16,cps40,spb16,xcd>"),
    (np.float32, 1025, "R16,cps72,spb8,xcd>"), (np.float32, 2047, "R16,cps128,spb8,xcd>")])
@pytest.mark.parametrize("sd", [1, 2])
def test_layout_and_solution(dtype, N, cfg, sd):
    spb = int(cfg.split("spb")[1].split(",")[0])
    for inc, pad in ((False, 0), (True, 3)):
        # one system more than 64, one fewer than 65 whole work-groups
        ns = 64 * spb + (1 if inc else spb - 1)
        dims = [ns, N, 1] if sd == 1 else [ns, 1, N]
        pads = [ns + pad] + dims[1:]
        run_case(dims, sd, dtype, inc, pads=pads, seed=N + sd)
        assert config().endswith(cfg), config()


@pytest.mark.parametrize("dtype,tol", [(np.float64, 1e-12), (np.float32, 2e-5)])
@pytest.mark.parametrize("N", [70, 150, 333, 600])
def test_adjoint(dtype, tol, N):
    """Gradients over three strided dimensions against 64-bit torch ones."""
    import torch
    from tridsolver_amd.autograd import trid_solve
    gen = torch.Generator(device="cuda").manual_seed(N)

    def rand(lo, hi):
        return (torch.rand((3, N, 1501), generator=gen, device="cuda", dtype=torch.float64)
                * (hi - lo) + lo).to(torch.float32 if dtype == np.float32 else torch.float64)

    a, c = rand(-1, -0.1), rand(-1, -0.1)
    b = a.abs() + c.abs() + rand(0.5, 1.5)
    d, g = rand(-1, 1), rand(-1, 1)
    leaves = [t.clone().requires_grad_(True) for t in (a, b, c, d)]
    x = trid_solve(*leaves, 1)
    got = torch.autograd.grad(x, leaves, g)
    # 64-bit Thomas of A x = d and A^T lam = g along dimension 1
    def thomas(a, b, c, d):
        cs, ds = [c[:, 0] / b[:, 0]], [d[:, 0] / b[:, 0]]
        for i in range(1, N):
            m = b[:, i] - a[:, i] * cs[-1]
            cs.append(c[:, i] / m)
            ds.append((d[:, i] - a[:, i] * ds[-1]) / m)
        out = [ds[-1]]
        for i in range(N - 2, -1, -1):
            out.append(ds[i] - cs[i] * out[-1])
        return torch.stack(out[::-1], 1)

    a, b, c, d, g = (t.double() for t in (a, b, c, d, g))
    zero = torch.zeros_like(a[:, :1])
    xr = thomas(a, b, c, d)
    lam = thomas(torch.cat([zero, c[:, :-1]], 1), b, torch.cat([a[:, 1:], zero], 1), g)
    want = (-lam * torch.cat([zero, xr[:, :-1]], 1), -lam * xr,
            -lam * torch.cat([xr[:, 1:], zero], 1), lam)
    for got_t, want_t in zip((x.detach(),) + got, (xr,) + want):
        err = (got_t.double() - want_t).norm() / want_t.norm()
        assert err <= tol, float(err)
