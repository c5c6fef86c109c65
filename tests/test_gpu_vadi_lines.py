"""Variable-diffusivity ADI on grids whose x lines are of any length: loss
and gradient against 64-bit torch autograd on the CPU (Thomas sweeps)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def thomas(a, b, c, d, dim):
    a, b, c, d = (t.movedim(dim, 0) for t in (a, b, c, d))
    n = d.shape[0]
    cs, ds = [c[0] / b[0]], [d[0] / b[0]]
    for i in range(1, n):
        m = b[i] - a[i] * cs[-1]
        cs.append(c[i] / m)
        ds.append((d[i] - a[i] * ds[-1]) / m)
    out = [ds[-1]]
    for i in range(n - 2, -1, -1):
        out.append(ds[i] - cs[i] * out[-1])
    import torch
    return torch.stack(out[::-1]).movedim(0, dim)


def step(u, kappa, lam):
    import torch
    inner = torch.zeros_like(u)
    inner[1:-1, 1:-1, 1:-1] = 1
    r, abc = torch.zeros_like(u), []
    for dim in (2, 1, 0):
        n = u.shape[dim]
        face = 0.5 * lam * (kappa.narrow(dim, 0, n - 1) + kappa.narrow(dim, 1, n - 1))
        flux = face * (u.narrow(dim, 1, n - 1) - u.narrow(dim, 0, n - 1))
        edge = torch.zeros_like(u.narrow(dim, 0, 1))
        r = r + torch.cat([flux, edge], dim) - torch.cat([edge, flux], dim)
        a, c = -torch.cat([edge, face], dim) * inner, -torch.cat([face, edge], dim) * inner
        abc.append((dim, a, 1.0 - a - c, c))
    r = r * inner
    for dim, a, b, c in abc:
        r = thomas(a, b, c, r, dim)
    return u + r


# lines at the edges of each chunk length and count, the longest (576), one
# past it (the general sweep), and enough lines for several waves per
# work-group with a partial last one
@pytest.mark.parametrize("nx,ny,nz", [
    (3, 5, 4), (9, 6, 5), (10, 5, 7), (27, 6, 5), (35, 7, 4), (36, 5, 3), (57, 4, 6), (113, 6, 5),
    (145, 4, 4), (289, 3, 5), (576, 4, 3), (577, 4, 3), (9, 211, 160), (33, 70, 61)])
def test_loss_grad_any_line(nx, ny, nz):
    import torch
    from tridsolver_amd.autograd import vadi_loss_grad
    rng = np.random.default_rng(nx)
    kap, u0, tgt = (torch.from_numpy(rng.uniform(lo, hi, (nz, ny, nx)))
                    for lo, hi in ((0.5, 1.5), (0, 1), (0, 1)))
    loss, gk, gu = vadi_loss_grad(kap.cuda(), u0.cuda(), tgt.cuda(), 3, 0.7, 2)
    k, u = kap.clone().requires_grad_(True), u0.clone().requires_grad_(True)
    x = u
    for _ in range(3):
        x = step(x, k, 0.7)
    want = 0.5 * (x - tgt).square().sum()
    ek, eu = torch.autograd.grad(want, (k, u))
    assert loss == pytest.approx(want.item(), rel=1e-12)
    assert oracle.rel_err(ek.numpy().ravel(), gk.cpu().numpy().ravel()) <= 1e-10
    assert oracle.rel_err(eu.numpy().ravel(), gu.cpu().numpy().ravel()) <= 1e-10
