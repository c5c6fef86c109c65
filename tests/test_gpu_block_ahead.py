"""Two-ended tiled block solves: rows loaded ahead (halves of every parity and
shorter than the rows ahead), one- and four-wave work-groups on either side of
the rule, and the gradients' row groups, against a dense solve."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def system(M, N, P, seed):
    import torch
    gen = torch.Generator().manual_seed(seed)

    def rand(*shape):
        return torch.rand(shape, generator=gen, dtype=torch.float64) * 2 - 1

    A, C, B = rand(N, P, M, M) / M, rand(N, P, M, M) / M, rand(N, P, M, M) / M
    B += torch.diag_embed(A.abs().sum(-1) + C.abs().sum(-1) + 1.0)
    return A, B, C, rand(N, P, M), rand(N, P, M)


def dense(A, B, C, d):
    """Solutions of the P systems, as one dense solve each."""
    import torch
    N, P, M = d.shape
    full = torch.zeros(P, N * M, N * M, dtype=torch.float64)
    for n in range(N):
        full[:, n * M:n * M + M, n * M:n * M + M] = B[n]
        if n:
            full[:, n * M:n * M + M, n * M - M:n * M] = A[n]
        if n + 1 < N:
            full[:, n * M:n * M + M, n * M + M:n * M + 2 * M] = C[n]
    x = torch.linalg.solve(full, d.permute(1, 0, 2).reshape(P, N * M, 1))
    return x.reshape(P, N, M).permute(1, 0, 2).contiguous(), full


def close(got, want):
    got, want = got.cpu(), want
    assert float((got - want).norm()) <= 1e-12 * max(float(want.norm()), 1e-300)


@pytest.mark.parametrize("M", [3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 6, 9])
def test_short_halves(M, N):
    import torch
    from tridsolver_amd.block import btsv, btsv_adjoint
    A, B, C, d, g = system(M, N, 13, 10 * M + N)
    A[0], C[N - 1] = float("nan"), float("nan")  # never used
    dev = [t.cuda() for t in (A, B, C, d, g)]
    u = btsv(*dev[:4], torch.empty_like(dev[3]))
    x, full = dense(A, B, C, d)
    close(u, x)
    gA, gB, gC, lam = btsv_adjoint(*dev[:3], u, dev[4])
    y = torch.linalg.solve(full.transpose(1, 2), g.permute(1, 0, 2).reshape(13, N * M, 1))
    y = y.reshape(13, N, M).permute(1, 0, 2)
    close(lam, y)
    zero = torch.zeros_like(x[:1])
    for got, v in ((gA, torch.cat([zero, x[:-1]])), (gB, x), (gC, torch.cat([x[1:], zero]))):
        close(got, -y.unsqueeze(-1) * v.unsqueeze(-2))


@pytest.mark.parametrize("M", [3, 4, 5, 8])
def test_work_group_rule(M):
    """Batches of one wave less than, exactly and one problem more than the
    four-wave limit; and the XCD order's remainder."""
    import torch
    from tridsolver_amd.block import btsv
    waves, per = (640 if M == 3 else 2048), 64 // (2 * M)
    for P in ((waves - 1) * per, waves * per - per + 1, (waves + 33) * per - 1):
        A, B, C, d, _ = system(M, 3, P, P)
        u = btsv(A.cuda(), B.cuda(), C.cuda(), d.cuda(), torch.empty_like(d).cuda())
        close(u, dense(A, B, C, d)[0])
