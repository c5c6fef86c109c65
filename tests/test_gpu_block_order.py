"""Two-ended tiled block solves on either side of the rules for the block order
and for the work-groups, with a remainder past the last 8 blocks, against a
dense solve of sampled systems and the residual of all."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu


def batch(M, N, P, dtype):
    import torch
    gen = torch.Generator().manual_seed(100 * M + P % 97)

    def rand(*shape):
        return torch.rand(shape, generator=gen, dtype=torch.float64) * 2 - 1

    A, C, B, d = rand(N, P, M, M), rand(N, P, M, M), rand(N, P, M, M), rand(N, P, M)
    B += torch.diag_embed(A.abs().sum(-1) + B.abs().sum(-1) + C.abs().sum(-1) + 1.0)
    return [t.to(dtype).cuda() for t in (A, B, C, d)]


def residual(A, B, C, d, u):
    """max |A u_{n-1} + B u_n + C u_{n+1} - d|, in FP64."""
    A, B, C, d, u = (t.double() for t in (A, B, C, d, u))

    def mul(m, v):
        return (m * v.unsqueeze(-2)).sum(-1)

    r = mul(B, u) - d
    r[1:] += mul(A[1:], u[:-1])
    r[:-1] += mul(C[:-1], u[1:])
    return float(r.abs().max())


# waves of 64/(2M) problems: 768 * 2^10 / (32 M) waves hold 6 MiB of FP64 per
# matrix row; M = 3 changes its work-groups at 640, 1024 and 4096 waves, the
# others at 1792
CASES = [(M, w) for M in (3, 4, 5, 6, 7, 8) for w in (24576 // M - 1, -(-24576 // M) + 29)]
CASES += [(3, w) for w in (639, 641, 1023, 1024 + 5, 4095, 4096 + 5)]
CASES += [(M, w) for M in (4, 5, 6, 7, 8) for w in (1791, 1792 + 5)]


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("M,waves", CASES)
def test_orders(M, waves, dtype):
    import torch
    from tridsolver_amd.block import btsv
    dt = getattr(torch, dtype)
    P = waves * (64 // (2 * M)) - 1  # the last group of the last wave is short
    A, B, C, d = batch(M, 4, P, dt)
    u = btsv(A, B, C, d, torch.empty_like(d))
    # rows are diagonally dominant: |u| <= 1, rows sum below 3 M + M + 1 in
    # magnitude, and a stable elimination leaves a few roundings of that
    eps = 2.0 ** -52 if dt == torch.float64 else 2.0 ** -23
    assert residual(A, B, C, d, u) <= 16 * M * (6 * M + 1) * eps
