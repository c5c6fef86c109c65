"""Differentiable wrappers over the adjoint kernels (include/trid_adjoint.h).

TridSolve: torch.autograd.Function for x = A^{-1} d along `solvedim` of
same-shaped tensors (a, b, c, d); backward runs the hand-written adjoint
kernel (transposed solve + fused coefficient gradients).  Used for the
gradient tests; it does not record anything for graph capture.

vadi_forward / vadi_loss_grad: the variable-diffusivity ADI forward pass and
its reverse-mode gradient (checkpoint every `ckpt` steps, recomputation).
"""
from __future__ import annotations

import ctypes as C

import torch

from . import _check, lib
from .api import _iv, dims_of, solve


def _sync(t) -> int:
    """0 where the library launches on the stream that torch works on for t's
    device: what follows there is ordered behind the call, and so is the reuse
    of its temporaries; elsewhere 1, and the call waits for its results.  The
    library launches on the current device, and the null streams of all devices
    have the same handle, so the device is compared as well.
    The waits kept the host from preparing the next launch: forward and
    backward of 1000 x 4000 FP32 took 176 us for 58 us of kernels."""
    dev = t.device.index
    if dev != torch.cuda.current_device():
        return 1
    return int((lib().tridGetStream() or 0) != torch.cuda.current_stream(dev).cuda_stream)


def _ordered(t) -> int:
    """_sync(t) for a call that is made next.  Where it is 1, torch's stream is
    waited for first: the library's stream is not ordered behind the copies of
    the operands or behind an earlier call that did not wait."""
    wait = _sync(t)
    if wait:
        torch.cuda.current_stream(t.device).synchronize()
    return wait


class TridSolve(torch.autograd.Function):
    @staticmethod
    def forward(ctx, a, b, c, d, solvedim: int):
        x = d.detach().clone().contiguous()
        solve(a.detach().contiguous(), b.detach().contiguous(), c.detach().contiguous(), x,
              solvedim, sync=_ordered(x))  # (the copies come first)
        ctx.solvedim = solvedim
        ctx.save_for_backward(a, b, c, x)
        return x

    @staticmethod
    def backward(ctx, gx):
        # the adjoint takes dense arrays; the copies, like gx's, are dropped on
        # torch's stream, behind the launch that reads them
        a, b, c, x = ctx.saved_tensors
        a, b, c, x = a.contiguous(), b.contiguous(), c.contiguous(), x.contiguous()
        gx = gx.contiguous()
        ga, gb, gc, gd = (torch.empty_like(x) for _ in range(4))
        dims = dims_of(x)
        fn = (lib().tridDmtsvStridedBatchAdjoint if x.dtype == torch.float64
              else lib().tridSmtsvStridedBatchAdjoint)
        _check(fn(a.data_ptr(), b.data_ptr(), c.data_ptr(), x.data_ptr(), gx.data_ptr(),
                  ga.data_ptr(), gb.data_ptr(), gc.data_ptr(), gd.data_ptr(), len(dims),
                  ctx.solvedim, _iv(dims), _iv(dims), _ordered(x)), "tridXmtsvStridedBatchAdjoint")
        return ga, gb, gc, gd, None


def trid_solve(a, b, c, d, solvedim: int):
    """x = A^{-1} d along `solvedim`.  Where the library launches on torch's
    stream the call does not wait; x is ordered on that stream, as the results
    of torch's own operations are."""
    return TridSolve.apply(a, b, c, d, solvedim)


def _grid(t):
    nz, ny, nx = t.shape
    return nx, ny, nz


def vadi_forward(kappa, u0, steps: int, lam: float):
    u = u0.clone().contiguous()
    kappa = kappa.contiguous()  # the library takes dense grids
    nx, ny, nz = _grid(u)
    _ordered(u)
    _check(lib().tridVadiForward(kappa.data_ptr(), u.data_ptr(), nx, ny, nz, int(steps),
                                 float(lam), 1), "tridVadiForward")
    return u


def vadi_loss_grad(kappa, u0, target, steps: int, lam: float, ckpt: int = 4):
    """Returns (loss, grad_kappa, grad_u0)."""
    nx, ny, nz = _grid(u0)
    kappa, u0, target = kappa.contiguous(), u0.contiguous(), target.contiguous()
    gk = torch.empty_like(kappa)
    gu = torch.empty_like(u0)
    loss = C.c_double(0.0)
    _ordered(u0)
    _check(lib().tridVadiLossGrad(kappa.data_ptr(), u0.data_ptr(), target.data_ptr(), nx, ny, nz,
                                  int(steps), float(lam), int(ckpt), C.byref(loss),
                                  gk.data_ptr(), gu.data_ptr()), "tridVadiLossGrad")
    return loss.value, gk, gu
