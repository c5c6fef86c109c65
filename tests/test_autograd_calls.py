"""What the differentiable wrappers hand to the library, on the CPU: the
library is replaced by one that solves with the oracle over the addresses it
is given."""
from __future__ import annotations

import ctypes as C
from types import SimpleNamespace

import numpy as np
import pytest
import torch

import oracle
from tests.helpers import dd_system, oracle_solve
from tridsolver_amd import autograd


class OracleLib:
    """The adjoint entry points over host arrays."""

    def _adjoint(self, a, b, c, x, g, ga, gb, gc, gd, ndim, sd, dims, pads, sync):
        dims = [dims[k] for k in range(ndim)]
        n = int(np.prod(dims))
        at = [np.ctypeslib.as_array((C.c_double * n).from_address(p))
              for p in (a, b, c, x, g, ga, gb, gc, gd)]
        exp = oracle.adjoint(*[v.copy() for v in at[:5]], ndim, sd, dims)
        for out, e in zip(at[5:], exp):
            out[:] = e
        return 0

    def __getattr__(self, name):
        if name == "tridDmtsvStridedBatchAdjoint":
            return self._adjoint
        raise AttributeError(name)


def _oracle_solve(a, b, c, d, sd, u=None, inc=False, sync=1):
    for t in (a, b, c, d):
        assert t.is_contiguous() and t.shape == d.shape
    dims = list(reversed(d.shape))
    x = oracle_solve(*[t.numpy().ravel() for t in (a, b, c, d)], None, dims, sd)
    d.copy_(torch.from_numpy(x.reshape(d.shape)))


@pytest.fixture
def on_host(monkeypatch):
    monkeypatch.setattr(autograd, "lib", lambda: OracleLib())
    monkeypatch.setattr(autograd, "solve", _oracle_solve)
    monkeypatch.setattr(autograd, "_sync", lambda t: 0)


def _transposed(t):
    return t.detach().transpose(0, 2).contiguous().transpose(0, 2)


def _sliced(t):
    wide = torch.full((*t.shape[:-1], t.shape[-1] + 3), float("nan"), dtype=t.dtype)
    wide[..., 2:-1] = t.detach()
    return wide[..., 2:-1]


def _expanded(t):
    """One plane for all (its storage holds whole planes for every index)."""
    room = torch.zeros_like(t)
    room[0] = t.detach()[0]
    return room[:1].expand(t.shape)


@pytest.mark.parametrize("sd", [0, 1, 2])
@pytest.mark.parametrize("make", [_transposed, _sliced, _expanded])
def test_coefficients_of_any_strides(on_host, make, sd):
    """Gradients with coefficients that are not contiguous are those with
    contiguous copies of them."""
    dims, shape = [6, 5, 4], (4, 5, 6)
    t = [torch.from_numpy(v).reshape(shape) for v in dd_system(dims, sd, np.float64, seed=2)]
    abc = [make(v) for v in t[:3]]
    assert not any(v.is_contiguous() for v in abc)
    g = torch.from_numpy(np.random.default_rng(1).uniform(-1, 1, shape))
    got, exp = [], []
    for out, coef in ((got, abc), (exp, [v.contiguous() for v in abc])):
        leaves = [v.detach().requires_grad_(True) for v in (*coef, t[3])]
        x = autograd.trid_solve(*leaves, sd)
        out.append(x.detach())
        out.extend(torch.autograd.grad(x, leaves, g))
    for a, b in zip(got, exp):
        assert torch.equal(a, b)


@pytest.mark.parametrize("device,library,torch_stream,wait",
                         [(0, 0, 0, 0), (0, 0, 7, 1), (0, 7, 0, 1), (0, 7, 7, 0),
                          (1, 0, 0, 1), (1, 7, 7, 1)])
def test_waits_unless_on_the_tensors_stream(monkeypatch, device, library, torch_stream, wait):
    """Null streams have the same handle on every device: a call for a tensor
    of another device than the current one waits whatever the handles."""
    class Lib:
        @staticmethod
        def tridGetStream():
            return library or None

    monkeypatch.setattr(autograd, "lib", Lib)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "current_stream",
                        lambda dev=None: SimpleNamespace(cuda_stream=torch_stream))
    assert autograd._sync(SimpleNamespace(device=torch.device("cuda", device))) == wait


@pytest.mark.parametrize("wait", [0, 1])
def test_other_streams_start_behind_torchs(on_host, monkeypatch, wait):
    """Where the library launches on another stream, what torch has on its own
    (the copies of the operands, an earlier call's results) is finished before
    the launch; elsewhere nothing waits."""
    log = []
    stream = SimpleNamespace(synchronize=lambda: log.append("wait"))

    class Lib(OracleLib):
        def _adjoint(self, *args):
            log.append(("adjoint", args[-1]))
            return super()._adjoint(*args)

    def solve(*args, sync):
        log.append(("solve", sync))
        _oracle_solve(*args)

    monkeypatch.setattr(autograd, "lib", lambda: Lib())
    monkeypatch.setattr(autograd, "solve", solve)
    monkeypatch.setattr(autograd, "_sync", lambda t: wait)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev=None: stream)
    dims = [6, 5]
    t = [torch.from_numpy(v).reshape(5, 6).requires_grad_(True)
         for v in dd_system(dims, 0, np.float64, seed=2)]
    autograd.trid_solve(*t, 0).sum().backward()
    start = ["wait"] * wait
    assert log == start + [("solve", wait)] + start + [("adjoint", wait)]


def test_saved_tensor_hooks_of_any_strides(on_host):
    """Hooks that give the saved tensors back with other strides change nothing."""
    dims, shape = [6, 5, 4], (4, 5, 6)
    t = [torch.from_numpy(v).reshape(shape) for v in dd_system(dims, 1, np.float64, seed=3)]
    g = torch.from_numpy(np.random.default_rng(2).uniform(-1, 1, shape))
    grads = []
    for unpack in (lambda v: v, _transposed):
        leaves = [v.clone().requires_grad_(True) for v in t]
        with torch.autograd.graph.saved_tensors_hooks(lambda v: v, unpack):
            x = autograd.trid_solve(*leaves, 1)
        grads.append(torch.autograd.grad(x, leaves, g))
    assert all(torch.equal(u, v) for u, v in zip(*grads))


class VadiLib:
    """The variable-diffusivity entry points over host arrays."""

    @staticmethod
    def _grid(p, n):
        return np.ctypeslib.as_array((C.c_double * n ** 3).from_address(p))

    def tridVadiForward(self, kappa, u, nx, ny, nz, steps, lam, sync):
        k, v = self._grid(kappa, nx), self._grid(u, nx)
        v[:] = oracle.vadi_forward(k.copy(), v.copy(), nx, steps, lam)
        return 0

    def tridVadiLossGrad(self, kappa, u0, target, nx, ny, nz, steps, lam, ckpt, loss, gk, gu):
        k, u, t = (self._grid(p, nx).copy() for p in (kappa, u0, target))
        loss._obj.value, a, b = oracle.vadi_grad(k, u, t, nx, steps, lam)
        self._grid(gk, nx)[:], self._grid(gu, nx)[:] = a, b
        return 0


@pytest.mark.parametrize("make", [_transposed, _sliced, _expanded])
def test_vadi_grids_of_any_strides(monkeypatch, make):
    """Grids that are not contiguous give what contiguous copies of them do."""
    monkeypatch.setattr(autograd, "lib", VadiLib)
    monkeypatch.setattr(autograd, "_sync", lambda t: 0)
    gen = torch.Generator().manual_seed(4)
    grids = [make(torch.rand(5, 5, 5, generator=gen, dtype=torch.float64) + 0.5)
             for _ in range(3)]
    assert not any(t.is_contiguous() for t in grids)
    kappa, u0, target = dense = [t.contiguous() for t in grids]
    assert torch.equal(autograd.vadi_forward(*grids[:2], 2, 0.5),
                       autograd.vadi_forward(kappa, u0, 2, 0.5))
    got = autograd.vadi_loss_grad(*grids, 2, 0.5)
    exp = autograd.vadi_loss_grad(*dense, 2, 0.5)
    assert got[0] == exp[0]
    assert torch.equal(got[1], exp[1]) and torch.equal(got[2], exp[2])


@pytest.mark.parametrize("wait", [0, 1])
def test_vadi_starts_behind_torchs_stream(monkeypatch, wait):
    """As for the solves: the copies of the grids are finished before a launch
    on another stream than torch's."""
    log = []

    class Lib(VadiLib):
        def tridVadiForward(self, *args):
            log.append("forward")
            return super().tridVadiForward(*args)

        def tridVadiLossGrad(self, *args):
            log.append("gradient")
            return super().tridVadiLossGrad(*args)

    monkeypatch.setattr(autograd, "lib", Lib)
    monkeypatch.setattr(autograd, "_sync", lambda t: wait)
    stream = SimpleNamespace(synchronize=lambda: log.append("wait"))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev=None: stream)
    kappa, u0, target = (torch.ones(4, 4, 4, dtype=torch.float64) for _ in range(3))
    autograd.vadi_forward(kappa, u0, 1, 0.5)
    autograd.vadi_loss_grad(kappa, u0, target, 1, 0.5)
    start = ["wait"] * wait
    assert log == start + ["forward"] + start + ["gradient"]
