"""The work that programs have this library do, as cases that can be timed.

Every case goes through a public entry point of tridsolver_amd with its
default settings (no autotuning, no forced layouts), with device arrays that
the program already holds, and enqueues without waiting (sync = 0) where the
entry point offers that.  Sizes are those of the benchmark (256^3 grids,
N = 128 block rows, lengths log-uniform in [8, 4096]), of the tests, or
ordinary grid sizes between the powers of two.

`op` of a case:
  solve      tridS/DmtsvStridedBatch[Padded][Inc]: `dims` "x,y,z" (dimension 0
             fastest), along dimension `sd`; `pad` elements of padding behind
             every line of dimension 0; `inc` adds the solution into u
  adi        AdiPlan.step: `steps` time steps on one grid
  ragged     RaggedPlan.solve: `nsys` systems of lengths log-uniform in
             [lo, hi]
  block      btsv: `P` systems of `N` block rows of M x M blocks
  block_grad btsv, then btsv_adjoint for an upstream gradient
  solve_grad trid_solve (autograd) forward and backward
  vadi_grad  vadi_loss_grad: loss and gradient of `steps` steps of the
             variable-diffusivity ADI, a checkpoint every `ckpt` steps
"""
import math

import numpy as np
import torch

import tridsolver_amd
from tridsolver_amd import api
from tridsolver_amd.adi import AdiPlan
from tridsolver_amd.autograd import trid_solve, vadi_loss_grad
from tridsolver_amd.block import btsv, btsv_adjoint
from tridsolver_amd.ragged import RaggedPlan

LISTED = [
    # one small batch inside a larger program: latency and launches
    dict(name="solve_x_small_f64", op="solve", dims="100,40", sd=0, dtype="f64", inc=False, pad=0),
    # the benchmark's plain solve along the contiguous dimension
    dict(name="solve_x_f64", op="solve", dims="256,256,256", sd=0, dtype="f64", inc=False, pad=0),
    # an implicit sweep along y of a single-precision grid of odd sizes
    dict(name="solve_y_f32", op="solve", dims="300,333,150", sd=1, dtype="f32", inc=False, pad=0),
    # the last sweep of a time step: along z, added into u, lines padded
    dict(name="solve_z_inc_f64", op="solve", dims="200,180,250", sd=2, dtype="f64", inc=True, pad=8),
    # a 2-d problem whose systems are longer than a work-group holds
    dict(name="solve_y_long_f64", op="solve", dims="48,150000", sd=1, dtype="f64", inc=False, pad=0),
    # the benchmark's time step
    dict(name="adi_f64", op="adi", dims="256,256,256", steps=10, dtype="f64"),
    # time steps of a single-precision grid of ordinary sizes
    dict(name="adi_f32", op="adi", dims="200,150,180", steps=10, dtype="f32"),
    # many systems of uneven length in one call
    dict(name="ragged_f64", op="ragged", nsys=50000, lo=8, hi=4096, dtype="f64"),
    # coupled equations: 4 unknowns per grid point
    dict(name="block_f64", op="block", M=4, N=128, P=16384, dtype="f64"),
    # the same with 3 unknowns, differentiated
    dict(name="block_grad_f64", op="block_grad", M=3, N=100, P=8000, dtype="f64"),
    # a differentiable single-precision solve of long rows
    dict(name="solve_grad_f32", op="solve_grad", dims="1000,4000", sd=0, dtype="f32"),
    # calibration of a diffusivity field against a target
    dict(name="vadi_grad_f64", op="vadi_grad", n=96, steps=8, ckpt=4),
]


def listed():
    return [dict(c) for c in LISTED]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges."""
    most = max(_cost(c) for c in LISTED)
    while True:
        op = rng.choice(["solve", "solve", "solve", "adi", "adi", "ragged", "block", "block",
                         "block_grad", "solve_grad", "vadi_grad"])
        dt = rng.choice(["f64", "f32"])
        if op == "solve":
            ndim = rng.choice([2, 3, 3])
            sd = rng.randrange(ndim)
            dims = [_log(rng, 8, 400) for _ in range(ndim)]
            # mostly grid lines, now and then systems past one work-group
            dims[sd] = _log(rng, 16, 2000) if rng.random() < 0.85 else _log(rng, 2000, 200000)
            c = dict(op=op, dims=",".join(map(str, dims)), sd=sd, dtype=dt,
                     inc=rng.random() < 0.3, pad=rng.choice([0, 0, 0, 1, 8]))
        elif op == "adi":
            dims = [_log(rng, 32, 300) for _ in range(3)]
            if rng.random() < 0.5:  # power-of-two lines, the other half as they come
                dims[0] = rng.choice([64, 128, 256])
            c = dict(op=op, dims=",".join(map(str, dims)), steps=rng.choice([1, 5, 10]), dtype=dt)
        elif op == "ragged":
            hi = rng.choice([64, 512, 4096, 6000])
            c = dict(op=op, nsys=_log(rng, 500, 50000), lo=rng.choice([4, 8, 32]), hi=hi, dtype=dt)
        elif op in ("block", "block_grad"):
            if op == "block_grad":
                dt = "f64"  # the adjoint's only precision
            c = dict(op=op, M=rng.randint(2, 8), N=_log(rng, 20, 256), P=_log(rng, 500, 32768),
                     dtype=dt)
        elif op == "solve_grad":
            ndim = rng.choice([2, 3])
            sd = rng.randrange(ndim)
            dims = [_log(rng, 8, 300) for _ in range(ndim)]
            dims[sd] = _log(rng, 16, 2000)
            c = dict(op=op, dims=",".join(map(str, dims)), sd=sd, dtype=dt)
        else:
            c = dict(op=op, n=_log(rng, 24, 128), steps=rng.choice([4, 8, 12]),
                     ckpt=rng.choice([2, 4]))
        if _cost(c) <= most and _values(c) >= 2000:
            return c


def _dims(case):
    return [int(v) for v in case["dims"].split(",")]


def _word(case):
    return 4 if case.get("dtype") == "f32" else 8


def _type(case):
    return torch.float32 if case.get("dtype") == "f32" else torch.float64


def _values(case):
    """Unknowns (block rows times M; grid points times steps) of one pass."""
    op = case["op"]
    if op in ("solve", "solve_grad"):
        return math.prod(_dims(case))
    if op == "adi":
        return math.prod(_dims(case)) * case["steps"]
    if op == "ragged":
        lo, hi = case["lo"], case["hi"]
        return int(case["nsys"] * (hi + 1 - lo) / math.log((hi + 1) / lo))
    if op in ("block", "block_grad"):
        return case["M"] * case["N"] * case["P"]
    return case["n"] ** 3 * case["steps"]


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def work(case):
    op, v, w = case["op"], _values(case), _word(case)
    if op == "solve":
        # a, b, c, d in, the solution out (Inc: u in as well)
        return dict(bytes=(6 if case["inc"] else 5) * w * v, flops=8 * v)
    if op == "adi":
        # per step u in and out; a step's three sweeps and 7-point stencil
        return dict(bytes=2 * w * v, flops=25 * v)
    if op == "ragged":
        return dict(bytes=5 * w * v + 8 * (case["nsys"] + 1), flops=8 * v)
    if op in ("block", "block_grad"):
        m, rows = case["M"], case["N"] * case["P"]
        fb, ff = 3 * m * m + 2 * m, 2 * m ** 3 * 7 // 3 + 6 * m * m
        if op == "block":
            return dict(bytes=fb * w * rows, flops=ff * rows)
        # the solve; then A, B, C, u, g in and four gradients out
        return dict(bytes=(fb + 6 * m * m + 3 * m) * w * rows, flops=(2 * ff + 3 * m * m) * rows)
    if op == "solve_grad":
        # the solve; then a, b, c, x, g in and four gradients out
        return dict(bytes=(5 + 9) * w * v, flops=20 * v)
    # kappa and u in, u out per step and again per step of the reverse pass
    return dict(bytes=6 * w * v, flops=100 * v)


# ---------------------------------------------------------------- inputs


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _uniform(shape, lo, hi, gen, dtype):
    return torch.rand(shape, generator=gen, device="cuda", dtype=dtype) * (hi - lo) + lo


def _system(shape, gen, dtype):
    """A diagonally dominant tridiagonal system per line: a, b, c, d."""
    a = _uniform(shape, -1.0, -0.1, gen, dtype)
    c = _uniform(shape, -1.0, -0.1, gen, dtype)
    b = a.abs() + c.abs() + _uniform(shape, 0.5, 1.5, gen, dtype)
    d = _uniform(shape, -1.0, 1.0, gen, dtype)
    return a, b, c, d


def _blocks(case, gen, dtype):
    n, p, m = case["N"], case["P"], case["M"]
    a = _uniform((n, p, m, m), -1.0, 1.0, gen, dtype) / m
    c = _uniform((n, p, m, m), -1.0, 1.0, gen, dtype) / m
    a[0] = 0
    c[n - 1] = 0
    b = _uniform((n, p, m, m), -1.0, 1.0, gen, dtype) / m
    b += torch.diag_embed(a.abs().sum(-1) + c.abs().sum(-1) + 1.0)
    return a, b, c, _uniform((n, p, m), -1.0, 1.0, gen, dtype)


def _kappa(n, gen):
    """exp(0.3 g), g a sum of eight Fourier modes with wave numbers in [-3, 3]."""
    x = torch.arange(n, device="cuda", dtype=torch.float64) / n
    z, y, x = torch.meshgrid(x, x, x, indexing="ij")
    k = torch.randint(-3, 4, (8, 3), generator=gen, device="cuda").double().tolist()
    amp = torch.randn(8, generator=gen, device="cuda", dtype=torch.float64) / math.sqrt(8)
    ph = torch.rand(8, generator=gen, device="cuda", dtype=torch.float64) * (2 * math.pi)
    g = torch.zeros_like(x)
    for i in range(8):
        g += amp[i] * torch.cos(2 * math.pi * (k[i][0] * x + k[i][1] * y + k[i][2] * z) + ph[i])
    return torch.exp(0.3 * g)


def _lengths(case, seed):
    """The quantiles of the log-uniform distribution, in an order of the seed's."""
    n, lo, hi = case["nsys"], case["lo"], case["hi"]
    q = (np.arange(n) + 0.5) / n
    lens = np.floor(lo * np.exp(q * np.log((hi + 1) / lo))).astype(np.int64)
    return np.random.default_rng(int(seed)).permutation(lens)


def _inputs(case, seed):
    """The tensors of a case, made from the seed alone."""
    op, g, dt = case["op"], _gen(seed), _type(case)
    if op == "solve":
        dims = _dims(case)
        shape = tuple(reversed([dims[0] + case["pad"]] + dims[1:]))
        t = dict(zip("abcd", _system(shape, g, dt)))
        if case["inc"]:
            t["u"] = _uniform(shape, -1.0, 1.0, g, dt)
        return t
    if op == "solve_grad":
        shape = tuple(reversed(_dims(case)))
        t = dict(zip("abcd", _system(shape, g, dt)))
        t["g"] = _uniform(shape, -1.0, 1.0, g, dt)
        return t
    if op == "adi":
        u = _uniform(tuple(reversed(_dims(case))), 0.0, 1.0, g, dt)
        inside = torch.zeros_like(u)
        inside[1:-1, 1:-1, 1:-1] = 1
        return dict(u=u * inside)
    if op == "ragged":
        off = np.concatenate([[0], np.cumsum(_lengths(case, seed))]).astype(np.int64)
        return dict(zip("abcd", _system((int(off[-1]),), g, dt)), off=torch.from_numpy(off).cuda())
    if op in ("block", "block_grad"):
        t = dict(zip("abcd", _blocks(case, g, dt)))
        if op == "block_grad":
            t["g"] = _uniform(t["d"].shape, -1.0, 1.0, g, dt)
        return t
    n = case["n"]
    return dict(kappa=_kappa(n, g), u0=_uniform((n, n, n), 0.0, 1.0, g, dt),
                target=_uniform((n, n, n), 0.0, 1.0, g, dt))


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"], op = case, case["op"]
    if op == "solve":
        dims = _dims(case)
        s["dims"], s["pads"] = dims, [dims[0] + case["pad"]] + dims[1:]
    elif op == "solve_grad":
        for k in "abcd":
            s[k].requires_grad_(True)
    elif op == "adi":
        s["du"] = torch.empty_like(s["u"])
        s["plan"] = AdiPlan(*_dims(case), _type(case))
    elif op == "ragged":
        s["plan"] = RaggedPlan(s["off"], _type(case))
    elif op in ("block", "block_grad"):
        s["u"] = torch.empty_like(s["d"])
    return s


_SOLVE = {
    ("f64", False, False): api.tridDmtsvStridedBatch,
    ("f64", True, False): api.tridDmtsvStridedBatchInc,
    ("f32", False, False): api.tridSmtsvStridedBatch,
    ("f32", True, False): api.tridSmtsvStridedBatchInc,
    ("f64", False, True): api.tridDmtsvStridedBatchPadded,
    ("f64", True, True): api.tridDmtsvStridedBatchPaddedInc,
    ("f32", False, True): api.tridSmtsvStridedBatchPadded,
    ("f32", True, True): api.tridSmtsvStridedBatchPaddedInc,
}


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "solve":
        fn = _SOLVE[case["dtype"], case["inc"], case["pad"] > 0]
        a, b, c, d, u, dims, pads = s["a"], s["b"], s["c"], s["d"], s.get("u"), s["dims"], s["pads"]
        if case["pad"]:
            st = fn(a, pads, b, pads, c, pads, d, pads, u, pads, len(dims), case["sd"], dims,
                    None, 0)
        else:
            st = fn(a, b, c, d, u, len(dims), case["sd"], dims, pads, None, 0)
        if st:
            raise RuntimeError(tridsolver_amd.last_error())
        return u if case["inc"] else d
    if op == "adi":
        s["plan"].step(s["u"], s["du"], case["steps"], sync=0)
        return s["u"]
    if op == "ragged":
        s["plan"].solve(s["a"], s["b"], s["c"], s["d"], sync=0)
        return s["d"]
    if op == "block":
        return btsv(s["a"], s["b"], s["c"], s["d"], s["u"], sync=0)
    if op == "block_grad":
        u = btsv(s["a"], s["b"], s["c"], s["d"], s["u"], sync=0)
        return (u,) + btsv_adjoint(s["a"], s["b"], s["c"], u, s["g"], sync=0)
    if op == "solve_grad":
        x = trid_solve(s["a"], s["b"], s["c"], s["d"], case["sd"])
        return (x.detach(),) + torch.autograd.grad(x, [s[k] for k in "abcd"], s["g"])
    return vadi_loss_grad(s["kappa"], s["u0"], s["target"], case["steps"], 1.0, case["ckpt"])


# ------------------------------------------------- the same in 64 bits


def _shift(x, k, dim, fill):
    """y_i = x_{i-k} along dim, `fill` where there is none."""
    n = x.shape[dim]
    pad = torch.full_like(x.narrow(dim, 0, min(abs(k), n)), fill)
    if abs(k) >= n:
        return pad
    if k > 0:
        return torch.cat([pad, x.narrow(dim, 0, n - k)], dim)
    return torch.cat([x.narrow(dim, -k, n + k), pad], dim)


def _pcr(a, b, c, d, dim):
    """Parallel cyclic reduction: all lines along dim at once."""
    n, k = d.shape[dim], 1
    zero = torch.zeros_like(a.narrow(dim, 0, 1))
    a = torch.cat([zero, a.narrow(dim, 1, n - 1)], dim)
    c = torch.cat([c.narrow(dim, 0, n - 1), zero], dim)
    while k < n:
        lo, hi = -a / _shift(b, k, dim, 1.0), -c / _shift(b, -k, dim, 1.0)
        b = b + lo * _shift(c, k, dim, 0.0) + hi * _shift(a, -k, dim, 0.0)
        d = d + lo * _shift(d, k, dim, 0.0) + hi * _shift(d, -k, dim, 0.0)
        a, c = lo * _shift(a, k, dim, 0.0), hi * _shift(c, -k, dim, 0.0)
        k *= 2
    return d / b


def _inside(shape, dim=None):
    m = torch.zeros(shape, device="cuda", dtype=torch.float64)
    at = [slice(None)] * 3
    for k in range(3) if dim is None else [dim]:
        at[k] = slice(1, -1)
    m[tuple(at)] = 1
    return m


def _vadi_step(u, kappa):
    """One variable-diffusivity step with lam = 1."""
    r = torch.zeros_like(u)
    abc = []
    for dim in (2, 1, 0):
        n = u.shape[dim]
        face = 0.5 * (kappa.narrow(dim, 0, n - 1) + kappa.narrow(dim, 1, n - 1))
        flux = face * (u.narrow(dim, 1, n - 1) - u.narrow(dim, 0, n - 1))
        edge = torch.zeros_like(face.narrow(dim, 0, 1))
        r = r + torch.cat([flux, edge], dim) - torch.cat([edge, flux], dim)
        m = _inside(u.shape, dim)
        a, c = -torch.cat([edge, face], dim) * m, -torch.cat([face, edge], dim) * m
        abc.append((dim, a, 1.0 - a - c, c))
    r = r * _inside(u.shape)
    for dim, a, b, c in abc:
        r = _pcr(a, b, c, r, dim)
    return u + r


def _inverse(x):
    """Gauss-Jordan inverses of a batch of (diagonally dominant) blocks."""
    m = x.shape[-1]
    w = torch.cat([x, torch.eye(m, device=x.device, dtype=x.dtype).expand_as(x)], -1)
    for i in range(m):
        row = w[..., i:i + 1, :] / w[..., i:i + 1, i:i + 1]
        w = w - w[..., :, i:i + 1] * row
        w[..., i:i + 1, :] = row
    return w[..., m:]


def _mul(x, y):
    """Products of a batch of small blocks (y: blocks or vectors)."""
    if y.dim() == x.dim():
        return (x.unsqueeze(-1) * y.unsqueeze(-3)).sum(-2)
    return (x * y.unsqueeze(-2)).sum(-1)


def _block_thomas(a, b, c, d):
    n, cs, ds = d.shape[0], [], []
    for i in range(n):
        x, r = b[i], d[i]
        if i:
            x, r = x - _mul(a[i], cs[-1]), r - _mul(a[i], ds[-1])
        inv = _inverse(x)
        cs.append(_mul(inv, c[i]))
        ds.append(_mul(inv, r))
    u = [ds[-1]]
    for i in range(n - 2, -1, -1):
        u.append(ds[i] - _mul(cs[i], u[-1]))
    return torch.stack(u[::-1])


def _outer(x, y):
    return x.unsqueeze(-1) * y.unsqueeze(-2)


def exact(case, seed):
    op = case["op"]
    t = {k: v.double() if v.is_floating_point() else v for k, v in _inputs(case, seed).items()}
    if op == "solve":
        dims = _dims(case)
        axis = len(dims) - 1 - case["sd"]
        view = [t[k][..., :dims[0]] for k in "abcd"]
        out = t["u"] if case["inc"] else t["d"]
        x = _pcr(*view, axis)
        out[..., :dims[0]] = out[..., :dims[0]] + x if case["inc"] else x
        return out
    if op == "adi":
        u, inner = t["u"], _inside(t["u"].shape)
        for _ in range(case["steps"]):
            r = -6.0 * u
            for dim in range(3):
                r = r + _shift(u, 1, dim, 0.0) + _shift(u, -1, dim, 0.0)
            r = r * inner
            for dim in (2, 1, 0):
                off = -_inside(u.shape, dim)
                r = _pcr(off, 1.0 - 2.0 * off, off, r, dim)
            u = u + r
        return u
    if op == "ragged":
        # the systems end to end, uncoupled where one ends
        off = t["off"]
        a, c = t["a"].clone(), t["c"].clone()
        a[off[:-1]] = 0
        c[off[1:] - 1] = 0
        n, k = a.numel(), 1
        b, d, top = t["b"], t["d"], case["hi"]
        while k < min(n, top):
            lo, hi = -a / _shift(b, k, 0, 1.0), -c / _shift(b, -k, 0, 1.0)
            b = b + lo * _shift(c, k, 0, 0.0) + hi * _shift(a, -k, 0, 0.0)
            d = d + lo * _shift(d, k, 0, 0.0) + hi * _shift(d, -k, 0, 0.0)
            a, c = lo * _shift(a, k, 0, 0.0), hi * _shift(c, -k, 0, 0.0)
            k *= 2
        return d / b
    if op in ("block", "block_grad"):
        a, b, c = t["a"], t["b"], t["c"]
        u = _block_thomas(a, b, c, t["d"])
        if op == "block":
            return u
        zero = torch.zeros_like(a[:1])
        at = torch.cat([zero, c[:-1].transpose(-1, -2)])
        ct = torch.cat([a[1:].transpose(-1, -2), zero])
        lam = _block_thomas(at, b.transpose(-1, -2), ct, t["g"])
        edge = torch.zeros_like(u[:1])
        return (u, -_outer(lam, torch.cat([edge, u[:-1]])), -_outer(lam, u),
                -_outer(lam, torch.cat([u[1:], edge])), lam)
    if op == "solve_grad":
        axis = len(_dims(case)) - 1 - case["sd"]
        a, b, c = t["a"], t["b"], t["c"]
        x = _pcr(a, b, c, t["d"], axis)
        lam = _pcr(_shift(c, 1, axis, 0.0), b, _shift(a, -1, axis, 0.0), t["g"], axis)
        return (x, -lam * _shift(x, 1, axis, 0.0), -lam * x, -lam * _shift(x, -1, axis, 0.0), lam)
    kappa, u0 = t["kappa"].requires_grad_(True), t["u0"].requires_grad_(True)
    u = u0
    for _ in range(case["steps"]):
        u = _vadi_step(u, kappa)
    loss = 0.5 * (u - t["target"]).square().sum()
    gk, gu = torch.autograd.grad(loss, (kappa, u0))
    return float(loss), gk, gu
