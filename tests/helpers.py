"""Shared helpers for the GPU parity tests: seeded input generation (the draw order the
benchmark configs use) and oracle evaluation on the exact values the GPU consumed."""
from __future__ import annotations

import torch

from oracle.formula import rel_err, tda_chunked, tda_grads  # noqa: F401

TOL = {torch.float32: 1e-4, torch.bfloat16: 2e-2}


def make_inputs(shape, seed, count, dtype, device="cuda"):
    """`count` i.i.d. N(0,1) tensors drawn in argument order from one CPU generator seeded
    with `seed`, rounded to `dtype` and moved to `device`."""
    g = torch.Generator("cpu").manual_seed(seed)
    xs = [torch.randn(shape, generator=g, dtype=torch.float32) for _ in range(count)]
    return [x.to(dtype).to(device) for x in xs]


def host(x, dtype=torch.float64):
    return None if x is None else x.detach().to("cpu", dtype)


def oracle_out(q1, q2, k1, k2, v, beta, lam, p, normalize, branches, heads=None, dtype=torch.float64):
    """The CPU oracle on the values the GPU saw (bf16 inputs are upcast exactly)."""
    return tda_chunked(host(q1, dtype), host(q2, dtype), host(k1, dtype), host(k2, dtype), host(v, dtype),
                       float(beta), float(lam), p, normalize, branches=branches, heads=heads, dtype=dtype)


def rel_norm(y, ref) -> float:
    """2-norm of the difference over the 2-norm of the reference."""
    y, ref = y.detach().double().cpu(), ref.detach().double().cpu()
    return ((y - ref).norm() / ref.norm().clamp_min(1e-300)).item()


def grads_on_gpu(rows, dout, beta, lam, p, normalize, branches, q_offset=0):
    """tda_grads of every head, evaluated in float64 on the GPU a batch entry at a time: a dict of out,
    the rows' gradients and the scalars', and for the scalars beta_scale and lambda_scale, the sums of
    their per-row contributions' magnitudes (what the rounding of sums of both signs is measured
    against)."""
    from oracle.formula import tda, tra
    names = ["dq1", "dq2", "dk1", "dk2", "dv"] if branches == 2 else ["dq1", "dk1", "dv"]
    n = rows[0].shape[2]
    res = {k: [] for k in ["out", *names]}
    res.update(dbeta=0.0, dlambda=0.0, beta_scale=0.0, lambda_scale=0.0)
    for b in range(rows[0].shape[0]):
        xs = [x.detach()[b:b + 1].double().cuda().requires_grad_(True) for x in rows]
        bt = torch.full((n,), float(beta), dtype=torch.float64, device="cuda", requires_grad=True)
        if branches == 2:
            lt = torch.full((n, 1), float(lam), dtype=torch.float64, device="cuda", requires_grad=True)
            out = tda(*xs, bt, lt, p, normalize, q_offset=q_offset)
            g = torch.autograd.grad(out, [*xs, bt, lt], dout[b:b + 1].double().cuda())
            res["dlambda"] += g[-1].sum().item()
            res["lambda_scale"] += g[-1].abs().sum().item()
            g = g[:-1]
        else:
            out = tra(*xs, bt, p, normalize, q_offset=q_offset)
            g = torch.autograd.grad(out, [*xs, bt], dout[b:b + 1].double().cuda())
        res["dbeta"] += g[-1].sum().item()
        res["beta_scale"] += g[-1].abs().sum().item()
        res["out"].append(out.detach())
        for name, x in zip(names, g):
            res[name].append(x)
    return {k: torch.cat(v) if isinstance(v, list) else v for k, v in res.items()}


def heads_of(x, heads):
    return torch.stack([x[b, h] for (b, h) in heads])
