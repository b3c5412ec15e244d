"""Normalised calls whose threshold scale lets a few per cent of the weights through: the candidate
and pair lists overflow, so the tile passes (fwd_pv_blk after the screen; bwd_tiles over the queue
of blocks, or bwd_dq_blk and bwd_dkv_blk without a queue) take most query and key tiles, beside
some that still fit.  Output and every gradient, beta's and lambda's too, against the fp64 oracle."""
import pytest
import torch

import tda_amd
from oracle.formula import rel_err, tda_grads
from tda_amd import ops
from tests.helpers import grads_on_gpu, rel_norm

pytestmark = pytest.mark.gpu
TOL = 2e-2  # bf16 weights, results and gradients (2^-9 each) in sums of up to a few hundred terms


def _inputs(b, h, nq, nk, d, br, dtype, seed):
    g = torch.Generator("cpu").manual_seed(seed)
    mk = lambda n: torch.randn((b, h, n, d), generator=g).to(dtype)  # noqa: E731
    return [mk(nq) for _ in range(br)] + [mk(nk) for _ in range(br + 1)], mk(nq)


@pytest.mark.parametrize("nq,nk,d,br,p,beta", [
    (33, 33, 64, 2, 2.0, 0.0),       # two query tiles, a partial block, every causal weight sign
    (128, 128, 128, 2, 2.0, 0.5),    # exactly one block of tiles
    (129, 129, 64, 1, 1.0, 0.4),     # a block of one tile with one row
    (300, 300, 64, 2, 1.5, 0.6),     # lists that fit beside lists that do not
    (520, 520, 128, 1, 2.0, 0.5),
    (100, 700, 64, 2, 2.0, 0.5),     # fewer query tiles than key tiles (a key cache)
    (200, 90, 128, 2, 3.0, 0.4),     # fewer key tiles than query tiles
    (33, 4200, 64, 2, 2.0, 0.5),     # more key tiles than the queue holds: no queue
    (40, 66000, 64, 1, 2.0, 0.7),    # more kept tiles than one listing of the walk (2048)
])
def test_overflowing_lists_against_the_oracle(nq, nk, d, br, p, beta):
    off = max(nk - nq, 0)
    rows, do = _inputs(1, 3 if nk < 10000 else 1, nq, nk, d, br, torch.bfloat16, 31)
    leaves = [x.cuda().requires_grad_(True) for x in rows]
    bt = torch.tensor(beta, device="cuda", requires_grad=True)
    lt = torch.tensor(0.4, device="cuda", requires_grad=True)
    if br == 2:
        out = tda_amd.differential_threshold_rela_triton(*leaves, bt, lt, relu_power=p, normalize=True)
        q1, q2, k1, k2, v = (x.double() for x in rows)
    else:
        out = tda_amd.threshold_rela_triton(*leaves, bt, relu_power=p, normalize=True)
        (q1, k1, v), q2, k2 = (x.double() for x in rows), None, None
    out.backward(do.cuda())
    ref = tda_grads(q1, q2, k1, k2, v, do.double(), beta, 0.4 if br == 2 else 0.0, p, True, br, q_offset=off)
    assert rel_err(out, ref["out"]) <= TOL
    names = ["dq1", "dq2", "dk1", "dk2", "dv"] if br == 2 else ["dq1", "dk1", "dv"]
    for leaf, name in zip(leaves, names):
        assert rel_err(leaf.grad, ref[name]) <= TOL, name
    # the scalars are sums of terms of both signs, each with the rounding of bf16 products' inputs only
    assert abs(bt.grad.item() - ref["dbeta"].item()) <= 1e-3 * abs(ref["dbeta"].item()) + 1e-5
    if br == 2:
        assert abs(lt.grad.item() - ref["dlambda"].item()) <= 1e-3 * abs(ref["dlambda"].item()) + 1e-5


@pytest.mark.parametrize("b,h,n,d,br,blocks", [(2, 16, 1500, 64, 2, 512), (3, 12, 1100, 128, 1, 256)])
def test_more_queued_blocks_than_workgroups(b, h, n, d, br, blocks):
    """bwd_tiles with more blocks in its queue than the GPU holds workgroups (`blocks`): they take
    further tickets, key blocks and then query blocks, in the same LDS.  Every head, in the 2-norm: bf16
    weights and results, 2^-9 at most each."""
    rows, do = _inputs(b, h, n, n, d, br, torch.bfloat16, 33)
    leaves = [x.cuda().requires_grad_(True) for x in rows]
    bt, lt = (torch.tensor(x, device="cuda", requires_grad=True) for x in (0.5, 0.4))
    if br == 2:
        out = tda_amd.differential_threshold_rela_triton(*leaves, bt, lt, normalize=True)
    else:
        out = tda_amd.threshold_rela_triton(*leaves, bt, normalize=True)
    out.backward(do.cuda())
    tiles = -(-n // 32)
    assert b * h * -(-tiles // 4) * (br + 1) * 0.8 > blocks  # (the first blocks' lists may fit)
    ref = grads_on_gpu(rows, do, 0.5, 0.4, 2.0, True, br)
    assert rel_norm(out, ref["out"]) <= 2.0 ** -8
    for leaf, name in zip(leaves, ["dq1", "dq2", "dk1", "dk2", "dv"] if br == 2 else ["dq1", "dk1", "dv"]):
        assert rel_norm(leaf.grad, ref[name]) <= 2.0 ** -8, name
    assert abs(bt.grad.item() - ref["dbeta"]) <= 1e-5 * ref["beta_scale"]
    if br == 2:
        assert abs(lt.grad.item() - ref["dlambda"]) <= 1e-5 * ref["lambda_scale"]


@pytest.mark.parametrize("d,br", [(64, 2), (128, 1)])
def test_queue_and_direct_launches_agree(d, br):
    """The backward from pair lists and a queue, and from the bitmask alone, give the same block
    sums for what both compute with the tile passes (bf16 rounding of dS apart in the rest)."""
    rows, do = _inputs(2, 2, 400, 400, d, br, torch.bfloat16, 32)
    xs = [x.cuda() for x in rows]
    do = do.cuda()
    q1, q2, k1, k2, v = xs if br == 2 else (xs[0], None, xs[1], None, xs[2])
    beta, lam = torch.tensor(0.3, device="cuda"), torch.tensor(0.5, device="cuda") if br == 2 else None
    norms, occ = ops.side_buffers(q1.shape, br, True, "cuda")
    pairs = ops.pair_buffer(q1.shape, br, "cuda")
    with torch.no_grad():
        ops.forward(q1, k1, q2, k2, v, beta, lam, 2.0, True, br, norms, occ, pairs=pairs)
        a = ops.backward(q1, k1, q2, k2, v, do, beta, lam, 2.0, True, br, norms, occ, pairs=pairs)
        again = ops.backward(q1, k1, q2, k2, v, do, beta, lam, 2.0, True, br, norms, occ, pairs=pairs)
        b = ops.backward(q1, k1, q2, k2, v, do, beta, lam, 2.0, True, br, norms, occ)
    for x, y, z in zip(a, again, b):
        if x is None:
            continue
        assert torch.equal(x, y)  # whatever order the queue was filled in
        assert rel_err(x, z.double().cpu()) <= TOL
