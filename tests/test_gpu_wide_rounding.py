"""head_dim 256 in bf16: what is rounded, and when.  Both branches' weights are combined in fp32 and
rounded once for the output and for dv; every pass contracts a score's row in one chain, so forward
and backward find the same weights."""
import pytest
import torch

import tda_amd
from oracle.formula import tda_grads

pytestmark = pytest.mark.gpu
D = 256


def _rows(n, seed, count, h=2):
    g = torch.Generator("cpu").manual_seed(seed)
    return [torch.randn((1, h, n, D), generator=g).bfloat16() for _ in range(count)]


def _step(rows, do, beta, lam, p, normalize, **kw):
    """(out, gradients of the rows) of one differential step."""
    leaves = [x.cuda().requires_grad_(True) for x in rows]
    out = tda_amd.differential_threshold_rela_triton(*leaves, beta, lam, relu_power=p, normalize=normalize, **kw)
    return out.detach(), torch.autograd.grad(out, leaves, do.cuda())


@pytest.mark.parametrize("normalize,n", [(True, 100), (False, 33), (True, 161)])
def test_equal_branches_cancel_exactly(normalize, n):
    """lambda = 1 and equal branches: every combined weight is exactly 0."""
    q, k, v, do = _rows(n, 51, 4)
    out, (dq1, dq2, dk1, dk2, dv) = _step([q, q, k, k, v], do, 0.3, 1.0, 2.0, normalize)
    assert not out.any() and not dv.any()
    assert dq1.any() and dk1.any()
    for a, b in ((dq1, dq2), (dk1, dk2)):  # each rounded once more
        assert (a.double() + b.double()).norm() <= 2.0 ** -8 * a.double().norm()


@pytest.mark.parametrize("normalize,p", [(True, 2.0), (False, 2.0), (False, 1.5)])
def test_combined_weights_are_rounded_once(normalize, p):
    """Branches that nearly cancel (A2 = 0.88 A1 or so): the combined weights' own rounding and the
    results' (2^-9 at most each, so 2^-8 in the 2-norm), not that of weights eight times larger."""
    q, k, v, do = _rows(130, 52, 4)
    q2 = (q.float() * 0.9375).bfloat16()
    k2 = k if not normalize else (k.float() + 0.02 * torch.randn(k.shape, generator=torch.Generator().manual_seed(1))).bfloat16()
    rows = [q, q2, k, k2, v]
    out, (_, _, _, _, dv) = _step(rows, do, 0.0, 1.0, p, normalize)
    ref = tda_grads(*(x.double() for x in rows), do.double(), 0.0, 1.0, p, normalize, 2)
    for got, want in ((out, ref["out"]), (dv, ref["dv"])):
        assert (got.double().cpu() - want).norm() <= 2.0 ** -8 * want.norm()


@pytest.mark.parametrize("br", [1, 2])
def test_forward_and_backward_find_the_same_weights(br):
    """Scores that are 0 but for the rounding of their own sum (the second half of every key is the
    negated first), a threshold of 0 and p = 0 (every weight 1): which pairs have a weight is decided by
    that rounding alone.  With v = 1 and dout = 1 a row of the output counts its weights and a row of
    dv its column's (at most 64 of one sign: exact in bf16)."""
    n = 64
    q, k = _rows(n, 53, 2, h=4)
    q[..., D // 2:] = q[..., :D // 2]
    k[..., D // 2:] = -k[..., :D // 2]
    one = torch.ones_like(q)
    if br == 1:
        leaves = [x.cuda().requires_grad_(True) for x in (q, k, one)]
        out = tda_amd.threshold_rela_triton(*leaves, 0.0, relu_power=0.0, normalize=False)
        dv = torch.autograd.grad(out, leaves, one.cuda())[2]
    else:  # the second branch has no weight at all (its scores are negative)
        out, grads = _step([q, -one, k, one, one], one, 0.0, 0.5, 0.0, False)
        dv = grads[4]
    rows, cols = out[..., 0].double().sum(-1), dv[..., 0].double().sum(-1)
    assert rows.sum() > 0  # some of the sums do round to a positive value
    assert torch.equal(rows, cols)
