"""bf16 training steps over many heads of one or two tiles: the block passes that take fewer tiles per
workgroup there (bwd_tiles with a queue longer than its grid, bwd_dq_blk, bwd_dkv_blk, the head_dim 256
forward), against the formula in 64 bits, every head.  2e-2: bf16 rows, weights and gradients, as in
the parity tests."""
import pytest
import torch

import tda_amd
from oracle.formula import rel_err
from tests.helpers import TOL, grads_on_gpu, rel_norm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,h,nq,nk,d,br,norm,p,beta", [
    (16, 64, 32, 32, 64, 2, True, 2.0, 0.3),    # one tile: up to 3072 queued blocks, 1792 workgroups
    (16, 64, 17, 17, 64, 1, True, 1.5, 0.3),
    (8, 64, 31, 31, 128, 2, True, 2.0, 0.3),    # 768 workgroups
    (8, 64, 32, 32, 128, 1, True, 1.5, 0.3),
    (16, 64, 33, 33, 64, 2, True, 2.0, 0.3),    # two tiles: 1024 workgroups
    (8, 64, 64, 64, 128, 2, True, 1.5, 0.3),    # 512
    (8, 64, 20, 50, 64, 2, True, 2.0, 0.3),     # one query tile, two key tiles
    (8, 64, 65, 65, 64, 2, True, 2.0, 0.3),     # three: blocks of four
    (4, 64, 32, 32, 64, 2, False, 2.0, 0.5), (4, 64, 9, 9, 128, 1, False, 1.5, 0.5),
    (4, 64, 32, 70, 64, 1, False, 2.0, 0.5),    # one query tile, three key tiles
    (4, 64, 32, 70, 128, 2, False, 2.0, 0.5),
    (4, 32, 32, 32, 256, 2, True, 2.0, 0.3), (4, 32, 1, 1, 256, 2, False, 2.0, 0.0),
    (4, 32, 17, 17, 256, 1, True, 1.5, 0.3), (4, 32, 31, 31, 256, 1, False, 2.0, 0.3),
    (4, 32, 20, 33, 256, 1, False, 2.0, 0.3),   # one query tile, two key tiles
])
def test_against_the_formula(b, h, nq, nk, d, br, norm, p, beta):
    g = torch.Generator("cpu").manual_seed(61)
    rows = [torch.randn((b, h, n, d), generator=g).bfloat16().cuda() for n in ([nq, nq, nk, nk, nk] if br == 2 else [nq, nk, nk])]
    do = torch.randn((b, h, nq, d), generator=g).bfloat16().cuda()
    leaves = [x.requires_grad_(True) for x in rows]
    bt, lt = (torch.tensor(x, device="cuda", requires_grad=True) for x in (beta, 0.4))
    if br == 2:
        out = tda_amd.differential_threshold_rela_triton(*leaves, bt, lt, relu_power=p, normalize=norm)
    else:
        out = tda_amd.threshold_rela_triton(*leaves, bt, relu_power=p, normalize=norm)
    out.backward(do)
    ref = grads_on_gpu(leaves, do, beta, 0.4, p, norm, br, q_offset=nk - nq)
    tol = TOL[torch.bfloat16]
    assert rel_err(out, ref["out"]) < tol and rel_norm(out, ref["out"]) < tol
    for x, name in zip(leaves, ["dq1", "dq2", "dk1", "dk2", "dv"] if br == 2 else ["dq1", "dk1", "dv"]):
        assert rel_err(x.grad, ref[name]) < tol and rel_norm(x.grad, ref[name]) < tol, name
    assert abs(bt.grad.item() - ref["dbeta"]) <= tol * ref["beta_scale"]
    if br == 2:
        assert abs(lt.grad.item() - ref["dlambda"]) <= tol * ref["lambda_scale"]


def test_more_work_items_than_one_grid_dimension_holds():
    """head_dim 256, 2^23 + 3 heads of one row: the query-major pass has 512 work-items per head, past
    2^32 - 1.  The first heads and the last against the formula at N = 1 (the threshold is 0 there): out =
    relu(q.k)^2 v, dq = 2 relu(q.k) (dout.v) k, in fp64; 2^-7 in the 2-norm: bf16 products' operands (dS) and
    results, 2^-9 each."""
    n = 2 ** 23 + 3
    g = torch.Generator("cuda").manual_seed(67)
    q, k, v, do = (torch.randn((1, n, 1, 256), generator=g, device="cuda", dtype=torch.bfloat16) for _ in range(4))
    q.requires_grad_(True), k.requires_grad_(True), v.requires_grad_(True)
    out = tda_amd.threshold_rela_triton(q, k, v, 1.0, relu_power=2.0, normalize=False)
    dq, dk, dv = torch.autograd.grad(out, [q, k, v], do)
    for at in (slice(0, 64), slice(n - 64, n)):
        qd, kd, vd, dd = (x.detach()[0, at, 0].double() for x in (q, k, v, do))
        x = (qd * kd).sum(-1, keepdim=True).clamp(min=0)
        dp = (dd * vd).sum(-1, keepdim=True)
        for got, want in ((out, x * x * vd), (dq, 2 * x * dp * kd), (dk, 2 * x * dp * qd), (dv, x * x * dd)):
            assert rel_norm(got[0, at, 0], want) < 2.0 ** -7
