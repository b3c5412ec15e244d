"""Non-finite values of v where no weight meets them, in the normalised bf16 tile passes (lists that
overflow): a tile whose weights are all zero adds nothing to the output, and a pair without a weight
adds nothing to a gradient, whatever v holds there."""
import pytest
import torch

import tda_amd
from oracle.formula import rel_err, tda_grads

pytestmark = pytest.mark.gpu
TOL = 2e-2  # bf16 weights, results and gradients (2^-9 each)
NAMES = {1: ["dq1", "dk1", "dv"], 2: ["dq1", "dq2", "dk1", "dk2", "dv"]}


def _call(rows, beta, lam, p, br):
    if br == 2:
        return tda_amd.differential_threshold_rela_triton(*rows, beta, lam, relu_power=p, normalize=True)
    return tda_amd.threshold_rela_triton(*rows, beta, relu_power=p, normalize=True)


def _oracle_rows(rows, br):
    rows = [x.double().cpu() for x in rows]
    return rows if br == 2 else [rows[0], None, rows[1], None, rows[2]]


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("d,br,p", [(64, 1, 2.0), (64, 2, 2.0), (128, 2, 2.0), (128, 1, 1.5), (256, 2, 2.0)])
def test_value_rows_without_a_weight(d, br, p, bad):
    """One key points away from every query (no weight in its column); its value row is not finite.
    Every gradient is what a finite row there gives."""
    n, j = 260, 70
    g = torch.Generator("cpu").manual_seed(61)
    mk = lambda: torch.randn((1, 2, n, d), generator=g)  # noqa: E731
    qs, ks = [mk() for _ in range(br)], [mk() for _ in range(br)]
    for q, k in zip(qs, ks):
        q[..., 0] = 3.0 + q[..., 0].abs()
        k[..., j, :] = 0.0
        k[..., j, 0] = -4.0
    rows = [x.bfloat16() for x in (*qs, *ks, mk())]
    do = mk().bfloat16()
    finite = [x.clone() for x in rows]
    finite[-1][..., j, :] = 0.0
    ref = tda_grads(*_oracle_rows(finite, br), do.double(), 0.4, 0.5, p, True, br)
    assert ref["dbeta"].abs() > 0
    rows[-1][..., j, :] = bad
    leaves = [x.cuda().requires_grad_(True) for x in rows]
    bt, lt = (torch.tensor(x, device="cuda", requires_grad=True) for x in (0.4, 0.5))
    out = _call(leaves, bt, lt, p, br)
    out.backward(do.cuda())
    for leaf, name in zip(leaves, NAMES[br]):
        assert torch.isfinite(leaf.grad).all(), name
        assert rel_err(leaf.grad, ref[name]) <= TOL, name
    assert abs(bt.grad.item() - ref["dbeta"].item()) <= 1e-3 * abs(ref["dbeta"].item()) + 1e-5
    if br == 2:
        assert abs(lt.grad.item() - ref["dlambda"].item()) <= 1e-3 * abs(ref["dlambda"].item()) + 1e-5


@pytest.mark.parametrize("d,br", [(64, 1), (64, 2), (128, 1), (128, 2), (256, 2)])
def test_kept_tiles_without_a_weight(d, br):
    """A key tile whose cosines lie just below the queries' thresholds, closer than the int8 screen
    can tell: it is walked, holds no weight, and its value rows (infinite) reach no output.  The other
    keys have weights with every query, so no list fits."""
    n, t0 = 256, 96  # the tile of keys 96 .. 127
    g = torch.Generator("cpu").manual_seed(62)
    off = 1000
    tau = torch.sqrt(2.0 * torch.log(torch.arange(off, off + n) + 1.0) / d)
    qs, ks = [], []
    for _ in range(br):
        # q = (tau - 0.004 along e0, 0.7 along e1, the rest of a unit vector spread over e2 ..)
        noise = torch.randn((1, 1, n, d), generator=g)
        noise[..., :2] = 0.0
        a = 0.9 * tau - 0.004
        rest = torch.sqrt(1.0 - a * a - 0.49)
        q = noise / noise.norm(dim=-1, keepdim=True) * rest.view(1, 1, n, 1)
        q[..., 0], q[..., 1] = a, 0.7
        k = 0.02 * torch.randn((1, 1, off + n, d), generator=g)
        k[..., 1] += 1.0
        k[..., t0:t0 + 32, :] = 0.0
        k[..., t0:t0 + 32, 0] = 1.0
        qs.append(q)
        ks.append(k)
    v = torch.randn((1, 1, off + n, d), generator=g)
    rows = [x.bfloat16() for x in (*qs, *ks, v)]
    finite = [x.clone() for x in rows]
    finite[-1][..., t0:t0 + 32, :] = 0.0
    do = torch.zeros_like(qs[0])
    ref = tda_grads(*_oracle_rows(finite, br), do.double(), 0.9, 0.5, 2.0, True, br, q_offset=off)["out"]
    big = [x.clone() for x in finite]  # what the tile adds with finite rows: no weight in the formula either
    big[-1][..., t0:t0 + 32, :] = 1e30
    assert torch.equal(ref, tda_grads(*_oracle_rows(big, br), do.double(), 0.9, 0.5, 2.0, True, br, q_offset=off)["out"])
    rows[-1][..., t0:t0 + 32, :] = float("inf")
    with torch.no_grad():
        out = _call([x.cuda() for x in rows], 0.9, 0.5, 2.0, br)
    assert torch.isfinite(out).all()
    assert rel_err(out, ref) <= TOL


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("normalize", [False, True])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_nan_scores_have_no_weight(d, normalize, bad):
    """A query row and a key row all of whose scores are NaN (Inf - Inf too): the query's output row is
    zero, and no other row has anything from them."""
    n, iq, jk = 140, 40, 90  # (the key after the query: their own score is infinite)
    g = torch.Generator("cpu").manual_seed(64)
    rows = [torch.randn((1, 1, n, d), generator=g) for _ in range(6)]
    for x in rows[:4]:
        x[..., :2] = x[..., :2].abs() + 0.5
    q1, q2, k1, k2, v, do = (x.bfloat16() for x in rows)
    beta = 0.4 if normalize else 0.4 * d ** 0.5
    clean = [x.clone() for x in (q1, q2, k1, k2, v)]
    for x, r in ((q1, iq), (q2, iq), (k1, jk), (k2, jk)):
        x[..., r, 0], x[..., r, 1] = bad, -bad
    # the same without them: rows of zeros, whose scores are below every threshold
    for x, r in zip(clean, (iq, iq, jk, jk)):
        x[..., r, :] = 0.0
    ref = tda_grads(*(x.double() for x in clean), do.double(), beta, 0.4, 2.0, normalize, 2)
    leaves = [x.cuda().requires_grad_(True) for x in (q1, q2, k1, k2, v)]
    out = tda_amd.differential_threshold_rela_triton(*leaves, beta, 0.4, normalize=normalize)
    dv = torch.autograd.grad(out, leaves, do.cuda())[4]
    assert not out[..., iq, :].any()
    assert rel_err(out, ref["out"]) <= TOL
    assert rel_err(dv, ref["dv"]) <= TOL
