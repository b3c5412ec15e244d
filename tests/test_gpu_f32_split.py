"""fp32 without normalisation: the split passes, one resident tile per workgroup, its streamed tiles
dealt to four, two or one waves (f32_split in tda_common.hpp: below 2048 resident tiles four; from
there two, and one for rows of at most 16 tiles or from 4096 tiles at d = 128), against the formula in
64 bits.  Sizes on both sides of each line, fewer streamed tiles than waves, ragged last tiles, a key
cache longer than the queries, and rows past one bitmask round (2048 key tiles).  1e-4 normwise: fp32
products and sums of at most 65600 terms of random signs (2^-24 sqrt(65600) = 1.5e-5), the power's
factor two, and the cancellation in score - tau."""
import pytest
import torch

import tda_amd
from oracle.formula import rel_err, tda_grads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,h,nq,nk,d,br,p", [
    (1, 2, 33, 33, 64, 1, 2.0),      # two tiles: two of the four waves idle
    (1, 3, 161, 161, 128, 2, 1.5),   # six tiles, ragged
    (2, 2, 40, 700, 64, 2, 2.0),     # two query tiles on a longer key cache
    (16, 32, 128, 128, 64, 1, 2.0),  # 2048 tiles, short rows: one wave
    (8, 15, 545, 545, 64, 1, 2.0),   # 2160 tiles of 18: two waves
    (8, 31, 545, 545, 128, 1, 2.0),  # 4464 tiles of 18 at d = 128: one wave
])
def test_against_the_formula(b, h, nq, nk, d, br, p):
    g = torch.Generator("cuda").manual_seed(nq + d)
    rows = [torch.randn((b, h, n, d), generator=g, device="cuda") for n in (nq, nq, nk, nk, nk, nq)]
    heads = sorted({0, b * h - 1})  # the heads that the formula checks
    q1, q2, k1, k2, v = (x.requires_grad_(True) for x in rows[:5])
    if br == 2:
        out = tda_amd.differential_threshold_rela_triton(q1, q2, k1, k2, v, 1.0, 0.4, relu_power=p, normalize=False)
        leaves = [q1, q2, k1, k2, v]
    else:
        out = tda_amd.threshold_rela_triton(q1, k1, v, 1.0, relu_power=p, normalize=False)
        leaves = [q1, k1, v]
    grads = torch.autograd.grad(out, leaves, rows[5])
    names = ["dq1", "dq2", "dk1", "dk2", "dv"] if br == 2 else ["dq1", "dk1", "dv"]
    for bh in heads:
        i, j = divmod(bh, h)
        one = [x.detach()[i:i + 1, j:j + 1].double().cpu() for x in rows]
        ref = tda_grads(*one, 1.0, 0.4, p, False, br, q_offset=nk - nq)
        assert rel_err(out[i:i + 1, j:j + 1], ref["out"]) < 1e-4
        for name, x in zip(names, grads):
            assert rel_err(x[i:i + 1, j:j + 1], ref[name]) < 1e-4, name


def test_rows_longer_than_a_bitmask_round():
    """65600 keys: 2050 key tiles, 65 bitmask words; the forward collects 64 words at a time."""
    g = torch.Generator("cuda").manual_seed(3)
    q, k, v = (torch.randn((1, 1, n, 64), generator=g, device="cuda") for n in (40, 65600, 65600))
    out = tda_amd.threshold_rela_triton(q, k, v, 1.0, relu_power=2.0, normalize=False)
    qd, kd, vd = (x[0, 0].double().cpu() for x in (q, k, v))
    pos = torch.arange(65560, 65600, dtype=torch.float64)
    x = qd @ kd.T - torch.sqrt(2.0 * torch.log(pos + 1.0) / 64).unsqueeze(1)
    x = torch.where((torch.arange(65600).unsqueeze(0) <= pos.unsqueeze(1)), x.clamp(min=0.0), torch.zeros_like(x))
    assert rel_err(out[0, 0], (x * x) @ vd) < 1e-4
