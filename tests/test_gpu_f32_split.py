"""fp32 without normalisation: the split passes, one resident tile per workgroup, its streamed tiles
dealt to four, two or one waves, and the block passes, four resident tiles per workgroup (f32_split in
tda_common.hpp: by the resident tiles against the 1024 or 2048 waves the GPU holds, and the streamed tiles), against the formula in
64 bits, every head and the gradients of beta and lambda.  Sizes on both sides of each line, fewer streamed tiles than waves, ragged last tiles, a key
cache longer than the queries, and rows past one bitmask round (2048 key tiles).  1e-4 normwise: fp32
products and sums of at most 65600 terms of random signs (2^-24 sqrt(65600) = 1.5e-5), the power's
factor two, and the cancellation in score - tau; the scalars 1e-6 of the sum of their rows' contributions
(sums of both signs, over the tiles in fp64).
Powers above 1: the derivative of p = 1 steps at the threshold, where a score within rounding of it moves a
whole term."""
import pytest
import torch

import tda_amd
from oracle.formula import rel_err
from tests.helpers import grads_on_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,h,nq,nk,d,br,p", [
    (1, 2, 33, 33, 64, 1, 2.0),      # two tiles: two of the four waves idle
    (1, 3, 161, 161, 128, 2, 1.5),   # six tiles, ragged
    (2, 2, 40, 700, 64, 2, 2.0),     # two query tiles on a longer key cache
    (16, 32, 128, 128, 64, 1, 2.0),  # 2048 tiles: two waves
    (8, 15, 545, 545, 64, 1, 2.0),   # 2160 tiles of 18: one wave
    (8, 31, 545, 545, 128, 1, 2.0),  # 4464 tiles of 18 at d = 128: blocks of four, the last of two
    (16, 32, 128, 128, 64, 2, 2.0),  # two branches, one wave
    (8, 15, 545, 545, 64, 2, 2.0),   # two branches, one wave
    (8, 15, 545, 545, 128, 1, 1.5),  # d = 128: one wave
    (8, 15, 545, 545, 128, 2, 2.0),  # d = 128: one wave, blocks in the query-major pass (4320 tiles)
    (4, 10, 545, 545, 64, 2, 2.0),   # 720 tiles of 18: two waves
    (4, 10, 545, 545, 128, 1, 1.5),  # d = 128: two waves
    (4, 10, 545, 545, 128, 2, 2.0),  # two waves, one in the query-major pass (1440 tiles)
    (8, 41, 545, 545, 64, 1, 2.0),   # 5904 tiles of 18: blocks
    (8, 21, 449, 545, 64, 2, 1.5),   # two branches, queries past the first keys: blocks, one wave in the query-major pass
    (8, 21, 545, 545, 64, 2, 2.0),   # two branches: blocks everywhere
    (8, 21, 500, 640, 128, 2, 2.0),  # d = 128: blocks
])
def test_against_the_formula(b, h, nq, nk, d, br, p):
    g = torch.Generator("cuda").manual_seed(nq + d)
    rows = [torch.randn((b, h, n, d), generator=g, device="cuda") for n in (nq, nq, nk, nk, nk, nq)]
    q1, q2, k1, k2, v, do = rows
    leaves = [x.requires_grad_(True) for x in ([q1, q2, k1, k2, v] if br == 2 else [q1, k1, v])]
    bt, lt = (torch.tensor(x, device="cuda", requires_grad=True) for x in (1.0, 0.4))
    if br == 2:
        out = tda_amd.differential_threshold_rela_triton(*leaves, bt, lt, relu_power=p, normalize=False)
    else:
        out = tda_amd.threshold_rela_triton(*leaves, bt, relu_power=p, normalize=False)
    out.backward(do)
    ref = grads_on_gpu(leaves, do, 1.0, 0.4, p, False, br, q_offset=nk - nq)
    assert rel_err(out, ref["out"]) < 1e-4
    for x, name in zip(leaves, ["dq1", "dq2", "dk1", "dk2", "dv"] if br == 2 else ["dq1", "dk1", "dv"]):
        assert rel_err(x.grad, ref[name]) < 1e-4, name
    assert abs(bt.grad.item() - ref["dbeta"]) <= 1e-6 * ref["beta_scale"]
    if br == 2:
        assert abs(lt.grad.item() - ref["dlambda"]) <= 1e-6 * ref["lambda_scale"]


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
