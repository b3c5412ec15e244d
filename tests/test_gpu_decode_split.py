"""Decode (one query tile) in both chunk sizes of the split-key kernels, bf16 and fp32: key counts at
the edges of a tile, of a chunk of 8 and of a bitmask word, one head (small chunks) and many (whole
words), against the fp64 oracle; the bitmask bytes past the last chunk are cleared.  In fp32 short
caches and many heads run a wave per head (one_wave_heads in tda_fwd.hip): both sides of its lines."""
import pytest
import torch

import tda_amd
from oracle.formula import rel_err, tda_grads
from tda_amd import ops

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-4, torch.bfloat16: 2e-2}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("b,h,nq,nk,d,br,norm,p", [
    (1, 1, 1, 1, 64, 2, True, 2.0), (1, 3, 1, 33, 64, 1, True, 2.0), (1, 2, 5, 255, 128, 2, True, 1.5),
    (1, 2, 1, 257, 64, 2, False, 2.0), (2, 2, 32, 1025, 64, 2, True, 2.0), (1, 8, 1, 1000, 64, 2, True, 2.0),
    (16, 32, 1, 97, 64, 1, True, 2.0),   # 512 heads: whole bitmask words
    (1, 2, 32, 64, 64, 2, True, 2.0), (1, 2, 1, 65, 128, 1, False, 2.0),            # two key tiles, three
    (8, 64, 32, 128, 128, 2, False, 2.0), (8, 64, 1, 129, 128, 1, True, 2.0),       # 512 heads: four, five
    (16, 64, 5, 255, 128, 1, True, 1.5), (16, 64, 1, 257, 64, 2, True, 2.0),        # 1024 heads: eight, nine
    (32, 64, 1, 300, 64, 2, True, 2.0), (32, 64, 7, 1100, 64, 1, False, 2.0),       # 2048: any
])
def test_decode_against_the_oracle(dtype, b, h, nq, nk, d, br, norm, p):
    g = torch.Generator("cpu").manual_seed(41)
    mk = lambda n: torch.randn((b, h, n, d), generator=g).to(dtype)  # noqa: E731
    rows, do = [mk(nq) for _ in range(br)] + [mk(nk) for _ in range(br + 1)], mk(nq)
    leaves = [x.cuda().requires_grad_(True) for x in rows]
    beta, lam = (0.4 if norm else 1.0), 0.4
    bt, lt = (torch.tensor(x, device="cuda", requires_grad=True) for x in (beta, lam))
    if br == 2:
        out = tda_amd.differential_threshold_rela_triton(*leaves, bt, lt, relu_power=p, normalize=norm)
        q1, q2, k1, k2, v = (x.double() for x in rows)
    else:
        out = tda_amd.threshold_rela_triton(*leaves, bt, relu_power=p, normalize=norm)
        (q1, k1, v), q2, k2 = (x.double() for x in rows), None, None
    out.backward(do.cuda())
    ref = tda_grads(q1, q2, k1, k2, v, do.double(), beta, lam if br == 2 else 0.0, p, norm, br, q_offset=nk - nq)
    assert rel_err(out, ref["out"]) <= TOL[dtype]
    for leaf, name in zip(leaves, ["dq1", "dq2", "dk1", "dk2", "dv"] if br == 2 else ["dq1", "dk1", "dv"]):
        assert rel_err(leaf.grad, ref[name]) <= TOL[dtype], name


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_bitmask_words_are_written_whole(dtype):
    g = torch.Generator("cpu").manual_seed(42)
    q = torch.randn((1, 2, 1, 64), generator=g).to(dtype).cuda()
    k, v = (torch.randn((1, 2, 300, 64), generator=g).to(dtype).abs().cuda() for _ in range(2))
    _, occ = ops.side_buffers(q.shape, 1, True, "cuda", 300)
    occ.fill_(-1)
    with torch.no_grad():
        ops.forward(q.abs(), k, None, None, v, torch.tensor(0.0, device="cuda"), None, 2.0, True, 1, None, occ,
                    q_offset=299)
    assert occ.tolist() == [(1 << 10) - 1] * 2  # ten key tiles, every one with a weight, nothing past them


def test_a_wave_per_head_writes_every_key_norm_and_the_counters():
    """fp32, 2048 heads, keys past the query's position: their norms are written too, the bitmask and the
    counters are the causal tiles'."""
    g = torch.Generator("cpu").manual_seed(43)
    q = torch.randn((32, 64, 3, 64), generator=g).cuda()
    k, v = (torch.randn((32, 64, 150, 64), generator=g).cuda() for _ in range(2))
    norms, occ = ops.side_buffers(q.shape, 1, True, "cuda", 150)
    norms.fill_(-1.0)
    occ.fill_(-1)
    stats = torch.zeros(3, dtype=torch.int64, device="cuda")
    with torch.no_grad():
        ops.forward(q, k, None, None, v, torch.tensor(0.0, device="cuda"), None, 2.0, True, 1, norms, occ, stats, q_offset=40)
    want = torch.cat([1.0 / x.norm(dim=-1).reshape(-1) for x in (q, k)])
    torch.testing.assert_close(norms[:want.numel()], want, rtol=1e-5, atol=0)
    assert occ.numel() == 2048 and set(occ.tolist()) <= {0b01, 0b10, 0b11}  # (two of five key tiles are seen, a third by the rows past Nq)
    assert stats[0] == 2048 * 3 and stats[1] == sum(bin(w).count("1") for w in occ.tolist()) and stats[2] == 0
