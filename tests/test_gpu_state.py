"""The state the forward hands to the backward (gmax, gsum) and to the trace is
in units of the scores themselves: the backward rebuilds P = exp(S - gmax) /
gsum from scores formed with the same rounded operands, so a max that went
through another unit (log2) would be off by its roundings.

A query at t = 0 sees one candidate at angle 0.  With q and k small integers
and a scale of 1/8 its score is exact in the split product and in fp32, so
gmax there is that score bit for bit, gsum is 1, and the bottom level's
traced max is the score too."""
import pytest
import torch

import htree_amd

pytestmark = pytest.mark.gpu

DEV = "cuda:0"

FORMS = [
    # B, T, H, Hkv, D, CR, TK, MTN
    (2, 300, 16, 2, 64, 16, 16, 128),    # register form
    (2, 300, 16, 2, 64, 32, 32, 256),    # streaming form, two levels
    (1, 300, 5, 1, 64, 32, 32, 1024),    # streaming form, one level
    (1, 300, 17, 1, 64, 16, 16, 128),    # streaming form, a KV-head pair with a padding head
    # (wide form, two levels: D = 128 takes the query of every slot from the
    # table; D <= 64 turns a batch's query on, which is not exact)
    (2, 300, 16, 2, 128, 16, 128, 64),
    (1, 300, 16, 1, 64, 16, 128, 2048),  # wide form, one level
    (1, 300, 34, 1, 64, 16, 32, 512),    # wide form, a quad with padding heads
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,H,Hkv,D,CR,TK,MTN", FORMS)
def test_max_is_a_score(B, T, H, Hkv, D, CR, TK, MTN, dtype):
    g = torch.Generator().manual_seed(3)
    q = torch.randint(-8, 9, (B, T, H, D), generator=g).to(dtype)
    k = torch.randint(-8, 9, (B, T, Hkv, D), generator=g).to(dtype)
    v = torch.randn(B, T, Hkv, D, generator=g).to(torch.bfloat16).to(dtype)
    want = (q[:, 0].double() * k[:, 0].double().repeat_interleave(H // Hkv, 1)).sum(-1) / 8
    out, _, gmax, gsum, _ = htree_amd.htree_forward_parents(q.to(DEV), k.to(DEV), v.to(DEV), CR, MTN, TK,
                                                            1 / 8)
    torch.cuda.synchronize()
    assert torch.equal(gmax[:, 0].cpu().double(), want)
    assert torch.equal(gsum[:, 0].cpu().double(), torch.ones_like(want))
    assert torch.equal(out[:, 0].cpu(), v[:, 0].repeat_interleave(H // Hkv, 1))
    _, tr = htree_amd.run_parallel_with_trace(q.to(DEV), k.to(DEV), v.to(DEV), CR, MTN, TK, 1 / 8,
                                              10000.0)
    torch.cuda.synchronize()
    assert torch.equal(tr["layers"][0].layer_max[:, 0].cpu().double(), want)


CONSISTENT = [
    # T, H, Hkv, D, CR, TK, MTN, dtype
    (8000, 4, 1, 32, 16, 512, 8192, torch.float32),   # wide form, one level
    (9001, 8, 1, 32, 16, 512, 8192, torch.float32),   # two levels
    (8000, 4, 1, 32, 16, 512, 8192, torch.bfloat16),  # two entries per dkv tile
    (8000, 4, 1, 128, 16, 512, 8192, torch.float32),
    (3000, 16, 1, 32, 64, 64, 4096, torch.float32),   # top_k 64 in four tiles each
    (3000, 8, 1, 64, 4, 512, 2048, torch.bfloat16),   # slots of four
    (4000, 34, 1, 32, 16, 16, 256, torch.float32),    # a quad, the merged top level
    (2000, 50, 1, 64, 16, 16, 128, torch.bfloat16),   # a quad, stored dS
    (8000, 8, 1, 64, 32, 32, 256, torch.float32),     # streaming form
    (4000, 8, 1, 64, 16, 16, 256, torch.float32),     # register form
]


@pytest.mark.parametrize("T,H,Hkv,D,CR,TK,MTN,dtype", CONSISTENT)
def test_probabilities_of_the_backward_sum_to_one(T, H, Hkv, D, CR, TK, MTN, dtype):
    """dO = e_i at D chosen queries (one head and one element i each) makes the
    sum of dv[..., i] over all tokens that query's sum of P as the backward
    rebuilds it.  Its scores and the forward's differ in the residuals of the
    queries' and keys' bf16 splits (at most 2^-17 of an element each, and
    2^-18 / sqrt(3) of it on average): with |q| of 2 sqrt(D), |k| of sqrt(D) and the
    scale 1 / sqrt(D) about 2^-17 = 7.6e-6 a score.  The bar is three times
    that.  (K~ at other angles in the two passes: 6e-5 in the first case.)"""
    g = torch.Generator().manual_seed(5)
    q = (2 * torch.randn(1, T, H, D, generator=g)).to(dtype).to(DEV)
    k = torch.randn(1, T, Hkv, D, generator=g).to(dtype).to(DEV)
    v = torch.randn(1, T, Hkv, D, generator=g).to(dtype).to(DEV)
    dO = torch.zeros_like(q)
    i = torch.arange(D)
    dO[0, torch.linspace(T // 2, T - 1, D).long(), i % H, i] = 1
    out, ctx = htree_amd.htree_forward(q, k, v, CR, MTN, TK, _save_for_backward=True)
    dv = htree_amd.htree_backward(dO, q, out, ctx)[2]
    torch.cuda.synchronize()
    off = (dv.double().sum((0, 1, 2)) - 1).abs().max().item()
    print(off, flush=True)
    assert off <= 2.3e-5


@pytest.mark.parametrize("H,D,TK,MTN", [(8, 32, 128, 2048), (16, 64, 128, 128), (64, 64, 16, 128)])
def test_wide_probabilities_beyond_bf16(H, D, TK, MTN):
    """The wide form at D <= 64 multiplies V by P in bf16 hi + lo for bf16 inputs
    too: with V = 1 a level's output is its sum of P.  The split leaves 2^-18
    of a P, the fp32 sums of up to 1500 terms a few 2^-24 each; P rounded to
    bf16 (2^-9) is off by 1e-3 where few candidates matter."""
    g = torch.Generator().manual_seed(9)
    q = torch.randn(1, 1500, H, D, generator=g).to(torch.bfloat16).to(DEV)
    k = torch.randn(1, 1500, 1, D, generator=g).to(torch.bfloat16).to(DEV)
    _, tr = htree_amd.run_parallel_with_trace(q, k, torch.ones_like(k), 16, MTN, TK, None, 10000.0)
    torch.cuda.synchronize()
    for lt in tr["layers"].values():
        some = lt.layer_sum > 0
        ratio = lt.layer_output[some].double() / lt.layer_sum[some].double()[:, None]
        assert (ratio - 1).abs().max().item() <= 2 ** -15 if some.any() else True
