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
