"""The wide forward (top_k > 64, or more than 64 tiles per level, or KV-head
quads) at the edges of its forms, against the oracle: levels that pass every
candidate down (at most top_k of them) and the first queries past that, a top
level that is also the bottom one, three levels, batches of four tiles cut
short (the bottom level's slots past the list), several tiles per slot and
several slots per tile, padding heads.  The bars are those of the other
forward tests (selection with its tie band, output and softmax state by dtype)."""
import pytest
import torch

import htree_amd
from tests.gpu_util import check_forward, inputs

pytestmark = pytest.mark.gpu

SHAPES = [
    # B, T, H, Hkv, D, dtype, CR, TK, MTN
    (1, 2090, 16, 1, 32, "float32", 16, 128, 2048),    # selects from query 2048 on
    (1, 2064, 8, 2, 64, "bfloat16", 16, 128, 2048),
    (1, 75, 6, 1, 32, "float16", 16, 128, 2048),       # one level, 1..75 candidates
    (2, 1100, 16, 1, 32, "bfloat16", 4, 128, 64),      # four levels, slots of 4
    (1, 1500, 12, 2, 128, "float32", 8, 128, 128),     # three levels, half tiles
    (1, 1300, 5, 1, 32, "float32", 64, 64, 16),        # four tiles per slot
    (1, 1601, 34, 1, 64, "float32", 16, 128, 1024),    # quads with padding heads
    (1, 700, 24, 1, 32, "bfloat16", 32, 128, 16),      # a pair, two tiles per slot
]


@pytest.mark.parametrize("B,T,H,Hkv,D,dtype,CR,TK,MTN", SHAPES)
def test_wide_forms_against_oracle(B, T, H, Hkv, D, dtype, CR, TK, MTN):
    q, k, v = inputs(B, T, H, Hkv, D, dtype, 7)[:3]
    dev = torch.device("cuda:0")
    out, par, gmax, gsum, _ = htree_amd.htree_forward_parents(q.to(dev), k.to(dev), v.to(dev), CR,
                                                              MTN, TK)
    torch.cuda.synchronize()
    check_forward(q, k, v, CR, TK, MTN, dtype, out_dev=out.float().cpu().numpy(),
                  parents_dev=par.cpu().numpy(), gmax_dev=gmax.cpu().numpy(), gsum_dev=gsum.cpu().numpy())
