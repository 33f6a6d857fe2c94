"""The work that a user of htree_amd has it do, as measured cases.

A pass is one call of the public entry points: the forward of an inference
call (`htree_forward`) or a training step of the attention layer
(`htree_forward_triton_autograd` and `out.backward(dO)`, the gradients of
q, k and v cleared first).  Shapes are those of bench.py's workloads, of the
tests and of the reference's timing scripts; `draw` gives others of the same
ranges, ragged lengths among them.
"""
import math

import numpy as np
import torch

import htree_amd

MODES = {
    # what the autograd forward keeps for its backward
    "default": {},
    "scores": {"_save_scores": True},
    "lean": {"_save_parents": False},
}


def _case(name, step, B, T, H, Hkv, D, dtype, CR, TK, MTN, mode="default", data="iid"):
    return dict(name=name, step=step, B=B, T=T, H=H, Hkv=Hkv, D=D, dtype=dtype, CR=CR, TK=TK,
                MTN=MTN, mode=mode, data=data)


def listed():
    return [
        # a short prompt through one layer: latency and launches
        _case("infer_1k", "infer", 1, 1024, 8, 1, 128, "bfloat16", 16, 8, 64),
        # the small fp32 configuration that is also run on the CPU
        _case("infer_2k_fp32", "infer", 1, 2048, 4, 1, 64, "float32", 16, 8, 64),
        # a short ragged fp16 training batch that keeps only the reference's
        # eight tensors between forward and backward
        _case("train_777_fp16_lean", "train", 2, 777, 8, 2, 64, "float16", 16, 8, 64, "lean"),
        # the headline: a 32k sequence, prefill and training step
        _case("infer_32k", "infer", 1, 32768, 32, 2, 128, "bfloat16", 16, 16, 128),
        _case("train_32k", "train", 1, 32768, 32, 2, 128, "bfloat16", 16, 16, 128),
        # an odd length with the candidate scores kept (the fastest backward)
        _case("train_20k_scores", "train", 1, 20011, 32, 2, 128, "bfloat16", 16, 16, 128, "scores"),
        # the batched training shape: groups of 8 heads
        _case("train_4x16k", "train", 4, 16384, 32, 4, 128, "bfloat16", 16, 16, 128),
        # clustered keys, queries around few clusters: very uneven selection
        _case("train_2x64k_skewed", "train", 2, 65536, 32, 2, 128, "bfloat16", 16, 16, 128,
              data="mixture"),
        # long-context prefill: 1024 candidates per level
        _case("infer_128k", "infer", 1, 131072, 64, 8, 128, "bfloat16", 32, 32, 256),
        # the entry points' default arguments (top_k 512 of up to 8192
        # candidates), at the sizes of the reference's timing scripts
        _case("infer_default_120k", "infer", 1, 120000, 64, 4, 32, "float32", 16, 512, 8192,
              data="slow"),
        _case("train_default_12k", "train", 1, 12000, 64, 4, 32, "float32", 16, 512, 8192),
        # the same arguments with 64 query heads over one KV head
        _case("infer_default_mqa_12k", "infer", 1, 12001, 64, 1, 64, "bfloat16", 16, 512, 8192),
    ]


def draw(rng):
    """A further case of the same ranges: short to 128k tokens, groups of 4
    to 64 heads, every dtype, both regimes of list length."""
    top = max(_cost(c) for c in listed())
    while True:
        step = rng.choice(["infer", "train"])
        if rng.random() < 0.7:  # short lists
            CR, TK, MTN = rng.choice([(16, 8, 64), (16, 16, 128), (16, 16, 128), (32, 32, 256),
                                      (16, 16, 256)])
            D = rng.choice([64, 128, 128])
            dtype = rng.choice(["bfloat16"] * 4 + ["float16", "float32"])
            G = rng.choice([4, 8, 16, 16])
            T = int(math.exp(rng.uniform(math.log(200), math.log(131072))))
            data = rng.choice(["iid", "iid", "iid", "mixture"])
        else:  # the default arguments' long lists
            CR = 16
            TK = rng.choice([128, 256, 512, 512])
            MTN = TK * CR
            D = rng.choice([32, 32, 64, 128])
            dtype = rng.choice(["float32", "float32", "bfloat16", "float16"])
            G = rng.choice([8, 16, 16, 64])
            T = int(math.exp(rng.uniform(math.log(500), math.log(120000))))
            data = "slow"
        if rng.random() < 0.5:
            T = T // 64 * 64 or 64
        Hkv = rng.choice([1, 2, 4, 8])
        B = rng.choice([1, 1, 2, 4])
        mode = rng.choice(["default", "default", "scores", "lean"]) if step == "train" else "default"
        c = _case("", step, B, T, Hkv * G, Hkv, D, dtype, CR, TK, MTN, mode, data)
        if B * T * Hkv * G * D <= 2 ** 30 and _cost(c) <= 0.7 * top:
            del c["name"]
            return c


def _levels(c):
    n = [c["T"]]
    while n[-1] > c["MTN"]:
        n.append(-(-n[-1] // c["CR"]))
    return n


def _rows(c):
    """(candidates scored, candidates accumulated) over all query groups."""
    T, CR, TK = c["T"], c["CR"], c["TK"]
    L = len(_levels(c))
    t = np.arange(T, dtype=np.int64)
    np_l = t // CR ** (L - 1) // CR + 1
    scored = acc = 0
    for l in range(L - 1, -1, -1):
        nc = (np_l - 1) * CR + t // CR ** l % CR + 1
        np_l = np.minimum(TK, nc)
        scored += int(nc.sum())
        acc += int((nc - np_l).sum() if l else nc.sum())
    groups = c["B"] * c["Hkv"]
    return scored * groups, acc * groups


def _cost(c):
    """Time of a pass, roughly: candidates times heads (a tile holds 16) and
    head dim, with the backward's five products."""
    scored, acc = _rows(c)
    G = -(-(c["H"] // c["Hkv"]) // 16) * 16
    train = c["step"] == "train"
    return (scored + acc * (9 if train else 1)) * G * c["D"] * (2 if c["dtype"] == "float32" and train else 1)


def work(case):
    """q, k, v (and dO) read once, the output (and gradients) written once;
    two products per scored / accumulated candidate, five in the backward."""
    c = case
    G, D, e = c["H"] // c["Hkv"], c["D"], 4 if c["dtype"] == "float32" else 2
    scored, acc = _rows(c)
    qb, kb = c["B"] * c["T"] * c["H"] * D * e, c["B"] * c["T"] * c["Hkv"] * D * e
    if c["step"] == "infer":
        return {"bytes": 2 * qb + 2 * kb, "flops": 2 * G * D * (scored + acc)}
    # q, dO, out, dq; k, v, dk, dv
    return {"bytes": 4 * qb + 4 * kb, "flops": 2 * G * D * (scored + acc) + 10 * G * D * acc}


def prepare(case, seed):
    """q, k, v (and dO) of one call.  "iid": N(0, 1).  "mixture": keys from a
    mixture of 64 components (means N(0, 4), sigma 0.5), queries around 4 of
    them.  "slow": N(0, 2) in the slower half of the RoPE pairs and N(0, 1/16)
    in the faster half, as heads that look far back have it: candidates are
    counted in list positions, so where one of two equal nodes is expanded
    instead of the other, the positions of all between them move by a node's
    children, which such heads hardly see (with iid queries over thousands of
    nodes one in a hundred has its edge within fp32 rounding, and its output
    then changes by 40 percent)."""
    c = case
    B, T, H, Hkv, D = c["B"], c["T"], c["H"], c["Hkv"], c["D"]
    dev, dtype = torch.device("cuda"), getattr(torch, c["dtype"])
    g = torch.Generator(device=dev).manual_seed(seed)
    rn = lambda *shape: torch.randn(*shape, generator=g, device=dev)
    if c["data"] == "mixture":
        mu = 2.0 * rn(64, D)
        hot = torch.randperm(64, generator=g, device=dev)[:4]
        k = mu[torch.randint(0, 64, (B, T, Hkv), generator=g, device=dev)] + 0.5 * rn(B, T, Hkv, D)
        q = mu[hot[torch.randint(0, 4, (B, T, H), generator=g, device=dev)]] + 0.5 * rn(B, T, H, D)
    else:
        k, q = rn(B, T, Hkv, D), rn(B, T, H, D)
        if c["data"] == "slow":
            pair = torch.arange(D, device=dev) % (D // 2)
            size = torch.where(pair < D // 4, 0.25, math.sqrt(2.0))
            k, q = k * size, q * size
    train = c["step"] == "train"
    state = dict(case=c, v=rn(B, T, Hkv, D).to(dtype), q=q.to(dtype), k=k.to(dtype))
    if train:
        state["dO"] = rn(B, T, H, D).to(dtype)
        for x in "qkv":
            state[x].requires_grad_(True)
    return state


def run(state):
    c, q, k, v = state["case"], state["q"], state["k"], state["v"]
    args = dict(compression_rate=c["CR"], max_top_nodes=c["MTN"], top_k_per_layer=c["TK"])
    if c["step"] == "infer":
        return htree_amd.htree_forward(q, k, v, **args)
    q.grad = k.grad = v.grad = None
    out = htree_amd.htree_forward_triton_autograd(q, k, v, **args, **MODES[c["mode"]])
    out.backward(state["dO"])
    return {"out": out.detach(), "dq": q.grad, "dk": k.grad, "dv": v.grad}


def tolerance(case):
    """About four times the distance from exact() (measured: bf16 up to
    0.009, its own rounding and that of the probabilities; fp16 and fp32 up
    to 0.004, the queries whose selection has a tie within the scores'
    rounding, where two correct implementations expand different nodes: a
    few rows, each off by as much as the two nodes' shares)."""
    return {"rel": {"bfloat16": 0.03, "float16": 0.016, "float32": 0.016}[case["dtype"]],
            "max": 0.99}


# The most candidate elements (groups x candidates x head dim, five times for
# a backward) that exact() takes: about 20 seconds.
EXACT_MOST = 1.5e12


def _rotate(x, cos, sin):
    h = x.shape[-1] // 2
    a, b = x[..., :h], x[..., h:]
    return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)


def exact(case, seed):
    """The same call in float64: the tree's levels as they are defined (fp32
    mean of the children, rounded to the dtype), scores and probabilities in
    float64, the selection by importances rounded to fp32 (where the
    definition's ties lie), the stable order at ties."""
    c = case
    scored, acc = _rows(c)
    if (scored + acc * (5 if c["step"] == "train" else 1)) * c["D"] > EXACT_MOST:
        return None
    s = prepare(c, seed)
    B, T, H, Hkv, D, CR, TK = (c[x] for x in ("B", "T", "H", "Hkv", "D", "CR", "TK"))
    q, k, v = (s[x].detach() for x in "qkv")
    train, G, dev, f64 = c["step"] == "train", H // Hkv, q.device, torch.float64
    sizes = _levels(c)
    L = len(sizes)

    def pool(x):
        n = -(-x.shape[1] // CR)
        y = torch.zeros(B, n * CR, Hkv, D, device=dev)
        y[:, :x.shape[1]] = x.float()
        y = y.view(B, n, CR, Hkv, D)
        a = y[:, :, 0].clone()
        for j in range(1, CR):
            a += y[:, :, j]
        cnt = torch.full((n,), float(CR), device=dev)
        cnt[-1] = x.shape[1] - (n - 1) * CR
        return (a / cnt[None, :, None, None]).to(x.dtype), cnt

    lk, lv, cnts = [k], [v], []
    for _ in sizes[1:]:
        a, cnt = pool(lk[-1])
        b, _ = pool(lv[-1])
        lk.append(a), lv.append(b), cnts.append(cnt)
    rows = max(c["MTN"] + 1024, TK * CR)
    inv = 1.0 / (10000.0 ** (torch.arange(0, D, 2, dtype=torch.float32) / D))
    ang = torch.outer(torch.arange(rows, dtype=torch.float32), inv)
    cos, sin = ang.cos().to(dev, f64), ang.sin().to(dev, f64)
    scale = D ** -0.5

    out = torch.empty(B, T, H, D, dtype=f64, device=dev)
    if train:
        dq = torch.empty(B, T, H, D, dtype=f64, device=dev)
        gk = [torch.zeros(B, Hkv, n, D, dtype=f64, device=dev) for n in sizes]
        gv = [torch.zeros(B, Hkv, n, D, dtype=f64, device=dev) for n in sizes]
    chunk = max(16, int(1.5e8 / (TK * CR * max(D, G))))
    slots = torch.arange(TK, device=dev)
    for b in range(B):
        for h in range(Hkv):
            K = [x[b, :, h].to(f64) for x in lk]
            V = [x[b, :, h].to(f64) for x in lv]
            for t0 in range(0, T, chunk):
                t = torch.arange(t0, min(T, t0 + chunk), device=dev)
                R = t.numel()
                qc = q[b, t0:t0 + R, h * G:h * G + G].to(f64)
                nvp = t // CR ** (L - 1) // CR + 1
                par = torch.where(slots[None] < nvp[:, None], slots[None], -1)
                kept = []
                for l in range(L - 1, -1, -1):
                    nc = ((par >= 0).sum(1) - 1) * CR + t // CR ** l % CR + 1
                    C = int(nc.max())
                    j = torch.arange(C, device=dev)
                    valid = j[None] < nc[:, None]
                    node = (par[:, j // CR] * CR + j % CR).clamp(0, sizes[l] - 1)
                    kr = _rotate(K[l][node], cos[j][None], sin[j][None])
                    qr = _rotate(qc, cos[nc - 1][:, None], sin[nc - 1][:, None]) * scale
                    S = torch.matmul(qr, kr.transpose(1, 2).contiguous())
                    S.masked_fill_(~valid[:, None], -math.inf)
                    keep = valid
                    if l:
                        imp = torch.exp(S - S.amax((1, 2), keepdim=True)).float().sum(1)
                        imp[~valid] = -1.0
                        imp.scatter_(1, (nc - 1)[:, None], 1e6)
                        take = min(TK, C)
                        pos = torch.sort(imp, dim=1, descending=True, stable=True)[1][:, :take]
                        chosen = torch.zeros_like(valid).scatter_(1, pos, True) & valid
                        keep = valid & ~chosen
                        big = 1 << 40
                        nxt = torch.where(chosen.gather(1, pos), node.gather(1, pos), big).sort(1)[0]
                        par = torch.full((R, TK), -1, dtype=torch.int64, device=dev)
                        par[:, :take] = torch.where(nxt < big, nxt, -1)
                    kept.append((l, node, keep, nc, S.masked_fill(~keep[:, None], -math.inf)))
                M = torch.stack([x[4].amax(2) for x in kept]).amax(0)
                P = [torch.exp(x[4] - M[:, :, None]) for x in kept]
                Z = sum(p.sum(2) for p in P)
                o = sum(torch.matmul(p, V[x[0]][x[1]]) for p, x in zip(P, kept)) / Z[:, :, None]
                out[b, t0:t0 + R, h * G:h * G + G] = o
                if not train:
                    continue
                dO = s["dO"][b, t0:t0 + R, h * G:h * G + G].to(f64)
                delta = (dO * o.to(q.dtype).to(f64)).sum(2, keepdim=True)
                dqc = torch.zeros_like(qc)
                for p, (l, node, keep, nc, _) in zip(P, kept):
                    j = torch.arange(node.shape[1], device=dev)
                    p = p / Z[:, :, None]
                    dP = torch.matmul(dO, V[l][node].transpose(1, 2).contiguous())
                    dS = p * (dP - delta)
                    pc, ps = cos[nc - 1][:, None], sin[nc - 1][:, None]
                    kr = _rotate(K[l][node], cos[j][None], sin[j][None])
                    dqc += scale * _rotate(torch.matmul(dS, kr), pc, -ps)
                    del kr, dP
                    qr = _rotate(qc, pc, ps) * scale
                    u = torch.matmul(dS.transpose(1, 2).contiguous(), qr)
                    u = _rotate(u, cos[j][None], -sin[j][None])
                    at = node[keep]
                    gk[l][b, h].index_add_(0, at, u[keep])
                    u = torch.matmul(p.transpose(1, 2).contiguous(), dO)
                    gv[l][b, h].index_add_(0, at, u[keep])
                    del u
                dq[b, t0:t0 + R, h * G:h * G + G] = dqc
    if not train:
        return out
    for g in (gk, gv):
        for l in range(L - 1, 0, -1):
            share = (g[l] / cnts[l - 1].to(f64)[:, None]).repeat_interleave(CR, 2)
            g[l - 1] += share[:, :, :sizes[l - 1]]
    return {"out": out, "dq": dq, "dk": gk[0].transpose(1, 2).contiguous(),
            "dv": gv[0].transpose(1, 2).contiguous()}
