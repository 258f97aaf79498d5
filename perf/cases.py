"""The work that a program on this framework has it do, one dict per case.

kind "ffn"    one layer's expert block on routed tokens, ops.ffn: decode
              (1 token), speculative verification and small batches, prefill
kind "route"  one layer's router, lookahead and slot lookup, ops.route
kind "stack"  a few tokens through the layers of a stack, every layer's
              router and expert block in one HIP graph (PrefillStack)
kind "token"  one token through a stack in one launch (DecodeStack)
kind "stream" tokens through a stack whose experts are read into a pool
              smaller than the model (StreamingStack, the native loop)

Sizes: the Qwen3-30B-A3B and gpt-oss-120b expert geometries, 128 experts
with Zipf(1.1) popularity, and the token counts of the benchmark workloads
(1, 8, 512) with smaller, odd and larger ones around them.
"""
import math

import numpy as np
import torch

from moe_stream_amd import geometry as G
from moe_stream_amd import ops, stack, synth
from moe_stream_amd.pool import SlotPool

GEOMS = {"qwen3": G.QWEN3_30B_A3B, "gptoss": G.GPT_OSS_120B}
ZIPF = 1.1


def listed():
    return [
        # bs=1 decode through the per-layer call: the smallest expert block
        dict(name="ffn-qwen3-1", kind="ffn", geom="qwen3", tokens=1, stored=False, f32=False),
        # a short draft verified at once, the fp32 output, experts in pool and store
        dict(name="ffn-qwen3-3", kind="ffn", geom="qwen3", tokens=3, stored=True, f32=True),
        # the benchmark's prefill
        dict(name="ffn-qwen3-512", kind="ffn", geom="qwen3", tokens=512, stored=True, f32=False),
        # a long prompt's chunk
        dict(name="ffn-qwen3-4096", kind="ffn", geom="qwen3", tokens=4096, stored=False, f32=False),
        # the other geometry (projection biases, clamped SwiGLU, 14 MB experts): decode, a small
        # batch of decoding sequences, a prompt
        dict(name="ffn-gptoss-1", kind="ffn", geom="gptoss", tokens=1, stored=False, f32=False),
        dict(name="ffn-gptoss-29", kind="ffn", geom="gptoss", tokens=29, stored=True, f32=False),
        dict(name="ffn-gptoss-700", kind="ffn", geom="gptoss", tokens=700, stored=False, f32=False),
        # the router of one decode layer, as the block calls it, and of a prompt
        dict(name="route-qwen3-1", kind="route", geom="qwen3", tokens=1, kept=False),
        dict(name="route-gptoss-1000", kind="route", geom="gptoss", tokens=1000, kept=True),
        # the benchmark's verification: 8 tokens, router and block, layer after layer
        dict(name="stack-qwen3-8", kind="stack", geom="qwen3", tokens=8, layers=12),
        # the benchmark's headline: one token through the 48 layers
        dict(name="token-qwen3-48", kind="token", geom="qwen3", layers=48),
        # the streaming pool, a third of the experts in HBM, the rest read over the host link
        dict(name="stream-qwen3-6", kind="stream", geom="qwen3", layers=6, tokens=16),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["ffn", "ffn", "ffn", "ffn", "route", "stack", "token", "stream"])
    geom = rng.choice(["qwen3", "gptoss"])
    if kind == "ffn":
        return dict(kind=kind, geom=geom, tokens=_log_int(rng, 1, 4096 if geom == "qwen3" else 1024),
                    stored=rng.random() < 0.5, f32=rng.random() < 0.25)
    if kind == "route":
        return dict(kind=kind, geom=geom, tokens=_log_int(rng, 1, 4096), kept=rng.random() < 0.5)
    if kind == "stack":
        return dict(kind=kind, geom="qwen3", tokens=rng.randint(2, 32), layers=rng.randint(3, 12))
    if kind == "token":
        return dict(kind=kind, geom=geom, layers=rng.randint(3, 48 if geom == "qwen3" else 8))
    return dict(kind=kind, geom="qwen3", layers=rng.randint(3, 6), tokens=rng.randint(4, 16))


# -- inputs -------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _records(geom, n, gen):
    """n synthetic expert records: uniform codes, |N(0, 0.02)| scales, biases
    of -8 scales, N(0, 0.02) projection biases."""
    rec = torch.zeros((n, geom.record_bytes), dtype=torch.uint8, device="cuda")
    comps = {c.name: c for c in geom.components}
    for name, c in comps.items():
        part = rec[:, c.offset:c.offset + c.nbytes]
        if name.endswith(".weight"):
            part.copy_(torch.randint(0, 256, part.shape, dtype=torch.uint8, generator=gen,
                                     device="cuda"))
        elif name.endswith(".biases"):
            s = comps[name.replace(".biases", ".scales")]
            v = rec[:, s.offset:s.offset + s.nbytes].view(torch.bfloat16)
            part.view(torch.bfloat16).copy_(v.float() * -8.0)
        else:
            v = torch.randn((n, c.nbytes // 2), generator=gen, device="cuda") * 0.02
            part.view(torch.bfloat16).copy_(v.abs() if name.endswith(".scales") else v)
    return rec


def _popularity(experts, gen):
    logp = -ZIPF * torch.log(torch.arange(1, experts + 1, device="cuda").float())
    return (logp - torch.logsumexp(logp, 0))[torch.randperm(experts, generator=gen, device="cuda")]


def _prepare_ffn(case, seed):
    geom, T = GEOMS[case["geom"]], case["tokens"]
    E, k = geom.n_experts, geom.top_k
    gen = _gen(seed)
    rec = _records(geom, E, gen)
    # half of the experts in pool slots and half read from the store, or all in slots
    n_slots = E // 2 if case["stored"] else E
    order = torch.randperm(E, generator=gen, device="cuda")
    table = -1 - torch.arange(E, device="cuda")
    table[order[:n_slots]] = torch.arange(n_slots, device="cuda")
    pool = SlotPool(geom, n_slots, "cuda", store=rec if case["stored"] else None)
    pool.fill(order[:n_slots].cpu().numpy(), np.arange(n_slots), src=rec)
    u = torch.rand((T, E), generator=gen, device="cuda").clamp_min(1e-20)
    z = _popularity(E, gen) - torch.log(-torch.log(u))
    top, ids = torch.topk(z, k, dim=1)
    scores = torch.softmax(top, dim=1).to(torch.bfloat16).float().contiguous()
    x = torch.randn((T, geom.d_model), generator=gen, device="cuda").to(torch.bfloat16)
    return dict(pool=pool, rec=rec, ids=ids, refs=table[ids].to(torch.int32).contiguous(),
                scores=scores, x=x, f32=case["f32"], geom=geom)


def _prepare_route(case, seed):
    geom, T = GEOMS[case["geom"]], case["tokens"]
    E = geom.n_experts
    gen = _gen(seed)
    W = (torch.randn((2, E, geom.d_model), generator=gen, device="cuda") * 0.02).to(torch.bfloat16)
    bias = None
    if geom.has_proj_bias:
        bias = torch.stack([_popularity(E, gen) for _ in range(2)]).to(torch.bfloat16)
    x = torch.randn((T, geom.d_model), generator=gen, device="cuda").to(torch.bfloat16)
    table = torch.randperm(E, generator=gen, device="cuda").to(torch.int32)
    k = geom.top_k
    bufs = ops.RouteBuffers(T, k, k, x.device) if case["kept"] else None
    return dict(x=x, W=W, bias=bias, table=table, bufs=bufs, geom=geom)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "ffn":
        st = _prepare_ffn(case, seed)
    elif kind == "route":
        st = _prepare_route(case, seed)
    else:
        geom, L = GEOMS[case["geom"]], case["layers"]
        slots = geom.n_experts * L // 3
        if kind == "stack":
            s = stack.PrefillStack(geom, L, slots, case["tokens"], block="auto", seed=seed)
            s.capture()
            x = synth.hidden_states(case["tokens"], L, geom.d_model, "cuda", seed + 5)
            x = x.transpose(0, 1).contiguous()
        elif kind == "token":
            s = stack.DecodeStack(geom, L, slots, seed=seed)
            x = synth.hidden_states(1, L, geom.d_model, "cuda", seed + 5)[0]
        else:
            s = stack.StreamingStack(geom, L, slots, seed=seed, native=True)
            x = synth.hidden_states(case["tokens"], L, geom.d_model, "cuda", seed + 5)
        st = dict(stack=s, x=x)
    st["kind"] = kind
    torch.cuda.synchronize()
    return st


# -- one pass -----------------------------------------------------------------
def run(st):
    kind = st["kind"]
    if kind == "ffn":
        out32 = torch.empty(st["x"].shape, device="cuda") if st["f32"] else None
        return {"y": ops.ffn(st["pool"], st["refs"], st["scores"], st["x"], out_f32=out32)}
    if kind == "route":
        g, W, b = st["geom"], st["W"], st["bias"]
        r = ops.route(st["x"], W[0], None if b is None else b[0], g.routing, g.norm_topk_prob,
                      g.top_k, W_next=W[1], bias_next=None if b is None else b[1],
                      k_pred=g.top_k, table=st["table"], bufs=st["bufs"])
        return {"ids": r.ids, "scores": r.scores, "refs": r.slot_refs, "pred": r.pred}
    s, x = st["stack"], st["x"]
    if kind == "stack":
        s.run_step(x)
        return {"y": s.y, "ids": [b.ids for b in s.bufs], "scores": [b.scores for b in s.bufs]}
    if kind == "token":
        s.token_persistent(x)
        return {"y": s.p_y, "ids": s.p_ids, "scores": s.p_scores}
    return {"y": torch.stack([s.token(t) for t in x])}


# -- what a pass cannot do without ---------------------------------------------
def _distinct(case):
    """Experts that a layer's tokens reach, by the Zipf popularity."""
    geom = GEOMS[case["geom"]]
    T = case.get("tokens", 1)
    rng = np.random.default_rng(1)
    logp = -ZIPF * np.log(np.arange(1, geom.n_experts + 1))
    z = logp + rng.gumbel(size=(T, geom.n_experts))
    return len(np.unique(np.argpartition(-z, geom.top_k - 1, axis=1)[:, :geom.top_k]))


def work(case):
    geom, kind = GEOMS[case["geom"]], case["kind"]
    D, F, E, k = geom.d_model, geom.d_ff, geom.n_experts, geom.top_k
    T, L = case.get("tokens", 1), case.get("layers", 1)
    ffn_flops = 6 * T * k * D * F
    ffn_bytes = T * (2 * D + 8 * k + (4 if case.get("f32") else 2) * D)
    route_flops, route_bytes = 4 * T * D * E, 4 * E * D + 2 * T * D + 16 * T * k
    if kind == "ffn":
        return {"bytes": ffn_bytes + _distinct(case) * geom.payload_bytes, "flops": ffn_flops}
    if kind == "route":
        return {"bytes": route_bytes, "flops": route_flops}
    # (tokens of a streaming loop come one after the other: k experts each)
    experts = T * k if kind == "stream" else _distinct(case)
    passes = T if kind == "stream" else 1
    return {"bytes": L * (experts * geom.payload_bytes + ffn_bytes + passes * 4 * E * D),
            "flops": L * (ffn_flops + route_flops)}


def tolerance(case):
    kind = case["kind"]
    if kind == "ffn":
        # bf16 activations between the projections, bf16 or fp32 results
        return {"rel": 1e-2}
    if kind == "route":
        # bf16 logits: sums in another order move a few by one step, which
        # swaps or replaces experts whose values tie or nearly tie
        return {"rel": 1e-2, "differ": 0.01}
    # a replaced expert changes its token's row by about its score
    return {"rel": 3e-2, "differ": 0.01}


# -- the same in 64 bits --------------------------------------------------------
def _bf16(v):
    """Rounded once, to nearest even, from 64 bits."""
    m, e = torch.frexp(v)
    return torch.ldexp(torch.round(m * 256.0), e - 8)


def _project(rec, geom, proj, v):
    """v [n, inputs] through one expert record's 4-bit projection, in fp64."""
    comps = {c.name: c for c in geom.components}

    def part(name):
        c = comps[proj + "." + name]
        return rec[c.offset:c.offset + c.nbytes]

    out = comps[proj + ".weight"].shape[0]
    b = part("weight").view(out, -1)
    q = torch.stack([b & 15, b >> 4], dim=2).view(out, -1, 64).double()
    s = part("scales").view(torch.bfloat16).view(out, -1, 1).double()
    o = part("biases").view(torch.bfloat16).view(out, -1, 1).double()
    r = v @ (q * s + o).view(out, -1).T
    if geom.has_proj_bias:
        r = r + part("bias").view(torch.bfloat16).double()
    return r


def _experts(records, geom, x, ids, scores):
    """sum_j scores[t, j] expert_{ids[t, j]}(x[t]) in fp64; records(e) is
    expert e's record on the GPU."""
    y = torch.zeros(x.shape, dtype=torch.float64, device="cuda")
    xd = x.double()
    for e in torch.unique(ids).tolist():
        t, j = torch.nonzero(ids == e, as_tuple=True)
        rec = records(e)
        g = _project(rec, geom, "gate_proj", xd[t])
        u = _project(rec, geom, "up_proj", xd[t])
        if geom.act == 0:
            h = g * torch.sigmoid(g) * u
        else:
            g = g.clamp(max=geom.limit)
            h = g * torch.sigmoid(geom.alpha * g) * (u.clamp(-geom.limit, geom.limit) + 1)
        y.index_add_(0, t, scores[t, j].double()[:, None] * _project(rec, geom, "down_proj", h))
    return y


def _top(v, k):
    """Values descending, ties to the lower expert."""
    return torch.sort(v, dim=1, descending=True, stable=True).indices[:, :k]


def _route(geom, x, W, bias):
    """ids and scores of one router, and its raw logits' top-k; the logits and
    probabilities are defined as bf16, the sums are in 64 bits."""
    z = x.double() @ W.double().T
    if bias is not None:
        z = z + bias.double()
    z = _bf16(z)
    pred = _top(z, geom.top_k)
    if geom.routing == 0:
        p = _bf16(torch.softmax(z, dim=1))
        ids = _top(p, geom.top_k)
        s = p.gather(1, ids)
        if geom.norm_topk_prob:
            s = _bf16(s / _bf16(s.sum(dim=1, keepdim=True)))
    else:
        ids = pred
        s = _bf16(torch.softmax(z.gather(1, ids), dim=1))
    return ids, s, pred


def exact(case, seed):
    st = prepare(case, seed)
    geom, kind = GEOMS[case["geom"]], case["kind"]
    if kind == "ffn":
        rec = st["rec"]
        return {"y": _experts(lambda e: rec[e], geom, st["x"], st["ids"], st["scores"])}
    if kind == "route":
        W, b = st["W"], st["bias"]
        ids, s, _ = _route(geom, st["x"], W[0], None if b is None else b[0])
        pred = _route(geom, st["x"], W[1], None if b is None else b[1])[2]
        return {"ids": ids, "scores": s, "refs": st["table"][ids], "pred": pred}
    s, x, L, E = st["stack"], st["x"], case["layers"], geom.n_experts
    if kind == "stream":
        x = x.transpose(0, 1)
        host = s.store.array
    ys, ids, scores = [], [], []
    for l in range(L):
        xl = x[l].reshape(-1, geom.d_model)
        i, sc, _ = _route(geom, xl, s.W[l], None if s.bias is None else s.bias[l])
        if kind == "stream":
            def records(e, l=l):
                return torch.from_numpy(host[l * E + e]).cuda()
        else:
            def records(e, l=l):
                return s.store[l * E + e]
        ys.append(_experts(records, geom, xl, i, sc))
        ids.append(i)
        scores.append(sc)
    if kind == "stream":
        return {"y": torch.stack(ys, dim=1)}
    if kind == "token":
        return {"y": torch.cat(ys), "ids": torch.cat(ids), "scores": torch.cat(scores)}
    return {"y": torch.stack(ys), "ids": ids, "scores": scores}
