"""Performance cases: the work a user of this package has it do, through its
public entry points, with the exact (64-bit) results beside it.

Kinds of a case (``case["kind"]``):

* ``expert``   expert_mlp_int4_fused: one INT4 SwiGLU expert over the tokens
               routed to it (the reference loop's call).
* ``linear``   Int4Linear.forward: an attention or dense projection held INT4.
* ``mixtral``  MixtralMoELayer.forward: router, 8 resident experts, combine.
* ``glm``      GLM4MoELayer.forward: sigmoid top-8 of 128 resident experts and
               the fp16 shared expert.
* ``attn``     Attention.forward over the KV cache (prefill of S tokens after
               ``past`` cached ones).
* ``decoder``  GraphDecoder.step: one greedy decode step of a Mixtral-shaped
               decoder, replayed from its captured graph.
* ``pack``     quantize_int4: the INT4 packer over one weight matrix.

Weights are drawn as INT4 codes and fp16 scales directly (codes of a normal
weight of deviation 0.02 at absmax / 7 scales).  The Mixtral routers see
hidden states with a component along the gate rows of the experts they prefer,
so the selection does not hang on the last bit of a logit.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

MIXTRAL = (4096, 14336)  # hidden, intermediate
GLM = (4096, 1408)
HEADS, KV_HEADS, HEAD_DIM = 32, 8, 128


# ----------------------------------------------------------------------------- the cases
def listed():
    return [
        # one decode token on one resident expert: the smallest drop-in call
        {"name": "expert_t1", "kind": "expert", "model": "mixtral", "tokens": 1},
        # an odd batch of decode tokens that all reached one expert
        {"name": "expert_t37", "kind": "expert", "model": "mixtral", "tokens": 37},
        # fused q/k/v projection of a 64-sequence decode step, held INT4
        {"name": "linear_m64", "kind": "linear", "k": 4096, "n": 6144, "group": 128, "m": 64,
         "bias": False},
        # a ragged prompt through an output projection at the group-64 fallback
        {"name": "linear_m333_g64", "kind": "linear", "k": 4096, "n": 4096, "group": 64, "m": 333,
         "bias": True},
        # one MoE layer of a 16-sequence decode step
        {"name": "mixtral_t16", "kind": "mixtral", "batch": 16, "seq": 1, "top_k": 2,
         "skew": 0.0},
        # a short prompt, unevenly routed
        {"name": "mixtral_t100", "kind": "mixtral", "batch": 1, "seq": 100, "top_k": 2,
         "skew": 1.1},
        # a long prompt (or several) in one prefill pass, unevenly routed
        {"name": "mixtral_t2048", "kind": "mixtral", "batch": 1, "seq": 2048, "top_k": 2,
         "skew": 1.1},
        # the many-small-experts layer of a 32-sequence decode step
        {"name": "glm_t32", "kind": "glm", "batch": 32, "seq": 1},
        # the same layer over a medium, odd-sized prompt
        {"name": "glm_t301", "kind": "glm", "batch": 1, "seq": 301},
        # attention of a prefill pass over a batch of odd-length prompts
        {"name": "attn_b8_s333", "kind": "attn", "batch": 8, "seq": 333, "past": 0},
        # a decode step of 64 sequences through two decoder layers and the LM head
        {"name": "decoder_b64", "kind": "decoder", "batch": 64, "past": 540, "layers": 2},
        # packing one expert projection of a checkpoint
        {"name": "pack_fp16", "kind": "pack", "n": 14336, "k": 4096, "group": 128, "mode": 0,
         "dtype": "float16"},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["expert", "linear", "mixtral", "mixtral", "glm", "attn", "decoder",
                       "pack"])
    if kind == "expert":
        return {"kind": kind, "model": rng.choice(["mixtral", "glm"]),
                "tokens": _logint(rng, 1, 700)}
    if kind == "linear":
        k, n = rng.choice([(4096, 6144), (4096, 4096), (4096, 1408), (1408, 4096),
                           (4096, 14336)])
        return {"kind": kind, "k": k, "n": n, "group": rng.choice([128, 128, 64, 32]),
                "m": _logint(rng, 1, 2048), "bias": rng.random() < 0.5}
    if kind == "mixtral":
        if rng.random() < 0.5:
            return {"kind": kind, "batch": _logint(rng, 1, 128), "seq": 1,
                    "top_k": rng.choice([1, 2]), "skew": 0.0}
        return {"kind": kind, "batch": 1, "seq": _logint(rng, 16, 2000), "top_k": 2, "skew": 1.1}
    if kind == "glm":
        if rng.random() < 0.5:
            return {"kind": kind, "batch": _logint(rng, 1, 128), "seq": 1}
        return {"kind": kind, "batch": 1, "seq": _logint(rng, 16, 1500)}
    if kind == "attn":
        b = rng.choice([1, 2, 4, 8])
        s = _logint(rng, 16, 900 if b <= 4 else 400)
        return {"kind": kind, "batch": b, "seq": s,
                "past": rng.choice([0, 0, rng.randint(1, 1000 - s)])}
    if kind == "decoder":
        return {"kind": kind, "batch": _logint(rng, 1, 64), "past": _logint(rng, 16, 900),
                "layers": 2}
    mode, dtype = rng.choice([(0, "float16"), (1, "float16"), (1, "float32")])
    n, k = rng.choice([(14336, 4096), (4096, 14336), (1408, 4096), (4096, 1408)])
    return {"kind": kind, "n": n, "k": k, "group": rng.choice([128, 64, 32]), "mode": mode,
            "dtype": dtype}


# ----------------------------------------------------------------------------- inputs
def _gen(seed, part):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 10007 + part)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _int4(g, n, k, group, sigma=0.02):
    """(packed [n, k/2] uint8, scales [n, k/group] fp16) of a normal [n, k] weight."""
    code = (_randn(g, n, k) * 2.7).round_().clamp_(-7, 7).add_(8).to(torch.uint8)
    packed = code[:, 0::2] | (code[:, 1::2] << 4)
    s = (sigma / 2.7) * (1 + 0.1 * _randn(g, n, k // group)).clamp_(0.5, 1.5)
    return packed.contiguous(), s.to(torch.float16)


def _dequant64(packed, scales):
    n, k = packed.shape[0], packed.shape[1] * 2
    code = torch.stack((packed & 15, packed >> 4), dim=2).view(n, k).to(torch.float64) - 8
    g = k // scales.shape[1]
    return (code.view(n, -1, g) * scales.double().unsqueeze(2)).view(n, k)


def _expert_tensors(seed, part, model, down_sigma=0.02, group=128):
    h, i = model
    g = _gen(seed, 100 + part)
    gate, up = _int4(g, i, h, group), _int4(g, i, h, group)
    down = _int4(g, h, i, group, down_sigma)
    return (*gate, *up, *down)


def _slot(tensors, model, idx, group=128):
    from hydranet_amd.cache.packed_expert_store import GpuExpertSlot
    slot = GpuExpertSlot(idx, model[0], model[1], group, torch.device("cuda"))
    names = ("gate_packed", "gate_scales", "up_packed", "up_scales", "down_packed", "down_scales")
    slot.load_from_tensors(dict(zip(names, tensors)))
    return slot


def _swiglu64(x, tensors):
    gate, up, down = (_dequant64(tensors[2 * j], tensors[2 * j + 1]) for j in range(3))
    return (F.silu(x @ gate.t()) * (x @ up.t())) @ down.t()


def _popularity(experts, skew, device):
    p = torch.arange(1, experts + 1, device=device, dtype=torch.float32) ** -skew
    return p / p.sum()


def _mixtral_inputs(case, seed):
    h, e, t = MIXTRAL[0], 8, case["batch"] * case["seq"]
    g = _gen(seed, 1)
    gate = (_randn(g, e, h) * 0.02).to(torch.float16)
    x = _randn(g, t, h)
    # the experts each token prefers, by popularity (Gumbel top-k), and the hidden
    # state's component along their gate rows
    gumbel = -torch.log(-torch.log(torch.rand(t, e, generator=g, device="cuda") + 1e-9) + 1e-9)
    pref = (_popularity(e, case["skew"], "cuda").log() + gumbel).topk(case["top_k"], -1).indices
    unit = F.normalize(gate.float(), dim=-1)
    for j in range(case["top_k"]):
        x += 7.0 * unit[pref[:, j]]
    return x.to(torch.float16), gate


def _attention_weights(seed, part):
    h = HEADS * HEAD_DIM
    g = _gen(seed, 50 + part)
    return {name: (_randn(g, n, h) * 0.02).to(torch.float16)
            for name, n in (("q_proj", h), ("k_proj", KV_HEADS * HEAD_DIM),
                            ("v_proj", KV_HEADS * HEAD_DIM), ("o_proj", h))}


def _cached(seed, part, batch, past, max_len):
    """Keys (transposed) and values of `past` cached positions, the rest zero."""
    g = _gen(seed, 70 + part)
    kt = torch.zeros(batch, KV_HEADS, HEAD_DIM, max_len, device="cuda", dtype=torch.float16)
    v = torch.zeros(batch, KV_HEADS, max_len, HEAD_DIM, device="cuda", dtype=torch.float16)
    if past:
        kt[..., :past] = _randn(g, batch, KV_HEADS, HEAD_DIM, past) * 1.28
        v[:, :, :past] = _randn(g, batch, KV_HEADS, past, HEAD_DIM) * 1.28
    return kt, v


def _max_len(case):
    n = case["past"] + case.get("seq", 1)
    return -(-n // 64) * 64


def _decoder_inputs(case, seed):
    """Embedding rows lean towards the gate row of one expert per token and layer
    (so the top-1 routing is decided); the sublayers write less than they read."""
    h, vocab, layers = MIXTRAL[0], 32000, case["layers"]
    g = _gen(seed, 2)
    gates = [(_randn(g, 8, h) * 0.02).to(torch.float16) for _ in range(layers)]
    embed = _randn(g, vocab, h)
    choice = torch.arange(vocab, device="cuda")
    for l, w in enumerate(gates):
        embed += 12.0 * F.normalize(w.float(), dim=-1)[(choice * 7 + choice // 8 + 3 * l) % 8]
    head = (_randn(g, vocab, h) * 0.02).to(torch.float16)
    tok = torch.randint(0, vocab, (case["batch"], 1), generator=g, device="cuda")
    return gates, embed.to(torch.float16), head, tok


def prepare(case, seed):
    kind = case["kind"]
    if kind == "expert":
        model = MIXTRAL if case["model"] == "mixtral" else GLM
        x = _randn(_gen(seed, 1), case["tokens"], model[0]).to(torch.float16)
        return {"kind": kind, "x": x, "slot": _slot(_expert_tensors(seed, 0, model), model, 0)}
    if kind == "linear":
        from hydranet_amd.kernels.int4_linear import Int4Linear
        g = _gen(seed, 1)
        x = _randn(g, case["m"], case["k"]).to(torch.float16)
        bias = _randn(g, case["n"]).to(torch.float16)
        lin = Int4Linear(case["k"], case["n"], case["bias"], case["group"], torch.device("cuda"))
        lin.load_quantized(*_int4(g, case["n"], case["k"], case["group"]), bias=bias)
        return {"kind": kind, "x": x, "layer": lin}
    if kind == "mixtral":
        from hydranet_amd.model.moe import MixtralMoELayer
        x, gate = _mixtral_inputs(case, seed)
        slots = [_slot(_expert_tensors(seed, e, MIXTRAL), MIXTRAL, e) for e in range(8)]
        with torch.device("cuda"):
            layer = MixtralMoELayer(MIXTRAL[0], 8, 2, slots=slots)
        layer = layer.to(torch.float16).eval()
        with torch.no_grad():
            layer.router.gate.weight.copy_(gate)
        return {"kind": kind, "x": x.view(case["batch"], case["seq"], -1), "layer": layer,
                "top_k": case["top_k"]}
    if kind == "glm":
        from hydranet_amd.model.moe import GLM4MoELayer
        x, weight, shared = _glm_inputs(case, seed)
        slots = [_slot(_expert_tensors(seed, e, GLM), GLM, e) for e in range(128)]
        with torch.device("cuda"):
            layer = GLM4MoELayer(GLM[0], GLM[1], 128, 8, slots=slots)
        layer.shared_expert.to(torch.float16)
        layer.eval()
        with torch.no_grad():
            layer.router.weight.copy_(weight)
            for name, w in shared.items():
                getattr(layer.shared_expert, name).weight.copy_(w)
        return {"kind": kind, "x": x.view(case["batch"], case["seq"], -1), "layer": layer}
    if kind == "attn":
        from hydranet_amd.model.decoder import (Attention, KVCache, MixtralDecoderConfig,
                                                RotaryEmbedding, causal_mask)
        cfg = MixtralDecoderConfig(num_layers=1)
        b, s, past, n = case["batch"], case["seq"], case["past"], _max_len(case)
        with torch.device("cuda"):
            att = Attention(cfg)
        att = att.to(torch.float16).eval()
        with torch.no_grad():
            for name, w in _attention_weights(seed, 0).items():
                getattr(att, name).weight.copy_(w)
        rope = RotaryEmbedding(HEAD_DIM, n, cfg.rope_theta, "cuda")
        cache = KVCache(1, b, KV_HEADS, HEAD_DIM, n, "cuda")
        cache.kt[0], cache.v[0] = _cached(seed, 0, b, past, n)
        x = _randn(_gen(seed, 1), b, s, cfg.hidden_dim).to(torch.float16)
        return {"kind": kind, "x": x, "att": att, "rope": rope, "cache": cache,
                "pos": torch.arange(past, past + s, device="cuda"), "len": past + s,
                "mask": causal_mask(past, s, "cuda") if s > 1 else None}
    if kind == "decoder":
        from hydranet_amd.model.decoder import (GraphDecoder, MixtralDecoder,
                                                MixtralDecoderConfig, RotaryEmbedding)
        cfg = MixtralDecoderConfig(num_layers=case["layers"])
        gates, embed, head, tok = _decoder_inputs(case, seed)
        slots = [[_slot(_expert_tensors(seed, 8 * l + e, MIXTRAL, 0.005), MIXTRAL, e)
                  for e in range(8)] for l in range(cfg.num_layers)]
        with torch.device("cuda"):
            m = MixtralDecoder(cfg, slots, device="cuda")
        m = m.to(torch.float16).eval()
        m.rotary = RotaryEmbedding(HEAD_DIM, cfg.max_position_embeddings, cfg.rope_theta, "cuda")
        with torch.no_grad():
            m.embed_tokens.weight.copy_(embed)
            m.lm_head.weight.copy_(head)
            for l, blk in enumerate(m.layers):
                blk.moe.router.gate.weight.copy_(gates[l])
                for name, w in _attention_weights(seed, l).items():
                    getattr(blk.self_attn, name).weight.copy_(w)
        past, n = case["past"], _max_len(case)
        cache = m.new_cache(case["batch"], n)
        for l in range(cfg.num_layers):
            kt, v = _cached(seed, l, case["batch"], past, n)
            cache.kt[l].copy_(kt)
            cache.v[l].copy_(v)
        cache.cur_len = past
        return {"kind": kind, "graph": GraphDecoder(m, cache, tok), "tok": tok, "past": past}
    dtype = getattr(torch, case["dtype"])
    w = (_randn(_gen(seed, 1), case["n"], case["k"]) * 0.02).to(dtype)
    return {"kind": kind, "w": w, "group": case["group"], "mode": case["mode"]}


def _glm_inputs(case, seed):
    h, i = GLM
    g = _gen(seed, 1)
    x = _randn(g, case["batch"] * case["seq"], h).to(torch.float16)
    weight = (torch.rand(128, h, generator=g, device="cuda") * 2 - 1) / math.sqrt(h)
    shared = {"gate_proj": (_randn(g, i, h) * 0.02).to(torch.float16),
              "up_proj": (_randn(g, i, h) * 0.02).to(torch.float16),
              "down_proj": (_randn(g, h, i) * 0.02).to(torch.float16)}
    return x, weight, shared


# ----------------------------------------------------------------------------- one pass
@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "expert":
        from hydranet_amd.kernels import expert_mlp_int4_fused
        s = state["slot"]
        return expert_mlp_int4_fused(state["x"], s.gate_packed, s.gate_scales, s.up_packed,
                                     s.up_scales, s.down_packed, s.down_scales, s.group_size)
    if kind in ("linear", "glm"):
        return state["layer"](state["x"])
    if kind == "mixtral":
        return state["layer"](state["x"], top_k=state["top_k"])
    if kind == "attn":
        c = state["cache"]
        out = state["att"](state["x"], state["rope"], state["pos"], c, 0, state["len"],
                           state["mask"])
        return {"out": out, "kt": c.kt[0], "v": c.v[0]}
    if kind == "decoder":
        # decode again from the same position: rewind the cache and the step's inputs
        g = state["graph"]
        g.cache.cur_len = state["past"]
        g.pos.fill_(state["past"])
        g.tok.copy_(state["tok"])
        g.step()
        return {"logits": g.logits, "kt": g.cache.kt, "v": g.cache.v}
    from hydranet_amd.kernels.int4_gemm import quantize_int4
    return quantize_int4(state["w"], state["group"], state["mode"])


# ----------------------------------------------------------------------------- what it must cost
def _int4_bytes(n, k, group=128):
    return n * k // 2 + n * (k // group) * 2


def _expert_bytes(model):
    return 3 * _int4_bytes(model[1], model[0])


def _experts_hit(experts, k, tokens, skew):
    """Expected number of distinct experts over the tokens' top-k choices."""
    p = [(i + 1) ** -skew for i in range(experts)]
    z = sum(p)
    p = [v / z for v in p]
    if k == 1:
        inc = p
    elif k == 2:
        inc = [p[i] + sum(p[j] * p[i] / (1 - p[j]) for j in range(experts) if j != i)
               for i in range(experts)]
    else:
        inc = [k / experts] * experts
    return sum(1 - (1 - min(v, 1.0)) ** tokens for v in inc)


def work(case):
    kind = case["kind"]
    if kind == "expert":
        model, t = (MIXTRAL if case["model"] == "mixtral" else GLM), case["tokens"]
        return {"bytes": _expert_bytes(model) + 4 * t * model[0],
                "flops": 6 * t * model[0] * model[1]}
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _int4_bytes(n, k, case["group"]) + 2 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "mixtral":
        t, k = case["batch"] * case["seq"], case["top_k"]
        hit = _experts_hit(8, k, t, case["skew"])
        return {"bytes": hit * _expert_bytes(MIXTRAL) + 4 * t * MIXTRAL[0] + 16 * MIXTRAL[0],
                "flops": 6 * t * k * MIXTRAL[0] * MIXTRAL[1]}
    if kind == "glm":
        t = case["batch"] * case["seq"]
        hit = _experts_hit(128, 8, t, 0.0)
        return {"bytes": hit * _expert_bytes(GLM) + 6 * GLM[0] * GLM[1] + 4 * 128 * GLM[0]
                + 4 * t * GLM[0],
                "flops": 6 * t * 9 * GLM[0] * GLM[1] + 2 * t * 128 * GLM[0]}
    if kind == "attn":
        b, s, past, h = case["batch"], case["seq"], case["past"], HEADS * HEAD_DIM
        kv = 2 * KV_HEADS * HEAD_DIM
        return {"bytes": 2 * (h * (2 * h + kv) + 2 * b * s * h + b * (past + 2 * s) * kv),
                "flops": 2 * b * s * h * (2 * h + kv) + 4 * b * h * s * (past + (s + 1) / 2)}
    if kind == "decoder":
        b, h = case["batch"], HEADS * HEAD_DIM
        kv = 2 * KV_HEADS * HEAD_DIM
        hit = _experts_hit(8, 1, b, 0.0)
        layer = hit * _expert_bytes(MIXTRAL) + 2 * h * (2 * h + kv) + 2 * b * case["past"] * kv
        flops = 2 * b * h * (2 * h + kv) + 4 * b * h * case["past"] + 6 * b * h * MIXTRAL[1]
        return {"bytes": case["layers"] * layer + 2 * 32000 * (h + b),
                "flops": case["layers"] * flops + 2 * b * h * 32000}
    n, k = case["n"], case["k"]
    size = 2 if case["dtype"] == "float16" else 4
    return {"bytes": n * k * size + _int4_bytes(n, k, case["group"]), "flops": 0}


def tolerance(case):
    # about four times the error against exact() measured over the ranges above
    # (expert 4.6e-4, linear 3.1e-4, mixtral 1.3e-3, glm 5.7e-4, attn 1.4e-3,
    # decoder 1.0e-3)
    return {"expert": {"rel": 2e-3}, "linear": {"rel": 1.5e-3}, "mixtral": {"rel": 5e-3},
            "glm": {"rel": 2.5e-3}, "attn": {"rel": 5e-3}, "decoder": {"rel": 4e-3},
            "pack": "exact"}[case["kind"]]


# ----------------------------------------------------------------------------- exact results
def _rotate64(x, pos, theta=1e6):
    inv = 1.0 / theta ** (torch.arange(0, HEAD_DIM, 2, device="cuda").double() / HEAD_DIM)
    ang = torch.outer(pos.double(), inv)
    cos, sin = torch.cat([ang.cos()] * 2, -1), torch.cat([ang.sin()] * 2, -1)
    half = HEAD_DIM // 2
    return x * cos + torch.cat((-x[..., half:], x[..., :half]), -1) * sin


def _attention64(x, weights, kt, v, past):
    """x [B, S, H] float64 -> (out, kt, v) with positions past .. past + S - 1 filled."""
    b, s, _ = x.shape
    pos = torch.arange(past, past + s, device="cuda")
    heads = {n: (x @ weights[n].double().t()).view(b, s, -1, HEAD_DIM).transpose(1, 2)
             for n in ("q_proj", "k_proj", "v_proj")}
    q, key = _rotate64(heads["q_proj"], pos), _rotate64(heads["k_proj"], pos)
    kt, v = kt.double(), v.double()
    kt[..., past:past + s] = key.transpose(2, 3)
    v[:, :, past:past + s] = heads["v_proj"]
    out = torch.empty(b, HEADS, s, HEAD_DIM, device="cuda", dtype=torch.float64)
    later = torch.arange(past + s, device="cuda") > pos.unsqueeze(1)
    for h in range(HEADS):
        g = h // (HEADS // KV_HEADS)
        for i in range(b):
            a = q[i, h] @ kt[i, g, :, :past + s] / math.sqrt(HEAD_DIM)
            out[i, h] = torch.softmax(a.masked_fill(later, -math.inf), -1) @ v[i, g, :past + s]
    return out.transpose(1, 2).reshape(b, s, -1) @ weights["o_proj"].double().t(), kt, v


def _moe64(x, logits, k, experts, weigh):
    """Sum over each row's top-k experts of weight * SwiGLU; experts(e) -> its tensors."""
    top, idx = logits.topk(k, -1)
    w = weigh(top)
    out = torch.zeros_like(x)
    for e in torch.unique(idx).tolist():
        row, slot = (idx == e).nonzero(as_tuple=True)
        out[row] += w[row, slot].unsqueeze(1) * _swiglu64(x[row], experts(e))
    return out


def _norm64(x, eps=1e-5):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "expert":
        model = MIXTRAL if case["model"] == "mixtral" else GLM
        x = _randn(_gen(seed, 1), case["tokens"], model[0]).to(torch.float16)
        return _swiglu64(x.double(), _expert_tensors(seed, 0, model))
    if kind == "linear":
        g = _gen(seed, 1)
        x = _randn(g, case["m"], case["k"]).to(torch.float16)
        bias = _randn(g, case["n"]).to(torch.float16)
        out = x.double() @ _dequant64(*_int4(g, case["n"], case["k"], case["group"])).t()
        return out + bias.double() if case["bias"] else out
    if kind == "mixtral":
        x, gate = _mixtral_inputs(case, seed)
        x = x.double()
        out = _moe64(x, x @ gate.double().t(), case["top_k"],
                     lambda e: _expert_tensors(seed, e, MIXTRAL), lambda t: torch.softmax(t, -1))
        return out.view(case["batch"], case["seq"], -1)
    if kind == "glm":
        x, weight, shared = _glm_inputs(case, seed)
        x = x.double()
        sh = {n: w.double() for n, w in shared.items()}
        out = (F.silu(x @ sh["gate_proj"].t()) * (x @ sh["up_proj"].t())) @ sh["down_proj"].t()
        out = out + _moe64(x, x @ weight.double().t(), 8, lambda e: _expert_tensors(seed, e, GLM),
                           lambda t: torch.sigmoid(t) / torch.sigmoid(t).sum(-1, keepdim=True))
        return out.view(case["batch"], case["seq"], -1)
    if kind == "attn":
        b, s, past = case["batch"], case["seq"], case["past"]
        x = _randn(_gen(seed, 1), b, s, MIXTRAL[0]).to(torch.float16)
        out, kt, v = _attention64(x.double(), _attention_weights(seed, 0),
                                  *_cached(seed, 0, b, past, _max_len(case)), past)
        return {"out": out, "kt": kt, "v": v}
    if kind == "decoder":
        gates, embed, head, tok = _decoder_inputs(case, seed)
        x = embed[tok].double()
        kts, vs = [], []
        for l in range(case["layers"]):
            a, kt, v = _attention64(_norm64(x), _attention_weights(seed, l),
                                    *_cached(seed, l, case["batch"], case["past"],
                                             _max_len(case)), case["past"])
            kts.append(kt)
            vs.append(v)
            x = x + a
            h = _norm64(x).squeeze(1)
            x = x + _moe64(h, h @ gates[l].double().t(), 1,
                           lambda e: _expert_tensors(seed, 8 * l + e, MIXTRAL, 0.005),
                           torch.ones_like).unsqueeze(1)
        return {"logits": _norm64(x) @ head.double().t(), "kt": kts, "v": vs}
    return None
