"""GPU tests of prefill attention (hn_attn_prefill) and of the RoPE + append
kernel for runs of tokens, against a float64 evaluation and against the
one-element-per-thread kernel, at the edges of their tiles."""
import math

import numpy as np
import pytest
import torch

from hydranet_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
HD = 128
INV = float(np.float32(1.0) / np.float32(math.sqrt(HD)))


def _operands(B, nkv, rep, S, L, max_len, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    q = torch.randn(B, nkv, rep * S, HD, generator=g, device=DEV).half()
    kt = torch.full((B, nkv, HD, max_len), float("nan"), dtype=torch.float16, device=DEV)
    v = torch.full((B, nkv, max_len, HD), float("nan"), dtype=torch.float16, device=DEV)
    kt[..., :L] = torch.randn(B, nkv, HD, L, generator=g, device=DEV).half()
    v[:, :, :L] = torch.randn(B, nkv, L, HD, generator=g, device=DEV).half()
    return q, kt, v  # positions past L hold NaN: nothing may read them into a result


def _run(q, kt, v, B, nkv, rep, S, L, mask, ld_o=None):
    out = torch.zeros(B * S, ld_o or nkv * rep * HD, dtype=torch.float16, device=DEV)
    n = _lib.lib().hn_attn_prefill_workspace_bytes(S, rep, L)
    work = torch.full((n,), 0xAB, dtype=torch.uint8, device=DEV)
    _lib.call("hn_attn_prefill", _lib.ptr(q), _lib.ptr(kt), _lib.ptr(v), kt.shape[3], B, nkv, rep,
              HD, S, L, _lib.ptr(mask), 0 if mask is None else mask.stride(0), INV,
              _lib.ptr(out), out.stride(0), _lib.ptr(work) if mask is not None else None,
              _lib.stream())
    return out[:, :nkv * rep * HD].view(B, S, nkv, rep, HD).permute(0, 2, 3, 1, 4)


def _ref(q, kt, v, B, nkv, rep, S, L, mask, rounded):
    """(out, sum p |v|) in float64; rounded: the scores' fp16 steps."""
    s = torch.matmul(q.double(), kt[..., :L].double()).view(B, nkv, rep, S, L)
    if rounded:
        s = (s.half().float() * INV).half().float()
        s = (s + mask.float()).half().double()
    else:
        s = s * INV
        if mask is not None:
            s = s + mask.double()
    p = torch.softmax(s, -1)
    vv = v[:, :, None, :L].double()
    return torch.matmul(p, vv), torch.matmul(p, vv.abs()), s


def _causal(S, L):
    m = torch.full((S, L), float("-inf"), dtype=torch.float16, device=DEV)
    return torch.triu(m, diagonal=L - S + 1)


def _check(got, ref, absum, L, extra=0.0):
    # probabilities rounded to fp16 (2^-11 of each, 2^-25 where subnormal), the
    # output rounded (2^-11), fp32 scores and exponentials (1e-5 covers them)
    bound = (2.0 ** -11 + 1e-5 + extra) * absum + 2.0 ** -11 * ref.abs() + L * 2.0 ** -25 * 5 + 1e-7
    err = (got.double() - ref).abs()
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("B,nkv,rep,S,L,max_len", [
    (2, 2, 4, 2, 2, 8),         # fewer rows than one wave, one ragged tile
    (1, 1, 1, 31, 31, 32), (1, 2, 2, 33, 64, 64), (1, 1, 1, 127, 127, 128),
    (1, 2, 1, 129, 129, 136), (2, 2, 4, 333, 333, 336),
    (1, 2, 4, 5, 1030, 1032),   # few tokens after a long past
    (1, 1, 3, 65, 4500, 4504),  # more than 64 tiles
])
@pytest.mark.parametrize("masked", [True, False])
def test_prefill_attention(B, nkv, rep, S, L, max_len, masked):
    q, kt, v = _operands(B, nkv, rep, S, L, max_len, S + L)
    mask = _causal(S, L) if masked else None
    got = _run(q, kt, v, B, nkv, rep, S, L, mask, ld_o=nkv * rep * HD + 8)
    ref, absum, _ = _ref(q, kt, v, B, nkv, rep, S, L, mask, False)
    _check(got, ref, absum, L)


@pytest.mark.parametrize("S,L,kind", [(70, 200, "finite"), (70, 200, "lowest"),
                                      (40, 130, "holes"), (40, 130, "row")])
def test_prefill_attention_masks(S, L, kind):
    """finite: any values; lowest: the type's lowest value for hidden
    positions, and a row of nothing else; holes: a random 0 / -inf mask; row:
    a row of -inf (NaN there, and there only)."""
    B, nkv, rep = 1, 2, 2
    q, kt, v = _operands(B, nkv, rep, S, L, L + 8 - L % 8, 3)
    g = torch.Generator(device=DEV).manual_seed(9)
    big = torch.full((S, L + 3), 0.0, dtype=torch.float16, device=DEV)
    mask = big[:, :L]  # odd row stride
    rnd = torch.rand(S, L, generator=g, device=DEV)
    if kind == "finite":
        mask.copy_(torch.where(rnd < 0.2, float("-inf"), 4 * rnd - 2).half())
    elif kind == "lowest":
        mask.copy_(torch.where(rnd < 0.5, -65504.0, 0.0).half())
        mask[7] = -65504.0
    elif kind == "holes":
        mask.copy_(torch.where(rnd < 0.9, float("-inf"), 0.0).half())
        mask[:, 100:] = float("-inf")
    else:
        mask[5] = float("-inf")
        mask[:, 64:] = float("-inf")
    got = _run(q, kt, v, B, nkv, rep, S, L, mask)
    rounded = kind in ("finite", "lowest")
    ref, absum, s = _ref(q, kt, v, B, nkv, rep, S, L, mask, rounded)
    if kind == "row":
        assert bool(got[:, :, :, 5].isnan().all())
        keep = [i for i in range(S) if i != 5]
        got, ref, absum = got[:, :, :, keep], ref[:, :, :, keep], absum[:, :, :, keep]
    # fp16 scores below 8 (and below 64 before the scale): an fp32 sum on the
    # other side of a rounding boundary moves the masked score by two ulps of 8
    _check(got, ref, absum, L, extra=2 * 2.0 ** -7 if rounded else 0.0)


def test_prefill_attention_graph_replays():
    B, nkv, rep, S, L = 2, 2, 4, 70, 150
    q, kt, v = _operands(B, nkv, rep, S, L, 152, 1)
    mask = _causal(S, L)
    want = _run(q, kt, v, B, nkv, rep, S, L, mask).clone()
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        _run(q, kt, v, B, nkv, rep, S, L, mask)
    torch.cuda.current_stream().wait_stream(st)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = _run(q, kt, v, B, nkv, rep, S, L, mask)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


@pytest.mark.parametrize("S,L,masked", [(2, 2, True), (33, 100, True), (130, 130, False)])
def test_attention_module_routes_agree(S, L, masked):
    """Attention.forward by hn_attn_prefill and by the two products (both over
    the appended cache): fp16 scores and probabilities on one side only, so
    they agree to a few parts in a thousand of the output's size."""
    from hydranet_amd.model.decoder import Attention, KVCache, MixtralDecoderConfig, RotaryEmbedding
    cfg = MixtralDecoderConfig(hidden_dim=512, num_attention_heads=4, num_kv_heads=2)
    torch.manual_seed(0)
    att = Attention(cfg).half().to(DEV)
    assert att.hd == HD
    rope = RotaryEmbedding(HD, 256, 1e6, device=DEV)
    x = torch.randn(2, S, 512, device=DEV).half()
    pos = torch.arange(L - S, L, device=DEV)
    outs = []
    with torch.no_grad():
        for on in (True, False):
            att.decode_kernel = on
            cache = KVCache(1, 2, 2, HD, 256, DEV)
            g = torch.Generator(device=DEV).manual_seed(4)
            cache.kt[0].normal_(generator=g)
            cache.v[0].normal_(generator=g)
            outs.append(att(x, rope, pos, cache, 0, L, _causal(S, L) if masked else None).float())
    rel = (outs[0] - outs[1]).norm() / outs[1].norm()
    assert rel.item() < 2e-3, rel.item()


@pytest.mark.parametrize("batch,dtype", [(4, torch.float16), (2, torch.float32)])
def test_attention_module_refuses_another_cache(batch, dtype):
    """Two sequences against a cache of four, or of fp32: an error, as by the products."""
    from hydranet_amd.model.decoder import Attention, KVCache, MixtralDecoderConfig, RotaryEmbedding
    cfg = MixtralDecoderConfig(hidden_dim=512, num_attention_heads=4, num_kv_heads=2)
    att = Attention(cfg).half().to(DEV)
    rope = RotaryEmbedding(HD, 256, 1e6, device=DEV)
    x = torch.randn(2, 130, 512, device=DEV).half()
    for on in (True, False):
        att.decode_kernel = on
        cache = KVCache(1, batch, 2, HD, 256, DEV, dtype)
        with pytest.raises(RuntimeError):
            with torch.no_grad():
                att(x, rope, torch.arange(130, device=DEV), cache, 0, 130, _causal(130, 130))


@pytest.mark.parametrize("B,S,nh,nkv", [(2, 8, 8, 2), (1, 63, 4, 1), (2, 65, 12, 3), (1, 333, 32, 8)])
def test_rope_append_runs_equal_elementwise(B, S, nh, nkv):
    """The kernel for runs of tokens against the one-element kernel (taken when
    a row stride is odd), bit for bit: positions out of order, one out of
    range (written by neither)."""
    ml = 512
    g = torch.Generator(device=DEV).manual_seed(S)
    w = (nh + 2 * nkv) * HD
    qkv = torch.randn(B * S, w, generator=g, device=DEV).half()
    odd = torch.zeros(B * S, w + 1, dtype=torch.float16, device=DEV)
    odd[:, :w] = qkv
    cos = torch.randn(ml, HD, generator=g, device=DEV)
    sin = torch.randn(ml, HD, generator=g, device=DEV)
    pos = torch.randperm(ml, generator=g, device=DEV)[:S]
    pos[S // 2] = ml
    res = []
    for t in (qkv, odd):
        o = [torch.full((B, nh, S, HD), 7.0, dtype=torch.float16, device=DEV),
             torch.full((B, nkv, HD, ml), 7.0, dtype=torch.float16, device=DEV),
             torch.full((B, nkv, ml, HD), 7.0, dtype=torch.float16, device=DEV)]
        p, ld = t.data_ptr(), t.stride(0)
        _lib.call("hn_rope_append", p, ld, p + 2 * nh * HD, ld, p + 2 * (nh + nkv) * HD, ld,
                  _lib.ptr(cos), _lib.ptr(sin), _lib.ptr(pos), B, S, nh, nkv, HD, _lib.ptr(o[0]),
                  _lib.ptr(o[1]), _lib.ptr(o[2]), ml, _lib.stream())
        res.append(o)
    for a, b in zip(*res):
        assert torch.equal(a, b)
