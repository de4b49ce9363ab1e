"""The kernels for a middle number of rows per weight matrix (csrc/hn_mid.hip)
against float64 products of the dequantised weights, at the edges of their tiles
(32 and 64 tokens, 256 weight rows), K splits (even, uneven, none) and group
sizes, single and grouped.

Tolerance: the repository's bar for fp16 matrix outputs, 1e-2 + 2e-3 |ref|: one
fp16 rounding of the result (2^-11 relative), for groups under 128 one more per
weight (2^-11, averaging out over K), fp32 sums.  For the SwiGLU the two
projections round to fp16 first (1e-2 covers 2^-11 of either at these sizes)."""
import ctypes

import pytest
import torch

from hydranet_amd import _lib
from hydranet_amd.kernels import int4_gemm as g
from hydranet_amd.model import moe

pytestmark = pytest.mark.gpu


def _weight(n, k, group, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    w = torch.randn(n, k, generator=gen, device="cuda").mul_(0.02).half()
    return g.quantize_int4(w, group)


def _deq(p, s):
    n, k = p.shape[0], 2 * p.shape[1]
    code = torch.stack((p & 15, p >> 4), 2).view(n, k).double() - 8
    return (code.view(n, s.shape[1], -1) * s.double().unsqueeze(2)).view(n, k)


def _x(m, k, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(m, k, generator=gen, device="cuda").half()


def _close(y, ref):
    err = (y.double() - ref).abs() - 2e-3 * ref.abs()
    assert bool(torch.isfinite(y).all()) and err.max().item() <= 1e-2, err.max().item()


def _form(mats, m, n, k, group):
    """How hn_mid.hip runs a product on 256 CUs: "other" not at all, "waves" K over a
    workgroup's waves, else tiles of 32 or 64 tokens, whole K or split over workgroups."""
    f = _lib.lib().hn_mid_linear_plan
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_int] + [ctypes.c_long] * 4
    r = f(mats, m, n, k, group)
    return {0: "other", -1: "waves"}.get(r) or ("whole" if r & 0xffff == 1 else "split") + str(r >> 16)


@pytest.mark.parametrize("m,n,k,group,form", [
    # K over a workgroup's waves: one stage each, uneven ranges, one row past a tile, two
    # and eight scales a load, columns that fill no tile, up to three rounds of tiles
    (17, 4096, 4096, 128, "waves"), (64, 6144, 4096, 128, "waves"), (65, 100, 1408, 128, "waves"),
    (40, 1408, 1408, 128, "waves"), (333, 4096, 4096, 64, "waves"), (19, 512, 4096, 32, "waves"),
    (512, 1000, 2048, 32, "waves"), (24, 4094, 4096, 128, "waves"), (17, 70, 1024, 128, "waves"),
    (45, 4096, 1408, 128, "waves"), (33, 1030, 2176, 128, "waves"), (49, 100, 2176, 64, "waves"),
    (37, 4096, 14336, 128, "waves"), (127, 4096, 2048, 64, "waves"), (700, 1408, 4096, 128, "waves"),
    (4096, 64, 1024, 32, "waves"),
    # tiles of 32 tokens: one and two row blocks, columns that fill no tile, short K
    (48, 1030, 640, 64, "whole32"), (33, 272, 896, 128, "whole32"), (480, 4096, 2048, 128, "whole32"),
    (481, 4096, 2048, 128, "whole32"), (65, 272, 128, 32, "whole32"),
    # tiles of 64: one to four row blocks of 16
    (200, 4096, 14336, 128, "waves"), (600, 4096, 4096, 64, "whole64"),
    (545, 4094, 4096, 128, "whole64"), (300, 14336, 4096, 128, "whole64"),
    # K over workgroups: even and uneven splits, both tiles
    (37, 512, 14336, 64, "split32"), (150, 1028, 14336, 32, "split32"),
    (333, 4096, 14336, 128, "split64"), (400, 4096, 14336, 128, "split64"),
    (560, 4096, 14336, 64, "split64"), (640, 4096, 11008, 128, "split64"),
    # left to the decode kernels and to the prefill GEMM
    (32, 256, 128, 128, "other"), (20, 256, 768, 128, "other"), (20, 4096, 14336, 128, "other"),
    (1100, 4096, 14336, 64, "other"),
])
def test_linear(m, n, k, group, form):
    print(f"[mid] linear m={m} n={n} k={k} group={group}", flush=True)
    assert _form(1, m, n, k, group) == form
    p, s = _weight(n, k, group, m + n)
    x = _x(m, k, m)
    y = g.int4_linear(x, p, s, group)
    _close(y, x.double() @ _deq(p, s).t())
    assert torch.equal(y, g.int4_linear(x, p, s, group))  # sums in split order: repeatable


@pytest.mark.parametrize("m,n,k,group,form", [
    # several runs of scales per tile: whole K and K splits, 32- and 64-token tiles, an odd
    # number of stages with a short last run, rows of scales that start on any half word
    (520, 2048, 4096, 32, "whole32"), (1030, 2048, 4096, 64, "whole64"),
    (600, 4096, 4096, 64, "whole64"), (700, 4096, 1408, 32, "whole32"),
    (1100, 1030, 2176, 32, "whole32"), (300, 512, 14336, 32, "split32"),
    (100, 512, 11008, 64, "split32"), (530, 2300, 5120, 128, "whole32"), (90, 1000, 17664, 128, "split32"),
])
def test_linear_scale_runs(m, n, k, group, form):
    print(f"[mid] scale runs m={m} n={n} k={k} group={group}", flush=True)
    assert _form(1, m, n, k, group) == form
    p, s = _weight(n, k, group, m + n)
    # every group its own size, so that a scale from another group shows
    s *= (2.0 ** (torch.arange(k // group, device="cuda") * 5 % 7 - 3)).half()
    x = _x(m, k, m)
    y = g.int4_linear(x, p, s, group)
    ref, size = x.double() @ _deq(p, s).t(), x.double().abs() @ _deq(p, s).abs().t()
    # fp32 sums of k products, below group 128 of weights rounded to fp16 (2^-11 each, all one
    # way at worst), one fp16 rounding of the result
    bound = (k * 2.0 ** -23 + (2.0 ** -11 if group < 128 else 0.0)) * size + 2.0 ** -10 * ref.abs() + 1e-6
    assert bool(((y.double() - ref).abs() <= bound).all()), ((y.double() - ref).abs() / bound).max().item()


@pytest.mark.parametrize("t,h,i,group,gate_up,down", [
    (17, 512, 768, 128, "other", "other"), (37, 4096, 14336, 128, "whole32", "waves"),
    (64, 1024, 1408, 64, "waves", "waves"), (130, 640, 2048, 128, "whole32", "waves"),
    (33, 2048, 1408, 128, "waves", "waves"), (47, 2304, 1088, 64, "waves", "other"),
    (1100, 4096, 512, 32, "whole32", "whole32"), (520, 4096, 2048, 128, "whole64", "whole32"),
    (160, 14336, 4096, 128, "split64", "whole64"), (40, 14336, 4096, 32, "split32", "waves"),
])
def test_expert(t, h, i, group, gate_up, down):
    print(f"[mid] expert t={t} h={h} i={i} group={group}", flush=True)
    assert (_form(2, t, i, h, group), _form(1, t, h, i, group)) == (gate_up, down)
    ws = [_weight(a, b, group, 7 + j) for j, (a, b) in enumerate(((i, h), (i, h), (h, i)))]
    x = _x(t, h, t)
    y = g.expert_mlp_int4_fused(x, *[v for w in ws for v in w], group_size=group)
    dg, du, dd = (_deq(*w) for w in ws)
    hid = torch.nn.functional.silu(x.double() @ dg.t()) * (x.double() @ du.t())
    _close(y, hid @ dd.t())


def _layer(e, h, i, seed):
    from hydranet_amd.preprocess.synthetic import make_expert_slot
    return [make_expert_slot(seed + j, h, i, 128, slot_idx=j) for j in range(e)]


def _expert_sum(x, idx, w, slots):
    """sum_k w[t, k] * expert idx[t, k] of x[t] in float64; idx and w on the CPU."""
    ref = torch.zeros(x.shape, dtype=torch.float64, device="cuda")
    for j, s in enumerate(slots):
        rows, slot = (idx == j).nonzero(as_tuple=True)
        if len(rows):
            xe = x[rows.cuda()].double()
            hid = torch.nn.functional.silu(xe @ _deq(s.gate_packed, s.gate_scales).t()) * (
                xe @ _deq(s.up_packed, s.up_scales).t())
            y = hid @ _deq(s.down_packed, s.down_scales).t()
            ref.index_add_(0, rows.cuda(), y * w[rows, slot].double().cuda().unsqueeze(1))
    return ref


@pytest.mark.parametrize("e,h,i,tokens,k", [
    (8, 512, 2048, 70, 2),     # down in one piece, over 64 tokens
    (8, 512, 6144, 60, 2),     # 48 stages: the down projection in K slices
    (4, 512, 2048, 300, 2),    # 150 rows per expert: past these kernels, the prefill GEMM
    (16, 256, 1408, 90, 4),    # ragged I
])
def test_experts_uneven(e, h, i, tokens, k):
    """Experts with no rows, one row, and most of the rows."""
    print(f"[mid] experts e={e} h={h} i={i} tokens={tokens} k={k}", flush=True)
    slots = _layer(e, h, i, 11)
    table = moe.ExpertTable.from_slots(slots)
    gen = torch.Generator().manual_seed(e + tokens)
    p = torch.tensor([0.0, 1e-4] + [2.0 ** -j for j in range(e - 2)]) + 1e-9
    idx = torch.multinomial(p.expand(tokens, e), k, generator=gen)
    idx[idx == 0] = e - 1                      # expert 0: no rows (duplicates are allowed)
    w = torch.rand(tokens, k, generator=gen).half()
    x = _x(tokens, h, 3)
    out = moe.moe_experts_forward(x, idx.int().cuda(), w.cuda(), table)
    ref = _expert_sum(x, idx, w, slots)
    # k roundings of the weighted rows and of their fp16 sum beside the products' own
    _close(out / k, ref / k)


def test_route_ignores_the_size_of_the_workspace():
    """16384 rows of 512 columns in four fp32 slices are more than the prefill workspace
    holds; a larger buffer left by another call changes neither the kernel nor a bit."""
    table = moe.ExpertTable.from_slots(_layer(128, 512, 4608, 3))
    gen = torch.Generator().manual_seed(4)
    idx = torch.randint(0, 128, (8192, 2), generator=gen, dtype=torch.int32).cuda()
    w = torch.rand(8192, 2, generator=gen).half().cuda()
    x = _x(8192, 512, 8)
    kept = dict(_lib._WORKSPACES)
    try:
        _lib._WORKSPACES.clear()
        want = moe.moe_experts_forward(x, idx, w, table)
        _lib.workspace(160 << 20, x.device)
        assert torch.equal(moe.moe_experts_forward(x, idx, w, table), want)
    finally:
        torch.cuda.synchronize()
        _lib._WORKSPACES.clear()
        _lib._WORKSPACES.update(kept)


@pytest.mark.parametrize("t,k,i", [(96, 2, 2048), (96, 2, 6144), (33, 4, 2048)])
def test_layer_graph_replay(t, k, i):
    """The layer's launches captured once and replayed: every replay as the eager run, and
    that as the float64 sum over the experts it routed to."""
    print(f"[mid] graph t={t} k={k} i={i}", flush=True)
    slots = _layer(8, 512, i, 5)
    layer = moe.MixtralMoELayer(512, 8, k, slots=slots).cuda().half().eval()
    x = _x(t, 512, 9).view(1, t, 512)
    with torch.no_grad():
        want = layer(x, top_k=k).clone()
        idx, w = (r.cpu() for r in layer.last_routing)
        _close(want[0] / k, _expert_sum(x[0], idx, w, slots) / k)
        st = torch.cuda.Stream()
        st.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(st):
            layer(x, top_k=k)
        torch.cuda.current_stream().wait_stream(st)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = layer(x, top_k=k)
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
            assert torch.equal(layer(x, top_k=k), want)
