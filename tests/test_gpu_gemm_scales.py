"""GPU test of the prefill GEMM's scale runs (hn_gemm.hip): eight groups of a
row loaded at once, by rows that start on any half word, with whole and partial
last runs, whole tiles and stream-K segments, against an fp32 product over the
oracle's dequantised weights."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from hydranet_amd import _lib

DEV = "cuda:0"
L, P = ctypes.c_long, ctypes.c_void_p


def _gemm(x, p, s, out, N, K, g, work):
    f = _lib.lib().hn_gemm_linear_impl
    f.restype = ctypes.c_int
    f.argtypes = [ctypes.c_int, P, L, P, P, P, P, L, L, P, L, L, L, L, L, P, L, P]
    st = torch.cuda.current_stream().cuda_stream
    return f(1, x.data_ptr(), x.stride(0), p.data_ptr(), s.data_ptr(), None, None, p.stride(0),
             s.stride(0), out.data_ptr(), out.stride(0), x.shape[0], N, K, g,
             None if work is None else work.data_ptr(), 0 if work is None else work.numel(), st)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,g,pad", [
    (65, 9, 128, 128, 0),       # 18 bytes of scales in all
    (70, 33, 11 * 128, 128, 0), # odd row stride, a run and three groups
    (130, 300, 17 * 128, 128, 0), (90, 64, 16 * 128, 128, 3), (300, 257, 640, 64, 0),
    (66, 100, 9 * 64, 64, 1), (65, 40, 320, 32, 0), (65, 70, 448, 32, 3),
    (80, 64, 9 * 192, 192, 0), (80, 64, 1024, 1024, 0), (257, 520, 4096, 128, 0),
])
def test_gemm_scale_runs(M, N, K, g, pad):
    gen = torch.Generator().manual_seed(M + K)
    w = (torch.randn(N, K, generator=gen) * 0.02).half()
    # every group its own size, so that a scale from another group shows
    w *= (2.0 ** (torch.arange(K // g) * 5 % 7 - 3)).repeat_interleave(g).half()
    x = torch.randn(M, K, generator=gen).half().to(DEV)
    q, sc = oracle.quantize(w.numpy(), g, mode=0)
    ref = x.float() @ torch.from_numpy(oracle.dequant(q, sc, g).astype(np.float32)).to(DEV).t()
    size = x.float().abs() @ torch.from_numpy(
        np.abs(oracle.dequant(q, sc, g)).astype(np.float32)).to(DEV).t()
    p = torch.from_numpy(q).to(DEV)
    s = torch.full((N, K // g + pad), float("nan"), dtype=torch.float16)
    s[:, :K // g] = torch.from_numpy(sc.copy())
    s = s.to(DEV)
    for work in (None, _lib.gemm_workspace(DEV)):
        out = torch.full((M, N), 7.0, dtype=torch.float16, device=DEV)
        assert _gemm(x, p, s, out, N, K, g, work) == 0
        # fp32 sums of K exact products (K 2^-24 of their sizes on either side),
        # one fp16 rounding
        bound = 2 * K * 2.0 ** -24 * size + 2.0 ** -10 * ref.abs() + 1e-6
        err = (out.float() - ref).abs()
        assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,g", [(65, 33, 11 * 128, 128), (130, 300, 17 * 128, 128),
                                     (66, 101, 9 * 64, 64), (65, 41, 320, 32), (257, 520, 4096, 128)])
@pytest.mark.parametrize("view", ["odd", "right"])
def test_gemm_scales_of_a_view(M, N, K, g, view):
    """Scales that start on the second half of a dword, and scales that are the last
    columns of a wider matrix (whose last row ends where the memory does)."""
    print(f"[scales] {view} M={M} N={N} K={K} g={g}", flush=True)
    gen = torch.Generator().manual_seed(M + K)
    w = (torch.randn(N, K, generator=gen) * 0.02).half()
    w *= (2.0 ** (torch.arange(K // g) * 5 % 7 - 3)).repeat_interleave(g).half()
    x = torch.randn(M, K, generator=gen).half().to(DEV)
    q, sc = oracle.quantize(w.numpy(), g, mode=0)
    deq = torch.from_numpy(oracle.dequant(q, sc, g).astype(np.float32)).to(DEV)
    p, kg = torch.from_numpy(q).to(DEV), K // g
    if view == "odd":
        s = torch.full((N * kg + 1,), float("nan"), dtype=torch.float16, device=DEV)[1:].view(N, kg)
        assert s.data_ptr() % 4 == 2
    else:
        s = torch.full((N, kg + 9), float("nan"), dtype=torch.float16, device=DEV)[:, 9:]
    s.copy_(torch.from_numpy(sc.copy()))
    ref = x.float() @ deq.t()
    bound = 2 * K * 2.0 ** -24 * (x.float().abs() @ deq.abs().t()) + 2.0 ** -10 * ref.abs() + 1e-6
    for work in (None, _lib.gemm_workspace(DEV)):
        out = torch.full((M, N), 7.0, dtype=torch.float16, device=DEV)
        assert _gemm(x, p, s, out, N, K, g, work) == 0
        assert bool(((out.float() - ref).abs() <= bound).all())


@pytest.mark.parametrize("ld_s,kg,odd", [(1, 1, 0), (1, 1, 2), (3, 3, 2), (11, 11, 0), (11, 11, 2),
                                         (40, 31, 0), (40, 31, 2), (32, 32, 2)])
@pytest.mark.parametrize("N", [9, 33, 100])
def test_scale_loads_stay_in_the_matrix(ld_s, kg, odd, N):
    """The byte ranges of the kernel's scale loads (its own arithmetic, on the host): every
    16 bytes from the dword of the first scale to the dword of the last, every scale that is
    read back inside what was loaded for it, whole tiles and later segments."""
    for first in range(0, kg, 2):                      # a segment's first group
        addr = 64 + odd + 2 * first                    # of the segment's first scale
        base = addr & ~3
        end = odd + 64 + 2 * ((N - 1) * ld_s + kg)     # past the last scale
        ns = ((addr & 2) + 2 * ((N - 1) * ld_s + kg - first) + 3) & ~3
        if ns < 16:
            continue                                   # not taken
        for row in {0, 1, N // 2, N - 2, N - 1}:
            vs = (addr & 2) + 2 * row * ld_s
            for g in range(kg - first):
                src = min((vs + 2 * (g & ~3)) & ~3, ns - 16)
                assert (64 + odd) & ~3 <= base + src and base + src + 16 <= (end + 3) & ~3
                assert 0 <= vs + 2 * g - src <= 14


@pytest.mark.gpu
@pytest.mark.parametrize("mats", [1, 2])
@pytest.mark.parametrize("M,N,K,g", [
    (1000, 8, 10240, 512), (70, 1, 4096, 4096), (300, 2, 8192, 4096), (65, 6, 4096, 4096),
    (130, 7, 4096, 4096), (200, 1, 10240, 512), (66, 3, 2048, 1024), (100, 8, 4096, 128),
])
def test_few_scales_need_no_workspace(M, N, K, g, mats):
    """More than 64 rows of a product with few columns and a handful of scales, with no
    workspace and with the prefill one."""
    print(f"[scales] few M={M} N={N} K={K} g={g} mats={mats}", flush=True)
    gen = torch.Generator().manual_seed(M + K)
    x = (torch.randn(M, K, generator=gen) * 0.25).half().to(DEV)
    deq, ptrs = [], []
    for _ in range(mats):
        q, sc = oracle.quantize((torch.randn(N, K, generator=gen) * 0.02).half().numpy(), g, mode=0)
        deq.append(torch.from_numpy(oracle.dequant(q, sc, g).astype(np.float32)).to(DEV))
        ptrs += [torch.from_numpy(q).to(DEV), torch.from_numpy(sc.copy()).to(DEV)]
    prod = [x.float() @ d.t() for d in deq]
    ref = prod[0] if mats == 1 else torch.nn.functional.silu(prod[0].half().float()) * prod[1].half().float()
    for work in (None, _lib.gemm_workspace(DEV)):
        out = torch.full((M, N), 7.0, dtype=torch.float16, device=DEV)
        tail = (_lib.ptr(out), N, M, N, K, g, _lib.ptr(work), 0 if work is None else work.numel(),
                _lib.stream())
        if mats == 1:
            _lib.call("hn_int4_linear", _lib.ptr(x), K, _lib.ptr(ptrs[0]), K // 2, _lib.ptr(ptrs[1]),
                      K // g, *tail)
        else:
            _lib.call("hn_int4_gate_up_silu", _lib.ptr(x), K, *[_lib.ptr(t) for t in ptrs], K // 2,
                      K // g, *tail)
        # the repository's bar for fp16 outputs
        assert bool(((out.float() - ref).abs() <= 1e-2 + 2e-3 * ref.abs()).all())
