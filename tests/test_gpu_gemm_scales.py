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

pytestmark = pytest.mark.gpu
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
