"""The coalesced quantiser kernel (contiguous rows) against the general one (reached
with a padded row stride), byte for byte: group sizes, remainders of a block,
every quotient of two 11-bit significands, and groups of zeros, subnormals,
infinities and NaN; and against the oracle for finite inputs."""
import numpy as np
import pytest
import torch

import oracle
from hydranet_amd import _lib

pytestmark = pytest.mark.gpu


def _quant(w, group, mode, pad):
    n, k = w.shape
    src = torch.zeros(n, k + pad, dtype=w.dtype, device="cuda")
    src[:, :k] = w
    p = torch.zeros(n, k // 2, dtype=torch.uint8, device="cuda")
    s = torch.zeros(n, k // group, dtype=torch.float16, device="cuda")
    _lib.call("hn_int4_quantize", _lib.ptr(src), k + pad, 0 if w.dtype == torch.float16 else 1,
              mode, _lib.ptr(p), k // 2, _lib.ptr(s), k // group, n, k, group, _lib.stream())
    return p, s.view(torch.int16)


def _same(w, group, mode):
    a, b = _quant(w, group, mode, 0), _quant(w, group, mode, 8)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    return a


@pytest.mark.parametrize("mode,dtype", [(0, torch.float16), (1, torch.float16),
                                        (1, torch.float32)])
@pytest.mark.parametrize("n,k,group", [(1, 8, 8), (3, 96, 32), (7, 1408, 128), (129, 4096, 64),
                                       (5, 1024, 512), (2, 288, 96), (33, 80, 16)])
def test_rows_equal_general(mode, dtype, n, k, group):
    print(f"[quant] n={n} k={k} group={group} mode={mode} {dtype}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(n * k)
    w = torch.randn(n, k, generator=gen, device="cuda").mul_(0.02).to(dtype)
    p, s = _same(w, group, mode)
    pr, sr = oracle.quantize(w.cpu().numpy(), group, mode)
    assert np.array_equal(p.cpu().numpy(), pr)
    assert np.array_equal(s.cpu().numpy().view(np.uint16), sr.view(np.uint16))


@pytest.mark.parametrize("mode", [0, 1])
def test_every_significand_pair(mode):
    """Group i: an absmax of significand 1024 + i (mode 0: 7 times it, so the scale
    is that) and every 11-bit significand below it, at three exponents."""
    div = torch.arange(1024, 2048, device="cuda").double()
    top = (div * (7 if mode == 0 else 1)).half().double()  # rounds; the scale follows it
    val = torch.arange(1024, 2048, device="cuda").double()
    w = torch.empty(1024, 25, 128, device="cuda", dtype=torch.float64)
    for e, scale in enumerate((1.0, 0.5, 0.25)):
        v = torch.minimum((val * scale).expand(1024, -1), top.unsqueeze(1))
        w[:, 8 * e:8 * e + 8] = torch.cat([v[:, :1016].view(1024, 8, 127),
                                           top.view(-1, 1, 1).expand(-1, 8, 1)], 2)
    w[:, 24] = torch.cat([-val[1016:].expand(1024, -1).minimum(top.unsqueeze(1)),
                          top.unsqueeze(1).expand(-1, 120)], 1)
    for shift in (-10, -14, -24):
        x = (w * 2.0 ** shift).half().view(1024, -1)
        _same(x, 128, mode)


@pytest.mark.parametrize("mode,dtype", [(0, torch.float16), (1, torch.float16),
                                        (1, torch.float32)])
def test_special_groups(mode, dtype):
    gen = torch.Generator(device="cuda").manual_seed(1)
    w = torch.randn(16, 4, 64, generator=gen, device="cuda")
    w[0] = 0
    w[1] *= 1e-7           # fp16 subnormals: scales of a few units, or zero
    w[2, :, 5] = float("inf")
    w[3, :, 9] = -float("inf")
    w[4, :, 0] = float("nan")
    w[5] = float("nan")
    w[6] *= 3e4            # near the largest fp16
    w[7, :, 1:] = 0        # one value
    w[8] = -w[8].abs()
    w[9] *= 2e-8           # rounds to zero or one unit in fp16
    _same(w.to(dtype).view(16, 256), 64, mode)
