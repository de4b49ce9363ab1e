"""GPU tests of the routing kernels' forms for many tokens: logits by tiles of 4
tokens x 4 experts against one dot product per wave (same bits), the counting
sort's prefix sums over up to 256 experts, and the unpermute's sorted list."""
import pytest
import torch

from hydranet_amd import _lib
from hydranet_amd.model import moe

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,E,H,fp32", [(2048, 8, 512, False), (2731, 6, 520, False),
                                        (129, 128, 1024, True), (65, 253, 8, True)])
def test_router_logits_tiles(T, E, H, fp32):
    g = torch.Generator(device=DEV).manual_seed(T)
    h = torch.randn(T, H, generator=g, device=DEV).half()
    w = torch.randn(E, H, generator=g, device=DEV) * 0.05
    w = w if fp32 else w.half()
    got = moe.router_logits(h, w)
    assert T * E >= 16384
    step = 16383 // E  # few enough products for the other kernel
    want = torch.cat([moe.router_logits(h[i:i + step].contiguous(), w) for i in range(0, T, step)])
    assert torch.equal(got, want)


@pytest.mark.parametrize("n,E", [(3000, 256), (1025, 129), (5, 256), (64, 1), (4000, 128)])
def test_permute_prefix_sums(n, E):
    g = torch.Generator().manual_seed(n)
    idx = torch.randint(-1, E + 1, (n,), generator=g, dtype=torch.int32)
    idx[idx % 5 == 3] = 0  # experts with no rows, and entries outside [0, E)
    d = idx.to(DEV)
    off, perm, inv = (torch.full((m,), 77, dtype=torch.int32, device=DEV) for m in (E + 1, n, n))
    act, na = torch.full((E,), 77, dtype=torch.int32, device=DEV), torch.zeros(
        1, dtype=torch.int32, device=DEV)
    _lib.call("hn_moe_permute", _lib.ptr(d), n, 1, E, _lib.ptr(off), _lib.ptr(perm),
              _lib.ptr(inv), _lib.ptr(act), _lib.ptr(na), _lib.stream())
    cnt = torch.tensor([(idx == e).sum() for e in range(E)])
    assert torch.equal(off.cpu().long(), torch.cat([torch.zeros(1, dtype=torch.long), cnt.cumsum(0)]))
    want = torch.cat([torch.nonzero(idx == e)[:, 0] for e in range(E)])
    assert torch.equal(perm[:len(want)].cpu().long(), want)
    pos = torch.full((n,), -1, dtype=torch.long)
    pos[want] = torch.arange(len(want))
    assert torch.equal(inv.cpu().long(), pos)
    hit = torch.nonzero(cnt)[:, 0]
    assert na.item() == len(hit) and torch.equal(act[:len(hit)].cpu().long(), hit)


@pytest.mark.parametrize("T,k,shared", [(3, 1, False), (70, 2, True), (5, 3, False),
                                        (65, 8, True), (7, 9, False), (66, 16, True)])
def test_unpermute_order_and_drops(T, k, shared):
    """fp16 accumulation in ascending expert id (equal ids in assignment order),
    dropped assignments (inv < 0) left out, a token with none of its own."""
    H, E = 264, 20
    g = torch.Generator().manual_seed(k)
    idx = torch.randint(0, E, (T, k), generator=g, dtype=torch.int32)
    inv = torch.randperm(T * k, generator=g).int().view(T, k)
    inv[torch.rand(T, k, generator=g) < 0.2] = -1
    inv[T // 2] = -1
    w = torch.rand(T, k, generator=g).half()
    y = torch.randn(T * k, H, generator=g).half()
    sh = torch.randn(T, H, generator=g).half()
    out = torch.empty(T, H, dtype=torch.float16, device=DEV)
    dev = [t.to(DEV).contiguous() for t in (y, inv, idx, w, sh)]
    _lib.call("hn_moe_unpermute", _lib.ptr(dev[0]), H, _lib.ptr(dev[1]), _lib.ptr(dev[2]),
              _lib.ptr(dev[3]), T, k, _lib.ptr(dev[4]) if shared else None, H, _lib.ptr(out), H, H,
              _lib.stream())
    want = torch.zeros(T, H, dtype=torch.float16)
    for t in range(T):
        for s in sorted(range(k), key=lambda s: int(idx[t, s])):
            if inv[t, s] >= 0:
                want[t] += (y[inv[t, s]].float() * w[t, s].float()).half()
    if shared:
        want = sh + want
    assert torch.equal(out.cpu(), want)
