"""Routing whose logits run as a launch of their own (hn_moe_route past the MFMA
logits' sizes): bit for bit the routing given those logits."""
import pytest
import torch

from hydranet_amd.model import moe

pytestmark = pytest.mark.gpu


def _x(m, k, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(m, k, generator=gen, device="cuda").half()


@pytest.mark.parametrize("t,e,k", [(65, 8, 2), (100, 8, 2), (40, 16, 4), (500, 8, 1)])
def test_route_logits_apart(t, e, k):
    """Routing whose logits run as a launch of their own: bit for bit the routing
    given those logits, and hn_router_logits' bits."""
    print(f"[mid] route t={t} e={e} k={k}", flush=True)
    h = _x(t, 512, t)
    gate = (_x(e, 512, 5) * 0.1).half()
    a = moe.moe_route(h, k, 0, gate_w=gate)
    logits = moe.router_logits(h, gate)
    b = moe.moe_route(h, k, 0, logits=logits)
    assert torch.equal(a.logits, logits)
    for name in ("idx", "w", "offsets", "perm", "inv", "x_perm", "n_active"):
        assert torch.equal(getattr(a, name), getattr(b, name)), name
