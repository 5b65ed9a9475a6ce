"""SparseMoE's router: logits are the f32 product of the widened activations whatever the step's size, the experts chosen are float64's but
where two scores lie within the bound of the sums, and gradients pass through the logits."""
import pytest
import torch
import torch.nn.functional as F

from light_vllm_amd import mix_ops
from light_vllm_amd.layers.moe import SparseMoE

pytestmark = pytest.mark.gpu
TOP = 4


def router(monkeypatch, T, E, W, seed=1):
    """(module, bf16 activations, list that takes the logits of every route)"""
    old = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        m = SparseMoE(W, 32, E, TOP).to("cuda")
    finally:
        torch.set_default_dtype(old)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    m.router_weight.data.normal_(0.0, W ** -0.5, generator=gen)
    m.correction.data.normal_(0.0, 0.1, generator=gen)
    h = torch.empty(T, W, dtype=torch.bfloat16, device="cuda").normal_(generator=gen)
    seen, choose = [], mix_ops.moe_route
    monkeypatch.setattr(mix_ops, "moe_route", lambda logits, *a, **k: seen.append(logits) or choose(logits, *a, **k))
    return m, h, seen


@torch.inference_mode()
@pytest.mark.parametrize("T", [1, 16, 256, 257, 1500, 5000])
@pytest.mark.parametrize("E,W", [(32, 2048), (33, 544)])
def test_logits_and_choice(monkeypatch, T, E, W):
    m, h, seen = router(monkeypatch, T, E, W)
    ids, weights, _ = m.route(h)
    assert torch.equal(seen[0], F.linear(h.float(), m.router_weight))
    exact = h.double() @ m.router_weight.double().t()
    score = torch.sigmoid(exact)
    c = score + m.correction.double()
    # W f32 additions in chains, each half a unit of the sum so far, through a slope of at most 1/4; and a score's own few roundings
    bound = (W * 2.0 ** -24 * (h.double().abs() @ m.router_weight.double().abs().t())).amax(1) / 4 + 2.0 ** -21
    chosen = torch.zeros_like(c, dtype=torch.bool).scatter_(1, ids.long(), True)
    assert bool((chosen.sum(1) == TOP).all())
    least = c.masked_fill(~chosen, float("inf")).amin(1)
    assert bool((least >= c.masked_fill(chosen, -float("inf")).amax(1) - 2 * bound).all())
    s = score.gather(1, ids.long())
    assert bool(((weights.double() - s / s.sum(1, keepdim=True)).abs() <= 4 * bound[:, None] + 2.0 ** -20).all())


@pytest.mark.parametrize("T", [8, 256, 300])
def test_gradients_pass_through_the_logits(monkeypatch, T):
    m, h, seen = router(monkeypatch, T, 32, 512)
    h.requires_grad_()
    with torch.enable_grad():
        logits = mix_ops.router_product(h, m.router_weight)
        m.route(h)
        assert seen[0].requires_grad
        for x in (logits, seen[0]):
            x.square().sum().backward()
            logits_grads = (h.grad.clone(), m.router_weight.grad.clone())
            h.grad = m.router_weight.grad = None
            seen.append(logits_grads)
    assert all(torch.equal(a, b) for a, b in zip(*seen[-2:]))
