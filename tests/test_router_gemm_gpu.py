"""Router logits (mix_ops.router_product, f32 products of widened bf16 activations) against float64: sizes around 64 rows, rows of a wider
tensor, values that are not finite."""
import pytest
import torch
import torch.nn.functional as F

from light_vllm_amd import mix_ops

pytestmark = pytest.mark.gpu


@torch.inference_mode()
@pytest.mark.parametrize("T", [1, 63, 64, 65, 300])
@pytest.mark.parametrize("E,K,pad", [(1, 32, 0), (8, 96, 8), (32, 2048, 0), (33, 544, 0), (256, 1024, 16)])
def test_against_float64(T, E, K, pad):
    gen = torch.Generator(device="cuda").manual_seed(T + E)
    h = torch.randn(T, K + pad, device="cuda", generator=gen).bfloat16()[:, pad:]
    w = torch.randn(E, K, device="cuda", generator=gen) * K ** -0.5
    ref = h.double() @ w.double().t()
    got, vendor = mix_ops.router_product(h, w), F.linear(h.float(), w)
    # K f32 additions in chains, each half a unit of the sum so far
    assert bool(((got.double() - ref).abs() <= K * 2.0 ** -24 * (h.double().abs() @ w.double().abs().t())).all())
    err = lambda x: float((x.double() - ref).norm() / ref.norm())    # noqa: E731
    assert err(got) <= max(1.1 * err(vendor), 2.0 ** -24)


@torch.inference_mode()
def test_values_that_are_not_finite():
    gen = torch.Generator(device="cuda").manual_seed(3)
    h = torch.randn(70, 256, device="cuda", generator=gen).bfloat16()
    w = torch.randn(40, 256, device="cuda", generator=gen)
    h[5, 17], h[66, 3], w[33, 8], w[2, 100] = float("inf"), float("nan"), -float("inf"), 3.4e38
    got, want = mix_ops.router_product(h, w), F.linear(h.double(), w.double())
    want = torch.where(want.abs() > torch.finfo(torch.float32).max, torch.copysign(torch.tensor(float("inf"), device="cuda").double(), want), want)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    plain = [i for i in range(40) if i != 2]              # column 2 may overflow on the way to a finite sum
    assert torch.equal(torch.isinf(got[:, plain]), torch.isinf(want[:, plain]))
