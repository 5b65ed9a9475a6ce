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


def tiles(h, w):
    from light_vllm_amd import _mixlib
    out = torch.empty(h.size(0), w.size(0), device="cuda")
    _mixlib.check(_mixlib.load().lv_router_tiles(h.data_ptr(), h.stride(0), w.data_ptr(), out.data_ptr(), h.size(0), h.size(1), w.size(0),
                                                 torch.cuda.current_stream().cuda_stream), "lv_router_tiles")
    return out


# the kernel by itself: rows around its 64, widths of one and more turns of its loop, every count of experts, rows of a wider tensor
@torch.inference_mode()
@pytest.mark.parametrize("T", [1, 63, 64, 65, 16447])
@pytest.mark.parametrize("E,K,pad", [(16, 256, 0), (32, 2304, 8), (48, 768, 0), (64, 512, 64)])
def test_tiles_against_float64(T, E, K, pad):
    gen = torch.Generator(device="cuda").manual_seed(T + E)
    h = torch.randn(T, K + pad, device="cuda", generator=gen).bfloat16()[:, pad:]
    w = torch.randn(E, K, device="cuda", generator=gen) * K ** -0.5
    ref = h.double() @ w.double().t()
    assert bool(((tiles(h, w).double() - ref).abs() <= K * 2.0 ** -24 * (h.double().abs() @ w.double().abs().t())).all())
    few = slice(0, min(T, 20))                            # a token's logits do not depend on the others
    assert torch.equal(tiles(h[few], w), tiles(h, w)[few])


# where router_product takes it, the vendor's bits: nearly tied experts stay in their order
@torch.inference_mode()
@pytest.mark.parametrize("T,E,K,pad", [(4500, 32, 512, 0), (4999, 32, 1024, 8), (4501, 32, 2048, 0), (16384, 32, 2048, 0), (6000, 32, 4096, 0),
                                       (9000, 64, 1024, 0), (12345, 64, 2048, 16)])
def test_bits_of_the_product_it_stands_in_for(T, E, K, pad):
    gen = torch.Generator(device="cuda").manual_seed(T + E)
    h = torch.randn(T, K + pad, device="cuda", generator=gen).bfloat16()[:, pad:]
    w = torch.randn(E, K, device="cuda", generator=gen) * K ** -0.5
    h[7, 9], h[300, 5], w[3, 8] = float("inf"), float("nan"), -float("inf")
    assert mix_ops.router_tiles_ok(h, w)
    got, want = mix_ops.router_product(h, w), F.linear(h.float(), w)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got.nan_to_num(0.0, 1.0, -1.0), want.nan_to_num(0.0, 1.0, -1.0))


def test_which_calls_take_the_tiles():
    h = torch.randn(5000, 1024, device="cuda").bfloat16()
    w = torch.randn(32, 1024, device="cuda")
    ok = mix_ops.router_tiles_ok
    with torch.inference_mode():
        assert ok(h, w)
    wide = torch.randn(5000, 1028, device="cuda").bfloat16()
    for a, b in [(h[:4499], w), (h.float(), w), (wide[:, :1024], w), (h[:, ::2].expand(5000, 512), w[:, :512].contiguous()), (h, w[:16]),
                 (h, w.t().contiguous().t()), (h.view(5, 1000, 1024), w), (h.clone().requires_grad_(), w), (h, w.clone().requires_grad_())]:
        assert not ok(a, b)
        assert torch.equal(mix_ops.router_product(a, b), F.linear(a.float(), b))


# the corners of the ranges, and counts just beyond, where the vendor's product sums in another order: the product itself
@torch.inference_mode()
@pytest.mark.parametrize("T,E,K,taken", [(4500, 32, 1024, True), (32768, 32, 512, True), (32767, 32, 1024, True), (24001, 32, 2048, True), (32768, 32, 4096, True), (9000, 64, 512, True),
                                         (16384, 64, 512, True), (16384, 64, 1024, True), (16383, 64, 2048, True), (16384, 64, 4096, True), (9000, 64, 4096, True),
                                         (16385, 64, 4096, False), (16448, 64, 512, False), (16448, 64, 1024, False), (16448, 64, 2048, False), (18496, 64, 4096, False)])
def test_bits_at_the_corners(T, E, K, taken):
    gen = torch.Generator(device="cuda").manual_seed(T + K)
    h = torch.randn(T, K, device="cuda", generator=gen).bfloat16()
    w = torch.randn(E, K, device="cuda", generator=gen) * K ** -0.5
    assert mix_ops.router_tiles_ok(h, w) == taken
    assert torch.equal(mix_ops.router_product(h, w), F.linear(h.float(), w))
