"""The weighted sum of expert rows: accesses of 16 and of 8 bytes, counts of choices beside four, choices that hand the token through."""
import pytest
import torch

from light_vllm_amd import mix_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,W,top,weighted,through,offset", [
    (1, 8, 1, True, False, 0), (3, 4, 4, True, False, 0), (5, 36, 3, False, False, 0), (70, 520, 5, True, True, 0),
    (33, 2048, 4, True, True, 4), (9, 2056, 8, False, False, 0), (17, 4104, 9, True, True, 0), (40, 2052, 2, True, True, 0)])
def test_sum_matches_float64(gpu, T, W, top, weighted, through, offset):
    g = torch.Generator().manual_seed(T * W + top)
    def act(n):
        flat = torch.empty(n * W + offset, dtype=torch.bfloat16)
        flat.copy_(torch.randn(n * W + offset, generator=g))
        return flat.to(gpu)[offset:].view(n, W)
    rows, h = act(T * top), act(T)
    inv = torch.randperm(T * top, generator=g).to(torch.int32).view(T, top).to(gpu)
    weights = torch.rand(T, top, generator=g).to(gpu) if weighted else None
    ids = torch.randint(0, 6, (T, top), generator=g, dtype=torch.int32).to(gpu) if through else None
    out = mix_ops.moe_combine(rows, inv, weights, ids, 4, h if through else None)
    picked = rows[inv.long()].double()
    if through:
        picked = torch.where((ids >= 4)[:, :, None], h.double()[:, None, :], picked)
    parts = picked * weights.double()[:, :, None] if weighted else picked
    # one rounding to bf16 (2^-9 of the sum) and `top` f32 roundings of partial sums of at most the sum of magnitudes
    bound = parts.sum(1).abs() * 2.0 ** -8 + parts.abs().sum(1) * top * 2.0 ** -23
    assert ((out.double() - parts.sum(1)).abs() <= bound).all()
