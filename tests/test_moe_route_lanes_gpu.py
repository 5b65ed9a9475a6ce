"""lv_moe_route_scored with 16, 32 and 64 lanes a token against the torch path, at the edges of each and with part of a wave's tokens."""
import pytest
import torch

from light_vllm_amd import mix_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,groups,top,keep", [(1, 1, 1, 1), (15, 3, 4, 2), (16, 4, 2, 2), (17, 1, 17, 1), (31, 1, 3, 1), (32, 4, 4, 2), (32, 32, 5, 7), (33, 3, 4, 1), (65, 5, 8, 3)])
@pytest.mark.parametrize("score,group_rank", [("sigmoid", "top2"), ("softmax", "max")])
def test_choices_and_weights(E, groups, top, keep, score, group_rank):
    gen = torch.Generator().manual_seed(E)
    for T in (1, 3, 4, 9, 67):
        # distinct scores 0.03 apart and more: neither path's rounding can change an order
        logits = (torch.stack([torch.randperm(E, generator=gen) for _ in range(T)]).float() - E / 2) * (4.0 / E) + 0.01 * torch.rand(T, 1, generator=gen)
        correction = torch.zeros(E)
        want = mix_ops.moe_route(logits, correction, top, groups, keep, score=score, group_rank=group_rank)
        got = mix_ops.moe_route(logits.cuda(), correction.cuda(), top, groups, keep, score=score, group_rank=group_rank)
        assert torch.equal(got[0].cpu().int(), want[0].int())
        for x, y in zip(got[1:], want[1:]):        # sums of up to 65 f32 terms, an exponential and a division on either side
            assert torch.allclose(x.cpu(), y, rtol=2.0 ** -18, atol=1e-9)
