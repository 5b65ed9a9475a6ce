"""Which steps of latent attention go to lv_latent_prompt_attn: none that the entry would refuse."""
import types

import pytest
import torch

from light_vllm_amd import mix_ops


def ok(lens, scale=0.1, H=4):
    bf16 = dict(dtype=torch.bfloat16)
    return mix_ops.latent_prompt_ok(torch.empty(40, H * 128, **bf16), torch.empty(2, 64, 256, **bf16), torch.empty(H, 64, 192, **bf16), torch.empty(H, 192, 64, **bf16),
                                    torch.empty(40, H, **bf16), types.SimpleNamespace(host_lens_q=lens, host_ctx_lens=[0] * len(lens)), H, 64, 64, 192, 64, False, scale)


@pytest.mark.parametrize("scale", [0.0, -0.1, float("nan")])
def test_scales_that_are_not_positive_stay_with_the_batched_products(scale):
    assert ok([17, 1]) and not ok([16, 1]) and not ok([])
    assert not ok([17, 1], scale)


def test_launches_of_two_to_the_31_workgroups_stay_with_the_batched_products():
    assert ok([32 << 25] + [0] * 62) and not ok([32 << 25] + [0] * 63)
    assert ok([32 << 25] + [0] * 30, H=8) and not ok([32 << 25] + [0] * 31, H=8)


@pytest.mark.parametrize("decoded,ctx,prompts,H,Dn,R,pays", [
    (0, 0, [17], 32, 128, 256, True), (31, 4000, [16384], 16, 128, 192, True), (250, 200, [1000, 1000], 16, 128, 192, True), (400, 100, [100], 16, 128, 192, False),
    (400, 100, [100], 32, 128, 256, False), (1000, 100, [1000], 16, 128, 256, False), (1000, 1000, [100], 16, 128, 256, True), (1000, 100, [1000], 16, 64, 256, True),
    (700, 300, [4000], 32, 128, 192, True)])
def test_where_one_launch_pays_beside_many_short_sequences(decoded, ctx, prompts, H, Dn, R, pays):
    step = types.SimpleNamespace(host_lens_q=[1] * decoded + prompts, host_ctx_lens=[ctx] * decoded + [0] * len(prompts))
    assert mix_ops._latent_prompt_pays(step, decoded + sum(prompts), H, Dn, R) == pays
