"""Which steps of latent attention go to lv_latent_prompt_attn: none that the entry would refuse."""
import types

import pytest
import torch

from light_vllm_amd import mix_ops


def ok(lens, scale=0.1, H=4):
    bf16 = dict(dtype=torch.bfloat16)
    return mix_ops.latent_prompt_ok(torch.empty(40, H * 128, **bf16), torch.empty(2, 64, 256, **bf16), torch.empty(H, 64, 192, **bf16), torch.empty(H, 192, 64, **bf16),
                                    torch.empty(40, H, **bf16), types.SimpleNamespace(host_lens_q=lens), H, 64, 64, 192, 64, False, scale)


@pytest.mark.parametrize("scale", [0.0, -0.1, float("nan")])
def test_scales_that_are_not_positive_stay_with_the_batched_products(scale):
    assert ok([17, 1]) and not ok([16, 1]) and not ok([])
    assert not ok([17, 1], scale)


def test_launches_of_two_to_the_31_workgroups_stay_with_the_batched_products():
    assert ok([32 << 25] + [0] * 62) and not ok([32 << 25] + [0] * 63)
    assert ok([32 << 25] + [0] * 30, H=8) and not ok([32 << 25] + [0] * 31, H=8)
