"""Prompt attention with several query heads of a group in a workgroup: every group size, prompts around the edges of its row tiles, packed
and paged, with and without splits of the keys, against the CPU f32 oracle."""
import pytest
import torch

from oracle.attention_oracle import prefill_ref
from tests._cases import make_prefill_case, to_dev

pytestmark = pytest.mark.gpu
TOL = 2e-2            # outputs and probabilities in bf16, values of unit size


def check(gpu, case, num_splits=0):
    from light_vllm_amd import ops
    d = to_dev(case, gpu)
    out = ops.prefill_attention(d["q"], d["k"], d["v"], d["cu_q"], d["cu_k"], d["max_q"], d["max_k"], d["scale"],
                                block_table=d["block_table"], num_splits=num_splits)
    ref = prefill_ref(case["q"], case["k"], case["v"], case["cu_q"], case["cu_k"], case["scale"], case["block_table"])
    assert (out.float().cpu() - ref).abs().max().item() <= TOL


@pytest.mark.parametrize("Hq,Hkv", [(8, 8), (16, 8), (24, 8), (32, 8), (40, 8), (48, 8), (64, 8), (12, 3)])
@pytest.mark.parametrize("num_splits", [1, 3])
def test_tile_edges(gpu, Hq, Hkv, num_splits):
    lens = [1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 0, 200]
    check(gpu, make_prefill_case(31, lens, lens, Hq, Hkv), num_splits)
    keys = [n + 256 * (i % 3) + 17 * (i % 2) for i, n in enumerate(lens)]
    check(gpu, make_prefill_case(32, lens, keys, Hq, Hkv, paged=True), num_splits)


@pytest.mark.parametrize("Hq,Hkv", [(32, 8), (64, 8)])
def test_many_prompts_of_few_tokens(gpu, Hq, Hkv):
    lens = [1 + 5 * i % 32 for i in range(40)]             # four heads a workgroup
    check(gpu, make_prefill_case(33, lens, lens, Hq, Hkv))
    check(gpu, make_prefill_case(34, lens, [n + 70 for n in lens], Hq, Hkv, paged=True))
