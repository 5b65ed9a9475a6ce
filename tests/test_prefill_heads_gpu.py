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


def outputs(q, k, v, case, num_splits):
    from light_vllm_amd import ops
    return ops.prefill_attention(q, k, v, case["cu_q"], case["cu_k"], case["max_q"], case["max_k"], case["scale"], block_table=case["block_table"],
                                 num_splits=num_splits)


@pytest.mark.parametrize("Hq,Hkv,lens", [(16, 8, [1, 31, 33, 63, 64, 65, 97, 128, 129, 0, 200]), (40, 8, [64, 1, 96, 130]), (64, 8, [1 + 5 * i % 32 for i in range(40)])])
@pytest.mark.parametrize("num_splits", [1, 3])
def test_column_views_and_neighbours_that_are_not_finite(gpu, Hq, Hkv, lens, num_splits):
    """Queries, keys and values as columns of one projection, bit for bit as separate tensors give; a sequence of NaNs and infinities, whose
    rows lie behind another one's last tile, changes that one in no bit, nor does what stale pages hold behind a sequence's last key."""
    case = to_dev(make_prefill_case(35, lens, lens, Hq, Hkv), gpu)
    clean = outputs(case["q"], case["k"], case["v"], case, num_splits)
    ref = prefill_ref(case["q"].cpu(), case["k"].cpu(), case["v"].cpu(), case["cu_q"].cpu(), case["cu_k"].cpu(), case["scale"], None)
    assert (clean.float().cpu() - ref).abs().max().item() <= TOL
    qkv = torch.cat([case[n].flatten(1) for n in "qkv"], 1)
    q, k, v = (x.view(len(qkv), -1, 128) for x in qkv.split([Hq * 128, Hkv * 128, Hkv * 128], 1))
    assert torch.equal(outputs(q, k, v, case, num_splits), clean)
    at, bad = case["cu_q"].tolist(), range(1, len(lens), 3)
    fine = torch.ones(len(qkv), dtype=torch.bool, device=gpu)
    for b in bad:
        qkv[at[b]:at[b + 1], ::2], qkv[at[b]:at[b + 1], 1::2] = float("nan"), float("inf")
        fine[at[b]:at[b + 1]] = False
    assert torch.equal(outputs(q, k, v, case, num_splits)[fine], clean[fine])
    keys = [n + 70 * (i % 2) for i, n in enumerate(lens)]
    case = to_dev(make_prefill_case(36, lens, keys, Hq, Hkv, paged=True), gpu)
    clean = outputs(case["q"], case["k"], case["v"], case, num_splits)
    used = torch.zeros(case["k"].shape[:2], dtype=torch.bool, device=gpu)
    for b, n in enumerate(keys):
        for i in range(-(-n // 256)):
            used[case["block_table"][b, i], :min(256, n - 256 * i)] = True
    case["k"][~used], case["v"][~used] = float("inf"), float("nan")
    assert torch.equal(outputs(case["q"], case["k"], case["v"], case, num_splits), clean)
