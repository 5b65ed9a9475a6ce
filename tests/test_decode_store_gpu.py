"""A decode step's rows stored by the attention launch (lv_decode_attn_store) against store_kvcache followed by the attention, and
the one-pass form of short contexts against forced splits: same caches bit for bit, same outputs up to the order of f32 sums."""
import pytest
import torch

from light_vllm_amd import Attention, ops, reset_context, set_context
from light_vllm_amd.decode_plan import build_plan

pytestmark = pytest.mark.gpu
D, BS = 128, 256
ATOL = 2 * 2.0 ** -8        # one rounding of an output below 2 to bf16, from sums in another order


def case(lens, Hq, Hkv, seed=0, spare=2):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    B = len(lens)
    need = [max(1, -(-n // BS)) for n in lens]
    blocks = sum(need) + spare
    perm = torch.randperm(blocks, generator=torch.Generator().manual_seed(seed)).tolist()
    tables, at = [], 0
    for k in need:
        tables.append(perm[at:at + k])
        at += k
    wide = max(need)
    i32 = dict(dtype=torch.int32, device="cuda")

    def rn(*shape):
        return torch.randn(*shape, device="cuda", generator=gen).bfloat16()

    qkv = rn(B, (Hq + 2 * Hkv) * D)
    q, k, v = qkv.split([Hq * D, Hkv * D, Hkv * D], dim=-1)
    slots = [t[(n - 1) // BS] * BS + (n - 1) % BS if n > 0 else -1 for n, t in zip(lens, tables)]
    return dict(q=q.view(B, Hq, D), k=k.view(B, Hkv, D), v=v.view(B, Hkv, D), kc=rn(blocks, BS, Hkv, D), vc=rn(blocks, BS, Hkv, D),
                ctx=torch.tensor(lens, **i32), table=torch.tensor([t + [-1] * (wide - len(t)) for t in tables], **i32), slots=slots,
                spare=perm[at:])


def both(c, slots, **kw):
    slots = torch.tensor(slots, dtype=torch.int32, device="cuda")
    kc, vc = c["kc"].clone(), c["vc"].clone()
    ops.store_kvcache(c["k"], c["v"], kc, vc, slots)
    want = ops.decode_attention(c["q"], kc, vc, c["ctx"], c["table"], D ** -0.5, **kw)
    kc2, vc2 = c["kc"].clone(), c["vc"].clone()
    got = ops.decode_attention(c["q"], kc2, vc2, c["ctx"], c["table"], D ** -0.5, new_kv=(c["k"], c["v"], slots), **kw)
    assert torch.equal(kc, kc2) and torch.equal(vc, vc2)
    assert bool(torch.isfinite(got.float()).all()) and (got.float() - want.float()).abs().max().item() <= ATOL
    return got


@pytest.mark.parametrize("Hq,Hkv", [(2, 2), (16, 8), (32, 8), (8, 1), (40, 8), (6, 2), (7, 1)])
@pytest.mark.parametrize("kernel", ["auto", "mfma"])
@pytest.mark.parametrize("splits", [0, 1, 3, 16])
def test_same_as_store_then_attend(Hq, Hkv, kernel, splits):
    for lens in ([1], [1, 0, 2, 31, 32, 33], [63, 64, 65, 255, 256, 257], [1000, 5, 513]):
        c = case(lens, Hq, Hkv, seed=len(lens) + Hq)
        both(c, c["slots"], num_splits=splits, kernel=kernel)


def test_vector_kernel_and_order():
    for Hq in (8, 16, 32, 64):
        c = case([300, 1, 700, 64, 129], Hq, 8, seed=Hq)
        order = torch.tensor([2, 0, 4, 3, 1], dtype=torch.int32, device="cuda")
        both(c, c["slots"], kernel="valu", seq_order=order)
        both(c, c["slots"], kernel="valu", seq_order=order, num_splits=4)


def test_slots_that_are_not_the_last_tokens_place():
    """Skipped slots, slots past the cache, and slots in blocks that no sequence reads: stored or not as store_kvcache does, and what
    is read stays what the cache holds."""
    c = case([300, 40, 700, 0, 5], 16, 8)
    total = c["kc"].size(0) * BS
    for splits in (0, 1, 5):
        both(c, [-1] * 5, num_splits=splits)
        both(c, [total, total + 7, -5, c["spare"][0] * BS + 3, c["spare"][1] * BS], num_splits=splits)
        both(c, [c["slots"][0], c["spare"][0] * BS, c["slots"][2], c["spare"][1] * BS + 255, -1], num_splits=splits)


def test_work_lists_store_on_their_own():
    c = case([3000, 40, 90, 200, 5], 32, 8)
    both(c, c["slots"], plan=build_plan([3000, 40, 90, 200, 5], 8, 4, max_splits=16).to("cuda"))


@pytest.mark.parametrize("Hq,Hkv", [(16, 8), (32, 8), (8, 1), (40, 8)])
@pytest.mark.parametrize("lens", [[1], [256] * 3, [200, 1, 0, 77], [256] * 31, [1024] * 21, [513] * 31, [100] * 32])
def test_one_pass_on_wide_workgroups(Hq, Hkv, lens):
    c = case(lens, Hq, Hkv, seed=len(lens))
    one = ops.decode_attention(c["q"], c["kc"], c["vc"], c["ctx"], c["table"], D ** -0.5)
    cut = ops.decode_attention(c["q"], c["kc"], c["vc"], c["ctx"], c["table"], D ** -0.5, num_splits=2)
    assert (one.float() - cut.float()).abs().max().item() <= ATOL


def test_attention_module_replays_in_a_graph():
    c = case([300, 17, 256, 1], 16, 8)
    slots = torch.tensor(c["slots"], dtype=torch.int32, device="cuda")
    attn = Attention(16, D, D ** -0.5, 8)
    attn.k_cache, attn.v_cache = c["kc"].clone(), c["vc"].clone()
    q, k, v = (c[x].reshape(4, -1).contiguous() for x in ("q", "k", "v"))
    set_context(False, slot_mapping=slots, context_lens=c["ctx"], block_tables=c["table"])
    attn(q, k, v)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = attn(q, k, v)
    reset_context()
    for seed in range(3):
        gen = torch.Generator(device="cuda").manual_seed(seed)
        for x in (q, k, v):
            x.copy_(torch.randn(x.shape, device="cuda", generator=gen))
        kc, vc = attn.k_cache.clone(), attn.v_cache.clone()
        ops.store_kvcache(k.view(4, 8, D), v.view(4, 8, D), kc, vc, slots)
        want = ops.decode_attention(q.view(4, 16, D), kc, vc, c["ctx"], c["table"], D ** -0.5)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(attn.k_cache, kc) and torch.equal(attn.v_cache, vc)
        assert (out.view(4, 16, D).float() - want.float()).abs().max().item() <= ATOL


def several_rows(ctx, rows, Hq, Hkv, seed=0):
    """`rows` tokens of one sequence behind `ctx` tokens, each a row of the batch with the same pages, and a sequence of its own."""
    c = case([ctx + rows, 70], Hq, Hkv, seed=seed)
    gen = torch.Generator(device="cuda").manual_seed(seed + 1)
    B = rows + 1

    def rn(*shape):
        return torch.randn(*shape, device="cuda", generator=gen).bfloat16()

    table = c["table"].tolist()
    slots = [table[0][j // BS] * BS + j % BS for j in range(ctx, ctx + rows)] + [table[1][0] * BS + 69]
    c.update(q=rn(B, Hq, D), k=rn(B, Hkv, D), v=rn(B, Hkv, D), table=torch.tensor([table[0]] * rows + [table[1]], dtype=torch.int32, device="cuda"),
             ctx=torch.tensor([ctx + i + 1 for i in range(rows)] + [70], dtype=torch.int32, device="cuda"), slots=slots)
    return c


@pytest.mark.parametrize("Hq,Hkv", [(16, 8), (32, 8), (8, 1), (40, 8)])
@pytest.mark.parametrize("kernel", ["auto", "mfma"])
@pytest.mark.parametrize("ctx,rows", [(0, 5), (30, 4), (250, 16), (500, 63), (500, 64)])
def test_rows_that_read_each_others_tokens(Hq, Hkv, kernel, ctx, rows):
    """Tokens of one sequence as rows of the batch: every row sees the tokens of the rows before it, as after a store."""
    c = several_rows(ctx, rows, Hq, Hkv, seed=ctx + rows)
    for splits in (0, 1, 3, 16):
        both(c, c["slots"], num_splits=splits, kernel=kernel)
    both(c, c["slots"], num_splits=2, kernel=kernel, seq_order=torch.arange(rows, -1, -1, dtype=torch.int32, device="cuda"))


@pytest.mark.parametrize("Hq,Hkv", [(16, 8), (32, 8), (8, 1)])
def test_slots_inside_contexts(Hq, Hkv):
    """A row stored over an earlier token of its own sequence, or over another sequence's token, is what that token reads as."""
    c = case([300, 700, 40, 513], Hq, Hkv, seed=Hq)
    table = c["table"].tolist()

    def at(b, j):
        return table[b][j // BS] * BS + j % BS

    for splits in (0, 1, 4, 16):
        both(c, [at(0, 17), at(1, 699), at(2, 0), at(3, 256)], num_splits=splits)
        both(c, [at(1, 3), at(1, 2), at(3, 512), at(1, 640)], num_splits=splits)


def test_an_order_that_leaves_rows_out_still_stores_them():
    c = case([300, 40, 700], 16, 8)
    order = torch.tensor([2, 2, 9], dtype=torch.int32, device="cuda")
    slots = torch.tensor(c["slots"], dtype=torch.int32, device="cuda")
    kc, vc = c["kc"].clone(), c["vc"].clone()
    ops.store_kvcache(c["k"], c["v"], kc, vc, slots)
    want = ops.decode_attention(c["q"], kc, vc, c["ctx"], c["table"], D ** -0.5)
    kc2, vc2 = c["kc"].clone(), c["vc"].clone()
    got = ops.decode_attention(c["q"], kc2, vc2, c["ctx"], c["table"], D ** -0.5, new_kv=(c["k"], c["v"], slots), seq_order=order)
    assert torch.equal(kc, kc2) and torch.equal(vc, vc2)
    assert (got[2].float() - want[2].float()).abs().max().item() <= ATOL
