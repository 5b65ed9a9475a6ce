"""Windowed and latent attention of steps of one token a sequence (decode_pool_kernel, and the merge of its splits) against the vector kernel
(f32 products of the same bf16 rows): tails of tiles, windows and chunks, pooled blocks, kept tokens, sinks, gates, head groups, empty
splits and sequences without a new token."""
import pytest
import torch

from light_vllm_amd import mix_ops
from tests._ragged import ragged_step

pytestmark = pytest.mark.gpu
# probabilities and outputs are rounded to bf16 (2^-9 each); an output is an average of values of magnitude 1 to 4
ATOL = 4 * 2.0 ** -8
REL = 3.0 ** 0.5 * 2.0 ** -9          # rounded probabilities and both kernels' rounded outputs, independent

SHAPES = [(4, 4, 64, 64, False), (16, 4, 128, 128, False), (6, 2, 128, 128, False), (40, 2, 64, 64, False), (16, 1, 256, 192, True),
          (20, 1, 256, 256, True), (32, 1, 256, 192, True), (16, 1, 128, 128, True), (8, 4, 128, 128, True), (20, 1, 64, 64, True),
          (8, 2, 256, 256, False)]


def both(monkeypatch, ctx, H, G, D, Dv, same, page=64, pool=0, gate=None, new=None, workgroups=256, out_pad=0, seed=0, **kw):
    step, pages = ragged_step(new or [1] * len(ctx), ctx, page, "cuda", seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    T = len(step.tok_seq)

    def rn(*shape):
        return torch.randn(*shape, device="cuda", generator=gen).bfloat16()

    q, kc = rn(T, H * D), rn(pages, page, G, D)
    vc = kc[..., :Dv] if same else rn(pages, page, G, Dv)
    pp = max(mix_ops.pooled_slots(page, pool), 1)
    kp, vp = (rn(pages, pp, G, D), rn(pages, pp, G, Dv)) if pool else (None, None)
    g = None if gate is None else rn(T, H if gate == "head" else H * Dv)
    monkeypatch.setattr(mix_ops, "SPLIT_WORKGROUPS", workgroups)
    got = []
    for kernel in ("valu", "auto"):
        monkeypatch.setattr(mix_ops, "WINDOW_ATTN_KERNEL", kernel)
        wide = torch.full((T, H * Dv + out_pad), 7.0, device="cuda", dtype=torch.bfloat16)
        mix_ops.window_pool_attention(q, kc, vc, kp, vp, g, step, H, G, D, Dv, kw.get("window", 1 << 30), pool, D ** -0.5,
                                      gate_per_head=gate == "head", out=wide[:, :H * Dv], **{k: v for k, v in kw.items() if k != "window"})
        assert bool((wide[:, H * Dv:] == 7.0).all())
        got.append(wide[:, :H * Dv].float())
    assert bool(torch.isfinite(got[1]).all())
    assert (got[0] - got[1]).abs().max().item() <= ATOL
    assert (got[0] - got[1]).norm().item() <= REL * got[0].norm().item()


@pytest.mark.parametrize("H,G,D,Dv,same", SHAPES)
@pytest.mark.parametrize("workgroups", [1, 64, 4096])
def test_lengths_and_splits(monkeypatch, H, G, D, Dv, same, workgroups):
    both(monkeypatch, [0, 30, 31, 32, 126, 127, 128, 700, 1, 2100], H, G, D, Dv, same, has_sink=False, workgroups=workgroups, seed=H)


@pytest.mark.parametrize("H,G,D,Dv,same", SHAPES)
@pytest.mark.parametrize("kw", [dict(window=70, has_sink=True), dict(window=33, keep_first=5, has_sink=False), dict(chunk=100, has_sink=False),
                                dict(window=1, has_sink=False), dict(sinks=True)])
def test_windows_chunks_and_sinks(monkeypatch, H, G, D, Dv, same, kw):
    if kw.get("sinks"):
        kw = dict(kw, sinks=torch.linspace(-2, 3, H, device="cuda"))
    both(monkeypatch, [0, 69, 70, 99, 100, 355, 1023], H, G, D, Dv, same, gate="head", workgroups=200, seed=G, **{"has_sink": True, **kw})


@pytest.mark.parametrize("pool,window", [(16, 40), (64, 128), (32, 1)])
def test_pooled_blocks_and_gates(monkeypatch, pool, window):
    for H, G, D in ((16, 4, 128), (8, 8, 64)):
        both(monkeypatch, [5, 40, 64, 500, 1500, 127], H, G, D, D, False, page=128, pool=pool, window=window, gate="channel", out_pad=8, seed=pool)


def test_sequences_without_a_new_token(monkeypatch):
    both(monkeypatch, [100, 300, 7], 16, 1, 256, 192, True, new=[1, 0, 1], has_sink=False)


@pytest.mark.parametrize("H,G,D,Dv,same", SHAPES + [(8, 2, 128, 64, False), (8, 1, 96, 96, True)])
@pytest.mark.parametrize("off", [False, True])
def test_splits_are_counted_for_the_kernel_that_runs(monkeypatch, H, G, D, Dv, same, off):
    """Workgroups of the launch, from the kernel's name and the rule: at most SPLIT_WORKGROUPS, in either kernel."""
    from torch.profiler import ProfilerActivity, profile
    ctx, page = [1500] * 6, 64
    step, pages = ragged_step([1] * 6, ctx, page, "cuda")
    q = torch.randn(6 * H * D + 8, device="cuda").bfloat16()[4 if off else 0:][:6 * H * D].view(6, H * D)
    kc = torch.randn(pages, page, G, D, device="cuda").bfloat16()
    vc = kc[..., :Dv] if same else torch.randn(pages, page, G, Dv, device="cuda").bfloat16()
    heads = mix_ops.decode_heads(q, kc, vc, None, None, G, D, Dv, 0)
    seen = []
    lib = mix_ops._mixlib.load()
    call = lib.lv_masked_attn_mfma
    monkeypatch.setattr(lib, "lv_masked_attn_mfma", lambda *a: seen.append(a[27]) or call(*a))
    run = lambda: mix_ops.window_pool_attention(q, kc, vc, None, None, None, step, H, G, D, Dv, 1 << 30, 0, D ** -0.5, has_sink=False)  # noqa: E731
    run()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        run()
        torch.cuda.synchronize()
    names = " ".join(e.key for e in prof.key_averages())
    assert ("decode_pool_kernel" in names) == (heads == 16) and ("window_pool_mfma_kernel" in names) == (heads == 4)
    assert seen[-1] == max(1, min(24 // (2 if heads == 16 else 1), 256 // (6 * G * -(-(H // G) // heads)), 32))


def exact(q, kc, vc, step, H, G, D, Dv, window, sinks):
    outs, rep = [], H // G
    for b, ctx in enumerate(step.host_ctx_lens):
        pages = torch.tensor(step.host_block_tables[b], device="cuda")
        k, v = (x[pages].reshape(-1, G, x.size(-1))[max(0, ctx - window + 1):ctx + 1].double() for x in (kc, vc))
        s = torch.einsum("grd,ngd->grn", q[b].view(G, rep, D).double(), k) * D ** -0.5
        if sinks is not None:
            s = torch.cat([s, sinks.double().view(G, rep, 1)], -1)
        outs.append(torch.einsum("grn,ngd->grd", torch.softmax(s, -1)[..., :k.size(0)], v).reshape(-1))
    return torch.stack(outs)


def run(q, kc, vc, step, H, G, D, Dv, window, sinks=None):
    return mix_ops.window_pool_attention(q, kc, vc, None, None, None, step, H, G, D, Dv, window, 0, D ** -0.5, has_sink=False, sinks=sinks)


def operands(ctx, H, G, D, Dv, same, page, seed):
    step, pages = ragged_step([1] * len(ctx), ctx, page, "cuda", seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kc = torch.randn(pages, page, G, D, device="cuda", generator=gen).bfloat16()
    vc = kc[..., :Dv] if same else torch.randn(pages, page, G, Dv, device="cuda", generator=gen).bfloat16()
    return step, torch.randn(len(ctx), H * D, device="cuda", generator=gen).bfloat16(), kc, vc


@pytest.mark.parametrize("H,G,D,Dv,same", SHAPES)
@pytest.mark.parametrize("sunk", [False, True])
def test_against_float64(H, G, D, Dv, same, sunk):
    """Sinks of minus infinity, which count nothing, among finite ones."""
    step, q, kc, vc = operands([0, 31, 64, 700, 2100], H, G, D, Dv, same, 64, H + D)
    sinks = torch.linspace(-3, 3, H, device="cuda") if sunk else None
    if sunk:
        sinks[::3] = float("-inf")
    got, want = run(q, kc, vc, step, H, G, D, Dv, 1500, sinks), exact(q, kc, vc, step, H, G, D, Dv, 1500, sinks)
    assert (got.double() - want).norm().item() <= 2 ** 0.5 * 2.0 ** -9 * want.norm().item()      # rounded probabilities and outputs, independent


@pytest.mark.parametrize("H,G,D,Dv,same", SHAPES)
def test_rows_that_are_not_finite_reach_only_the_queries_that_see_them(H, G, D, Dv, same):
    ctx, page, window = [100, 63, 500], 64, 80
    step, q, kc, vc = operands(ctx, H, G, D, Dv, same, page, 3)
    clean = run(q, kc, vc, step, H, G, D, Dv, window)
    table = step.host_block_tables
    for rows in ({kc.data_ptr(): kc, vc.data_ptr(): vc}).values():
        for b, c in enumerate(ctx):
            rows[table[b][c // page], c % page + 1:] = float("nan")                 # behind the last token
        rows[torch.tensor(table[2][:421 // page])] = float("inf")                   # whole pages in front of the window's first token, 421
    assert torch.equal(run(q, kc, vc, step, H, G, D, Dv, window), clean)
    for at in (90, 100):                                                            # inside the window, and the last token
        keep = vc[table[0][at // page], at % page, 0, 3].clone()
        vc[table[0][at // page], at % page, 0, 3] = float("inf")
        got = run(q, kc, vc, step, H, G, D, Dv, window)
        first = got[0, :H // G * Dv].view(-1, Dv)                                   # the kv head's query heads
        assert torch.equal(got[1:], clean[1:]) and torch.equal(got[0, H // G * Dv:], clean[0, H // G * Dv:])
        assert not torch.isfinite(first[:, 3]).any()
        if not same:                                                                # (a key with an infinity takes its head along)
            assert torch.equal(first[:, 4:], clean[0, :H // G * Dv].view(-1, Dv)[:, 4:])
        vc[table[0][at // page], at % page, 0, 3] = keep
