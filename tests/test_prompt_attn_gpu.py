"""The 32-query form of the windowed attention (prompt_attn_kernel) at the edges of its tiles, windows, pages and head groups,
against the vector kernel (f32 products of the same bf16 rows), and the rule that takes a launch to it."""
import pytest
import torch

from light_vllm_amd import mix_ops
from light_vllm_amd.utils.context import RaggedStep

pytestmark = pytest.mark.gpu
# probabilities and outputs are rounded to bf16 (2^-9 each); an output is an average of values of magnitude 1 to 4
ATOL = 4 * 2.0 ** -8
# the same over all outputs: rounded probabilities and both kernels' rounded outputs, each within 2^-9 of its value and independent
REL = 3.0 ** 0.5 * 2.0 ** -9


def make_step(new, ctx, page, seed):
    cu, tok = [0], []
    for b, n in enumerate(new):
        cu.append(cu[-1] + n)
        tok += [b] * n
    need = [-(-(n + c) // page) for n, c in zip(new, ctx)]
    perm = torch.randperm(sum(need), generator=torch.Generator().manual_seed(seed)).tolist()
    tables, at = [], 0
    for k in need:
        tables.append(perm[at:at + k])
        at += k
    wide = max(need)
    i32 = dict(dtype=torch.int32, device="cuda")
    return RaggedStep(torch.tensor(cu, **i32), torch.tensor(ctx, **i32), torch.arange(len(new), **i32), torch.tensor(tok, **i32),
                      torch.tensor([t + [-1] * (wide - len(t)) for t in tables], **i32), new, ctx, list(range(len(new))), tables), sum(need)


def both(monkeypatch, new, ctx, H, G, D, Dv, page=256, same=False, gate=None, ext=False, pool=0, out_pad=0, seed=0, **kw):
    step, pages = make_step(new, ctx, page, seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    T = sum(new)

    def rn(*shape):
        return torch.randn(*shape, device="cuda", generator=gen).bfloat16()

    q, kc = rn(T, H * D), rn(pages, page, G, D)
    vc = kc[..., :Dv] if same else rn(pages, page, G, Dv)
    pp = max(mix_ops.pooled_slots(page, pool), 1)
    kp, vp = (rn(pages, pp, G, D), rn(pages, pp, G, Dv)) if pool else (None, None)
    g = None if gate is None else rn(T, H if gate == "head" else H * Dv)
    if ext:
        kw.update(key_scale=torch.rand(pages, page, G, device="cuda", generator=gen) + 0.5,
                  dist_bias=torch.randn(H, ext, device="cuda", generator=gen))
    got = []
    for kernel in ("valu", "prompt"):
        monkeypatch.setattr(mix_ops, "WINDOW_ATTN_KERNEL", kernel)
        wide = torch.full((T, H * Dv + out_pad), 7.0, device="cuda", dtype=torch.bfloat16)
        out = wide[:, :H * Dv]
        mix_ops.window_pool_attention(q, kc, vc, kp, vp, g, step, H, G, D, Dv, kw.get("window", 1 << 30), pool, D ** -0.5,
                                      gate_per_head=gate == "head", out=out, **{k: v for k, v in kw.items() if k != "window"})
        assert bool((wide[:, H * Dv:] == 7.0).all())
        got.append(out.float())
    assert bool(torch.isfinite(got[1]).all())
    assert (got[0] - got[1]).abs().max().item() <= ATOL
    assert (got[0] - got[1]).norm().item() <= REL * got[0].norm().item()


@pytest.mark.parametrize("n", [17, 31, 32, 33, 63, 64, 65, 129])
@pytest.mark.parametrize("ctx", [0, 1, 63, 200])
def test_tiles(monkeypatch, n, ctx):
    both(monkeypatch, [n, 1, 40], [ctx, ctx, 0], 4, 1, 64, 64, has_sink=False, seed=n + ctx)


@pytest.mark.parametrize("H,G", [(1, 1), (2, 1), (3, 1), (4, 1), (6, 2), (8, 1), (8, 4)])
def test_head_groups(monkeypatch, H, G):
    both(monkeypatch, [70, 150], [5, 0], H, G, 128, 128, window=100, gate="channel", has_sink=True, seed=H)


@pytest.mark.parametrize("D,Dv", [(256, 192), (256, 256), (128, 128)])
def test_values_inside_the_key_rows(monkeypatch, D, Dv):
    both(monkeypatch, [65, 200], [130, 0], 8, 1, D, Dv, same=True, has_sink=False, out_pad=64, seed=D)
    both(monkeypatch, [65, 200], [130, 0], 8, 1, D, Dv, same=True, window=90, sinks=torch.randn(8, device="cuda"), seed=D)


@pytest.mark.parametrize("window", [1, 31, 64, 65, 100])
@pytest.mark.parametrize("pool", [0, 16, 64])
def test_windows_and_pooled_blocks(monkeypatch, window, pool):
    both(monkeypatch, [300, 33], [0, 270], 4, 2, 64, 64, page=64, window=window, pool=pool, gate="head", seed=window)


@pytest.mark.parametrize("kw", [dict(window=50, keep_first=3), dict(window=64, keep_first=130), dict(window=1, chunk=48),
                                dict(window=1, chunk=128, keep_first=5), dict(window=70, softcap=5.0), dict(softcap=20.0),
                                dict(window=90, ext=32), dict(ext=1500), dict(window=1, chunk=100, ext=7)])
@pytest.mark.parametrize("D", [64, 128])
def test_masks_and_scores(monkeypatch, kw, D):
    kw = dict(kw)
    both(monkeypatch, [210, 20, 64], [0, 140, 64], 4, 1, D, D, has_sink=kw.get("window", 0) % 2 == 0, seed=D, **kw)


def test_other_pages_and_sizes_keep_their_kernel(monkeypatch):
    """Pages that do not hold whole tiles, head sizes without an instance, latent rows with kept tokens, a scale of another sign."""
    both(monkeypatch, [80, 20], [9, 0], 4, 2, 64, 64, page=48, window=60)
    both(monkeypatch, [80, 20], [9, 0], 4, 2, 48, 80, window=60)
    both(monkeypatch, [80, 20], [9, 0], 4, 1, 256, 192, same=True, window=60, keep_first=4)
    both(monkeypatch, [80, 20], [9, 0], 4, 1, 256, 192, window=60)


@pytest.mark.parametrize("D,Dv,G", [(64, 64, 2), (128, 128, 1), (256, 192, 1)])
@pytest.mark.parametrize("window", [1, 100, 1 << 30])
def test_sinks_of_minus_infinity_count_nothing(monkeypatch, D, Dv, G, window):
    monkeypatch.setattr(mix_ops, "WINDOW_ATTN_KERNEL", "prompt")
    step, pages = make_step([300, 33], [140, 0], 256, D)
    gen = torch.Generator(device="cuda").manual_seed(D)
    H, T = 4, 333
    q, kc = (torch.randn(*s, device="cuda", generator=gen).bfloat16() for s in ((T, H * D), (pages, 256, G, D)))
    vc = kc[..., :Dv]
    if D != Dv:
        args = (q, kc, vc, None, None, None, step, H, G, D, Dv, window, 0, D ** -0.5)
    else:
        args = (q, kc, torch.randn(pages, 256, G, Dv, device="cuda", generator=gen).bfloat16(), None, None, None, step, H, G, D, Dv, window, 0, D ** -0.5)
    none = mix_ops.window_pool_attention(*args, has_sink=False)
    some = mix_ops.window_pool_attention(*args, has_sink=True, sinks=torch.tensor([-float("inf"), -3e38, 0.5, 2.0], device="cuda"))
    assert bool(torch.isfinite(some.float()).all())
    assert torch.equal(some.view(T, H, Dv)[:, :2], none.view(T, H, Dv)[:, :2])
    assert not torch.equal(some.view(T, H, Dv)[:, 2:], none.view(T, H, Dv)[:, 2:])


@pytest.mark.parametrize("D,Dv,same", [(64, 64, False), (128, 128, False), (256, 192, True)])
@pytest.mark.parametrize("n,window,sink,sharp", [(200, 1 << 30, True, 1.0), (200, 1 << 30, False, 4.0), (1500, 1024, True, 1.0), (600, 100, False, 2.0)])
def test_as_precise_as_the_16_query_form(D, Dv, same, n, window, sink, sharp):
    """Against float64 on the same rows, which the 16-query form serves from pages that do not hold whole tiles. Both round every
    probability to bf16; a query's largest one is exact where the running maximum follows it."""
    H, G = 4, 1
    gen = torch.Generator(device="cuda").manual_seed(D + n)

    def rn(*shape):
        return torch.randn(*shape, device="cuda", generator=gen).bfloat16()

    q, k = rn(n, H * D) * sharp, rn(n, G, D)
    v = k[..., :Dv] if same else rn(n, G, Dv)
    s = q.double().view(n, H, D).transpose(0, 1) @ k[:, 0].double().T.contiguous() * D ** -0.5
    i = torch.arange(n, device="cuda")
    s.masked_fill_((i[None] > i[:, None]) | (i[:, None] - i[None] >= window), -float("inf"))
    top = s.amax(-1, keepdim=True).clamp_min(0.0)
    e = torch.exp(s - top)
    want = (e @ v[:, 0].double() / (e.sum(-1, keepdim=True) + (torch.exp(-top) if sink else 0.0))).transpose(0, 1).reshape(n, H * Dv)
    err = []
    for page in (48, 64):
        step, pages = make_step([n], [0], page, 1)
        rows = torch.tensor([step.host_block_tables[0][j // page] * page + j % page for j in range(n)], device="cuda")
        kc = torch.zeros(pages * page, G, D, device="cuda", dtype=torch.bfloat16)
        kc[rows] = k
        vc = torch.zeros(pages * page, G, Dv, device="cuda", dtype=torch.bfloat16)
        vc[rows] = v
        kc, vc = kc.view(pages, page, G, D), vc.view(pages, page, G, Dv)
        o = mix_ops.window_pool_attention(q, kc, kc[..., :Dv] if same else vc, None, None, None, step, H, G, D, Dv, window, 0, D ** -0.5,
                                          has_sink=sink)
        err.append(((o.double() - want).norm() / want.norm()).item())
    assert err[1] <= 1.005 * err[0], err


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("D,Dv,same,kw", [(64, 64, False, dict(window=100)), (64, 64, False, dict(window=64, pool=16, page=64)), (128, 128, False, dict()),
                                          (128, 128, False, dict(window=70, keep_first=3, softcap=20.0)), (64, 64, False, dict(window=1, chunk=96)),
                                          (64, 64, False, dict(window=90, ext=32)), (256, 192, True, dict()), (256, 256, True, dict(window=120))])
def test_a_bad_token_reaches_only_who_sees_it(D, Dv, same, kw, bad):
    """An infinity or a NaN in the value row of one cached token makes the outputs of the queries that see it not finite and leaves
    all others as they are: queries before it, behind its window or chunk, and other sequences."""
    kw = dict(kw)
    window, pool, page, ext = kw.pop("window", 1 << 30), kw.pop("pool", 0), kw.pop("page", 256), kw.pop("ext", 0)
    H, G, new, ctx = 4, 1, [290, 40], [37, 5]
    step, pages = make_step(new, ctx, page, 3)
    gen = torch.Generator(device="cuda").manual_seed(D + Dv)

    def rn(*shape):
        return torch.randn(*shape, device="cuda", generator=gen).bfloat16()

    T = sum(new)
    q, kc = rn(T, H * D), rn(pages, page, G, D)
    vc = kc[..., :Dv] if same else rn(pages, page, G, Dv)
    pp = max(mix_ops.pooled_slots(page, pool), 1)
    kp, vp = (rn(pages, pp, G, D), rn(pages, pp, G, Dv)) if pool else (None, None)
    if ext:
        kw.update(key_scale=torch.rand(pages, page, G, device="cuda", generator=gen) + 0.5, dist_bias=torch.randn(H, ext, device="cuda", generator=gen))

    def run(cache):
        v = cache if not same else cache[..., :Dv]
        return mix_ops.window_pool_attention(q, kc if not same else cache, v, kp, vp, None, step, H, G, D, Dv, window, pool, D ** -0.5, **kw).float()

    base = kc if same else vc
    clean = run(base)
    pos = torch.cat([torch.arange(c, c + n) for n, c in zip(new, ctx)]).cuda()
    first = torch.arange(T, device="cuda") < new[0]
    for at in (1, 40, 63, 64, 100, 170, 255, 326):
        cache = base.clone()
        cache.view(-1, G, base.size(-1))[step.host_block_tables[0][at // page] * page + at % page] = bad
        o = run(cache)
        sees = first & (pos >= at)
        if kw.get("chunk"):
            sees &= pos // kw["chunk"] == at // kw["chunk"]
        elif at >= kw.get("keep_first", 0):
            sees &= pos - at < window
        assert not bool(torch.isfinite(o[sees]).any()), at
        assert (o[~sees] - clean[~sees]).abs().max().item() <= 2.0 ** -6, at      # sums in another order: a rounding of values up to 4


@pytest.mark.parametrize("H,G,D,new,ctx,wide", [
    # us, 16 / 32 queries a wave: 8.4 / 13.2, 10.0 / 15.6, 31 / 37, 9.1 / 10.0, 9.8 / 13.2, 7.4 / 8.9
    (8, 8, 64, [100], [0], False), (8, 8, 128, [100], [0], False), (8, 8, 64, [100], [1000], False), (16, 8, 64, [100], [0], False),
    (6, 2, 64, [100], [0], False), (8, 8, 64, [60], [0], False),
    # 82.7 / 23.8, 36 / 34, 43.1 / 33.4, level; four heads a kv head
    (8, 8, 64, [500] * 16, [0] * 16, True), (16, 8, 64, [100], [1000], True), (8, 8, 64, [64] * 16, [1000] * 16, True), (6, 2, 64, [60], [0], True),
    (8, 2, 64, [100], [0], True), (8, 2, 64, [60], [0], True)])
def test_which_launches_take_32_queries_a_wave(monkeypatch, H, G, D, new, ctx, wide):
    """Small launches with fewer than four query heads a kv head keep the 16-query form: bit for bit what it gives on pages that do not
    hold whole tiles, and not what the other form gives."""
    gen = torch.Generator(device="cuda").manual_seed(H + len(new))
    T, total = sum(new), sum(new) + sum(ctx)
    q, k, v = (torch.randn(n, h * D, device="cuda", generator=gen).bfloat16() for n, h in ((T, H), (total, G), (total, G)))
    got = {}
    for page, kernel in ((256, "auto"), (256, "prompt"), (272, "auto")):
        step, pages = make_step(new, ctx, page, 1)
        at = torch.tensor([step.host_block_tables[b][j // page] * page + j % page for b in range(len(new)) for j in range(new[b] + ctx[b])], device="cuda")
        kc, vc = (torch.zeros(pages * page, G * D, device="cuda", dtype=torch.bfloat16).index_copy(0, at, x).view(pages, page, G, D) for x in (k, v))
        monkeypatch.setattr(mix_ops, "WINDOW_ATTN_KERNEL", kernel)
        got[page, kernel] = mix_ops.window_pool_attention(q, kc, vc, None, None, None, step, H, G, D, D, 1 << 30, 0, D ** -0.5)
    assert not torch.equal(got[256, "prompt"], got[272, "auto"])
    assert torch.equal(got[256, "auto"], got[256, "prompt"] if wide else got[272, "auto"])
