"""The work that a serving step does in one kind of layer, as cases to be timed: the paged attention of Qwen3 and the
sequence mixers and expert feed-forwards of the other model families, on prompts and on decoded tokens.

Every case drives a public layer module under the step context that the engine would set: `Attention` (a layer's K/V store and
attention, as light_vllm_amd.models.qwen3 calls it) and the modules of light_vllm_amd.layers that own their projections. Prompt
steps run eagerly and decode steps replay a hipGraph over `layers` layers with weights and caches of their own, which is how the
engine runs both by default. Sizes are those of the repository's benchmark and tests: Qwen3-0.6B / 8B / 14B heads and one rank's
share of Qwen3-32B; the mixers' 2k and 4k designs.

`exact` restates each layer in float64 torch ops on whole sequences.
"""
from __future__ import annotations

import math
import random

import torch
import torch.nn.functional as F

PAGE = 256               # tokens per cache page, the engine's default
EPS = 1e-6
MAX_MODEL_LEN = 4096     # bound that a captured decode step of the mixers is laid out for
F64 = torch.float64
SIZES = {"2k": dict(width=2048, heads=16, kv_heads=4, q_rank=768, thin=64, ff=1536),
         "4k": dict(width=4096, heads=32, kv_heads=8, q_rank=1536, thin=128, ff=3072)}
KV_RANK, EXPERTS, TOP, GROUPS, KEEP, TAPS = 192, 32, 4, 4, 2, 4


def listed():
    att = dict(kind="attention", ragged=False, cached=0)
    mix = dict(size="2k", dim=128, ragged=False, cached=0)
    return [
        # a few interactive sessions on Qwen3-0.6B: every launch is a few microseconds of work
        dict(name="qwen_decode_few", **{**att, "ragged": True}, phase="decode", heads=16, kv_heads=8, seqs=4, tokens=512, layers=28),
        # the batch that a loaded Qwen3-8B server decodes
        dict(name="qwen_decode_batch", **att, phase="decode", heads=32, kv_heads=8, seqs=256, tokens=1024, layers=4),
        # the same model over long documents
        dict(name="qwen_decode_long", **att, phase="decode", heads=32, kv_heads=8, seqs=32, tokens=32768, layers=1),
        # Qwen3-8B reading four 4k prompts in one step
        dict(name="qwen_prefill", **att, phase="prompt", heads=32, kv_heads=8, seqs=4, tokens=4096, layers=1),
        # chat turns: a few hundred new tokens each behind a prefix that the block manager found in the cache
        dict(name="qwen_prefill_cached", **{**att, "ragged": True, "cached": 1024}, phase="prompt", heads=16, kv_heads=8, seqs=13,
             tokens=300, layers=1),
        # Kagalorn's delta-rule layer: a full prompt step, and a decode step over its four layers
        dict(name="delta_prompt", kind="delta", **mix, phase="prompt", per_channel=False, seqs=16, tokens=1024, layers=1),
        dict(name="delta_decode", kind="delta", **mix, phase="decode", per_channel=False, seqs=64, tokens=1, layers=4),
        # Kagalorn's windowed attention with pooled blocks, prompts of mixed lengths
        dict(name="window_prompt", kind="window", **{**mix, "ragged": True}, phase="prompt", window=1024, pool=64, seqs=11, tokens=1500,
             layers=1),
        # Bokulorn's latent attention
        dict(name="latent_prompt", kind="latent", **mix, phase="prompt", rot=64, seqs=16, tokens=1024, layers=1),
        # Bisuzen's lightning attention
        dict(name="lightning_prompt", kind="lightning", **mix, phase="prompt", seqs=16, tokens=1024, layers=1),
        # Feditar's state-space layer
        dict(name="ssm_prompt", kind="ssm", **{**mix, "ragged": True}, phase="prompt", seqs=7, tokens=2000, layers=1),
        # Bokulorn's expert feed-forward on a prompt step
        dict(name="moe_prompt", kind="moe", **mix, phase="prompt", seqs=16, tokens=1024, layers=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attention", "attention", "attention", "delta", "delta", "window", "latent", "lightning", "ssm", "moe"])
    phase = rng.choice(["prompt", "prompt", "decode"])
    case = dict(kind=kind, ragged=rng.random() < 0.6, cached=0, phase=phase)
    if kind == "attention":
        heads, kv_heads = rng.choice([(16, 8), (32, 8), (40, 8), (8, 1)])
        case.update(heads=heads, kv_heads=kv_heads)
        if phase == "decode":
            tokens = _log(rng, 32, 32768)
            rows = (1 << 20) * 8 // kv_heads if tokens > 4096 else 1 << 18
            seqs = _log(rng, 1, max(1, min(256, rows // tokens)))
            case.update(seqs=seqs, tokens=tokens, layers=max(1, min(16, (1 << 18) // (seqs * tokens))))
        else:
            tokens = _log(rng, 16, 4096)
            case.update(seqs=_log(rng, 1, max(1, min(32, 16384 // tokens))), tokens=tokens, layers=1)
            if rng.random() < 0.4:
                case["cached"] = PAGE * rng.randint(1, 12)
                case["seqs"] = max(1, case["seqs"] // 2)
        return case
    size = rng.choice(["2k", "2k", "4k"])
    case.update(size=size, dim=rng.choice([64, 128, 128]) if kind != "moe" else 128)
    if phase == "decode":
        case.update(seqs=_log(rng, 1, 64), tokens=1, cached=_log(rng, 1, MAX_MODEL_LEN - 2), layers=2)
    else:
        most = 16384 if size == "2k" else 6144
        tokens = _log(rng, 16, 4096)
        case.update(seqs=_log(rng, 1, max(1, min(32, most // tokens))), tokens=tokens, layers=1)
        if rng.random() < 0.3:
            case["cached"] = _log(rng, 1, 2048)        # a later portion of each prompt
            case["seqs"] = max(1, case["seqs"] // 2)
    if kind == "delta":
        case["per_channel"] = rng.random() < 0.4       # Bokulorn's form of the decay
    if kind == "window":
        case["window"], case["pool"] = rng.choice([(1024, 64), (2048, 128), (512, 32)])
    if kind == "latent":
        case["rot"] = rng.choice([64, 0])
    return case


# ------------------------------------------------------------------------------------------------ steps
def _lens(case):
    """New tokens of each sequence. Ragged prompts spread from an eighth of `tokens` to fifteen eighths of it."""
    n, B = case["tokens"], case["seqs"]
    if not case["ragged"] or n == 1:
        return [n] * B
    r = random.Random(1000 * B + n)
    return [max(1, min(n * (r.randint(1, 15)) // 8 + r.randint(-7, 7), 2 * n)) for _ in range(B)]


def _contexts(case):
    """Tokens that each sequence already has in the cache or the state."""
    c, B = case["cached"], case["seqs"]
    if not case["ragged"] or c < 2 or case["kind"] == "attention":
        return [c] * B
    r = random.Random(c)
    return [r.randint(max(1, c // 2), c) for _ in range(B)]


def _i32(v, dev):
    return torch.tensor(v, dtype=torch.int32, device=dev)


def _pages(totals, gen):
    """A random assignment of pages to sequences of these many tokens: one list of page numbers each, and the number of pages."""
    need = [-(-max(t, 1) // PAGE) for t in totals]
    perm = torch.randperm(sum(need), generator=gen).tolist()
    out, at = [], 0
    for n in need:
        out.append(perm[at:at + n])
        at += n
    return out, sum(need)


def _table(pages, dev, fill=-1):
    width = max(len(p) for p in pages)
    return _i32([p + [fill] * (width - len(p)) for p in pages], dev)


def _cu(lens):
    out = [0]
    for n in lens:
        out.append(out[-1] + n)
    return out


def _ragged_step(lens, ctx, pages, dev, static=False):
    from light_vllm_amd.utils.context import RaggedStep
    B = len(lens)
    cu = _cu(lens)
    tok = [b for b, n in enumerate(lens) for _ in range(n)]
    if static:
        width = -(-MAX_MODEL_LEN // PAGE)
        tables = _i32([p + [p[-1]] * (width - len(p)) for p in pages], dev)
        return RaggedStep(_i32(cu, dev), _i32(ctx, dev), _i32(list(range(B)), dev), _i32(tok, dev), tables, lens,
                          [MAX_MODEL_LEN - 1] * B, list(range(B)), None, static=True)
    return RaggedStep(_i32(cu, dev), _i32(ctx, dev), _i32(list(range(B)), dev), _i32(tok, dev), _table(pages, dev), lens, ctx,
                      list(range(B)), pages)


# ------------------------------------------------------------------------------------------------ attention of Qwen3
def _prepare_attention(case, seed, dev):
    from light_vllm_amd import Attention, ops
    from light_vllm_amd.decode_plan import build_plan, worth_planning
    Hq, Hkv, D, L = case["heads"], case["kv_heads"], 128, case["layers"]
    host = torch.Generator().manual_seed(seed)
    gen = torch.Generator(device=dev).manual_seed(seed)
    lens = _lens(case)
    if case["phase"] == "decode":
        total, new = lens, [1] * len(lens)
    else:
        total, new = [n + case["cached"] for n in lens], lens
    pages, count = _pages(total, host)
    kv = torch.empty(2, L, count, PAGE, Hkv, D, dtype=torch.bfloat16, device=dev).normal_(generator=gen)
    T = sum(new)
    qkv = torch.empty(L, T, (Hq + 2 * Hkv) * D, dtype=torch.bfloat16, device=dev).normal_(generator=gen)
    a, b = Hq * D, (Hq + Hkv) * D
    qkv = [tuple(x.split([a, b - a, Hkv * D], dim=-1)) for x in qkv]
    mods = []
    for i in range(L):
        m = Attention(Hq, D, D ** -0.5, Hkv)
        m.k_cache, m.v_cache = kv[0, i], kv[1, i]
        mods.append(m)
    slots = [pages[s][j // PAGE] * PAGE + j % PAGE for s in range(len(new)) for j in range(total[s] - new[s], total[s])]
    if case["phase"] == "decode":
        plan = order = None
        if worth_planning(total, Hkv, Hq // Hkv):
            plan = build_plan(total, Hkv, Hq // Hkv, max_splits=16).to(dev)
        elif max(total) - min(total) > max(total) // 4:
            order = _i32(sorted(range(len(total)), key=lambda j: -total[j]), dev)
        ctx = dict(args=(False,), kw=dict(slot_mapping=_i32(slots, dev), context_lens=_i32(total, dev), block_tables=_table(pages, dev),
                                          seq_order=order, decode_plan=plan))
    else:
        table = _table(pages, dev) if case["cached"] else None
        tiles = ops.prefill_tile_order(new, total, Hq, Hkv, dev, paged=table is not None)
        ctx = dict(args=(True, _i32(_cu(new), dev), _i32(_cu(total), dev), max(new), max(total), _i32(slots, dev), None, table),
                   kw=dict(tile_order=tiles))
    return dict(mods=mods, inputs=qkv, ctx=ctx, state=[kv], keep=dict(pages=pages, total=total, new=new, slots=slots, D=D))


def _softmax_rows(q, k, v, scale, see, extra=0.0):
    """q [H, n, D], k [H or 1, m, D], v [H or 1, m, Dv], see [n, m] (true: visible) -> [H, n, Dv]; `extra` is added to the denominator
    (a sink of score 0)."""
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale
    s.masked_fill_(~see, -math.inf)
    top = s.amax(-1, keepdim=True).clamp_min(0.0) if extra else s.amax(-1, keepdim=True)
    e = torch.exp(s.sub_(top))
    den = e.sum(-1, keepdim=True) + (extra * torch.exp(-top) if extra else 0.0)
    return torch.matmul(e, v.contiguous()) / den


def _causal(n, m, dev):
    i = torch.arange(m - n, m, device=dev)[:, None]
    return torch.arange(m, device=dev)[None, :] <= i


def _exact_attention(case, st):
    Hq, Hkv, k_ = case["heads"], case["kv_heads"], st["keep"]
    D, rep, kv = k_["D"], Hq // Hkv, st["state"][0]
    slots = torch.tensor(k_["slots"], device=kv.device)
    outs = []
    for i, (q, k, v) in enumerate(st["inputs"]):
        kc, vc = kv[0, i].view(-1, Hkv, D), kv[1, i].view(-1, Hkv, D)
        kc[slots], vc[slots] = k.view(-1, Hkv, D), v.view(-1, Hkv, D)
        rows, at = [], 0
        for s, (n, total) in enumerate(zip(k_["new"], k_["total"])):
            where = torch.tensor(k_["pages"][s], device=kv.device)
            ks = kc.view(-1, PAGE, Hkv, D)[where].view(-1, Hkv, D)[:total].permute(1, 0, 2).to(F64)
            vs = vc.view(-1, PAGE, Hkv, D)[where].view(-1, Hkv, D)[:total].permute(1, 0, 2).to(F64)
            qs = q[at:at + n].view(n, Hq, D).permute(1, 0, 2).to(F64)
            see = _causal(n, total, kv.device)
            o = [_softmax_rows(qs[g * rep:(g + 1) * rep], ks[g:g + 1], vs[g:g + 1], D ** -0.5, see) for g in range(Hkv)]
            rows.append(torch.cat(o).permute(1, 0, 2).reshape(n, Hq * D))
            at += n
        outs.append(torch.cat(rows))
    return outs, [kv]


# ------------------------------------------------------------------------------------------------ mixers and experts
def _build(case, dev):
    """One layer's module; bf16 matrices, f32 small parameters, as the models build it."""
    from light_vllm_amd.layers.delta_rule import GatedDeltaRule
    from light_vllm_amd.layers.latent_attention import LatentAttention
    from light_vllm_amd.layers.lightning_attention import LightningAttention
    from light_vllm_amd.layers.moe import SparseMoE
    from light_vllm_amd.layers.state_space import StateSpaceMixer
    from light_vllm_amd.layers.window_pool_attention import WindowPoolAttention
    z, D, kind = SIZES[case["size"]], case["dim"], case["kind"]
    W, H, G = z["width"], z["heads"], z["kv_heads"]
    old = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.device(dev):
            if kind == "delta":
                thin = dict(decay="channel", decay_rank=z["thin"], gate_rank=z["thin"], gate_act="sigmoid") if case["per_channel"] else {}
                return GatedDeltaRule(W, H, G, D, D, TAPS, norm_eps=EPS, **thin)
            if kind == "window":
                return WindowPoolAttention(W, H, G, D, D, case["window"], case["pool"], D ** -0.5, norm_eps=EPS)
            if kind == "latent":
                if case["rot"]:
                    return LatentAttention(W, H, D, D, z["q_rank"], KV_RANK, (D + 64) ** -0.5, rot_dim=64, rot_dims=64, gate="head",
                                           norm_eps=EPS)
                return LatentAttention(W, H, D, D, z["q_rank"], KV_RANK + 64, D ** -0.5, gate="channel", norm_eps=EPS)
            if kind == "lightning":
                return LightningAttention(W, H, D, D, [1.0 - 2.0 ** (-5.0 - 5.0 * i / max(H - 1, 1)) for i in range(H)], norm_eps=EPS)
            if kind == "ssm":
                return StateSpaceMixer(W, W // 64, 64, D, 8, TAPS, norm_groups=8, norm_eps=EPS)
            return SparseMoE(W, z["ff"], EXPERTS, TOP, groups=GROUPS, keep=KEEP)
    finally:
        torch.set_default_dtype(old)


def _states(kind, m):
    return {"delta": lambda: [m.state, m.conv_state], "window": lambda: [m.k_cache, m.v_cache, m.k_pool, m.v_pool],
            "latent": lambda: [m.cache], "lightning": lambda: [m.state], "ssm": lambda: [m.state, m.conv_state], "moe": lambda: []}[kind]()


@torch.no_grad()
def _prepare_mixer(case, seed, dev):
    from light_vllm_amd import mix_ops
    from light_vllm_amd.utils.context import reset_context, set_context
    kind, W, L = case["kind"], SIZES[case["size"]]["width"], case["layers"]
    host = torch.Generator().manual_seed(seed)
    gen = torch.Generator(device=dev).manual_seed(seed)
    new, ctx = _lens(case), _contexts(case)
    total = [n + c for n, c in zip(new, ctx)]
    pages, count = _pages(total, host)
    B, T = len(new), sum(new)
    decode = case["phase"] == "decode"
    step = _ragged_step(new, ctx, pages, dev, static=decode)
    mods, fill = [], []
    for _ in range(L):
        m = _build(case, dev)
        for name, p in m.named_parameters():
            if "norm" in name:
                p.normal_(1.0, 0.1, generator=gen)
            elif p.dim() >= 2 and not name.startswith("conv"):
                p.normal_(0.0, (p.shape[-1] if p.dim() == 2 else p.shape[1]) ** -0.5, generator=gen)
            else:
                p.normal_(0.0, 0.5 if name != "correction" else 0.1, generator=gen)
        if kind == "moe":       # the down matrices of the experts lie side by side: each sums over one expert's ff inputs
            m.down_weight.mul_(EXPERTS ** 0.5)
        else:
            m.bind_cache(count, PAGE, B, dev, torch.bfloat16)
            for x in _states(kind, m):
                if x.numel() and (decode or case["cached"]):
                    x.normal_(0.0, 1.0 if x.dtype == torch.bfloat16 else 0.3, generator=gen)
            if kind == "window" and max(ctx) > 0:       # what earlier steps left: the means of the blocks that they completed
                past = _ragged_step([max(c, 1) for c in ctx], [0] * B, pages, dev)
                mix_ops.pool_update(m.k_cache, m.v_cache, m.k_pool, m.v_pool, past, m.G, m.D, m.Dv, m.pool)
        mods.append(m)
    inputs = [(x,) for x in torch.empty(L, T, W, dtype=torch.bfloat16, device=dev).normal_(generator=gen)]
    st = dict(mods=mods, inputs=inputs, ctx=dict(args=(any(n > 1 for n in new),), kw=dict(ragged=step)),
              state=[x for m in mods for x in _states(kind, m)], keep=dict(pages=pages, total=total, new=new, cached=ctx, B=B))
    return st


def _f(p):
    return p.detach().to(F64)


def _rms(x, eps=EPS):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _rotate(x, pos, base=10000.0):
    d = x.shape[-1]
    a = pos.to(F64)[:, None] * (base ** (-torch.arange(0, d, 2, dtype=F64, device=x.device) / d))[None]
    while a.dim() < x.dim():
        a = a.unsqueeze(1)
    u, v = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([u * torch.cos(a) - v * torch.sin(a), v * torch.cos(a) + u * torch.sin(a)], -1)


def _conv_silu(x, w, bias, before):
    """x [n, C] behind `before` [taps - 1, C], last tap on the current token."""
    full = torch.cat([before, x])
    y = sum(full[i:i + x.shape[0]] * w[:, i] for i in range(w.shape[1]))
    return F.silu(y + bias if bias is not None else y), full[-(w.shape[1] - 1):]


def _history(conv_state, b, ctx):
    h = _f(conv_state[b]).clone()
    h[:max(0, h.shape[0] - ctx)] = 0
    return h


def _padded(rows, B, new, value=0.0):
    """[T, ...] packed rows -> [B, longest, ...]."""
    out = rows.new_full((B, max(new)) + rows.shape[1:], value)
    for b, (a, n) in enumerate(zip(_cu(new), new)):
        out[b, :n] = rows[a:a + n]
    return out


def _packed(x, new):
    return torch.cat([x[b, :n] for b, n in enumerate(new)])


def _start(state, ctx):
    s = _f(state).clone()
    s[torch.tensor([c == 0 for c in ctx], device=s.device)] = 0
    return s


def _exact_layer(case, m, h, keep):
    """(y, states in the order of _states) of one layer."""
    kind, new, ctx, total, B = case["kind"], keep["new"], keep["cached"], keep["total"], keep["B"]
    dev, cu, T = h.device, _cu(keep["new"]), h.shape[0]
    h = h.to(F64)
    if kind in ("delta", "ssm"):
        proj = h @ _f(m.in_proj.weight).T
        off = 0 if kind == "delta" else m.inner
        bias = None if kind == "delta" else _f(m.conv_bias)
        conv, tails = [], []
        for b in range(B):
            y, tail = _conv_silu(proj[cu[b]:cu[b + 1], off:off + m.channels], _f(m.conv_weight), bias, _history(m.conv_state, b, ctx[b]))
            conv.append(y)
            tails.append(tail)
        conv, tails = torch.cat(conv), torch.stack(tails)
    if kind == "delta":
        G, H, D, Dv = m.G, m.H, m.D, m.Dv
        unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        q = unit(conv[:, :G * D].view(T, G, D)).repeat_interleave(H // G, 1) * D ** -0.5
        k = unit(conv[:, G * D:2 * G * D].view(T, G, D)).repeat_interleave(H // G, 1)
        v = conv[:, 2 * G * D:].view(T, H, Dv)
        beta = torch.sigmoid(proj[:, m.off_b:m.off_b + H])
        a, gate = proj[:, m.off_a:m.off_a + m.decay_in], proj[:, m.off_gate:m.off_gate + m.gate_in]
        if m.decay_up is not None:
            a, gate = a @ _f(m.decay_up.weight).T, gate @ _f(m.gate_up.weight).T
        rate = torch.exp(_f(m.A_log))[None, :, None]
        g = torch.exp(-rate * F.softplus((a + _f(m.dt_bias)).view(T, H, -1)))                    # [T, H, 1 or D]
        q, k, v, beta = (_padded(x, B, new) for x in (q, k, v, beta))
        g = _padded(g, B, new, 1.0)
        S = _start(m.state, ctx)
        o = torch.empty_like(v)
        for t in range(max(new)):
            S = S * g[:, t][..., None]
            u = beta[:, t][..., None] * (v[:, t] - (k[:, t].unsqueeze(-2) @ S).squeeze(-2))
            S = S + k[:, t][..., None] * u[..., None, :]
            o[:, t] = (q[:, t].unsqueeze(-2) @ S).squeeze(-2)
        o = _rms(_packed(o, new)) * _f(m.out_norm_weight)
        act = F.silu(gate) if m.gate_act == "silu" else torch.sigmoid(gate)
        return (o.reshape(T, H * Dv) * act) @ _f(m.o_proj.weight).T, [S, tails]
    if kind == "ssm":
        H, Dv, N, G = m.H, m.Dv, m.N, m.G
        x, Bm, C = conv.split([m.inner, G * N, G * N], dim=1)
        dt = F.softplus(proj[:, m.inner + m.channels:] + _f(m.dt_bias))
        g = torch.exp(-torch.exp(_f(m.A_log)) * dt)
        x = x.reshape(T, H, Dv)
        Bm, C = (y.reshape(T, G, N).repeat_interleave(H // G, 1) for y in (Bm, C))
        xp, kp, cp = _padded(x, B, new), _padded(Bm * dt[..., None], B, new), _padded(C, B, new)
        gp = _padded(g, B, new, 1.0)
        S = _start(m.state, ctx)
        o = torch.empty_like(xp)
        for t in range(max(new)):
            S = S * gp[:, t][..., None, None] + kp[:, t][..., None] * xp[:, t][..., None, :]
            o[:, t] = (cp[:, t].unsqueeze(-2) @ S).squeeze(-2)
        y = (_packed(o, new) + _f(m.skip)[:, None] * x).reshape(T, m.inner) * F.silu(proj[:, :m.inner])
        y = _rms(y.view(T, m.norm_groups, -1)).reshape(T, m.inner) * _f(m.out_norm_weight)
        return y @ _f(m.o_proj.weight).T, [S, tails]
    if kind == "lightning":
        H, D, Dv = m.H, m.D, m.Dv
        q, k, v, gate = (h @ _f(m.in_proj.weight).T).split(m.sizes, dim=1)
        q, k, v = F.silu(q).view(T, H, D), F.silu(k).view(T, H, D), F.silu(v).view(T, H, Dv)
        q, k, v = (_padded(x, B, new) for x in (q, k, v))
        decay = torch.tensor(m.decay_values, dtype=F64, device=dev).expand(T, H)
        decay = _padded(decay, B, new, 1.0)
        S = _start(m.state, ctx)
        o = torch.empty_like(v)
        for t in range(max(new)):
            S = S * decay[:, t][..., None, None] + k[:, t][..., None] * v[:, t][..., None, :]
            o[:, t] = (q[:, t].unsqueeze(-2) @ S).squeeze(-2)
        y = _rms(_packed(o, new).reshape(T, H * Dv)) * _f(m.out_norm_weight) * torch.sigmoid(gate)
        return y @ _f(m.o_proj.weight).T, [S]
    if kind == "moe":
        s = torch.sigmoid(h @ _f(m.router_weight).T)
        c = s + _f(m.correction)
        best = c.view(T, GROUPS, -1).topk(2, -1).values.sum(-1)
        kept = torch.zeros(T, GROUPS, dtype=torch.bool, device=dev).scatter_(1, best.topk(KEEP, -1).indices, True)
        c = c.masked_fill(~kept.repeat_interleave(EXPERTS // GROUPS, 1), -math.inf)
        ids = c.topk(TOP, -1).indices
        w = torch.zeros(T, EXPERTS, dtype=F64, device=dev).scatter_(1, ids, s.gather(1, ids) / s.gather(1, ids).sum(-1, keepdim=True))
        y = torch.zeros_like(h)
        for e in range(EXPERTS):
            rows = w[:, e].nonzero()[:, 0]
            up = h[rows] @ _f(m.up_weight[e * m.ff:(e + 1) * m.ff]).T
            y.index_add_(0, rows, (torch.relu(up) ** 2 @ _f(m.down_weight[:, e * m.ff:(e + 1) * m.ff]).T) * w[rows, e:e + 1])
        return y, []
    proj = h @ _f(m.in_proj.weight).T
    outs = []
    if kind == "window":
        H, G, D, Dv, rep, P = m.H, m.G, m.D, m.Dv, m.H // m.G, m.pool
        q, k, v, gate = proj.split(m.sizes, dim=1)
        q = (_rms(q) * _f(m.q_norm_weight)).view(T, H, D)
        k = (_rms(k) * _f(m.k_norm_weight)).view(T, G, D)
        v = v.view(T, G, Dv)
        for b in range(B):
            where = torch.tensor(keep["pages"][b], device=dev)
            ks = torch.cat([_f(m.k_cache[where]).view(-1, G, D)[:ctx[b]], k[cu[b]:cu[b + 1]]]).permute(1, 0, 2)
            vs = torch.cat([_f(m.v_cache[where]).view(-1, G, Dv)[:ctx[b]], v[cu[b]:cu[b + 1]]]).permute(1, 0, 2)
            n, nb = total[b], total[b] // P
            i = torch.arange(ctx[b], n, device=dev)[:, None]
            j = torch.arange(n, device=dev)[None]
            see = (j <= i) & (i - j < m.window)
            if nb:
                end = (torch.arange(nb, device=dev)[None] + 1) * P - 1
                see = torch.cat([see, end <= i - m.window], 1)
                ks = torch.cat([ks, ks[:, :nb * P].reshape(G, nb, P, D).mean(2)], 1)
                vs = torch.cat([vs, vs[:, :nb * P].reshape(G, nb, P, Dv).mean(2)], 1)
            qs = q[cu[b]:cu[b + 1]].permute(1, 0, 2)
            o = [_softmax_rows(qs[g * rep:(g + 1) * rep], ks[g:g + 1], vs[g:g + 1], m.scale, see, 1.0) for g in range(G)]
            outs.append(torch.cat(o).permute(1, 0, 2).reshape(-1, H * Dv))
        return (torch.cat(outs) * torch.sigmoid(gate)) @ _f(m.o_proj.weight).T, [None] * 4
    H, R, Dn, Dr, Dv = m.H, m.R, m.Dn, m.Dr, m.Dv
    cq, ckv, gate = proj.split(m.sizes, dim=1)
    q = ((_rms(cq) * _f(m.q_norm_weight)) @ _f(m.uq.weight).T).view(T, H, Dn + Dr)
    c = _rms(ckv[:, :R]) * _f(m.kv_norm_weight)
    pos = torch.cat([torch.arange(a, t, device=dev) for a, t in zip(ctx, total)])
    if Dr:
        q = torch.cat([q[..., :Dn], _rotate(q[..., Dn:], pos)], -1)
        c = torch.cat([c, _rotate(ckv[:, R:], pos)], -1)
    for b in range(B):
        where = torch.tensor(keep["pages"][b], device=dev)
        rows = torch.cat([_f(m.cache[where]).view(-1, R + Dr)[:ctx[b]], c[cu[b]:cu[b + 1]]])
        see = _causal(new[b], total[b], dev)
        o = []
        for hh in range(H):
            ks = torch.cat([rows[:, :R] @ _f(m.uk[hh]).T, rows[:, R:]], -1)
            o.append(_softmax_rows(q[cu[b]:cu[b + 1], hh][None], ks[None], (rows[:, :R] @ _f(m.uv[hh]))[None], m.scale, see)[0])
        outs.append(torch.stack(o, 1))
    o = torch.cat(outs)
    g = torch.sigmoid(gate)
    o = o * (g[..., None] if not m.gate_per_channel else g.view(T, H, Dv))
    return o.reshape(T, H * Dv) @ _f(m.o_proj.weight).T, [None]


# ------------------------------------------------------------------------------------------------ the interface
def _forward(st):
    return [m(*x) for m, x in zip(st["mods"], st["inputs"])]


def prepare(case, seed):
    from light_vllm_amd.utils.context import reset_context, set_context
    dev = torch.device("cuda", torch.cuda.current_device())
    st = (_prepare_attention if case["kind"] == "attention" else _prepare_mixer)(case, seed, dev)
    if case["phase"] == "decode":       # the engine captures its decode step once and replays it
        before = [x.clone() for x in st["state"]] if case["kind"] in ("delta", "lightning", "ssm") else None
        with torch.inference_mode():
            set_context(*st["ctx"]["args"], **st["ctx"]["kw"])
            _forward(st)
            torch.cuda.synchronize()
            st["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(st["graph"]):
                st["outs"] = _forward(st)
            reset_context()
        for x, y in zip(st["state"], before or []):     # the run before the capture moved the recurrent states
            x.copy_(y)
        torch.cuda.synchronize()
    return st


@torch.inference_mode()
def run(st):
    from light_vllm_amd.utils.context import reset_context, set_context
    if "graph" in st:
        st["graph"].replay()
        return {"outs": st["outs"], "state": st["state"]}
    set_context(*st["ctx"]["args"], **st["ctx"]["kw"])
    outs = _forward(st)
    reset_context()
    return {"outs": outs, "state": st["state"]}


@torch.no_grad()
def exact(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    if case["kind"] == "attention":
        outs, state = _exact_attention(case, _prepare_attention(case, seed, dev))
        return {"outs": outs, "state": state}
    st = _prepare_mixer(case, seed, dev)
    got = [_exact_layer(case, m, x[0], st["keep"]) for m, x in zip(st["mods"], st["inputs"])]
    return {"outs": [y for y, _ in got], "state": [s for _, states in got for s in states]}


def work(case):
    """Inputs, weights and visible cache or state entries read once, outputs and new entries written once; the products of the
    projections, of the visible (query, key) pairs and of the recurrence's state."""
    new, L = _lens(case), case["layers"]
    if case["kind"] == "attention":
        Hq, Hkv, D = case["heads"], case["kv_heads"], 128
        if case["phase"] == "decode":
            total, new = new, [1] * len(new)
        else:
            total = [n + case["cached"] for n in new]
        pairs = sum(n * t - n * (n - 1) // 2 for n, t in zip(new, total))
        keys = sum(total) if case["phase"] == "decode" or case["cached"] else sum(new)
        nbytes = keys * Hkv * D * 4 + sum(new) * (2 * Hq + 4 * Hkv) * D * 2 - (sum(new) * Hkv * D * 4 if keys == sum(new) else 0)
        return {"bytes": L * nbytes, "flops": L * pairs * Hq * D * 4}
    z, D, ctx = SIZES[case["size"]], case["dim"], _contexts(case)
    W, H, G, T, B, kind = z["width"], z["heads"], z["kv_heads"], sum(new), len(new), case["kind"]
    if kind == "moe":
        used = min(EXPERTS, T * TOP)
        return {"bytes": L * (T * W * 4 + used * 2 * W * z["ff"] * 2 + EXPERTS * W * 4),
                "flops": L * T * (TOP * 4 * W * z["ff"] + 2 * W * EXPERTS)}
    pairs = 0
    for n, c in zip(new, ctx):
        if kind == "window":
            pairs += sum(min(i + 1, case["window"]) + max(0, (i - case["window"] + 1) // case["pool"]) for i in range(c, c + n))
        else:
            pairs += n * (n + c) - n * (n - 1) // 2
    if kind == "delta":
        wide = H * D if case["per_channel"] else 0
        cols = 2 * G * D + H * D + H + (2 * z["thin"] if wide else H * D + H)
        mats, mix, state = W * (cols + H * D) + 2 * z["thin"] * wide, T * H * D * D * 6, B * H * D * D * 8
    elif kind == "ssm":
        inner = W
        cols = 2 * inner + 16 * D + W // 64
        mats, mix, state = W * (cols + inner), T * inner * D * 4, B * inner * D * 8
    elif kind == "lightning":
        mats, mix, state = W * 5 * H * D, T * H * D * D * 4, B * H * D * D * 8
    elif kind == "window":
        mats, mix = W * ((2 * H + 2 * G) * D + H * D), pairs * H * D * 4
        seen = sum(min(n + c, case["window"] + n) for n, c in zip(new, ctx))
        state = seen * G * D * 4 + T * G * D * 4
    else:
        R = KV_RANK if case["rot"] else KV_RANK + 64
        mats = W * (z["q_rank"] + KV_RANK + 64 + (H if case["rot"] else H * D)) + z["q_rank"] * H * (D + case["rot"]) + W * H * D + 2 * H * D * R
        mix = pairs * H * (2 * D + case["rot"]) * 2
        state = sum(n + c for n, c in zip(new, ctx)) * 512 + T * 512
    return {"bytes": L * (T * W * 4 + mats * 2 + state), "flops": L * (2 * T * mats + mix)}


def tolerance(case):
    if case["kind"] == "attention":
        return {"rel": 6e-3, "max": 0.1}          # bf16 outputs and probabilities
    return {"rel": 1.5e-2, "max": 0.5}            # several bf16 tensors behind one another
