"""The chunked recurrences (lv_chunk_scan) against the recurrence in float64, at the edges of their chunks and segments, and the
rule that takes a step to them against the token loop."""
import math

import pytest
import torch
import torch.nn.functional as F

from light_vllm_amd import mix_ops
from light_vllm_amd.utils.context import RaggedStep

pytestmark = pytest.mark.gpu
F64 = torch.float64
# f32 products and sums: a read-out is a sum over at most 128 rows of the state and 32 tokens of the chunk, each addition off
# by half a unit in the last place at most, and the state carries the errors of as many additions
REL = (128 + 2 * 32) * 2.0 ** -24


@pytest.fixture(autouse=True)
def chunks(monkeypatch):
    """The chunked kernel wherever it serves; which steps it pays on is tested on the CPU."""
    monkeypatch.setattr(mix_ops, "SCAN_KERNEL", "chunk")


def make_step(new, ctx, static=False):
    cu, tok = [0], []
    for b, n in enumerate(new):
        cu.append(cu[-1] + n)
        tok += [b] * n
    i32 = dict(dtype=torch.int32, device="cuda")
    B = len(new)
    slots = list(reversed(range(B)))
    return RaggedStep(torch.tensor(cu, **i32), torch.tensor(ctx, **i32), torch.tensor(slots, **i32), torch.tensor(tok, **i32),
                      torch.zeros(B, 1, **i32), new, ctx, slots, [[0]] * B, static=static)


def recurrence(q, k, v, g, beta, state, step):
    """q, k [T, H, D], v [T, H, Dv], g [T, H] in float64; beta [T, H]: delta rule. -> (o, state)."""
    S_all, o = state.to(F64).clone(), torch.empty_like(v)
    at = 0
    for b, n in enumerate(step.host_lens_q):
        slot = step.host_slots[b]
        S = S_all[slot] if step.host_ctx_lens[b] > 0 else torch.zeros_like(S_all[slot])
        for t in range(at, at + n):
            S = S * g[t][:, None, None]
            u = v[t] if beta is None else beta[t][:, None] * (v[t] - torch.einsum("hdv,hd->hv", S, k[t]))
            S = S + k[t][:, :, None] * u[:, None, :]
            o[t] = torch.einsum("hdv,hd->hv", S, q[t])
        if n > 0:
            S_all[slot] = S
        at += n
    return o, S_all


def case(kind, new, H, G, D, Dv, seed, pad=4, zeros=False):
    """(call(state, step), float64 arguments of recurrence, skip) on seeded inputs; rows are views of a wider tensor."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    T, rep = sum(new), H // G

    def rn(*shape):
        return torch.randn(*shape, device="cuda", generator=gen)

    def heads(x):
        return x.to(F64).view(T, G, D).repeat_interleave(rep, 1)

    if kind == "delta":
        q, k, v = F.normalize(rn(T, G, D), dim=-1) * D ** -0.5, F.normalize(rn(T, G, D), dim=-1), rn(T, H, Dv)
        beta, g = torch.sigmoid(rn(T, H)), torch.exp(-torch.exp(0.5 * rn(H)) * F.softplus(rn(T, H)))
        if zeros:
            g[::5] = 0.0
        return (lambda st, step: mix_ops.gated_delta_rule(q, k, v, beta, g, st, step),
                (heads(q), heads(k), v.to(F64), g.to(F64), beta.to(F64)), 0.0)
    if kind == "step":
        u = (0.6 * rn(T, 2 * G * D + H * Dv + pad)).bfloat16()[:, pad:]
        a, p0, p1, p2 = rn(T, H).bfloat16(), 0.5 * rn(H), 0.5 * rn(H), rn(H)
        q, k, v = u[:, :G * D], u[:, G * D:2 * G * D], u[:, 2 * G * D:]
        dt = F.softplus(a.to(F64) + p0.to(F64))
        v64 = v.to(F64).view(T, H, Dv)
        return (lambda st, step: mix_ops.gated_scan(mix_ops.SCAN_STEP, q, k, v, a, p0, p1, step, st, H, G, D, Dv, p2=p2),
                (heads(q), heads(k) * dt[..., None], v64, torch.exp(-torch.exp(p1.to(F64)) * dt), None), p2.to(F64)[:, None] * v64)
    proj = rn(T, 2 * H * D + H * Dv + pad).bfloat16()
    decay = torch.tensor([0.0 if zeros and h == 0 else 1.0 - 2.0 ** (-5.0 - 5.0 * h / H) for h in range(H)], device="cuda")
    x = F.silu(proj[:, pad:].to(F64))
    return (lambda st, step: mix_ops.lightning_attention(proj, pad, pad + H * D, pad + 2 * H * D, decay, st, step, H, D, Dv),
            (x[:, :H * D].view(T, H, D), x[:, H * D:2 * H * D].view(T, H, D), x[:, 2 * H * D:].reshape(T, H, Dv),
             decay.to(F64).expand(T, H), None), 0.0)


def rel(x, y):
    return ((x.to(F64) - y).norm() / y.norm()).item()


@pytest.mark.parametrize("kind,H,G,D,Dv", [("delta", 4, 2, 64, 64), ("delta", 3, 1, 128, 64), ("delta", 4, 1, 128, 128), ("delta", 2, 2, 64, 256),
                                           ("step", 6, 3, 128, 64), ("step", 3, 3, 64, 64), ("step", 2, 1, 64, 128),
                                           ("const", 2, 2, 64, 64), ("const", 3, 3, 128, 128), ("const", 2, 2, 64, 256)])
@pytest.mark.parametrize("new,ctx", [([96], [0]), ([97, 1, 31, 32, 33], [0, 7, 0, 1, 0]), ([128, 0, 64, 65], [3, 0, 0, 2])])
def test_chunks_match_the_recurrence(kind, H, G, D, Dv, new, ctx):
    call, args, skip = case(kind, new, H, G, D, Dv, seed=D + Dv + len(new))
    step = make_step(new, ctx)
    state = 0.3 * torch.randn(len(new), H, D, Dv, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    want_o, want_s = recurrence(*args, state, step)
    o = call(state, step)
    assert rel(o, want_o + skip) < REL and rel(state, want_s) < REL


@pytest.mark.parametrize("kind", ["step", "const"])
@pytest.mark.parametrize("new", [[1024], [1500, 40, 1057]])
def test_segments_match_the_recurrence(kind, new):
    """Long portions on few sequences are cut into segments."""
    H, D, Dv = 2, 64, 64
    call, args, skip = case(kind, new, H, H, D, Dv, seed=sum(new))
    step = make_step(new, [5] * len(new))
    state = 0.3 * torch.randn(len(new), H, D, Dv, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    want_o, want_s = recurrence(*args, state, step)
    o = call(state, step)
    # decays of 1 - 2^-7.5: the state of `const` sums about 200 tokens, whose additions add their errors
    assert rel(o, want_o + skip) < 2 * REL and rel(state, want_s) < 2 * REL


@pytest.mark.parametrize("kind", ["delta", "const"])
def test_decays_of_zero(kind):
    new = [85, 40]
    call, args, _ = case(kind, new, 2, 2, 64, 64, seed=5, zeros=True)
    step = make_step(new, [0, 3])
    state = torch.randn(2, 2, 64, 64, device="cuda")
    want_o, want_s = recurrence(*args, state, step)
    o = call(state, step)
    assert rel(o, want_o) < REL and rel(state, want_s) < REL


@pytest.mark.parametrize("kind", ["step", "const"])
@pytest.mark.parametrize("pad", [1, 2, 3])
def test_misaligned_rows_and_captured_steps_take_the_token_loop(kind, pad, monkeypatch):
    """Rows that do not lie on four entries, and steps that are captured, run where they ran before."""
    new = [96, 5]
    state = torch.randn(2, 2, 64, 64, device="cuda")
    monkeypatch.setattr(mix_ops, "SCAN_KERNEL", "token")
    call, args, skip = case(kind, new, 2, 2, 64, 64, seed=pad, pad=pad)
    s_token = state.clone()
    o_token = call(s_token, make_step(new, [0, 2]))
    monkeypatch.setattr(mix_ops, "SCAN_KERNEL", "chunk")
    s_auto = state.clone()
    o_auto = call(s_auto, make_step(new, [0, 2]))
    assert torch.equal(o_auto, o_token) and torch.equal(s_auto, s_token)
    call, args, skip = case(kind, new, 2, 2, 64, 64, seed=pad, pad=4)
    s_token, s_static, s_auto = state.clone(), state.clone(), state.clone()
    monkeypatch.setattr(mix_ops, "SCAN_KERNEL", "token")
    o_token = call(s_token, make_step(new, [0, 2]))
    monkeypatch.setattr(mix_ops, "SCAN_KERNEL", "chunk")
    o_static = call(s_static, make_step(new, [0, 2], static=True))
    assert torch.equal(o_static, o_token) and torch.equal(s_static, s_token)
    o_auto = call(s_auto, make_step(new, [0, 2]))        # aligned and not captured: the same numbers in another order
    assert rel(o_auto, o_token.to(F64)) < REL and rel(s_auto, s_token.to(F64)) < REL


def test_silu_of_large_arguments():
    """Constant decays read their rows through silu: zero far below zero (not a small multiple of the argument), the argument far
    above. Values of 1e-36 and less are taken as zero."""
    H, D, Dv, new = 2, 64, 64, [96]
    gen = torch.Generator(device="cuda").manual_seed(9)
    proj = torch.randn(96, 2 * H * D + H * Dv, device="cuda", generator=gen).bfloat16()
    proj[3, ::3] = -3e38
    proj[7, 1::2] = -1e30
    proj[11, ::5] = -88.5
    proj[13, ::4] = -86.0
    proj[17, ::7] = 200.0
    decay = torch.full((H,), 0.9, device="cuda")
    x = F.silu(proj.to(F64))
    q, k, v = x[:, :H * D].view(96, H, D), x[:, H * D:2 * H * D].view(96, H, D), x[:, 2 * H * D:].reshape(96, H, Dv)
    step, state = make_step(new, [0]), torch.zeros(1, H, D, Dv, device="cuda")
    want_o, want_s = recurrence(q, k, v, decay.to(F64).expand(96, H), None, state, step)
    o = mix_ops.lightning_attention(proj, 0, H * D, 2 * H * D, decay, state, step, H, D, Dv)
    assert rel(o, want_o) < REL and rel(state, want_s) < REL


def test_a_bad_token_reaches_no_earlier_one():
    """An infinity or a NaN in a token's query, key, value, write strength or decay leaves the outputs of every token before it and of
    every other sequence and head as they were (bit for bit before its chunk; inside, sums in another order); outputs behind a bad
    key or value are not finite."""
    G, H, D, Dv, new = 2, 4, 128, 128, [100, 70]
    gen = torch.Generator(device="cuda").manual_seed(4)

    def rn(*shape):
        return torch.randn(*shape, device="cuda", generator=gen)

    T, step = sum(new), make_step(new, [3, 0])
    delta = dict(q=F.normalize(rn(T, G, D), dim=-1), k=F.normalize(rn(T, G, D), dim=-1), v=rn(T, H, Dv), beta=torch.sigmoid(rn(T, H)),
                 decay=torch.sigmoid(rn(T, H) + 2))
    steps = {n: rn(T, c).bfloat16() for n, c in (("q", G * D), ("k", G * D), ("v", H * Dv), ("a", H))}
    const = rn(T, 2 * H * D + H * Dv).bfloat16()
    small = [0.5 * rn(H) for _ in range(3)]
    rate = torch.full((H,), 0.95, device="cuda")

    def run_delta(x, st):
        return mix_ops.gated_delta_rule(x["q"], x["k"], x["v"], x["beta"], x["decay"], st, step)

    def run_step(x, st):
        return mix_ops.gated_scan(mix_ops.SCAN_STEP, x["q"], x["k"], x["v"], x["a"], small[0], small[1], step, st, H, G, D, Dv, p2=small[2])

    def run_const(x, st):
        return mix_ops.lightning_attention(x["p"], 0, H * D, 2 * H * D, rate, st, step, H, D, Dv)

    for run, inputs, carried in ((run_delta, delta, ("k", "v", "beta", "decay")), (run_step, steps, ("k", "v", "a")), (run_const, dict(p=const), ("p",))):
        state = rn(2, H, D, Dv)
        clean = run(inputs, state.clone())
        for name, x in inputs.items():
            for at in (0, 5, 15, 16, 31, 32, 50, 99):
                for bad in (float("nan"), float("inf")):
                    y = x.clone()
                    y[at] = bad                        # (silu leaves +inf, softplus too)
                    st = state.clone()
                    o = run({**inputs, name: y}, st)
                    chunk = at // 32 * 32
                    assert torch.equal(o[:chunk], clean[:chunk]) and torch.equal(o[100:], clean[100:]), (name, at, bad)
                    assert at == chunk or rel(o[chunk:at], clean[chunk:at].to(F64)) < REL, (name, at, bad)
                    if name in carried and name != "beta" and not (bad > 0 and name in ("a", "decay")):
                        assert not bool(torch.isfinite(o[at]).any()) and not bool(torch.isfinite(st[1]).any()), (name, at, bad)
    # one value column of one head: the others stay clean, bit for bit
    y = {**delta, "v": delta["v"].clone()}
    y["v"][40, 1, 17] = float("inf")
    st = torch.zeros(2, H, D, Dv, device="cuda")
    clean = run_delta(delta, st.clone())
    o = run_delta(y, st)
    keep = torch.ones(H, Dv, dtype=torch.bool, device="cuda")
    keep[1, 17] = False
    assert torch.equal(o[:32], clean[:32]) and rel(o[:40], clean[:40].to(F64)) < REL and rel(o[:, keep], clean[:, keep].to(F64)) < REL
    assert not bool(torch.isfinite(o[40:100, 1, 17]).any())


@pytest.mark.parametrize("kind,H,G,D,Dv", [("delta", 4, 2, 64, 64), ("delta", 4, 1, 128, 128), ("step", 4, 2, 128, 64), ("step", 2, 1, 64, 128),
                                           ("const", 2, 2, 64, 64), ("const", 3, 3, 128, 128)])
@pytest.mark.parametrize("new", [[96], [300, 97], [1500, 40]])
def test_as_precise_as_the_token_loop(kind, H, G, D, Dv, new, monkeypatch):
    """Outputs are no further from float64 than the token loop's (a tenth for the draw), states by at most a quarter of a rounding:
    what a token writes is rounded once more on its way into the state."""
    call, args, skip = case(kind, new, H, G, D, Dv, seed=3)
    step = make_step(new, [5] * len(new))
    state = 0.3 * torch.randn(len(new), H, D, Dv, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    want_o, want_s = recurrence(*args, state, step)
    err = []
    for kernel in ("token", "chunk"):
        monkeypatch.setattr(mix_ops, "SCAN_KERNEL", kernel)
        s = state.clone()
        o = call(s, step)
        err.append((rel(o, want_o + skip), rel(s, want_s)))
    assert err[1][0] <= 1.1 * err[0][0] and err[1][1] <= 1.1 * err[0][1] + 2.0 ** -26


@pytest.mark.parametrize("kind,H,G,D,Dv", [("delta", 2, 1, 64, 64), ("step", 2, 1, 64, 64), ("const", 2, 2, 64, 64)])
@pytest.mark.parametrize("new", [[1] * 63 + [130], [200] + [1] * 63, [1] * 64 + [97], [0] * 70 + [33, 0, 64] + [1] * 60 + [0], [31, 32, 33] * 45])
def test_many_sequences(kind, H, G, D, Dv, new):
    """The places of chunks among those of all sequences, which a wave looks up 64 sequences at a time."""
    call, args, skip = case(kind, new, H, G, D, Dv, seed=len(new))
    step = make_step(new, [i % 3 for i in range(len(new))])
    state = 0.3 * torch.randn(len(new), H, D, Dv, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    want_o, want_s = recurrence(*args, state, step)
    o = call(state, step)
    assert rel(o, want_o + skip) < REL and rel(state, want_s) < REL


@pytest.mark.parametrize("kind,H,G,D,Dv", [("step", 4, 2, 128, 64), ("step", 8, 2, 64, 64), ("step", 3, 3, 128, 64), ("step", 2, 1, 128, 256), ("const", 2, 2, 128, 128),
                                           ("const", 2, 2, 64, 128), ("const", 3, 3, 128, 64)])
@pytest.mark.parametrize("new,seg", [([1000, 256, 513, 255, 1, 0, 512], 256), ([96, 33, 65, 31], 32), ([700, 1400], 512)])
def test_segments_of_every_instance(kind, H, G, D, Dv, new, seg, monkeypatch):
    """Sequences shorter than a segment, of whole segments, one token past them and empty, cut as asked for, on the workgroups of one
    head, of two heads of a group and of four waves; and what the cut costs in precision against none: nothing but the draw."""
    assert any(n > seg for n in new)
    call, args, skip = case(kind, new, H, G, D, Dv, seed=D + H)
    step = make_step(new, [i % 2 for i in range(len(new))])
    state = 0.3 * torch.randn(len(new), H, D, Dv, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    want_o, want_s = recurrence(*args, state, step)
    err, asked = [], []
    for length in (0, seg):
        monkeypatch.setattr(mix_ops, "_segment_length", lambda *a: asked.append(length) or length)
        s = state.clone()
        o = call(s, step)
        assert rel(o, want_o + skip) < 2 * REL and rel(s, want_s) < 2 * REL
        err.append(rel(o, want_o + skip))
    assert asked == [0, seg] and err[1] <= 1.15 * err[0]


# launches of more than 128 workgroups: eight waves each, and the delta rule's states of 128 rows grow by products of bf16 pieces
@pytest.mark.parametrize("H,G,Dv", [(32, 8, 128), (48, 8, 64), (24, 24, 128)])
def test_large_delta_launches(H, G, Dv):
    new = [33, 64, 95, 1, 40, 71, 130]
    call, args, _ = case("delta", new, H, G, 128, Dv, seed=H + Dv)
    step = make_step(new, [0, 4, 0, 9, 1, 0, 2])
    state = 0.3 * torch.randn(len(new), H, 128, Dv, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    want_o, want_s = recurrence(*args, state, step)
    o = call(state, step)
    assert rel(o, want_o) < REL and rel(state, want_s) < REL


@pytest.mark.parametrize("bad", [float("inf"), float("nan"), -3e38])
def test_large_delta_launches_with_values_that_are_not_finite(bad):
    """A key, a value, a state entry or sums that are not finite reach the tokens behind them and no earlier or other row."""
    H, G, D, Dv, new = 32, 8, 128, 128, [100] * 6
    gen = torch.Generator(device="cuda").manual_seed(2)
    T = sum(new)
    q, k = (F.normalize(torch.randn(T, G, D, device="cuda", generator=gen), dim=-1) for _ in range(2))
    v = torch.randn(T, H, Dv, device="cuda", generator=gen)
    beta, g = torch.rand(T, H, device="cuda", generator=gen), 0.5 + 0.5 * torch.rand(T, H, device="cuda", generator=gen)
    state = torch.randn(6, H, D, Dv, device="cuda", generator=gen)
    s0 = state.clone()
    want = mix_ops.gated_delta_rule(q, k, v, beta, g, s0, make_step(new, [3] * 6))
    k[140, 2, 7], v[270, 9, 5], v[310, 3, 100] = bad, bad, bad      # sequences 1, 2 and 3
    state[1, 20, 3, 4] = bad                                        # slot 1: sequence 4
    s1 = state.clone()
    got = mix_ops.gated_delta_rule(q, k, v, beta, g, s1, make_step(new, [3] * 6))
    heads = [h for h in range(H) if not 8 <= h < 12]                # heads that do not read the key
    cols = [c for c in range(Dv) if c not in (4, 5, 100)]
    # a wave that sees such a value sums its chunk in another order: what it does not reach is off by the two sums' roundings
    for x, y in [(got[:140], want[:140]), (got[140:200, heads], want[140:200, heads]), (got[200:270], want[200:270]), (got[300:310], want[300:310]),
                 (got[200:][:, :, cols], want[200:][:, :, cols]), (s1[0], s0[0]), (s1[5], s0[5]), (s1[1][:, :, cols], s0[1][:, :, cols])]:
        assert rel(x, y.to(F64)) < 2 * REL
    if not math.isfinite(bad):                                      # a bad key reaches every column of its heads, in the state too
        for x in (got[140:200, 8:12], s1[4, 8:12], got[270:300, 9, 5], s1[3, 9, :, 5], got[310:400, 3, 100], s1[2, 3, :, 100], got[400:500, 20, 4], s1[1, 20, :, 4]):
            assert not bool(torch.isfinite(x).any())


# constant decays on launches of more than 128 workgroups form P in the scan: whole and partial chunks, fewer chunks than are staged ahead, segments
@pytest.mark.parametrize("H,D,Dv,new,ctx", [(32, 128, 128, [33, 64, 1, 95, 32, 130, 161], [0, 4, 0, 9, 1, 0, 2]), (64, 64, 64, [40, 97, 129, 0, 31, 66], [3, 0, 0, 5, 1, 2]),
                                            (8, 128, 128, [2100, 1500, 1700], [0, 3, 0])])
def test_large_launches_of_constant_decays(H, D, Dv, new, ctx):
    call, args, _ = case("const", new, H, H, D, Dv, seed=H + D)
    step = make_step(new, ctx)
    state = 0.3 * torch.randn(len(new), H, D, Dv, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    want_o, want_s = recurrence(*args, state, step)
    o = call(state, step)
    assert rel(o, want_o) < 2 * REL and rel(state, want_s) < 2 * REL


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_large_launches_of_constant_decays_with_values_that_are_not_finite(bad):
    """q, k and v entries that are not finite reach their own tokens and those behind them in the same head, and no earlier or other one."""
    H, D, Dv, new = 32, 128, 128, [100] * 6
    gen = torch.Generator(device="cuda").manual_seed(2)
    proj = torch.randn(sum(new), 3 * H * D, device="cuda", generator=gen).bfloat16()
    decay = torch.linspace(0.9, 0.999, H, device="cuda")
    run = lambda x, st: mix_ops.lightning_attention(x, 0, H * D, 2 * H * D, decay, st, make_step(new, [0] * 6), H, D, Dv).view(-1, H, Dv)  # noqa: E731
    s0, s1 = torch.zeros(6, H, D, Dv, device="cuda"), torch.zeros(6, H, D, Dv, device="cuda")
    want = run(proj, s0)
    proj[150, 3 * D + 7], proj[250, H * D + 9 * D + 4], proj[350, 2 * H * D + 5 * D + 100] = bad, bad, bad      # q of head 3, k of head 9, v of head 5
    got = run(proj, s1)
    assert not torch.isfinite(got[150, 3]).any() and not torch.isfinite(got[250, 9]).any() and not torch.isfinite(got[350:400, 5, 100]).any()
    ok = torch.ones(sum(new), H, Dv, dtype=torch.bool, device="cuda")
    ok[150, 3] = ok[250:300, 9] = ok[350:400, 5, 100] = False
    # a wave that sees such a value goes through its block of tokens one by one: another order of the same sums
    assert rel(torch.where(ok, got, 0.0), torch.where(ok, want, 0.0).to(F64)) < 4 * REL
    rest = [h for h in range(H) if h not in (5, 9)]
    assert torch.equal(s1[:, rest], s0[:, rest])


# key sizes, value sizes and lengths on either side of the rule, whole and in segments; head 0 decays at once
@pytest.mark.parametrize("H,D,Dv,new,seg,own", [
    (48, 128, 128, [33, 130, 95], 0, True), (48, 128, 128, [330, 40], 128, True), (24, 128, 128, [300] + [9] * 9, 0, False),
    (32, 128, 64, [33, 64, 1, 95, 32, 130, 161, 70, 97], 0, False), (48, 128, 64, [230, 97, 33], 64, False),
    (48, 64, 128, [200, 180, 150], 0, True), (48, 64, 128, [400, 33, 95], 0, False), (96, 64, 128, [130, 100, 120], 0, True),
    (96, 64, 128, [64, 65, 63], 0, False), (48, 64, 128, [256, 250, 240], 128, True), (96, 64, 64, [200, 180, 150], 0, True),
    (96, 64, 64, [64, 65, 63, 33, 40, 64], 0, False), (96, 64, 64, [256, 250, 240], 128, True), (96, 64, 64, [230, 97, 33], 64, False)])
def test_where_constant_decays_form_their_products_in_the_scan(H, D, Dv, new, seg, own, monkeypatch):
    """Launches of more than 128 workgroups have no launch in front where that is faster, and are the recurrence either way."""
    from torch.profiler import ProfilerActivity, profile
    call, args, _ = case("const", new, H, H, D, Dv, seed=H + D + Dv, zeros=True)
    step = make_step(new, [i % 2 for i in range(len(new))])
    monkeypatch.setattr(mix_ops, "_segment_length", lambda *a: seg)
    state = 0.3 * torch.randn(len(new), H, D, Dv, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    want_o, want_s = recurrence(*args, state, step)
    s = state.clone()
    o = call(s, step)
    assert rel(o, want_o) < 2 * REL and rel(s, want_s) < 2 * REL
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        call(state, step)
        torch.cuda.synchronize()
    names = " ".join(e.key for e in prof.key_averages())
    assert "chunk_scan_kernel" in names and ("chunk_prep_kernel" in names) != own and ("chunk_combine_kernel" in names) == (seg > 0)


# eight waves with the state's growth from pieces (128 rows), and without; constant decays with their products in the scan, whole and in segments
@pytest.mark.parametrize("kind,H,G,D,Dv,new,seg", [
    ("delta", 32, 8, 128, 128, [160, 97, 33, 64, 200], 0), ("delta", 48, 24, 128, 64, [160, 97, 33, 64, 200, 31], 0), ("delta", 32, 8, 64, 128, [160, 97, 33, 64, 200], 0),
    ("const", 48, 48, 128, 128, [160, 97, 200], 0), ("const", 48, 48, 64, 128, [160, 180, 200], 0), ("const", 96, 96, 64, 64, [160, 180, 200], 0),
    ("const", 48, 48, 128, 128, [160, 300], 128), ("const", 96, 96, 64, 64, [160, 256, 256], 128)])
def test_large_launches_are_as_precise_as_the_token_loop(kind, H, G, D, Dv, new, seg, monkeypatch):
    """More than 128 workgroups, errors as in test_as_precise_as_the_token_loop (in segments by what test_segments_of_every_instance allows
    them more). Leaving out one of the pieces' products above a rounding makes outputs 1.1e-6 and states 1e-5 wrong; f32 errors are 1e-7."""
    call, args, skip = case(kind, new, H, G, D, Dv, seed=11)
    step = make_step(new, [5] * len(new))
    state = 0.3 * torch.randn(len(new), H, D, Dv, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    want_o, want_s = recurrence(*args, state, step)
    monkeypatch.setattr(mix_ops, "_segment_length", lambda *a: seg)
    err = []
    for kernel in ("token", "chunk"):
        monkeypatch.setattr(mix_ops, "SCAN_KERNEL", kernel)
        s = state.clone()
        o = call(s, step)
        err.append((rel(o, want_o + skip), rel(s, want_s)))
    more = 1.1 * 1.15 if seg else 1.1
    assert err[1][0] <= more * err[0][0] and err[1][1] <= more * err[0][1] + 2.0 ** -26
