"""The delta rule's decode steps (one new token a sequence): preparation with the carried inputs in one launch, and rule, norm and gate in
one launch, against the launches that they stand for and against float64."""
import pytest
import torch

from light_vllm_amd import mix_ops
from tests.test_chunk_scan_gpu import make_step

pytestmark = pytest.mark.gpu
NEW, CTX = [1, 1, 0, 1, 1, 1] * 16, [0, 1, 4, 2, 3, 700] * 16


@pytest.mark.parametrize("G,H,D,taps", [(2, 4, 64, 4), (1, 3, 128, 4), (2, 2, 256, 2), (2, 4, 128, 3)])
@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_preparation(G, H, D, taps, channel, dtype):
    preparation(G, H, D, taps, channel, dtype, NEW, CTX)


# tiles of two and five tokens, each a sequence of its own, the last tile cut short
@pytest.mark.parametrize("G,H,D,taps,times", [(1, 1, 64, 4, 214), (1, 2, 128, 3, 530), (1, 2, 64, 2, 531)])
@pytest.mark.parametrize("channel", [False, True])
def test_preparation_of_many_sequences(G, H, D, taps, times, channel):
    preparation(G, H, D, taps, channel, torch.bfloat16, NEW[:6] * times + [1], CTX[:6] * times + [2])


# no more tokens than sequences, but not one each: the launches that longer steps take
@pytest.mark.parametrize("new,ctx", [([3, 0, 0], [5, 4, 0]), ([0, 2, 1, 0], [0, 1, 2, 9])])
def test_preparation_of_uneven_steps(new, ctx):
    preparation(2, 4, 128, 4, False, torch.bfloat16, new, ctx)


def preparation(G, H, D, taps, channel, dtype, NEW, CTX):
    gen = torch.Generator(device="cuda").manual_seed(G + D)
    rn = lambda *s: torch.randn(*s, device="cuda", generator=gen)    # noqa: E731
    T, C, wide = sum(NEW), 2 * G * D + H * D, H * D if channel else H
    step = make_step(NEW, CTX)
    proj, a = rn(T, C + 2 * H + 4 - 2 * H % 4).to(dtype), rn(T, wide).to(dtype)
    w, A_log, dt = rn(C, taps), rn(H), rn(wide)
    state = rn(len(NEW), taps - 1, C).to(dtype)
    ours, theirs = state.clone(), state.clone()
    args = (A_log, dt, step, G, H, D, D, taps, C, a, 1e-6, channel)
    got = mix_ops.delta_prep(proj, w, ours, *args, carry_on=True)
    want = mix_ops.delta_prep(proj, w, theirs, *args)
    mix_ops.conv_state_update(proj, theirs, step, C, taps)
    assert all(torch.equal(x, y) for x, y in zip(got, want)) and torch.equal(ours, theirs)


@pytest.mark.parametrize("G,H,D", [(2, 4, 64), (1, 3, 128), (4, 4, 128)])
@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("dtype,act", [(torch.bfloat16, "silu"), (torch.float32, "sigmoid")])
def test_rule_norm_gate(G, H, D, channel, dtype, act):
    gen = torch.Generator(device="cuda").manual_seed(H + D)
    rn = lambda *s: torch.randn(*s, device="cuda", generator=gen)    # noqa: E731
    T, step = sum(NEW), make_step(NEW, CTX)
    q, k = (torch.nn.functional.normalize(rn(T, G, D), dim=-1) for _ in range(2))
    v, beta, decay = rn(T, H, D), torch.sigmoid(rn(T, H)), torch.sigmoid(rn(*((T, H, D) if channel else (T, H))))
    gate, w, state = rn(T, H * D + 8)[:, 4:-4].to(dtype), rn(D), rn(len(NEW), H, D, D)
    ours, theirs = state.clone(), state.clone()
    got = mix_ops.delta_rule_norm_gate(q, k, v, beta, decay, ours, step, gate, w, 1e-6, dtype, act)
    want = mix_ops.head_norm_gate(mix_ops.gated_delta_rule(q, k, v, beta, decay, theirs, step), gate, w, 1e-6, dtype, act)
    S, o, at = state.double(), torch.zeros(T, H, D, dtype=torch.float64, device="cuda"), 0
    for b, n in enumerate(NEW):
        if n == 0:
            continue
        s = S[step.host_slots[b]] if CTX[b] > 0 else torch.zeros_like(S[0])
        kk, qq = (x[at].double().repeat_interleave(H // G, 0) for x in (k, q))
        s = s * (decay[at].double()[..., None] if channel else decay[at].double()[:, None, None])
        u = beta[at].double()[:, None] * (v[at].double() - (s * kk[..., None]).sum(1))
        s = s + kk[..., None] * u[:, None]
        o[at], S[step.host_slots[b]] = (s * qq[..., None]).sum(1), s
        at += 1
    y = o / torch.sqrt(o.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()
    g = gate.double().view(T, H, D)
    y = (y * (g * torch.sigmoid(g) if act == "silu" else torch.sigmoid(g))).view(T, H * D)
    err = lambda x, r: float((x.double() - r).norm() / r.norm())     # noqa: E731
    # f32 sums in another order: as far from float64 as the two launches, but for the luck of some hundred heads' norms
    assert err(ours, S) <= 1.05 * err(theirs, S) + 1e-9 and err(got, y) <= 1.05 * err(want, y) + 1e-9
    still = step.host_slots[NEW.index(0)]
    assert torch.equal(ours[still], state[still])


@pytest.mark.parametrize("new,ctx", [([3, 0, 0], [5, 4, 0]), ([0, 2, 1, 0], [0, 1, 2, 9])])
def test_rule_of_uneven_steps(new, ctx):
    gen = torch.Generator(device="cuda").manual_seed(3)
    rn = lambda *s: torch.randn(*s, device="cuda", generator=gen)    # noqa: E731
    T, G, H, D, step = sum(new), 2, 4, 128, make_step(new, ctx)
    q, k = (torch.nn.functional.normalize(rn(T, G, D), dim=-1) for _ in range(2))
    v, beta, decay, gate, w = rn(T, H, D), torch.sigmoid(rn(T, H)), torch.sigmoid(rn(T, H)), rn(T, H * D).bfloat16(), rn(D)
    state = rn(len(new), H, D, D)
    ours, theirs = state.clone(), state.clone()
    got = mix_ops.delta_rule_norm_gate(q, k, v, beta, decay, ours, step, gate, w, 1e-6, torch.bfloat16)
    want = mix_ops.head_norm_gate(mix_ops.gated_delta_rule(q, k, v, beta, decay, theirs, step), gate, w, 1e-6, torch.bfloat16)
    assert torch.equal(got, want) and torch.equal(ours, theirs)
