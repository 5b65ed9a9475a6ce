"""The delta rule's chunks with norm and gate in the scan (lv_chunk_delta_norm) against the two launches that they replace: partial and whole
chunks, sequences with and without state and new tokens, both gates, all head sizes, gates as views of wider rows."""
import pytest
import torch

from light_vllm_amd import mix_ops
from tests._ragged import close, ragged_step

pytestmark = pytest.mark.gpu


def inputs(new, ctx, H, G, D, Dv, seed):
    step, _ = ragged_step(new, ctx, 64, "cuda", seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    T = sum(new)

    def rn(*shape):
        return torch.randn(*shape, device="cuda", generator=gen)

    unit = lambda x: x / x.norm(dim=-1, keepdim=True)  # noqa: E731
    a = dict(qn=unit(rn(T, G, D)) * D ** -0.5, kn=unit(rn(T, G, D)), v=rn(T, H, Dv), beta=torch.sigmoid(rn(T, H)), decay=torch.sigmoid(rn(T, H) + 2))
    return step, a, rn(len(new), H, D, Dv), rn(T, H * Dv + 24).bfloat16()[:, 8:8 + H * Dv], 1 + 0.2 * rn(Dv)


@pytest.mark.parametrize("H,G,D,Dv", [(8, 2, 128, 128), (8, 4, 64, 128), (16, 4, 64, 64), (16, 8, 128, 64)])
@pytest.mark.parametrize("gate_act", ["silu", "sigmoid"])
@pytest.mark.parametrize("new,ctx", [([97, 1, 31, 32, 33, 64, 0, 5] * 5, [0, 3] * 20), ([128] * 24, [0] * 24)])
def test_norm_and_gate_with_the_scan(monkeypatch, H, G, D, Dv, gate_act, new, ctx):
    monkeypatch.setattr(mix_ops, "SCAN_KERNEL", "chunk")
    step, a, state, gate, w = inputs(new, ctx, H, G, D, Dv, H + Dv)
    s0, s1 = state.clone(), state.clone()
    want = mix_ops.head_norm_gate(mix_ops.gated_delta_rule(**a, state=s0, step=step), gate, w, 1e-6, torch.bfloat16, gate_act)
    assert mix_ops._chunk_norm_ok(a["qn"], a["kn"], a["v"], a["decay"], s1, step, gate, torch.bfloat16)
    got = mix_ops.delta_rule_norm_gate(**a, state=s1, step=step, gate=gate, norm_w=w, eps=1e-6, act_dtype=torch.bfloat16, gate_act=gate_act)
    assert torch.equal(s0, s1)
    assert close(got, want.cpu(), torch.bfloat16)


def test_a_bad_token_reaches_no_earlier_one(monkeypatch):
    monkeypatch.setattr(mix_ops, "SCAN_KERNEL", "chunk")
    new = [100] * 24
    step, a, state, gate, w = inputs(new, [0] * 24, 8, 2, 128, 128, 5)
    run = lambda: mix_ops.delta_rule_norm_gate(**a, state=state.clone(), step=step, gate=gate, norm_w=w, eps=1e-6, act_dtype=torch.bfloat16)  # noqa: E731
    clean = run()
    a["v"][250] = float("nan")                     # token 50 of the third sequence
    y = run()
    bad = y.isnan().any(-1).nonzero()[:, 0].tolist()
    assert bad == list(range(250, 300))
    keep = ~y.isnan().any(-1)
    assert close(y[keep], clean[keep].cpu(), torch.bfloat16)      # (the chunk with it goes token by token)


def test_what_stays_with_two_launches(monkeypatch):
    monkeypatch.setattr(mix_ops, "SCAN_KERNEL", "chunk")
    step, a, state, gate, w = inputs([128] * 24, [0] * 24, 8, 2, 128, 128, 1)
    ok = lambda **kw: mix_ops._chunk_norm_ok(*{**dict(qn=a["qn"], kn=a["kn"], v=a["v"], decay=a["decay"], state=state, step=step, gate=gate,  # noqa: E731
                                                      act_dtype=torch.bfloat16), **kw}.values())
    assert ok() and not ok(act_dtype=torch.float32) and not ok(gate=gate.float(), act_dtype=torch.float32)
    few, b, s, g, _ = inputs([400] * 3, [0] * 3, 8, 2, 128, 128, 1)
    assert not ok(qn=b["qn"], kn=b["kn"], v=b["v"], decay=b["decay"], state=s, step=few, gate=g)
    assert not ok(decay=torch.ones(24 * 128, 8, 128, device="cuda"))
