"""The chunked scan with step sizes where a value is not finite: infinities and NaNs appear where the token loop has them and nowhere else."""
import pytest
import torch

from light_vllm_amd import mix_ops
from tests.test_chunk_scan_gpu import REL, case, make_step, recurrence

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,Dv,H,G", [(128, 64, 4, 2), (64, 64, 3, 3), (64, 128, 2, 1)])
@pytest.mark.parametrize("where", ["state", "q", "k", "v", "nan", "huge", "none"])
def test_like_the_token_loop(monkeypatch, D, Dv, H, G, where):
    new = [100, 1, 64, 300]
    T = sum(new)
    gen = torch.Generator(device="cuda").manual_seed(7)
    u = (0.6 * torch.randn(T, 2 * G * D + H * Dv, device="cuda", generator=gen)).bfloat16()
    q, k, v = u[:, :G * D], u[:, G * D:2 * G * D], u[:, 2 * G * D:]
    a = torch.randn(T, H, device="cuda", generator=gen).bfloat16()
    p0, p1, p2 = (0.5 * torch.randn(H, device="cuda", generator=gen) for _ in range(3))
    state = torch.randn(4, H, D, Dv, device="cuda", generator=gen)
    t = 100 + 1 + 40                                     # inside the second chunk of the third sequence
    if where == "state":
        state[0, H - 1, 5, 7] = float("inf")
    elif where == "huge":
        state[0, H - 1, 5, 7] = 1e38
    elif where in ("q", "k", "v"):
        dict(q=q, k=k, v=v)[where][t, 3] = float("inf")
    elif where == "nan":
        v[t, 3] = float("nan")
    got = []
    for kernel in ("token", "chunk"):
        monkeypatch.setattr(mix_ops, "SCAN_KERNEL", kernel)
        st = state.clone()
        step = make_step(new, [9, 9, 0, 9])
        got.append((mix_ops.gated_scan(mix_ops.SCAN_STEP, q, k, v, a, p0, p1, step, st, H, G, D, Dv, p2=p2).view(T, H, Dv), st))
    for x, y in zip(*got):
        assert torch.equal(torch.isfinite(x), torch.isfinite(y))
        if where not in ("q", "v"):
            # one infinity a sum on both sides: the same sign. (An infinite v fills a column of the state, which a later token sums with the
            # signs of its q; the chunk multiplies it by one sum of q and k. An infinite q the other way round.)
            assert torch.equal(torch.isnan(x), torch.isnan(y)) and torch.equal(torch.isposinf(x), torch.isposinf(y))
        ok = torch.isfinite(x)
        # f32 sums of D + T terms on both sides, relative to their terms: the state's huge entry dominates the outputs that it reaches
        assert bool(((x - y)[ok].abs() <= 2.0 ** -24 * (D + 64) * 8 * (1 + x[ok].abs())).all())
    if where == "huge":
        far = got[1][0][sum(new[:3]):, H - 1, 7].abs()
        assert float(far[0]) > 1e30 and float(got[1][0].abs().amax()) < 1.1e38
    assert where in ("none", "huge") or not bool(torch.isfinite(got[1][0]).all())


@pytest.mark.parametrize("kind", ["delta", "const"])
@pytest.mark.parametrize("H,G,D,Dv,B", [(4, 4, 128, 128, 32), (4, 4, 128, 128, 33), (4, 2, 64, 64, 64), (4, 2, 64, 64, 65), (2, 2, 128, 256, 3), (2, 1, 128, 64, 2)])
def test_both_workgroup_sizes(monkeypatch, kind, H, G, D, Dv, B):
    """Launches on both sides of the rule that cuts workgroups in two, against float64 as the other shapes are."""
    monkeypatch.setattr(mix_ops, "SCAN_KERNEL", "chunk")
    G = H if kind == "const" else G
    new, ctx = [33 + i % 40 for i in range(B)], [3 * (i % 2) for i in range(B)]
    step = make_step(new, ctx)
    call, args, skip = case(kind, new, H, G, D, Dv, 11)
    state = torch.randn(B, H, D, Dv, device="cuda", generator=torch.Generator(device="cuda").manual_seed(12))
    want_o, want_s = recurrence(*args, state, step)
    o = call(state, step).view(sum(new), H, Dv)
    assert float((o.double() - want_o - skip).norm() / want_o.norm()) <= REL and float((state.double() - want_s).norm() / want_s.norm()) <= REL
