"""Latent attention of prompt steps in one launch (lv_latent_prompt_attn) against float64 torch, at the edges of its query tiles, pages,
windows and head sizes, beside the path of batched products that it replaces, and the calls that stay with that path."""
import pytest
import torch

from light_vllm_amd import mix_ops
from light_vllm_amd.layers.latent_attention import LatentAttention
from light_vllm_amd.utils.context import reset_context, set_context
from tests._ragged import ragged_step

pytestmark = pytest.mark.gpu
# absorbed queries, probabilities, sums and outputs are rounded to bf16 (2^-9 of the value each, independent); a query's rounding
# moves a score of magnitude 1 by about 2^-9 too, and its probability with it
REL = 5.0 ** 0.5 * 2.0 ** -9


def layer(H, dim, rot, gate, window=1 << 30, sink=False, page=64, new=(), ctx=(), seed=0):
    old = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        R = 192 if rot else 256
        m = LatentAttention(256, H, dim, dim, 64, R, (dim + rot) ** -0.5, rot_dim=rot, rot_dims=rot, gate=gate, window=window, sink=sink).cuda()
    finally:
        torch.set_default_dtype(old)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    with torch.no_grad():
        for p in m.parameters():
            p.normal_(0.0, p.shape[-1] ** -0.5 if p.dim() == 2 else p.shape[1] ** -0.5 if p.dim() == 3 else 0.5, generator=gen)
    step, pages = ragged_step(list(new), list(ctx), page, "cuda", seed)
    m.bind_cache(pages, page, len(new), "cuda", torch.bfloat16)
    m.cache.normal_(generator=gen)
    h = torch.randn(sum(new), 256, device="cuda", generator=gen).bfloat16()
    return m, step, h


def inner(m, step, h):
    """Gated head outputs of the layer, [T, H * dim]: what o_proj is given."""
    seen = []
    hook = m.o_proj.register_forward_pre_hook(lambda mod, args: seen.append(args[0]))
    set_context(True, ragged=step)
    with torch.no_grad():
        m(h)
    reset_context()
    hook.remove()
    return seen[0]


@torch.no_grad()
def exact(m, step, h):
    """The same from the layer's own bf16 queries, cache rows and gates, in float64."""
    H, R, Dn, Dr = m.H, m.R, m.Dn, m.Dr
    proj = m.in_proj(h)
    cq = mix_ops.latent_prep(proj, 0, m.Rq, m.q_norm_weight, m.kv_norm_weight, m.inv_freq, m.cache, step, m.Rq, R, Dr, m.rot_dims, m.norm_eps)
    q = m.uq(cq).double().view(-1, H, Dn + Dr)
    gate = torch.sigmoid(proj[:, m.sizes[0] + m.sizes[1]:].double())
    rows, outs, at = m.cache.double(), [], 0
    for b, (n, c) in enumerate(zip(step.host_lens_q, step.host_ctx_lens)):
        k = torch.cat([rows[p] for p in step.host_block_tables[b]])[:c + n]
        pos = torch.arange(c, c + n, device="cuda")
        x = q[at:at + n]
        a = torch.einsum("thd,hdr->htr", x[..., :Dn], m.uk.double())
        if Dr:
            u, v = x[..., Dn:Dn + Dr // 2], x[..., Dn + Dr // 2:]
            ang = (pos.float()[:, None] * m.inv_freq[None]).double()[:, None]
            a = torch.cat([a, torch.cat([u * ang.cos() - v * ang.sin(), v * ang.cos() + u * ang.sin()], -1).transpose(0, 1)], -1)
        s = a @ k.t() * m.scale
        d = pos[:, None] - torch.arange(c + n, device="cuda")[None]
        s = s.masked_fill((d < 0) | (d >= m.window), float("-inf"))
        if m.sink is not None:
            s = torch.cat([s, m.sink.double()[:, None, None].expand(H, n, 1)], -1)
        p = torch.softmax(s, -1)[..., :c + n]
        o = torch.einsum("htr,hrd->thd", p @ k[:, :R], m.uv.double())
        g = gate[at:at + n]
        outs.append((o * (g.view(n, H, Dn) if m.gate_per_channel else g[:, :, None])).reshape(n, H * Dn))
        at += n
    return torch.cat(outs)


@pytest.mark.parametrize("H,dim,rot,gate", [(4, 64, 64, "head"), (16, 128, 64, "head"), (8, 128, 0, "channel"), (4, 64, 0, "channel"), (12, 128, 64, "channel")])
@pytest.mark.parametrize("new,ctx,kw", [([17], [0], {}), ([32, 33, 1], [0, 31, 64], {}), ([130, 64, 7], [0, 1, 300], dict(page=128)),
                                        ([300, 90], [5, 0], dict(window=70)), ([65, 200], [63, 0], dict(sink=True))])
def test_against_float64(H, dim, rot, gate, new, ctx, kw, monkeypatch):
    m, step, h = layer(H, dim, rot, gate, new=new, ctx=ctx, seed=H + new[0], **kw)
    calls = []
    one = mix_ops.latent_prompt_attention
    monkeypatch.setattr(mix_ops, "latent_prompt_attention", lambda *a, **k: calls.append(1) or one(*a, **k))
    got = inner(m, step, h)
    assert calls
    monkeypatch.setattr(mix_ops, "latent_prompt_ok", lambda *a: False)
    general, want = inner(m, step, h), exact(m, step, h)
    err = [(x.double() - want).norm().item() / want.norm().item() for x in (got, general)]
    assert err[0] <= REL and err[0] <= 1.02 * err[1], err


@pytest.mark.parametrize("dim,rot,gate", [(128, 64, "head"), (64, 0, "channel")])
def test_rows_that_are_not_finite_reach_only_the_queries_that_see_them(dim, rot, gate):
    new, ctx, page = [100, 45], [0, 70], 64
    m, step, h = layer(4, dim, rot, gate, window=50, page=page, new=new, ctx=ctx, seed=9)
    want = inner(m, step, h)
    m.cache[step.host_block_tables[1][0], 40, 3] = float("inf")                 # position 40 of the second: its queries up to position 89 see it
    h = h.clone()
    got = inner(m, step, h)
    bad = ~torch.isfinite(got.float()).all(-1)
    assert bad.nonzero()[:, 0].tolist() == list(range(100, 100 + 20))
    assert torch.allclose(got[~bad].float(), want[~bad].float(), rtol=2.0 ** -6, atol=2.0 ** -6)


def test_what_stays_with_the_batched_products():
    m, step, h = layer(4, 64, 64, "head", new=[40], ctx=[0])
    q, gate = torch.empty(40, 4 * 128, device="cuda", dtype=torch.bfloat16), torch.empty(40, 4, device="cuda", dtype=torch.bfloat16)

    def ok(**kw):
        a = dict(q=q, cache=m.cache, uk=m.uk, uv=m.uv, gate=gate, step=step, H=4, Dn=64, Dr=64, R=192, rot_dims=64, gate_per_channel=False)
        return mix_ops.latent_prompt_ok(*{**a, **kw}.values())

    assert ok()
    short, _ = ragged_step([16, 3], [0, 9], 64, "cuda")
    assert not ok(step=short) and not ok(rot_dims=32) and not ok(H=6) and not ok(q=q.float())
    assert not ok(cache=torch.empty(2, 48, 256, device="cuda", dtype=torch.bfloat16))
    assert not ok(uk=torch.empty(4, 192, 64, device="cuda", dtype=torch.bfloat16).transpose(1, 2))
    assert not ok(uv=torch.empty(4 * 192 * 64 + 4, device="cuda", dtype=torch.bfloat16)[4:].view(4, 192, 64))
    assert not ok(gate=torch.empty(40, 4 * 64 + 2, device="cuda", dtype=torch.bfloat16)[:, 2:], gate_per_channel=True)


@pytest.mark.parametrize("H,dim,rot", [(4, 64, 64), (16, 128, 64), (8, 128, 0)])
def test_outputs_are_those_of_the_separate_launches(H, dim, rot, monkeypatch):
    """With matrices that hand entries through, sums have one term and any order is the same: rotation, attention and a gate per head
    leave the bits that they leave in launches of their own."""
    m, step, h = layer(H, dim, rot, "head", new=[130, 33, 1], ctx=[70, 0, 64], seed=H)
    with torch.no_grad():
        m.uk.copy_(torch.eye(dim, m.R))
        m.uv.copy_(torch.eye(m.R, dim))
    got = inner(m, step, h)
    monkeypatch.setattr(mix_ops, "latent_prompt_ok", lambda *a: False)
    assert torch.equal(got, inner(m, step, h))


@pytest.mark.parametrize("scale", [0.0, -0.07])
def test_scales_that_are_not_positive(scale):
    m, step, h = layer(4, 128, 64, "head", new=[40, 3], ctx=[0, 70], seed=2)
    m.scale = scale
    got, want = inner(m, step, h), exact(m, step, h)
    assert (got.double() - want).norm().item() <= REL * want.norm().item()


@pytest.mark.parametrize("new", [[40, 3], [9, 3]])
def test_the_output_projection_keeps_its_gradient(new, monkeypatch):
    """The kernels between carry none, on steps of either length and with either form of the products: the same weights have one."""
    m, step, h = layer(4, 64, 64, "head", new=new, ctx=[0, 70], seed=1)
    m.requires_grad_(True)
    set_context(True, ragged=step)
    try:
        grads = []
        for general in (False, True):
            if general:
                monkeypatch.setattr(mix_ops, "latent_prompt_ok", lambda *a: False)
            m.zero_grad()
            m(h).float().square().sum().backward()
            grads.append({n for n, p in m.named_parameters() if p.grad is not None})
        assert grads == [{"o_proj.weight"}] * 2
    finally:
        reset_context()


@pytest.mark.parametrize("H,dim,rot,gate", [(4, 128, 64, "head"), (8, 64, 0, "channel")])
def test_a_prompt_beside_many_decoded_sequences(H, dim, rot, gate, monkeypatch):
    """One query of a wave's 32 in use, or none, at contexts around tiles and pages."""
    new, ctx = [1] * 30 + [37, 0, 1], [63 * i % 200 for i in range(30)] + [0, 5, 64]
    m, step, h = layer(H, dim, rot, gate, new=new, ctx=ctx, seed=4)
    calls = []
    one = mix_ops.latent_prompt_attention
    monkeypatch.setattr(mix_ops, "latent_prompt_attention", lambda *a, **k: calls.append(1) or one(*a, **k))
    got, want = inner(m, step, h), exact(m, step, h)
    assert calls and (got.double() - want).norm().item() <= REL * want.norm().item()
