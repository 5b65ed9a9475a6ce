"""Queries joined in place (lv_latent_q_finish without q_lat), the four-entry output gate, and a latent attention layer under
autograd's default mode."""
import pytest
import torch

from light_vllm_amd import mix_ops
from light_vllm_amd.layers.latent_attention import LatentAttention
from light_vllm_amd.utils.context import reset_context, set_context
from tests._ragged import close, ragged_step

pytestmark = pytest.mark.gpu
NEW, CTX = [1, 40, 7], [3, 0, 33]


@pytest.mark.parametrize("H,Dn,Dr,R,dims", [(2, 8, 8, 16, 8), (16, 128, 64, 192, 64), (3, 12, 16, 20, 8), (2, 8, 12, 16, 12), (2, 6, 6, 10, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rotation_beside_the_absorbed_part(H, Dn, Dr, R, dims, dtype):
    gen = torch.Generator().manual_seed(Dr)
    T = sum(NEW)
    q, lat = torch.randn(T, H * (Dn + Dr), generator=gen).to(dtype), torch.randn(T, H, R, generator=gen).to(dtype)
    got = []
    for dev in ("cpu", "cuda"):
        step, _ = ragged_step(NEW, CTX, 16, dev)
        out = torch.full((T, H, R + Dr), 9.0, dtype=dtype, device=dev)
        out[:, :, :R] = lat.to(dev)
        mix_ops.latent_q_finish(q.to(dev), None, mix_ops.rotary_inv_freq(dims, 10000.0, dev), step, H, Dn, Dr, R, dims,
                                out=out.view(T, H * (R + Dr)))
        got.append(out)
    assert torch.equal(got[1][:, :, :R].cpu(), lat)
    assert (got[1].cpu().float() - got[0].float()).abs().max().item() <= (4 * 2.0 ** -7 if dtype == torch.bfloat16 else 2e-5)


@pytest.mark.parametrize("H,Dv,pad", [(2, 4, 0), (16, 128, 4), (3, 20, 2), (2, 6, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_output_gate(H, Dv, pad, dtype):
    gen = torch.Generator().manual_seed(H)
    o, gate = torch.randn(H, 37, Dv, generator=gen).to(dtype), torch.randn(37, H * Dv + pad, generator=gen).to(dtype)
    want = mix_ops.latent_out_gate(o, gate[:, pad:], True)
    assert close(mix_ops.latent_out_gate(o.cuda(), gate.cuda()[:, pad:], True), want, dtype)


@pytest.mark.parametrize("gate,rot", [("head", 8), ("channel", 0)])
def test_layer_runs_with_and_without_gradients(gate, rot):
    old = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        m = LatentAttention(64, 4, 32, 32, 48, 40, 32 ** -0.5, rot_dim=rot, rot_dims=rot, gate=gate).cuda()
    finally:
        torch.set_default_dtype(old)
    for p in m.parameters():
        torch.nn.init.normal_(p, std=0.2)
    step, pages = ragged_step(NEW, [0, 0, 0], 64, "cuda")
    m.bind_cache(pages, 64, 3, "cuda", torch.bfloat16)
    h = torch.randn(sum(NEW), 64, device="cuda").bfloat16()
    set_context(True, ragged=step)
    y = m(h)
    with torch.inference_mode():
        z = m(h)
    reset_context()
    assert torch.equal(y.detach(), z)
