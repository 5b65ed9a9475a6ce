"""A latent attention layer on the CPU is torch ops throughout: every parameter and the input get gradients."""
import pytest
import torch

from light_vllm_amd.layers.latent_attention import LatentAttention
from light_vllm_amd.utils.context import reset_context, set_context
from tests._ragged import ragged_step


@pytest.mark.parametrize("gate,rot", [("head", 8), ("channel", 0)])
def test_gradients_on_the_cpu(gate, rot):
    gen = torch.Generator().manual_seed(3)
    m = LatentAttention(64, 4, 32, 32, 48, 40, 32 ** -0.5, rot_dim=rot, rot_dims=rot, gate=gate)
    for p in m.parameters():
        torch.nn.init.normal_(p, std=0.2, generator=gen)
    step, pages = ragged_step([1, 9, 4], [0, 0, 0], 16, "cpu")
    m.bind_cache(pages, 16, 3, "cpu", torch.float32)
    h, probe = torch.randn(14, 64, generator=gen), torch.randn(14, 64, generator=gen)
    set_context(True, ragged=step)
    try:
        x = h.clone().requires_grad_()
        loss = (m(x) * probe).sum()
        loss.backward()
        assert x.grad is not None and all(p.grad is not None for p in m.parameters())
        # the slope along the up projections' gradient, from two more passes: f32 passes of about 1e-6, a step of 1e-3
        g = {p: p.grad.clone() for p in (m.uk, m.uv)}
        size = sum((v * v).sum() for v in g.values()).sqrt()
        ends = []
        for sign in (1.0, -1.0):
            with torch.no_grad():
                for p, v in g.items():
                    p.add_(v, alpha=sign * 1e-3 / size.item())
                ends.append((m(h) * probe).sum().item())
                for p, v in g.items():
                    p.sub_(v, alpha=sign * 1e-3 / size.item())
        assert (ends[0] - ends[1]) / 2e-3 == pytest.approx(size.item(), rel=0.05)
    finally:
        reset_context()
