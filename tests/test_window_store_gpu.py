"""The four-entry forms of lv_qk_fullnorm_store and lv_pool_update against the torch restatements on the CPU: the largest and
smallest rows they take, rows they leave to the general form, blocks that straddle pages and steps."""
import pytest
import torch

from light_vllm_amd import mix_ops
from tests._ragged import close, ragged_step

pytestmark = pytest.mark.gpu
NEW, CTX = [1, 40, 7, 90], [3, 0, 33, 70]


@pytest.mark.parametrize("H,G,D,Dv,pad", [(2, 1, 4, 4, 0), (16, 4, 128, 128, 0), (32, 8, 128, 64, 4), (32, 8, 128, 128, 0), (33, 3, 128, 128, 0),
                                          (16, 16, 80, 128, 0), (4, 2, 6, 5, 1), (4, 2, 64, 64, 2)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_norm_and_store(H, G, D, Dv, pad, dtype):
    gen = torch.Generator().manual_seed(H + D)
    a, b, c = H * D, (H + G) * D, (H + G) * D + G * Dv
    wide = torch.randn(sum(NEW), c + pad, generator=gen).to(dtype)
    q_w, k_w = torch.randn(H * D, generator=gen), torch.randn(G * D, generator=gen)
    got = []
    for dev in ("cpu", "cuda"):
        step, pages = ragged_step(NEW, CTX, 16, dev)
        proj = wide.to(dev)[:, pad:]
        kc, vc = torch.zeros(pages, 16, G, D, dtype=dtype, device=dev), torch.zeros(pages, 16, G, Dv, dtype=dtype, device=dev)
        q = mix_ops.qk_fullnorm_store(proj[:, :a], proj[:, a:b], proj[:, b:c], q_w.to(dev), k_w.to(dev), kc, vc, step, H, G, D, Dv, 1e-6)
        got.append((q, kc, vc))
    assert close(got[1][0], got[0][0], dtype) and close(got[1][1], got[0][1], dtype)
    assert torch.equal(got[1][2].cpu(), got[0][2])


@pytest.mark.parametrize("P", [1, 3, 8, 16, 20, 64])
@pytest.mark.parametrize("G,D,Dv", [(1, 4, 4), (4, 128, 128), (2, 64, 32), (1, 6, 3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_pooled_means(P, G, D, Dv, dtype):
    gen = torch.Generator().manual_seed(P + D)
    _, pages = ragged_step(NEW, CTX, 16, "cpu")
    kc, vc = torch.randn(pages, 16, G, D, generator=gen).to(dtype), torch.randn(pages, 16, G, Dv, generator=gen).to(dtype)
    pp = mix_ops.pooled_slots(16, P)
    got = []
    for dev in ("cpu", "cuda"):
        step, _ = ragged_step(NEW, CTX, 16, dev)
        kp, vp = torch.zeros(pages, pp, G, D, dtype=dtype, device=dev), torch.zeros(pages, pp, G, Dv, dtype=dtype, device=dev)
        mix_ops.pool_update(kc.to(dev), vc.to(dev), kp, vp, step, G, D, Dv, P)
        got.append((kp, vp))
    for a, b in zip(got[1], got[0]):
        assert (a.cpu().float() - b.float()).abs().max().item() <= (2.0 ** -7 if dtype == torch.bfloat16 else 1e-6) * max(1.0, b.abs().max().item())
