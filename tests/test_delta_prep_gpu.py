"""lv_delta_prep's tiled form (heads of 64, 128 and 256, up to four taps) against the torch restatement on the CPU: tiles that
meet the ends of sequences, portions shorter than the filter, aligned and misaligned rows."""
import pytest
import torch

from light_vllm_amd import mix_ops
from tests._ragged import ragged_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,G,H", [(64, 1, 3), (128, 2, 4), (256, 1, 2), (32, 2, 2)])
@pytest.mark.parametrize("taps", [1, 2, 4, 5])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("per_channel", [False, True])
def test_against_the_restatement(D, G, H, taps, dtype, per_channel):
    for new, ctx, pad in (([1, 1, 1], [0, 1, 9], 0), ([17, 1, 2, 40, 3], [0, 2, 1, 0, 7], 4), ([700, 0, 5, 900], [1, 3, 0, 0], 2)):
        gen = torch.Generator().manual_seed(D + taps + len(new))
        T, nd = sum(new), D if per_channel else 1
        C = 2 * G * D + H * D
        wide = torch.randn(T, C + H + H * nd + pad + 2, generator=gen).to(dtype)
        conv_w, state = torch.randn(C, taps, generator=gen) * 0.5, torch.randn(len(new), taps - 1, C, generator=gen).to(dtype)
        A_log, dt_bias = 0.5 * torch.randn(H, generator=gen), 0.5 * torch.randn(H * nd, generator=gen)
        got = []
        for dev in ("cpu", "cuda"):
            step, _ = ragged_step(new, ctx, 16, dev)
            proj = wide.to(dev)[:, pad:]
            got.append(mix_ops.delta_prep(proj, conv_w.to(dev), state.to(dev), A_log.to(dev), dt_bias.to(dev), step, G, H, D, D, taps, C,
                                          proj[:, C + H:C + H + H * nd], 1e-6, per_channel))
        for a, b, name in zip(got[1], got[0], ("q", "k", "v", "beta", "decay")):
            # silu and the decays' exponentials are a few roundings off the CPU's; unit vectors have entries near zero
            assert (a.cpu() - b).abs().max().item() <= 2e-5 * max(1.0, b.abs().max().item()), name
