"""lv_latent_prep with four entries an access (a wave a token) against the torch path, at the edges of its rows and launches."""
import pytest
import torch

from light_vllm_amd import mix_ops
from tests._ragged import close, ragged_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Rq,R,Dr,dims", [(768, 192, 64, 64), (1536, 256, 0, 0), (4, 4, 8, 8), (2048, 512, 64, 32), (772, 196, 60, 56), (260, 640, 128, 128)])
@pytest.mark.parametrize("new,ctx", [([1], [0]), ([19, 1, 2], [40, 0, 63]), ([2045, 1, 5], [3, 100, 0])])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_norms_and_rotation(Rq, R, Dr, dims, new, ctx, dtype):
    gen = torch.Generator().manual_seed(Rq + new[0])
    T, page = sum(new), 64
    proj = torch.randn(T, Rq + R + Dr + 12, generator=gen).to(dtype)
    qw, kw = 1 + 0.3 * torch.randn(Rq, generator=gen), 1 + 0.3 * torch.randn(R, generator=gen)
    got = []
    for dev in ("cpu", "cuda"):
        step, pages = ragged_step(new, ctx, page, dev)
        cache = torch.full((pages, page, R + Dr), 9.0, dtype=dtype, device=dev)
        cq = mix_ops.latent_prep(proj.to(dev), 4, 8 + Rq, qw.to(dev), kw.to(dev), mix_ops.rotary_inv_freq(max(dims, 2), 10000.0, dev), cache, step,
                                 Rq, R, Dr, dims, 1e-6)
        got.append((cq, cache))
    assert close(got[1][0], got[0][0], dtype)
    # rotated entries are a sum of two products, each rounded: up to a rounding of the larger one, and of an angle of up to 2000
    tol = 2.0 ** -6 if dtype == torch.bfloat16 else 2.0 ** -11
    assert (got[1][1].cpu().float() - got[0][1].float()).abs().max().item() <= tol * 4
    untouched = got[0][1] == 9.0
    assert bool((got[1][1].cpu()[untouched] == 9.0).all())


@pytest.mark.parametrize("Rq,R,Dr,dims", [(768, 192, 64, 64), (1536, 256, 0, 0), (4, 4, 8, 8), (2048, 512, 64, 32), (772, 196, 60, 56), (260, 640, 128, 128)])
@pytest.mark.parametrize("new,ctx", [([70, 1, 6], [5, 0, 63]), ([2045, 1, 5], [3, 100, 0])])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_do_not_depend_on_the_kernel(Rq, R, Dr, dims, new, ctx, dtype):
    """Rows whose stride is no multiple of four go through the kernel of a thread an entry: the same bits."""
    gen = torch.Generator(device="cuda").manual_seed(R)
    T, page = sum(new), 64
    rows = torch.randn(T, Rq + R + Dr, device="cuda", generator=gen).to(dtype)
    qw, kw = (1 + 0.3 * torch.randn(n, device="cuda", generator=gen) for n in (Rq, R))
    step, pages = ragged_step(new, ctx, page, "cuda")
    got = []
    for pad in (0, 1):
        proj = torch.zeros(T, Rq + R + Dr + pad, dtype=dtype, device="cuda")
        proj[:, :Rq + R + Dr] = rows
        cache = torch.zeros(pages, page, R + Dr, dtype=dtype, device="cuda")
        cq = mix_ops.latent_prep(proj, 0, Rq, qw, kw, mix_ops.rotary_inv_freq(max(dims, 2), 10000.0, "cuda"), cache, step, Rq, R, Dr, dims, 1e-6)
        got.append((cq, cache))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
