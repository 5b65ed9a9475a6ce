"""lv_rows_gemm (projections of up to 64 rows) against float64, over the edges of its tiles and its k loop, and which calls take it."""
import pytest
import torch
import torch.nn.functional as F

from light_vllm_amd import mix_ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def case(M, N, K, seed, lead=0, lead_w=0):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.empty(M, K + lead, dtype=torch.bfloat16, device=DEV).normal_(generator=gen)[:, lead:]
    w = torch.empty(N, K + lead_w, dtype=torch.bfloat16, device=DEV).normal_(0.0, K ** -0.5, generator=gen)[:, lead_w:]
    return x, w


@torch.inference_mode()
@pytest.mark.parametrize("M", [1, 16, 17, 33, 48, 64])
@pytest.mark.parametrize("N,K,lead", [(1, 32, 0), (15, 64, 8), (16, 96, 0), (33, 544, 0), (132, 2080, 64), (1040, 2048, 0), (2600, 1024, 0),
                                      (5152, 512, 0), (8208, 768, 8), (10304, 256, 0)])
def test_against_float64(M, N, K, lead):
    check(M, N, K, lead)


# both halves of a last piece of k, first and last rows of a tile and columns that leave remainders, in tiles (16-row blocks, 16-column
# blocks) of 1 x 1, 1 x 2, 2 x 2, 3 x 2 and 4 x 2; rows of x and of w inside wider ones
@torch.inference_mode()
@pytest.mark.parametrize("Ms,N", [((1, 15, 33, 48), 1041), ((2, 16), 5170), ((49, 63), 1045), ((17, 31, 32), 5170), ((50, 64), 2607), ((33, 47, 48), 5170),
                                  ((49, 63, 64), 5170)])
@pytest.mark.parametrize("K", [32, 544, 576])
@pytest.mark.parametrize("lead,lead_w", [(0, 0), (8, 24)])
def test_tiles(Ms, N, K, lead, lead_w):
    for M in Ms:
        check(M, N, K, lead, lead_w)


def check(M, N, K, lead=0, lead_w=0):
    x, w = case(M, N, K, 1000 * M + N, lead, lead_w)
    y = mix_ops._rows_gemm(x, w, (M, N, K, K + lead, K + lead_w, x.get_device()))       # whether or not it pays
    assert not mix_ops.rows_gemm_ok(x, w) or torch.equal(y, mix_ops.linear(x, w))
    ref = x.double() @ w.double().t()
    # one rounding to bf16 (half a unit in the last place, 2^-9 of the value at most) and K f32 additions in chains of their own
    bound = ref.abs() * 2.0 ** -8 + (x.double().abs() @ w.double().abs().t()) * K * 2.0 ** -24
    assert y.shape == (M, N) and bool(((y.double() - ref).abs() <= bound).all())


@torch.inference_mode()
def test_a_row_does_not_depend_on_the_others():
    x, w = case(64, 5152, 2048, 5)
    whole = mix_ops.linear(x, w)
    for rows in (slice(0, 1), slice(3, 20), slice(16, 49), slice(30, 64)):
        assert torch.equal(mix_ops.linear(x[rows], w), whole[rows])


@torch.inference_mode()
def test_a_graph_replays_it():
    x, w = case(9, 2048, 2048, 6)
    mix_ops.linear(x, w)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = mix_ops.linear(x, w)
    for i in range(3):
        x.copy_(case(9, 2048, 2048, 7 + i)[0])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, mix_ops.linear(x, w))


def test_calls_that_stay_with_torch():
    x, w = case(8, 64, 64, 8)
    assert mix_ops.rows_gemm_ok(x, w)
    with torch.inference_mode():
        assert not mix_ops.rows_gemm_ok(*case(65, 64, 64, 8)) and not mix_ops.rows_gemm_ok(x[:0], w)
        assert not mix_ops.rows_gemm_ok(*case(8, 64, 48, 8)) and not mix_ops.rows_gemm_ok(*case(8, 64, 64, 8, lead=1))
        assert not mix_ops.rows_gemm_ok(x.float(), w.float()) and not mix_ops.rows_gemm_ok(x.view(2, 4, 64), w)
        assert not mix_ops.rows_gemm_ok(x, w.t()) and not mix_ops.rows_gemm_ok(x[:, ::2], w[:, ::2])
        assert not mix_ops.rows_gemm_ok(*case(64, 20480, 4096, 8)) and mix_ops.rows_gemm_ok(*case(32, 20480, 4096, 8))
        assert not mix_ops.rows_gemm_ok(*case(17, 10304, 4096, 8)) and mix_ops.rows_gemm_ok(*case(16, 10304, 4096, 8))
        with torch.autocast("cuda", dtype=torch.float16):
            assert not mix_ops.rows_gemm_ok(x, w)
        with torch.device("cuda"):               # a default device, as the engine sets one
            assert mix_ops.rows_gemm_ok(x, w)
    with torch.no_grad():
        several = torch.func.vmap(lambda row: mix_ops.linear(row, w))(x.view(2, 4, 64))
        assert torch.allclose(several.view(8, 64).float(), F.linear(x, w).float(), atol=0.05)
        with torch.autograd.forward_ad.dual_level():
            tangent = torch.autograd.forward_ad.unpack_dual(mix_ops.linear(torch.autograd.forward_ad.make_dual(x, x), w)).tangent
        assert tangent is not None


def test_gradients():
    x, w = case(8, 96, 64, 9)
    got, want = [], []
    for f, to in ((mix_ops.linear, got), (F.linear, want)):
        a, b = x.clone().requires_grad_(), torch.nn.Parameter(w.clone())
        y = f(a, b)
        y.square().sum().backward()
        to += [y.detach(), a.grad, b.grad]
    with torch.inference_mode():
        assert torch.equal(got[0], mix_ops.linear(x, w))
    for a, b in zip(got, want):                 # the outputs differ by roundings to bf16, the gradients with them
        assert float((a.double() - b.double()).norm() / b.double().norm()) < 2.0 ** -7
    once = mix_ops.linear(x.clone().requires_grad_(), w)
    assert once.grad_fn is not None and mix_ops.linear(x, w).grad_fn is None
