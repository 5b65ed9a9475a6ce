"""Up to 64 columns of a projection of many rows (lv_columns_gemm) against float64, and projections in two launches (mix_ops.linear) against
torch's linear: which calls take them, and that a row's values are the product's."""
import pytest
import torch
import torch.nn.functional as F

from light_vllm_amd import _mixlib, mix_ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def case(M, N, K, seed, lead=0):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.empty(M, K + lead, dtype=torch.bfloat16, device=DEV).normal_(generator=gen)[:, lead:]
    w = torch.empty(N, K + lead, dtype=torch.bfloat16, device=DEV).normal_(0.0, K ** -0.5, generator=gen)[:, lead:]
    return x, w


def bound(x, w):
    """One rounding to bf16 and K f32 additions."""
    ref = x.double() @ w.double().t()
    return ref, ref.abs() * 2.0 ** -8 + (x.double().abs() @ w.double().abs().t()) * x.size(1) * 2.0 ** -24


# rows around the 32 of a workgroup, columns around its tiles of 16, 32 and 64, k in halves of a piece and in fewer pieces than waves
@torch.inference_mode()
@pytest.mark.parametrize("M", [1, 31, 33, 4097])
@pytest.mark.parametrize("N", [1, 16, 17, 32, 33, 63, 64])
@pytest.mark.parametrize("K,lead", [(32, 0), (416, 8), (2048, 0)])
def test_columns(M, N, K, lead):
    x, w = case(M, N, K, 100 * M + N, lead)
    y = torch.full((M, N + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    _mixlib.check(_mixlib.load().lv_columns_gemm(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), y.data_ptr() + 8, N + 8, M, N, K,
                                                 torch.cuda.current_stream().cuda_stream), "lv_columns_gemm")
    ref, most = bound(x, w)
    assert bool(((y[:, 4:4 + N].double() - ref).abs() <= most).all())
    assert bool((y[:, :4] == 7).all()) and bool((y[:, 4 + N:] == 7).all())


@torch.inference_mode()
@pytest.mark.parametrize("M,N,K,lead", [(4096, 4128, 1024, 0), (8192, 2064, 1024, 8), (16384, 1040, 2048, 0)])
def test_in_two_launches(M, N, K, lead):
    x, w = case(M, N, K, M + N, lead)
    assert mix_ops._split_sizes(x, w) is not None
    y = mix_ops.linear(x, w)
    ref, most = bound(x, w)
    assert y.shape == (M, N) and y.is_contiguous() and bool(((y.double() - ref).abs() <= most).all())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        z = mix_ops.linear(x, w)
    for _ in range(3):
        z.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(z, y)


def test_which_calls_are_split():
    x, w = case(4096, 4128, 1024, 3)
    with torch.inference_mode():
        assert mix_ops._split_sizes(x, w) is not None
    odd, _ = case(4096, 8, 1028, 4)
    for a, b in [(x[:4095], w), (x, w[:4096]), (x, w[:4064]), (x[:, :960], w[:, :960]), (odd[:, :1024], w), (x.float(), w.float()),
                 (x.view(4, 1024, 1024), w), (x.t().contiguous().t(), w), (x, w.t().contiguous().t())]:
        assert mix_ops._split_sizes(a, b) is None
        assert torch.equal(mix_ops.linear(a, b), F.linear(a, b))
    a, b = x.clone().requires_grad_(), w.clone().requires_grad_()
    for p, q in [(a, w), (x, b)]:
        assert mix_ops._split_sizes(p, q) is None and mix_ops.linear(p, q).requires_grad


# rows whose last tile of 256 is a part (of one row, of all but one), in whole rounds all the same
@torch.inference_mode()
@pytest.mark.parametrize("M,N,K,lead", [(7937, 2064, 1024, 0), (8191, 2112, 1088, 8), (16129, 1040, 1024, 0), (16300, 1028, 1024, 0)])
def test_in_two_launches_of_odd_rows(M, N, K, lead):
    x, w = case(M, N, K, M + N, lead)
    assert mix_ops._split_sizes(x, w) is not None and mix_ops._split_sizes(x[:M // 256 * 256 - 256], w) is None
    y = mix_ops.linear(x, w)
    ref, most = bound(x, w)
    assert y.shape == (M, N) and y.is_contiguous() and bool(((y.double() - ref).abs() <= most).all())
