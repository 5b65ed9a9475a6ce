"""The autograd function around the projections' own kernel, with torch's product in the kernel's place: what it keeps and what it gives."""
import pytest
import torch
import torch.nn.functional as F

from light_vllm_amd import mix_ops


@pytest.fixture
def product(monkeypatch):
    monkeypatch.setattr(mix_ops, "_rows_gemm", lambda x, w, *a: torch.mm(x, w.t()))
    return lambda x, w: mix_ops._RowsLinear.apply(x, w, None)


def operands(gx, gw):
    gen = torch.Generator().manual_seed(4)
    return torch.randn(6, 8, generator=gen).requires_grad_(gx), torch.randn(5, 8, generator=gen).requires_grad_(gw)


@pytest.mark.parametrize("gx,gw", [(True, True), (True, False), (False, True)])
def test_keeps_what_torch_keeps(product, gx, gw):
    """An operand is kept only for the other one's gradient: what is not kept may be overwritten before the backward."""
    results = []
    for f in (product, F.linear):
        kept = []
        x, w = operands(gx, gw)
        h = x * 2 if gx else x                             # (no leaf: it may be written in place)
        with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(tuple(t.shape)) or t, lambda t: t):
            y = f(h, w)
        with torch.no_grad():
            if not gw:
                h.add_(1.0)
            if not gx:
                w.add_(1.0)
        y.square().sum().backward()
        results.append((sorted({(min(s), max(s)) for s in kept}), [t.grad for t in (x, w)]))
    (ours, got), (theirs, want) = results
    assert ours == theirs
    assert all(a is None and b is None or torch.allclose(a, b, rtol=1e-6) for a, b in zip(got, want))


def test_second_derivatives_and_batched_gradients(product):
    for f in (product, F.linear):
        x, w = (t.double().detach().requires_grad_() for t in operands(True, True))
        assert torch.autograd.gradgradcheck(f, (x, w))
    x, w = operands(True, True)
    dy = torch.randn(3, 6, 5, generator=torch.Generator().manual_seed(5))
    got = torch.autograd.grad(product(x, w), (x, w), dy, is_grads_batched=True)
    want = torch.autograd.grad(F.linear(x, w), (x, w), dy, is_grads_batched=True)
    assert all(torch.allclose(a, b, rtol=1e-5, atol=1e-6) for a, b in zip(got, want))


@pytest.mark.parametrize("N,K,pays,not_pays", [
    (48, 2048, (1, 64), ()), (4096, 6400, (1, 16, 17, 64), ()), (256, 8192, (), (1, 16, 64)), (4096, 12288, (), (1, 17, 64)), (5120, 17408, (1, 32), (33, 64)),
    (8192, 4096, (1, 17, 32, 48), (49, 64)), (8192, 3584, (1, 64), ()), (5120, 5120, (), (1, 17, 33, 64)), (10304, 4096, (1, 16), (17, 32, 33, 64)),
    (12800, 5120, (), (1, 16, 32, 64)), (34816, 5120, (1, 16), (17, 64)), (9000, 3072, (1, 16), (17, 33)), (12288, 2048, (16, 32), (33, 64)),
    (14336, 1024, (32,), (64,)), (16384, 4096, (32,), (64,)), (20480, 4096, (16, 32), (33, 64)), (26000, 4096, (16,), (32,)), (65536, 2048, (), (1, 32))])
def test_where_the_kernel_pays(N, K, pays, not_pays):
    """Both sides of the measured rule."""
    assert all(mix_ops.rows_gemm_pays(M, N, K) for M in pays) and not any(mix_ops.rows_gemm_pays(M, N, K) for M in not_pays)
