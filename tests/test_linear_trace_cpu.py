"""The linear layers under what traces or rewrites torch's operators, and on operands that are no matrices: as torch's own linear."""
import pytest
import torch
import torch.nn.functional as F

from light_vllm_amd import mix_ops
from light_vllm_amd.layers.linear import ColumnParallelLinear, ReplicatedLinear, RowParallelLinear

K, N = 64, 32


def layer(cls):
    m = cls(K, N)
    for i, p in enumerate(m.parameters()):
        p.data.normal_(generator=torch.Generator().manual_seed(i))
    return m


class Projection(torch.nn.Module):
    def __init__(self):
        super().__init__()
        self.weight = torch.nn.Parameter(torch.randn(N, K, generator=torch.Generator().manual_seed(3)))

    def forward(self, x):
        return mix_ops.linear(x, self.weight)


def forms():
    return [layer(ReplicatedLinear), layer(ColumnParallelLinear), Projection()]


def rows(n):
    return torch.randn(n, K, generator=torch.Generator().manual_seed(n))


@pytest.mark.parametrize("i", range(3))
def test_symbolic_trace(i):
    m = forms()[i]
    traced = torch.fx.symbolic_trace(m)
    for n in (3, 64, 65):
        assert torch.equal(traced(rows(n)), F.linear(rows(n), m.weight))


@pytest.mark.parametrize("i", range(2))
def test_script(i):
    m = forms()[i]
    scripted = torch.jit.script(m)
    assert torch.equal(scripted(rows(5)), F.linear(rows(5), m.weight))


@pytest.mark.parametrize("m", [*forms(), layer(RowParallelLinear)])
def test_trace_export_compile(m):
    import warnings
    with warnings.catch_warnings():
        warnings.simplefilter("error", torch.jit.TracerWarning)        # nothing that a trace would fix
        traced = torch.jit.trace(m, rows(8))
    # any number of rows: neither the 64 that a kernel takes nor the example's
    dyn = torch.export.export(m, (rows(8),), dynamic_shapes=({0: torch.export.Dim("t", min=2, max=4096)},)).module()
    count = []

    def backend(g, _):
        count.append(g)
        return g.forward
    torch._dynamo.reset()
    whole = torch.compile(m, backend=backend, fullgraph=True)
    for n in (8, 9, 64, 65, 300):
        want = F.linear(rows(n), m.weight)
        assert torch.equal(traced(rows(n)), want) and torch.equal(dyn(rows(n)), want) and torch.equal(whole(rows(n)), want)
    assert len(count) == 2                                             # the first size, then any


@pytest.mark.parametrize("m", forms())
def test_operands_that_are_no_matrices(m):
    for x in (torch.tensor(1.0), [1.0], None):
        with pytest.raises(Exception) as want:
            F.linear(x, m.weight)
        with pytest.raises(want.type):
            m(x)
    for shape in ((K,), (0, K), (2, 3, K)):
        x = torch.randn(shape)
        assert torch.equal(m(x), F.linear(x, m.weight))
    assert torch.func.vmap(m)(torch.randn(2, 8, K)).shape == (2, 8, N)


def test_few_rows_are_not_asked_what_only_many_can_have(monkeypatch):
    """Eager steps of few tokens are bound by the host: a projection of theirs looks for the kernel of few rows only, one between for none."""
    asked = []
    for name in ("_split_sizes", "_rows_gemm_sizes"):
        monkeypatch.setattr(mix_ops, name, lambda x, w, name=name: asked.append((name, len(x))))
    m = layer(ReplicatedLinear)
    with torch.no_grad():
        for n in (8, 64, 65, 4095, 4096):
            assert torch.equal(m(rows(n)), F.linear(rows(n), m.weight))
    assert asked == [("_rows_gemm_sizes", 8), ("_rows_gemm_sizes", 64), ("_split_sizes", 4096), ("_rows_gemm_sizes", 4096)]
