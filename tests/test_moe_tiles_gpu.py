"""The experts' products on LDS tiles (lv_moe_tiled_ff) against the sum in float64, at sizes where tiles end: one row, blocks of 64 and tiles of
256 rows and one more, widths beside a multiple of the 256 columns, k of half a step of 64 and in whole pairs of steps, experts without
rows, experts that hand their input through.

Bound: the intermediate row, the expert's output row and the result are each rounded to bf16 once (2^-9 relative; the gelus
also read a rounded product, whose error they pass on at most 1.13 times), sums are in f32. So the error of an element is at
most 2^-9 (2 S + |y|) with S = sum_k w_k |m_k| |W_down|, where |m| grows by 1.13 |z| for the gelus; 3.5 S covers |y| <= S and the
f32 sums."""
import pytest
import torch

from light_vllm_amd import mix_ops

pytestmark = pytest.mark.gpu

#        T     W    F    E  top  act         through   rows per expert about
CASES = [(1, 32, 32, 4, 2, "relu2", 0),
         (257, 64, 96, 1, 1, "relu2", 0),          # one expert: 257 rows, one past a tile
         (129, 288, 32, 2, 1, "gelu_tanh", 0),     # one past two blocks of 64 rows; k of half a step
         (256, 160, 288, 1, 1, "gelu", 0),
         (333, 32, 32, 16, 5, "relu2", 3),
         (2500, 544, 224, 5, 3, "relu2", 1),       # several runs of the sort
         (9000, 128, 128, 70, 2, "relu2", 0)]      # more experts than a wave scans at once
# more tiles than a round of 256 workgroups holds uncut: one row past the last tile, a part tile, several experts with one that no one
# chose, handed through
TALL = [(4097, 2080, 96, 1, 1, "relu2", 0), (4200, 2080, 224, 1, 1, "gelu", 0), (3000, 1568, 160, 4, 2, "relu2", 0),
        (1500, 2336, 288, 5, 4, "gelu_tanh", 2)]


def operands(T, W, F, E, top, through, ups, seed):
    g = torch.Generator().manual_seed(seed)
    h = torch.randn(T, W, generator=g).bfloat16()
    up = (torch.randn(E * ups * F, W, generator=g) * W ** -0.5).bfloat16()
    down = (torch.randn(W, E * F, generator=g) * F ** -0.5).bfloat16()
    score = torch.rand(T, E + through, generator=g)
    if E + through - 1 >= top and E > 2:
        score[:, 1] = -1.0                         # an expert without rows
    ids = score.topk(top, 1).indices.int().contiguous()
    return [x.cuda() for x in (h, ids, torch.rand(T, top, generator=g) + 0.1, up, down)]


def exact(h, ids, w, up, down, E, F, act, glu=None):
    y = torch.zeros(h.shape, dtype=torch.float64, device=h.device)
    S = torch.zeros_like(y)
    for e in range(int(ids.max()) + 1):
        r, k = (ids == e).nonzero(as_tuple=True)
        x, f = h[r].double(), w[r, k].double()[:, None]
        if e >= E:
            y.index_add_(0, r, x * f)
            S.index_add_(0, r, x.abs() * f)
            continue
        down_e = down[:, e * F:(e + 1) * F].double().T.contiguous()
        if glu is not None:
            z = x @ up[e * 2 * F:(e + 1) * 2 * F].double().T.contiguous() * f
            gate, lin = z[:, :F].clamp(max=glu[0]), z[:, F:].clamp(-glu[0], glu[0])
            m, f = gate * torch.sigmoid(glu[1] * gate) * (lin + 1.0), torch.ones_like(f)
            size = m.abs()
        else:
            z = x @ up[e * F:(e + 1) * F].double().T.contiguous()
            m = torch.relu(z) ** 2 if act == "relu2" else torch.nn.functional.gelu(z, approximate="tanh" if act == "gelu_tanh" else "none")
            size = m.abs() + (0 if act == "relu2" else 1.13 * z.abs())
        y.index_add_(0, r, (m @ down_e) * f)
        S.index_add_(0, r, (size @ down_e.abs()) * f)
    return y, S


@pytest.mark.parametrize("T,W,F,E,top,act,through", CASES + TALL)
def test_tiles_match_the_exact_sum(gpu, T, W, F, E, top, act, through):
    h, ids, w, up, down = operands(T, W, F, E, top, through, 1, T + F)
    assert mix_ops.moe_tiles_ok(h, up, down, E, F, 1, act, through)
    y = mix_ops.moe_sorted_ff(h, ids, w, up, down, E, F, act, through)
    ref, S = exact(h, ids, w, up, down, E, F, act)
    assert ((y.double() - ref).abs() <= 3.5 * 2.0 ** -9 * S + 1e-6).all()


@pytest.mark.parametrize("T,W,F,E,top,act,uneven", [(70, 256, 256, 1, 1, "relu2", 0), (600, 384, 256, 3, 1, "relu2", 0.3), (1500, 256, 640, 6, 2, "gelu", 1.0),
                                                    (2000, 2048, 512, 5, 4, "relu2", 1.0), (9000, 512, 1280, 3, 2, "gelu_tanh", 2.0),
                                                    (24000, 256, 256, 7, 3, "relu2", 2.0)])
def test_tiles_in_a_chain_match_the_exact_sum(gpu, T, W, F, E, top, act, uneven):
    """k in whole pairs of steps: workgroups go from tile to tile. Experts of 0 to 256 rows past a whole tile, fewer tiles than
    workgroups, a last round cut in two or four, and rounds that are whole."""
    h, _, w, up, down = operands(T, W, F, E, top, 0, 1, T + E)
    score = torch.rand(T, E, generator=torch.Generator().manual_seed(E)) + uneven * torch.linspace(0, 1, E)
    ids = score.topk(top, 1).indices.int().contiguous().cuda()
    for _ in range(2):                             # and the workgroups of a second launch behind those of the first
        y = mix_ops.moe_sorted_ff(h, ids, w, up, down, E, F, act)
    ref, S = exact(h, ids, w, up, down, E, F, act)
    assert ((y.double() - ref).abs() <= 3.5 * 2.0 ** -9 * S + 1e-6).all()


@pytest.mark.parametrize("T,W,F,E,top,through", [(3000, 256, 384, 5, 3, 2), (9000, 512, 256, 2, 2, 3), (40, 256, 256, 3, 1, 1)])
def test_chains_pass_over_the_tiles_of_experts_that_hand_through(gpu, T, W, F, E, top, through):
    h, ids, w, up, down = operands(T, W, F, E, top, through, 1, T + through)
    y = mix_ops.moe_sorted_ff(h, ids, w, up, down, E, F, "relu2", through)
    ref, S = exact(h, ids, w, up, down, E, F, "relu2")
    assert ((y.double() - ref).abs() <= 3.5 * 2.0 ** -9 * S + 1e-6).all()


@pytest.mark.parametrize("T,W,F", [(43000, 1024, 128), (43000, 128, 1024)])
def test_rows_written_past_the_caches(gpu, T, W, F):
    """Two choices of 43000 tokens: 176 MB of rows of 1024, the outputs of either product; every 41st token."""
    E, top = 3, 2
    h, ids, w, up, down = operands(T, W, F, E, top, 0, 1, W)
    y = mix_ops.moe_sorted_ff(h, ids, w, up, down, E, F)
    some = torch.arange(0, T, 41, device=h.device)
    ref, S = exact(h[some], ids[some], w[some], up, down, E, F, "relu2")
    assert ((y[some].double() - ref).abs() <= 3.5 * 2.0 ** -9 * S + 1e-6).all()


@pytest.mark.parametrize("T,W,F,E,top", [(1, 32, 32, 4, 2), (257, 96, 160, 1, 1), (700, 256, 288, 4, 2), (3000, 160, 96, 5, 3),
                                           (4097, 2080, 96, 1, 1), (2500, 1568, 224, 4, 2), (1100, 96, 2080, 5, 3),
                                           (3000, 512, 384, 5, 3)])
def test_gated_tiles_match_the_exact_sum(gpu, T, W, F, E, top):
    h, ids, w, up, down = operands(T, W, F, E, top, 0, 2, T)
    wide = torch.zeros(W, E * F + 64, dtype=torch.bfloat16, device=h.device)        # the experts' columns of a wider weight
    wide[:, :E * F] = down
    y = mix_ops.moe_sorted_glu_ff(h, ids, w, up, wide[:, :E * F], E, F, 2.0, 1.702)
    ref, S = exact(h, ids, w, up, down, E, F, None, (2.0, 1.702))
    assert ((y.double() - ref).abs() <= 3.5 * 2.0 ** -9 * S + 1e-6).all()


def test_operands_beside_the_rule_take_the_general_path(gpu):
    """Weights off the 16-byte grid, a strided input and 64-bit choices are multiplied as before, to the same sum."""
    T, W, F, E, top = 300, 64, 96, 4, 2
    h, ids, w, up, down = operands(T, W, F, E, top, 0, 1, 7)
    ref, S = exact(h, ids, w, up, down, E, F, "relu2")
    off = torch.empty(up.numel() + 1, dtype=up.dtype, device=up.device)[1:].view_as(up).copy_(up)
    strided = torch.zeros(T, 2 * W, dtype=h.dtype, device=h.device)[:, :W].copy_(h)
    for a, b in ((h, off), (strided, up)):
        assert not mix_ops.moe_tiles_ok(a, b, down, E, F)
        y = mix_ops.moe_sorted_ff(a, ids, w, b, down, E, F)
        # this path also rounds the product and its relu's square: two more roundings of m, the first doubled by the square
        assert ((y.double() - ref).abs() <= 6.5 * 2.0 ** -9 * S + 1e-6).all()


@pytest.mark.parametrize("T,W", [(600, 64), (9000, 1056)])
def test_a_bad_token_stays_alone(gpu, T, W):
    """A NaN in one token's row reaches that token's result and no other's."""
    F, E, top = 64, 2, 1
    h, ids, w, up, down = operands(T, W, F, E, top, 0, 1, 3)
    clean = mix_ops.moe_sorted_ff(h, ids, w, up, down, E, F)
    h[123, 5] = float("nan")
    y = mix_ops.moe_sorted_ff(h, ids, w, up, down, E, F)
    assert y[123].isnan().all()
    keep = torch.arange(T, device=h.device) != 123
    assert torch.equal(y[keep], clean[keep])
