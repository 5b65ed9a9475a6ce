"""lv_chunk_scan rejects bad arguments on the host, before any launch, and which calls of the recurrences take it."""
import ctypes

import pytest
import torch

from light_vllm_amd import mix_ops
from tests._ragged import ragged_step
from tests._route import device, record


def test_argument_validation():
    from light_vllm_amd import _mixlib
    lib = _mixlib.load()
    buf = ctypes.create_string_buffer(256)
    p = (ctypes.addressof(buf) + 15) & ~15

    def call(kind=1, q=p, ldq=256, ldk=256, ldv=256, a=p, decay=p, p0=p, ws=p, nbytes=1 << 40, T=64, B=1, longest=64, H=2, G=2, D=64, Dv=64,
             seg=0):
        return lib.lv_chunk_scan(kind, q, ldq, p, ldk, p, ldv, a, 2, decay, p0, p, p, p, p, p, p, p, ws, nbytes, T, B, longest, H, G, D, Dv,
                                 seg, None)

    assert call(B=0) == 0 and call(T=0) == 0                        # nothing to do
    for bad in (dict(q=None), dict(ws=None), dict(kind=3), dict(kind=0, p0=None), dict(decay=None), dict(kind=2, a=None), dict(D=96),
                dict(Dv=96), dict(H=3), dict(ldq=100), dict(ldk=130), dict(q=p + 4), dict(kind=2, q=p + 8), dict(ws=p + 4), dict(seg=48),
                dict(longest=65), dict(longest=0)):
        assert call(**bad) == -1, bad
    assert call(nbytes=64) == -3
    need = lib.lv_chunk_scan_workspace_bytes
    assert need(1, 64, 1, 64, 2, 64, 64, 0) >= 64 * 2 * 34 * 4
    assert need(2, 64, 1, 64, 2, 64, 64, 32) >= 64 * 2 * 66 * 4      # the delta rule is never cut
    assert need(1, 64, 1, 64, 2, 64, 64, 32) > need(1, 64, 1, 64, 2, 64, 64, 64)
    assert need(1, -1, 1, 64, 2, 64, 64, 0) < 0


def lightning(off_q, off_k, off_v, width, H=2, D=64, Dv=64):
    step, _ = ragged_step([96, 3], [0, 0], 16, "cpu")
    proj = device(torch.zeros(99, width, dtype=torch.bfloat16))
    state = torch.zeros(2, H, D, Dv)
    return mix_ops.lightning_attention(proj, off_q, off_k, off_v, torch.full((H,), 0.9), state, step, H, D, Dv)


def test_columns_outside_the_row_are_refused(monkeypatch):
    """A head's columns that do not lie in the row of the projection are an argument error on long steps as on short ones."""
    calls = record(monkeypatch, real=("lv_lightning_attn",))
    lightning(0, 128, 256, 384)
    assert calls == ["lv_chunk_scan"]
    for bad in ((0, 128, 260, 384), (260, 0, 128, 384), (0, 400, 128, 384), (-4, 128, 256, 384), (0, 128, 256, 256)):
        with pytest.raises(RuntimeError):
            lightning(*bad)
    assert calls == ["lv_chunk_scan"]


def delta_call(state, D=64, Dv=64, H=2):
    step, _ = ragged_step([96, 3], [0, 0], 16, "cpu")
    rows = [device(torch.zeros(99, H, n)) for n in (D, D, Dv)]
    return mix_ops.gated_delta_rule(*rows, torch.zeros(99, H), torch.ones(99, H), state, step)


def test_state_off_a_16_byte_boundary_takes_the_token_loop(monkeypatch):
    """The chunked kernel's combine step reads states four entries at a time; a state that lies elsewhere is still served."""
    calls = record(monkeypatch, real=("lv_chunk_scan",))
    flat = torch.zeros(2 * 2 * 64 * 64 + 1)
    delta_call(flat[1:].view(2, 2, 64, 64))
    assert calls == ["lv_gated_delta_rule"]


def step_call(a_ld, H=2, D=64, Dv=64):
    step, _ = ragged_step([96, 3], [0, 0], 16, "cpu")
    q, k, v = (device(torch.zeros(99, H * n, dtype=torch.bfloat16)) for n in (D, D, Dv))
    a = torch.zeros(99, a_ld, dtype=torch.bfloat16)[:, :H] if a_ld >= H else torch.zeros(1, H, dtype=torch.bfloat16).expand(99, H)
    one = torch.zeros(H)
    return mix_ops.gated_scan(mix_ops.SCAN_STEP, q, k, v, a, one, one, step, torch.zeros(2, H, D, Dv), H, H, D, Dv, p2=one)


def test_step_sizes_that_share_a_row_are_refused(monkeypatch):
    """Row strides below the heads' count are an argument error on long steps as on short ones."""
    calls = record(monkeypatch, real=("lv_gated_scan",))
    step_call(4)
    assert calls == ["lv_chunk_scan"]
    record(monkeypatch, real=("lv_gated_scan", "lv_chunk_scan"))
    with pytest.raises(RuntimeError, match="bad sizes|strides"):
        step_call(0)


@pytest.mark.parametrize("kind,H,D,Dv,lens,chunks", [
    # measured, us, token loop / chunks: 30 / 25, 67 / 73, 228 / 119, 123 / 239, 61 / 74, 1030 / 328
    (2, 16, 128, 128, [32], True), (2, 16, 128, 128, [64] + [1] * 63, False), (2, 16, 128, 128, [256] + [1] * 63, True),
    (2, 16, 128, 128, [64] + [1] * 255, False), (2, 16, 64, 64, [32] + [1] * 255, False), (2, 16, 128, 128, [1024] * 16, True),
    # 159 / 209, 476 / 284, 57 / 40, 105 / 217
    (0, 32, 128, 64, [160] + [1] * 255, False), (0, 32, 128, 64, [640] + [1] * 255, True), (0, 32, 128, 64, [160], True),
    (0, 32, 128, 64, [80] + [1] * 255, False),
    # 19 / 21, 35 / 25, 104 / 149, 596 / 280; below every threshold
    (1, 32, 64, 64, [80], False), (1, 32, 64, 64, [160], True), (1, 32, 64, 64, [160] + [1] * 255, False), (1, 16, 128, 128, [1024] * 16, True),
    (1, 16, 128, 128, [1] * 64, False), (2, 16, 128, 128, [31], False)])
def test_which_steps_take_chunks(kind, H, D, Dv, lens, chunks):
    """A portion of a prompt beside many decoded tokens is the token loop's, where a chunk for every sequence would cost more."""
    assert mix_ops._chunk_pays(kind, lens, H, D, Dv) == chunks


@pytest.mark.parametrize("lens,wgs,seg", [([1024] * 16, 16, 0), ([4096], 16, 256), ([900, 3750, 2000, 1500, 2500, 1200, 2150], 16, 256), ([255], 16, 0),
                                          ([1, 1, 1], 16, 0), ([2048] * 8, 16, 512), ([5000], 2, 256)])
def test_segment_lengths(lens, wgs, seg):
    """Few long sequences are cut into multiples of a chunk; what fills the chip by itself, and short portions, are not."""
    got = mix_ops._segment_length(lens, wgs, wgs * 128 * 128 * 4)
    assert got == seg or (seg and got % 32 == 0 and 256 <= got < max(lens)), got
    assert (got > 0) == (seg > 0)


def test_segments_keep_their_states_within_256_mb():
    assert mix_ops._segment_length([4096] * 40, 1, 1 << 24) == 0
    for n in (1, 3, 40):
        seg = mix_ops._segment_length([4096] * n, 1, 1 << 20)
        assert seg == 0 or n * -(-4096 // seg) * (1 << 20) <= 1 << 28


@pytest.mark.parametrize("lens,H,Dv,pays", [([1024] * 16, 16, 128, True), ([500] * 32, 16, 64, True), ([60] * 30, 16, 128, True), ([900] * 6 + [100] * 6, 32, 128, False),
                                            ([4000] + [40] * 20, 16, 128, False)])
def test_where_the_norm_rides_with_the_scan(lens, H, Dv, pays):
    assert mix_ops._chunk_norm_pays(lens, H, Dv) == pays


@pytest.mark.parametrize("lens,H,Dv,D,pays", [
    ([750, 50, 400, 600] * 8, 16, 128, 128, False), ([750, 50, 400, 600] * 8, 32, 64, 64, True),
    ([700, 100, 350, 600] * 4, 32, 64, 128, False), ([1024] * 9, 16, 128, 128, False), ([64] * 9, 16, 128, 128, True)])
def test_where_the_norm_rides_by_head_sizes(lens, H, Dv, D, pays):
    assert mix_ops._chunk_norm_pays(lens, H, Dv, D) == pays


@pytest.mark.parametrize("lens,seg,H,D,Dv,front", [
    ([1024] * 16, 0, 16, 128, 128, False), ([1000], 0, 16, 128, 128, True), ([4000] + [300] * 12, 0, 16, 128, 128, True), ([1024] * 16, 0, 32, 128, 64, True),
    ([1024] * 16, 0, 32, 64, 64, False), ([64] * 256, 0, 32, 64, 64, True), ([120] * 128, 0, 32, 64, 64, False), ([4000] + [300] * 12, 0, 32, 64, 64, True),
    ([4096], 256, 32, 64, 64, False), ([4096], 256, 16, 128, 64, True), ([64] * 128, 0, 16, 64, 128, True)])
def test_workspace_of_constant_decays(lens, seg, H, D, Dv, front):
    """Launches that form their products in the scan keep none in memory: only the segments' states are asked for."""
    from light_vllm_amd import _mixlib
    T, B, segs = sum(lens), len(lens), -(-max(lens) // seg) if seg else 1
    got = _mixlib.load().lv_chunk_scan_workspace_bytes(1, T, B, max(lens), H, D, Dv, seg)
    assert got == 4 * ((T * H * 32 + 2 * (-(-T * H // 4) * 4) if front else 0) + (B * segs * H * (D * Dv + 1) if segs > 1 else 0))
