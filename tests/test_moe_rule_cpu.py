"""Which eager steps multiply the experts' sorted rows on LDS tiles."""
import pytest

from light_vllm_amd.layers.moe import sorted_pays


@pytest.mark.parametrize("experts,width,ff,rows,tiled", [
    # measured, us, tiled / gathered: 57 / 39, 60 / 50, 61 / 111, 36 / 29, 31 / 35, 107 / 162, 47 / 39, 28 / 39
    (4, 2048, 1536, 16, False), (4, 2048, 1536, 32, False), (4, 2048, 1536, 48, True), (16, 1024, 512, 16, False), (64, 512, 256, 16, True),
    (32, 2048, 1536, 16, True), (16, 2048, 256, 32, False), (4, 512, 256, 48, True), (32, 2048, 1536, 15, False)])
def test_tiles_pay(experts, width, ff, rows, tiled):
    assert sorted_pays(True, rows * experts, experts, width, ff) == tiled


def test_other_weights_from_256_rows():
    assert not sorted_pays(False, 255 * 8, 8, 4096, 3072) and sorted_pays(False, 256 * 8, 8, 4096, 3072) and sorted_pays(True, 256 * 8, 8, 32, 32)
