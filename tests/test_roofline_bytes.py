"""The byte counts that the roofline fractions of Loop64 and Loop32 go by are
those of what runs: every fragment's target listed, every fragment read once
by its tile's composite, every image element written; no slots, whatever K."""
import pytest

from vk_order_independent_transparency_amd import roofline


@pytest.mark.parametrize("F,P", [(0, 64), (1000, 437), (12_762_550, 1920 * 1080)])
@pytest.mark.parametrize("K", [1, 8, 32])
def test_tiled_frames_count_stream_and_image(F, P, K):
    for stages in (roofline.loop64_stage_bytes(F, P, K), roofline.loop32_stage_bytes(F, P, K),
                   roofline.loop64_stage_bytes(F, P, K, occupied=F // 2, tail=False),
                   roofline.loop32_stage_bytes(F, P, K, occupied=F // 2), roofline.tile_stage_bytes(F, P)):
        assert stages == {"clear": 0, "store": 4 * F, "resolve": 24 * F + 16 * P}
    with_runs = roofline.tile_stage_bytes(F, P, runs=77)
    assert sum(with_runs.values()) == 28 * F + 16 * P + 2 * 8 * 77
