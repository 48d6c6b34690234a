"""Which tiles the fp32 experts' products take (llm_sharding_amd/ops/moe.py tile_rows)."""
import pytest

from llm_sharding_amd.ops.moe import tile_rows


@pytest.mark.parametrize("mean,experts,cols,rows", [
    (12, 32, 2048, 16), (16, 32, 2048, 32), (24, 32, 2048, 32), (25, 32, 2048, 64), (42, 32, 2048, 64), (95, 64, 1024, 64), (112, 64, 1024, 64),
    (50, 16, 2048, 64), (70, 16, 2048, 64), (115, 24, 2048, 128), (125, 8, 2048, 64), (125, 8, 4096, 128), (200, 32, 2048, 128)])
def test_fp32_tiles(mean, experts, cols, rows):
    """Tall tiles from 113 pairs an expert on, where there are 160 of them."""
    assert tile_rows(mean * experts, experts, True, cols) == rows
    assert tile_rows(mean * experts, experts, True) == (128 if mean > 112 else rows)
