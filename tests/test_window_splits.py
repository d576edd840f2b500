"""How many key splits a windowed token step takes (``seqmix.window_token_splits``)."""
import pytest

from loqa_hub_amd.ops import seqmix


@pytest.mark.parametrize("ctx,window,keep,tiles", [(2048, 1024, 0, 32), (2048, 1024, 4, 33), (2048, 1023, 33, 34), (1026, 1024, 4, 33), (1024, 1024, 4, 32),
                                                   (700, 1024, 4, 22), (2048, 0, 4, 64), (1, 0, 0, 1), (2049, 0, 0, 65), (40, 1, 0, 1)])
def test_tiles_are_those_of_the_kernel(ctx, window, keep, tiles):
    assert seqmix.window_token_tiles(ctx, window, keep) == tiles
    # as the kernel has them for the last row, and for no earlier one more
    def rows(pos):
        hi, lo = pos, max(0, pos - window + 1) if window else 0
        kept = min(keep, lo, hi + 1) if window else 0
        return -(-kept // 32) + max(hi - lo + 32, 0) // 32
    assert max(rows(p) for p in range(ctx)) == tiles


@pytest.mark.parametrize("window,rows,D,splits", [(1024, 32, 128, 8), (1024, 64, 128, 8), (1024, 128, 128, 4), (512, 32, 128, 4), (512, 128, 128, 4),
                                                  (512, 32, 64, 1), (1024, 32, 64, 8), (300, 32, 128, 1), (1024, 256, 128, 2)])
def test_splits_of_whole_windows(window, rows, D, splits):
    assert seqmix.window_token_splits(seqmix.window_token_tiles(2048, window, 0), rows, D) == seqmix._window_token_plan(2048, window, 0, rows, D) == splits
