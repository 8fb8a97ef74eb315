"""Rows per block of the expert GEMMs of prompts: blocks of 320 rows where they were measured ahead."""
import pytest

from semi_pd_amd import ops
from semi_pd_amd.layers import moe


# (calls on both sides of the line, and the quotient of their times with blocks of 256 or 128 rows and of 320)
@pytest.mark.parametrize("E,K,F,top,tokens,quotient", [
    (64, 2048, 1408, 6, 500, 1.12), (64, 2048, 1408, 6, 3001, 1.34), (64, 2048, 1408, 6, 8192, 1.11), (128, 2048, 768, 8, 2048, 1.19), (256, 2048, 512, 8, 1500, 1.17),
    (8, 4096, 14336, 2, 500, 1.28), (8, 4096, 14336, 2, 2048, 1.18), (8, 4096, 1792, 2, 2048, 1.39), (8, 4096, 1792, 2, 2600, 0.85), (8, 2048, 1024, 2, 4096, 1.25),
    (8, 2048, 1024, 2, 3001, 0.91), (8, 2048, 1024, 2, 5000, 0.86), (16, 4096, 1024, 4, 2048, 1.36), (16, 4096, 1024, 4, 2600, 0.87), (32, 1024, 512, 4, 2048, 0.92),
    (32, 1024, 512, 4, 4096, 1.49), (32, 1024, 512, 4, 6000, 0.95), (32, 2048, 1024, 4, 2048, 1.39), (32, 2048, 1024, 4, 2600, 0.93)])
def test_blocks_of_320_rows_where_they_are_ahead(monkeypatch, E, K, F, top, tokens, quotient):
    monkeypatch.setitem(ops._DENSE_GEMM, "cus", 0)
    numel = tokens * top
    block_m = 256 if numel >= moe.MOE_TALL_MIN_ROWS and numel >= moe.MOE_TALL_MIN_ROWS_PER_EXPERT * E else 128
    assert moe._tall_block(block_m, tokens, top, E, K, F) == (320 if quotient > 1 else block_m)


def test_rounds_are_those_of_the_share(monkeypatch):
    """8 experts of 4096 x 1792, 3500 tokens: as many rounds of either tiles on the whole chip, fewer of 320 rows on 192 CUs (403 / 349 us)."""
    took = []
    for cus in (0, 256, 192):
        monkeypatch.setitem(ops._DENSE_GEMM, "cus", cus)
        took.append(moe._tall_block(256, 3500, 2, 8, 4096, 1792))
    assert took == [256, 256, 320]
