"""Grouped GEMM of up to 320 routed rows a workgroup (csrc/moe_gemm_rows.h): its bodies for every 32 rows, and an entry's row by a
multiplication instead of a division."""
import pytest
import torch

import test_gpu_moe_rows as rows

pytestmark = pytest.mark.gpu


# (one, powers of two, what 2^32 leaves a rest of, more than there are entries)
@pytest.mark.parametrize("div", [1, 3, 6, 7, 8, 641, 100003])
def test_row_of_an_entry(div):
    rows.test_rows_of_every_body([130, 1, 320, 331, 40], 128, 64, div, torch.bfloat16)


# a tile is as long as its rows ask for in steps of 32, its second half shorter than its first at every other of them: on both sides of each step, in
# the last row tile of an expert too (its weights have another reader), with and without the entries' weights, SiLU * up
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,K,n_out", [([128, 129, 160, 161, 192, 193, 224, 225, 256, 257, 288, 289, 320], 128, 112),
                                            ([320 + 159, 320 + 161, 320 + 224, 320 + 226, 640 + 287, 640 + 289, 31], 384, 144)])
def test_every_count_of_row_fragments(counts, K, n_out, dtype):
    rows.test_rows_of_every_body(counts, K, n_out, 2, dtype)
