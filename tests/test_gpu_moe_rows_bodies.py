"""Grouped GEMM of up to 320 routed rows a workgroup (csrc/moe_gemm_rows.h): an entry's row by a multiplication instead of a division."""
import pytest
import torch

import test_gpu_moe_rows as rows

pytestmark = pytest.mark.gpu


# (one, powers of two, what 2^32 leaves a rest of, more than there are entries)
@pytest.mark.parametrize("div", [1, 3, 6, 7, 8, 641, 100003])
def test_row_of_an_entry(div):
    rows.test_rows_of_every_body([130, 1, 320, 331, 40], 128, 64, div, torch.bfloat16)
