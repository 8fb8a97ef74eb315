"""Decode steps of the recurrences where a workgroup's convolution channels meet the two a thread that are fetched in front of the state:
as many, fewer and more of them, and more taps than that form has (ssm_step_kernel, delta_step_kernel)."""
import pytest
import torch

import test_gpu_recurrence_chunks as steps

pytestmark = pytest.mark.gpu


# (channels of a workgroup of 256: 512, 504, 576, 40, 192, 576; taps in and beyond the early form)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,N,E,taps", [(6, 2, 240, 32, 3), (12, 1, 244, 16, 4), (4, 2, 256, 64, 4), (300, 4, 4, 32, 4), (10, 2, 64, 64, 5), (4, 2, 256, 64, 7)])
def test_state_space_step_channels(dtype, H, G, N, E, taps):
    steps.test_state_space_decode_step(dtype, H, G, N, E, taps, 1)


# (2 D + E H / G channels: 2336 for 512 threads, 1024 for 512, 384 for 1024, a head each of several workgroups; taps in and beyond the early form)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,D,E,taps", [(774, 86, 16, 256, 4), (6, 1, 128, 128, 4), (4, 1, 64, 64, 3), (24, 1, 128, 64, 4), (774, 86, 16, 256, 6), (8, 2, 128, 128, 5)])
def test_delta_rule_step_channels(dtype, H, G, D, E, taps):
    steps.test_delta_rule_decode_step(dtype, H, G, D, E, taps)
