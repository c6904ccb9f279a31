"""Steps in two launches whose values are replayed beside the keys (at most eight waves of keys per CU): segments around the
units that the values' waves hold (whole groups of eight, at most 24, 16 where waves are many), up to the most waves of either form
and one unit beyond."""
import pytest
import torch

from tests.test_gpu_segment_step import test_against_the_three_calls as against_the_calls

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hq,H,D,bits", [(3, 3, 256, 4), (3, 3, 512, 4), (6, 3, 128, 4), (12, 3, 128, 4), (24, 3, 128, 4), (3, 3, 128, 2), (12, 3, 128, 2)])
@pytest.mark.parametrize("T", [63, 64, 79, 80, 128, 191, 192, 199, 200, 208, 256, 257, 320, 449, 512])
def test_segments_around_what_is_held(gpu, oracle, Hq, H, D, bits, T):
    against_the_calls(gpu, oracle, 2, Hq, H, D, T, bits, 256, torch.float16)


# 512 units of two waves (256 of four) on 256 CUs, twice that, and four more of either; one query head, grouped, 2-bit, wide
@pytest.mark.parametrize("B,Hq,H,D,T,bits", [(2, 32, 32, 128, 2000, 4), (2, 32, 32, 128, 2100, 4), (4, 32, 16, 128, 2048, 4), (4, 32, 16, 128, 2049, 4),
                                             (8, 64, 8, 128, 2000, 4), (2, 32, 32, 128, 1999, 2), (2, 16, 16, 256, 2000, 4), (2, 16, 16, 256, 2064, 4),
                                             (4, 32, 32, 128, 2047, 4), (4, 32, 32, 128, 1800, 2), (8, 32, 16, 128, 2048, 4), (5, 32, 8, 128, 6400, 4),
                                             (5, 64, 8, 128, 5633, 4), (4, 16, 16, 256, 2040, 4), (3, 8, 8, 512, 2500, 4), (1, 8, 8, 512, 8192, 4)])
def test_most_waves(gpu, oracle, B, Hq, H, D, T, bits):
    against_the_calls(gpu, oracle, B, Hq, H, D, T, bits, 256, torch.bfloat16)
