"""Steps in two launches with one channel per lane (a KV head over two, four or eight waves): its workgroup sizes and the
sizes just beyond it, and the ends of supergroups, tiles and groups of tiles."""
import re

import pytest
import torch

from adkv_amd import _lib
from tests.test_gpu_segment_step import test_against_the_three_calls, test_error_against_64_bits, test_masked_segments_and_rows

pytestmark = pytest.mark.gpu


def _runs(B, Hq, H, D, T, bits, S):
    """What the library says a step starts with: the waves of a step_lone_kernel's workgroup, 0 for the other kernel."""
    tps = 32 // bits
    name = _lib.lib().adkv_decode_step_kernel_name(B, Hq, H, T, D, bits, (T + tps) // S + 1 if S else 0, S, 0).decode()
    return 0 if name == "step_segments_kernel" else int(re.fullmatch(r"step_lone_kernel, (\d+)-wave workgroups", name)[1])


@pytest.mark.parametrize("B,Hq,H,D,T,S,waves", [
    (4, 32, 32, 128, 1300, 256, 4), (5, 32, 32, 128, 1800, 256, 12), (6, 32, 32, 128, 2041, 256, 12), (7, 32, 32, 128, 2041, 256, 0),
    (4, 32, 16, 128, 1500, 256, 4), (8, 32, 16, 128, 1793, 256, 8), (9, 32, 16, 128, 2047, 256, 12), (13, 32, 16, 128, 2047, 256, 0),
    (2, 32, 8, 128, 6000, 256, 4), (3, 32, 8, 128, 9001, 256, 8), (6, 32, 8, 128, 7680, 256, 12), (7, 32, 8, 128, 7169, 256, 0),
    (3, 64, 8, 128, 4799, 256, 4), (5, 64, 8, 128, 5632, 256, 8), (9, 64, 8, 128, 3800, 256, 0),
    (2, 16, 16, 256, 3900, 256, 4), (2, 16, 16, 256, 5021, 256, 12), (4, 8, 8, 256, 7171, 256, 16), (5, 8, 8, 256, 7170, 256, 0),
    (1, 8, 8, 512, 3333, 256, 8), (3, 8, 8, 512, 3584, 256, 16), (10, 8, 8, 512, 1799, 256, 0),
])
def test_workgroup_sizes(gpu, oracle, B, Hq, H, D, T, S, waves):
    assert _runs(B, Hq, H, D, T, 4, S) == waves
    test_against_the_three_calls(gpu, oracle, B, Hq, H, D, T, 4, S, torch.float16)


@pytest.mark.parametrize("Hq,H,D", [(2, 2, 256), (3, 3, 512), (4, 2, 128), (4, 1, 128), (8, 1, 128)])
@pytest.mark.parametrize("T,S", [(0, 0), (1, 0), (7, 0), (8, 256), (63, 0), (72, 256), (80, 256), (129, 0), (255, 256), (256, 0),
                                 (257, 256), (264, 256), (281, 256), (330, 256), (512, 256), (200, 64)])
def test_ends_of_segments(gpu, oracle, Hq, H, D, T, S):
    """No supergroup, a half tile, a tile, a group of four and one more; 256 tokens and the appended one; segments of 64."""
    if S == 64 and Hq == H:
        pytest.skip("segments below 128 tokens of one query head per KV head keep the separate launches")
    assert _runs(2, Hq, H, D, T, 4, S) > 0
    test_against_the_three_calls(gpu, oracle, 2, Hq, H, D, T, 4, S, torch.bfloat16)


@pytest.mark.parametrize("Hq,H", [(2, 2), (4, 2), (4, 1), (8, 1)])
@pytest.mark.parametrize("T,S", [(0, 0), (1, 0), (15, 0), (16, 256), (17, 0), (40, 0), (144, 256), (255, 256), (256, 0), (257, 256),
                                 (271, 256), (272, 256), (330, 256), (512, 256), (200, 64)])
def test_two_bits(gpu, oracle, Hq, H, T, S):
    """A word of codes is a whole tile: no word, ragged ones of one to fifteen tokens, an odd and an even number of them."""
    assert _runs(2, Hq, H, 128, T, 2, S) > 0
    test_against_the_three_calls(gpu, oracle, 2, Hq, H, 128, T, 2, S, torch.float16)


@pytest.mark.parametrize("B,Hq,H,T,waves", [(4, 32, 32, 1300, 4), (6, 32, 32, 1900, 12), (7, 32, 32, 1900, 0), (8, 32, 16, 1793, 8),
                                            (12, 32, 16, 1800, 12), (3, 32, 8, 9001, 8), (6, 32, 8, 7680, 12), (2, 64, 8, 4000, 4),
                                            (5, 64, 8, 5632, 8), (8, 64, 8, 8000, 0)])
def test_two_bits_workgroup_sizes(gpu, oracle, B, Hq, H, T, waves):
    assert _runs(B, Hq, H, 128, T, 2, 256) == waves
    test_against_the_three_calls(gpu, oracle, B, Hq, H, 128, T, 2, 256, torch.bfloat16)


@pytest.mark.parametrize("low", [torch.finfo(torch.float32).min, float("-inf")])
@pytest.mark.parametrize("Hq,H,D", [(4, 4, 512), (8, 1, 128), (4, 2, 128)])
def test_masks(gpu, Hq, H, D, low):
    assert _runs(3, Hq, H, D, 768, 4, 256) > 0
    test_masked_segments_and_rows(gpu, 3, Hq, H, D, 768, low)


@pytest.mark.parametrize("q_scale", [0.3, 1.0])
@pytest.mark.parametrize("B,Hq,H,D,T,bits", [(9, 8, 8, 512, 700, 4), (6, 16, 16, 256, 1290, 4), (4, 32, 32, 128, 1100, 4), (12, 8, 2, 128, 1100, 4),
                                             (12, 16, 2, 128, 1500, 2)])
def test_no_further_from_64_bits(gpu, oracle, B, Hq, H, D, T, bits, q_scale):
    """One query head on the vector pipe and, with 512 channels, on the matrix cores; four and eight of them."""
    assert _runs(B, Hq, H, D, T, bits, 256) > 0
    test_error_against_64_bits(gpu, oracle, B, Hq, H, D, T, bits, q_scale)
