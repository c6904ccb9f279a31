"""Steps in one launch, whose values are replayed beside the keys: segments around the tokens that the values' waves
hold (whole groups of 64), one to four segments, with a tail and without."""
import pytest

from tests.test_gpu_lone import test_the_step_and_the_calls_agree_bit_for_bit as agree

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,S", [(63, 0), (64, 0), (71, 0), (72, 0), (127, 0), (128, 0), (255, 256), (256, 256), (263, 0), (328, 0), (1535, 0),
                                 (300, 256), (319, 256), (320, 256), (511, 256), (512, 256), (1024, 512), (577, 256), (640, 256), (767, 256),
                                 (768, 256), (1152, 512), (831, 256), (832, 256), (904, 256), (1023, 256), (1024, 256), (1300, 512)])
def test_values_beside_keys(gpu, T, S):
    agree(gpu, T, S)
