"""-m gpu: prompt GEMMs on codes with a team of waves for each quarter of the scale groups (csrc/lm_prefill.hip, k_gemm_pf_codes in up to 512 tiles of 64 x 64): two, three and five
groups (quarters of none, of one and of two), quarters of equal and of unequal length, a part of a tile in both directions - the comparisons of test_gpu_prompt_codes.py."""
import pytest

from test_gpu_prompt_codes import test_prompts_on_codes as prompts_on_codes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden, heads, ff, bits, total", [(320, 1, 192, 8, 101), (320, 1, 192, 4, 150), (1088, 3, 1216, 8, 193), (2048, 16, 4160, 8, 300), (2048, 16, 4160, 4, 417)])
def test_quarters(hidden, heads, ff, bits, total):
    prompts_on_codes(hidden, heads, ff, bits, total)
