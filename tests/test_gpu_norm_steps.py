"""RMSNorm on both sides of every number of loads that a row may take from the threads of its workgroup: the entry point, and the norm in front of the
first projection of a prompt."""
import pytest

import test_gpu_norm_widths as widths
import test_gpu_prompt_angles as prompt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [d for k in range(2, 8) for d in (1024 * k - 4, 1024 * k, 1024 * k + 4)])
@pytest.mark.parametrize("offset", [0, 1])
def test_rows(d, offset):
    widths.test_against_64_bits(d, offset)


@pytest.mark.parametrize("d_model", [1280, 2048, 2560, 3072, 4608, 5120, 6400, 7168, 8192, 8704])
def test_prompt(d_model):
    prompt.check(dict(n_layers=1, d_model=d_model, n_heads=2, n_kv_heads=1, head_dim=64, d_ff=256), 41)
