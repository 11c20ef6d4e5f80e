"""Tree kernels whose chunks end in a tile of 32 or of 64 of 96 samples, in both primary trees, with
staggered subbands and two batches, bit for bit against the oracle."""

import pytest

from gpu_cases import CASES
from gpu_harness import run_and_compare

pytestmark = pytest.mark.gpu


# 320 = 3 x 96 + 32 and 160 = 96 + 64 samples; 640 = 6 x 96 + 64 and 320
@pytest.mark.parametrize('dtype,chunk', [('float32', 320), ('float32', 640), ('float16', 640), ('bfloat16', 640)])
def test_remainders(dtype, chunk):
    print(f'[tree remainders] {dtype} {chunk}', flush=True)
    bad, _, _ = run_and_compare(dict(CASES['half_tile'], dtype=dtype, time_samples_per_chunk=chunk), 3, seed=chunk, log=print)
    assert not bad, f'first mismatch: {bad[0]}'
