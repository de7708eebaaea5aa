"""The estimate of the prompt product's time (csrc/hip/gemm_prompt.hip) that the choice of the kernel at 257 - 512 rows goes by."""
import random

import pytest

from bigdl_amd import qtypes as Q
from bigdl_amd.ops import hip


@pytest.mark.parametrize("pair", [0, 1])
def test_every_format_is_priced_at_the_plan_that_is_launched(pair):
    """A plan's time is a + b f, with f the format's time of a k tile (sym_int4 1, nf4 1.26, fp6 1.39), and there is one plan for all formats:
    the three times lie on a line"""
    lib, rng = hip.lib(), random.Random(0)
    for _ in range(2000):
        m, n, k = rng.randint(257, 512), 8 * rng.randint(128, 1792), 128 * rng.randint(4, 112)
        t = [lib.bigdl_gemm_prompt_us(m, n, k, Q.ggml_tensor_qtype[f], pair) for f in ("sym_int4", "nf4", "fp6")]
        assert 0 < t[0] < t[1] < t[2]
        assert (t[1] - t[0]) / 0.26 == pytest.approx((t[2] - t[0]) / 0.39, rel=1e-4), (m, n, k, t)
