"""Host inputs and results of op-level calls: through the context's 1 MiB of
pinned memory where they fit, through the runtime's copies where they do not."""
import numpy as np
import pytest

from dotllm_amd import SamplingOptions
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 4097, 87296, 87381, 131072, 131073, 262144, 262145])
def test_two_inputs_and_a_result(hip, n):
    """Both inputs and the result inside; the result outside; the second input
    and the result outside; nothing inside.  Sums of two floats are exact to compare."""
    rng = np.random.default_rng(n)
    a, b = rng.standard_normal(n, dtype=np.float32), rng.standard_normal(n, dtype=np.float32)
    y = np.zeros(n, dtype=np.float32)
    for _ in range(2):
        hip.add(a, b, y)
        assert np.array_equal(y, a + b)
        a = -a


@pytest.mark.parametrize("n,recent", [(262077, 64), (262078, 65), (262143, 0), (5, 3)])
def test_sample_inputs(hip, n, recent):
    """Logits, recent tokens, draw and counter just inside and just outside."""
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n, dtype=np.float32) * 3
    rec = [int(i) for i in rng.integers(0, n, size=recent)]
    opt = SamplingOptions(top_k=3, top_p=0.9)
    for r in (0.0, 0.4, 0.99):
        want = O.sample(x, opt.temperature, opt.top_k, opt.top_p, opt.repeat_penalty, opt.repeat_penalty_window_size, rec, r)
        assert hip.sample(x, opt, rec, r) == want
