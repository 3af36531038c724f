"""Steps of several tokens whose workgroups walk several units of the weights: as many as are in flight, more, and a last one that is
ragged; rows of one unit, of two, and such that end inside one.  Reference and bound are those of test_gpu_linear_step."""
import numpy as np
import pytest

import lopazen_cases as lc
import test_gpu_linear_step as steps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [2, 5, 8])
@pytest.mark.parametrize("n", [4096, 8197, 12293, 16400, 24600])
@pytest.mark.parametrize("k", [960, 2048, 3001, 4096])
def test_units(k, n, tokens):
    if k > 2048 and n > 12293:
        n //= 2
    r = np.random.default_rng(k + n + tokens)
    x = r.standard_normal((tokens, k)).astype(np.float32)
    w = lc.round_bf16(r.standard_normal((n, k)).astype(np.float32))
    steps.near(steps.step(x, w, "bfloat16", n_split=n // 4 * 2)[0], x, w[:n // 4 * 2])
