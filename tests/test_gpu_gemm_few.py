"""bfloat16 products of few rows and many columns, one pass over the weights: every number of 16 rows, a k in one unit and in two that ends
inside one, tiles that do not fill the last round; each form of the outputs.  Reference and bounds are those of the tests of the tiles."""
import pytest

import test_gpu_decoder_sizes as floats

pytestmark = pytest.mark.gpu

FEW = [(1, 8192), (9, 8196), (16, 12310), (17, 8192), (32, 16390)]
K = [64, 960, 1088, 2048, 2112, 4096]
# k that ends inside a unit and still fills it well enough for this pass, by the rows of A that it is made for
FILLED = {16: [512, 576, 832, 960, 1536, 2048, 3136, 4096], 32: [1792, 2048, 3648, 4096]}


@pytest.mark.parametrize("k", K)
@pytest.mark.parametrize("split,glu", [("all", 0), ("all", 1), ("half", 2), ("none", 0)])
@pytest.mark.parametrize("m,n", FEW)
def test_few_rows(m, n, split, glu, k):
    floats.test_gemm_tiles(m, n, {"all": n, "half": n // 64 * 32, "none": 0}[split], glu, k, "bfloat16")


@pytest.mark.parametrize("split,glu", [("all", 0), ("half", 2)])
@pytest.mark.parametrize("m,n", FEW)
def test_units_that_are_not_full(m, n, split, glu):
    for k in FILLED[16 if m <= 16 else 32]:
        if k not in K:
            floats.test_gemm_tiles(m, n, {"all": n, "half": n // 64 * 32}[split], glu, k, "bfloat16")


def test_infinite_weights_behind_a_part():
    """What lies behind the k of a row is not looked at: an infinite weight at the end of a row meets its own value alone."""
    import numpy as np
    from flexllm_amd import ops, to_device
    from flexllm_amd.loader import from_bf16, to_bf16
    import lopazen_cases as lc
    r = np.random.default_rng(3)
    a, w = lc.round_bf16(r.uniform(0.5, 1.0, (11, 576))), lc.round_bf16(r.standard_normal((8192, 576)))
    w[5, 575] = np.inf
    y = from_bf16(ops.linear_float(to_device(to_bf16(a)), to_device(to_bf16(w)))[0].numpy())
    assert np.isposinf(y[:, 5]).all() and np.isfinite(np.delete(y, 5, 1)).all()
