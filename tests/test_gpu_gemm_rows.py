"""GEMMs on tiles of 256 columns: every number of rows that a workgroup takes, with the last row tile and the last columns not filled and as
many stages of k as the ring holds and more.  References and bounds are those of the tests of the other tiles."""
import pytest

import test_gpu_decoder_sizes as floats
import test_gpu_gemm_tiles as ints
from test_gpu_prefill import fx  # noqa: F401

pytestmark = pytest.mark.gpu

# rows of a workgroup: rows and columns of a product
FLOAT = {96: (371, 12272), 128: (589, 12272), 160: (1299, 12272), 192: (1632, 12288), 224: (2076, 6128), 256: (1151, 12272)}
FLOAT_K = [320, 576]
INT = {(128, 1152): (300, 12284), (160, 1152): (1558, 6144), (192, 1152): (1632, 6140), (224, 384): (2076, 6144), (224, 1152): (1928, 6140),
       (256, 384): (1151, 12284), (256, 1152): (1151, 12288)}


@pytest.mark.parametrize("k", FLOAT_K)
@pytest.mark.parametrize("split,glu", [("all", 0), ("all", 1), ("all", 2), ("half", 0), ("half", 2), ("none", 0), ("odd", 0)])
@pytest.mark.parametrize("rows", FLOAT)
def test_rows_bfloat16(rows, split, glu, k):
    """Outputs on either side of a split between waves; a split inside a wave's columns goes to other tiles."""
    m, n = FLOAT[rows]
    floats.test_gemm_tiles(m, n, {"all": n, "half": n // 512 * 256 + 128, "none": 0, "odd": n // 512 * 256 + 64}[split], glu, k, "bfloat16")


@pytest.mark.parametrize("rows", FLOAT)
def test_bias(rows):
    """Added in float32 ahead of the rounding, on both sides of the split, columns that do not fill the last wave among them."""
    import numpy as np
    import lopazen_cases as lc
    from flexllm_amd import ops, to_device
    from flexllm_amd.loader import from_bf16, to_bf16
    (m, n), k = FLOAT[rows], 320
    split, r = n // 512 * 256, np.random.default_rng(rows)
    a, w, bias = lc.round_bf16(r.standard_normal((m, k))), lc.round_bf16(r.standard_normal((n, k))), r.standard_normal(n).astype(np.float32)
    y, y32 = ops.linear_float(to_device(to_bf16(a)), to_device(to_bf16(w)), split, bias=to_device(bias))
    want = a.astype(np.float64) @ w.astype(np.float64).T + bias
    d = 1e-5 * np.sqrt(k)                                 # as for the tiles
    assert np.all(np.abs(from_bf16(y.numpy()) - want[:, :split]) <= 2.0 ** -8 * np.abs(want[:, :split]) + d)
    assert np.all(np.abs(y32.numpy() - want[:, split:]) <= 1e-5 * np.abs(want[:, split:]) + d)


@pytest.mark.parametrize("rows,k", INT)
def test_rows_int8(fx, oracle, rows, k):  # noqa: F811
    m, n = INT[rows, k]
    ints.test_tiles(fx, oracle, m, k, n)
    ints.test_half_line_tiles_with_the_gated_unit(fx, m, k, n)


def test_outputs_of_4_gib(fx):  # noqa: F811
    """The bytes of the rows behind a tile's first one need more than 32 bits: first rows, rows on both sides of 2 GiB, last rows."""
    import numpy as np
    from flexllm_amd import synth
    m, k, n = 65536, 1024, 16384
    assert fx.lib().flexllm_linear_i8_gemm_rows(m, k, n, 0) == 256      # on the wide tiles
    a, w = synth.device_i8((m, k), 3), synth.device_i8((n, k), 4)
    s_x, w_s, res = synth.device_uniform_f32((m,), 5, 0.01, 0.02), synth.device_uniform_f32((n,), 6, 1e-3, 1e-2), synth.device_uniform_f32((m, n), 7, -1, 1)
    rows = np.r_[0:4, 126:130, 32766:32770, 65404:65412, 65534:65536]
    ha, hw = a.numpy()[rows].astype(np.float64), w.numpy().astype(np.float64)
    want = (ha @ hw.T).astype(np.int64).astype(np.int32)
    some = lambda y: np.stack([y.view(4 * n * int(r), (n,)).numpy() for r in rows])  # noqa: E731
    acc = fx.ops.linear_i8_gemm(a, w)
    assert np.array_equal(some(acc), want)
    del acc
    y = fx.ops.linear_i8_gemm_dequant(a, s_x, w, w_s, residual=res)
    assert np.array_equal(some(y), (want.astype(np.float32) * s_x.numpy()[rows, None]) * w_s.numpy() + some(res))
