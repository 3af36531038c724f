"""Every tile of the int8 GEMM on the GPU: rows and columns that do not fill the last tile, fewer and more stages than the ring
holds, each epilogue; exact against integer products and the oracle's arithmetic."""
import numpy as np
import pytest

import test_gpu_prefill as prefill
from test_gpu_prefill import fx  # noqa: F401

pytestmark = pytest.mark.gpu

TILES = [(1024, 128, 16384), (1021, 256, 16380), (1000, 128, 8192), (897, 384, 8188), (1000, 1024, 4096), (1023, 1024, 3972), (1000, 512, 2048),
         (961, 128, 1924), (100, 640, 1028), (1, 128, 4), (200, 192, 516), (100, 2048, 1028), (3700, 1152, 2060),
         (1021, 640, 16380), (1000, 1024, 8188), (900, 1152, 2052), (1530, 128, 4092), (700, 640, 4092), (700, 384, 2052)]
# k a multiple of 64 alone: stages of 64-byte rows, fewer and more of them than the four of the ring
HALF = [(1021, 320, 16380), (1024, 2112, 16384), (1000, 64, 8192), (897, 320, 8188), (1023, 2112, 3972), (1000, 192, 4096), (961, 64, 1924), (1000, 1088, 2048),
        (1, 64, 4), (100, 448, 1028), (900, 2112, 8188), (900, 2112, 2052)]
QKV = [(1056, 33, 11, 64, 2048), (640, 96, 32, 0, 2048), (1024, 16, 4, 0, 2048), (1056, 33, 11, 64, 1088), (640, 96, 32, 0, 64), (1024, 16, 4, 0, 320),
       (96, 8, 2, 64, 192), (1120, 24, 4, 64, 512), (640, 96, 32, 0, 2112), (1024, 16, 4, 0, 2112), (96, 8, 2, 64, 256)]


@pytest.mark.parametrize("m,k,n", TILES + HALF)
def test_tiles(fx, oracle, m, k, n):  # noqa: F811
    r = np.random.default_rng(m + k + n)
    a, w = r.integers(-128, 128, (m, k)).astype(np.int8), r.integers(-128, 128, (n, k)).astype(np.int8)
    ref = (a.astype(np.float64) @ w.astype(np.float64).T).astype(np.int64).astype(np.int32)      # exact: |sum| < 2^31
    da, dw = fx.to_device(a), fx.to_device(w)
    assert np.array_equal(fx.ops.linear_i8_gemm(da, dw).numpy(), ref)
    s_x, w_s = r.uniform(0.01, 0.02, m).astype(np.float32), r.uniform(1e-3, 1e-2, n).astype(np.float32)
    res = r.standard_normal((m, n)).astype(np.float32)
    y = fx.ops.linear_i8_gemm_dequant(da, fx.to_device(s_x), dw, fx.to_device(w_s), residual=fx.to_device(res)).numpy()
    assert np.array_equal(y, oracle.residual(oracle.dequant(ref, s_x, w_s), res))
    b_x, w_sum = r.uniform(-1, 0, m).astype(np.float32), r.uniform(-1, 1, n).astype(np.float32)
    y = fx.ops.linear_i8_gemm_dequant_asym(da, fx.to_device(s_x), fx.to_device(b_x), dw, fx.to_device(w_s), fx.to_device(w_sum)).numpy()
    assert np.array_equal(y, oracle.dequant(ref, s_x, w_s, b_x=b_x, w_sum=w_sum))


@pytest.mark.parametrize("m,k,n", HALF)
def test_half_line_tiles_with_the_gated_unit(fx, m, k, n):  # noqa: F811
    """SiLU(gate) * up in the epilogue is the dequantising product and the gate layer, bit for bit."""
    r = np.random.default_rng(m + k + n)
    a, w = [fx.to_device(r.integers(-127, 128, s).astype(np.int8)) for s in ((m, k), (n, k))]
    s_x, w_s, b_x, w_sum = [fx.to_device(r.uniform(lo, hi, c).astype(np.float32)) for lo, hi, c in ((.01, .02, m), (1e-3, 1e-2, n), (-1, 0, m), (-1, 1, n))]

    def unit(y):
        return fx.ops.swiglu_f32(*(fx.to_device(np.ascontiguousarray(y.numpy()[:, i::2])) for i in (0, 1))).numpy()

    assert np.array_equal(fx.ops.linear_i8_gemm_swiglu(a, s_x, w, w_s).numpy(), unit(fx.ops.linear_i8_gemm_dequant(a, s_x, w, w_s)))
    assert np.array_equal(fx.ops.linear_i8_gemm_swiglu_asym(a, s_x, b_x, w, w_s, w_sum).numpy(),
                          unit(fx.ops.linear_i8_gemm_dequant_asym(a, s_x, b_x, w, w_s, w_sum)))


# tiles of 128 x 128 and 128 x 256: several heads per tile, the last head alone in its tile, half a block of tokens in the last row tile
@pytest.mark.parametrize("m,qh,kvh,pos0,k", QKV)
def test_qkv_tiles(fx, oracle, m, qh, kvh, pos0, k):  # noqa: F811
    prefill.test_gemm_qkv_rope_cache_fused(fx, oracle, m, qh, kvh, pos0, k)
