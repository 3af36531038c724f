"""Which tile a product runs on is arithmetic on the host: the tests on the GPU reach every tile, and wide products take wide ones."""
import ctypes as C

import pytest

import test_gpu_gemm_tiles as gpu


def tile(m, k, n, qkv=False):
    from flexllm_amd import lib
    rows, cols = C.c_int(), C.c_int()
    assert lib().flexllm_linear_i8_gemm_tile(m, k, n, int(qkv), C.byref(rows), C.byref(cols)) == 0
    return rows.value, cols.value


ALL = {(256, 256), (128, 256), (128, 128), (64, 128), (64, 64)}


def test_every_int8_tile_is_under_test():
    assert {tile(*s) for s in gpu.TILES if s[1] % 128 == 0} == ALL
    assert {tile(*s) for s in gpu.HALF} == ALL
    assert {tile(m, k, (qh + 2 * kvh) * 64, True) for m, qh, kvh, _, k in gpu.QKV} == ALL - {(256, 256)}


@pytest.mark.parametrize("k", [2048, 2112])
def test_wide_int8_products_take_wide_tiles(k):
    assert tile(4096, k, 16384) == tile(1024, k, 16384) == (256, 256)
    assert tile(4096, 4 * k, 2048) == (128, 256)
    assert tile(2048, k, 2048) == (128, 128)
    assert tile(1024, k, 2048) == (64, 128)
    assert tile(32, k, 2048) == (64, 64)
