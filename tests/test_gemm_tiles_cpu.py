"""Which tile a product runs on is arithmetic on the host: the tests on the GPU reach every tile, and products take the ones that
measured best."""
import ctypes as C

import pytest

import test_gpu_decoder_sizes as floats
import test_gpu_gemm_tiles as gpu


def ask(name, *sizes):
    from flexllm_amd import lib
    out = [C.c_int() for _ in range(3)]
    assert getattr(lib(), name)(*sizes, *(C.byref(v) for v in out)) == 0
    return tuple(v.value for v in out)


def tile(m, k, n, qkv=False):
    return ask("flexllm_linear_i8_gemm_tile", m, k, n, int(qkv))


def float_tile(m, k, n, dtype="bfloat16"):
    return ask("flexllm_linear_float_gemm_tile", m, k, n, int(dtype == "float32"))


ONE = {(256, 256, 1), (128, 256, 1), (128, 128, 1), (64, 128, 1), (64, 64, 1)}      # rows, columns, workgroups per CU
TWO, THREE = {(128, 128, 2)}, {(64, 64, 3)}


def test_every_int8_tile_is_under_test():
    assert {tile(*s) for s in gpu.TILES if s[1] % 128 == 0} == ONE | TWO | THREE
    assert {tile(*s) for s in gpu.HALF} == ONE
    for half in (0, 64):
        assert {tile(m, k, (qh + 2 * kvh) * 64, True) for m, qh, kvh, _, k in gpu.QKV if k % 128 == half} == ONE - {(256, 256, 1)}


def test_every_float_tile_is_under_test():
    at = {k: {float_tile(m, k, n) for m, n, _, _ in floats.GEMM} for k in floats.GEMM_K}
    assert at[448] == at[576] == ONE | TWO
    assert at[256] == {(128, 128, 1), (64, 128, 1), (64, 64, 1)} | TWO                        # short k never runs on the wide tiles,
    assert at[64] == at[128] == {(128, 128, 1), (64, 64, 1)} | TWO                            # nor the shortest on 64 x 128
    at = {k: {float_tile(m, k, n, "float32") for m, n, _, _ in floats.GEMM} for k in floats.GEMM_K}
    assert at[576] == {(128, 128, 1), (64, 128, 1), (64, 64, 1)}
    assert all(at[k] == {(128, 128, 1), (64, 64, 1)} for k in floats.GEMM_K if k < 512)


@pytest.mark.parametrize("k", [2048, 2112])
def test_wide_int8_products_take_wide_tiles(k):
    assert tile(4096, k, 16384) == tile(1024, k, 16384) == (256, 256, 1)
    assert tile(4096, 4 * k, 2048) == (128, 256, 1)
    assert tile(2048, k, 2048) == (128, 128, 1)
    assert tile(1024, k, 2048) == (64, 128, 1)
    assert tile(32, k, 2048) == (64, 64, 1)


def test_tiles_that_measured_best():
    """Sizes at which another tile was 5 to 40 % slower."""
    assert float_tile(3700, 8576, 2064) == tile(3700, 8576, 2064) == (128, 128, 2)      # 493 tiles
    assert float_tile(3700, 4096, 28672) == float_tile(3072, 4096, 28672) == (256, 256, 1)
    assert float_tile(1621, 320, 22276) == (128, 256, 1)
    assert float_tile(2409, 256, 5608) == float_tile(1468, 128, 23752) == float_tile(639, 128, 16380) == (128, 128, 2)
    assert float_tile(2070, 5632, 9468) == float_tile(3072, 2048, 6144) == (128, 256, 1)
    assert float_tile(288, 1664, 23660) == (128, 128, 1)
    assert float_tile(777, 4096, 28672) == (256, 256, 1)
    assert float_tile(1531, 2048, 16384) == (128, 256, 1)
    assert float_tile(777, 14336, 4096) == (128, 128, 1)
    assert float_tile(1024, 2048, 2048) == (64, 128, 1)
    assert tile(917, 704, 19348) == tile(1621, 320, 22276) == tile(838, 192, 10668) == (128, 128, 1)
    assert tile(3575, 192, 2548) == tile(260, 64, 3440) == tile(530, 192, 3580) == (64, 64, 1)
    assert tile(1536, 2048, 2048) == tile(2176, 512, 2048) == tile(1536, 512, 2048) == tile(393, 128, 9536) == (64, 64, 3)
    assert tile(2528, 2048, 16384) == (256, 256, 1) and tile(1024, 2048, 3072, True) == tile(3072, 2048, 3072, True) == (128, 128, 1)
    assert tile(2528, 2048, 8192) == tile(3072, 2048, 2048) == (128, 256, 1)
    assert float_tile(266, 128, 18912, "float32") == (64, 64, 1)


def parts(m, k, n, dtype="bfloat16", most=8):
    from flexllm_amd import lib
    return lib().flexllm_linear_float_gemm_parts(m, k, n, int(dtype == "float32"), most)


def test_parts_of_k():
    """Shared out for few rows; not for next to nothing, nor where the sums leave the caches (measured slower in parts)."""
    assert parts(64, 14336, 4096) == 8 and parts(200, 8192, 2048) == 8 and parts(200, 8192, 2048, most=4) == 4
    assert parts(64, 8192, 2048, "float32") == 8
    assert parts(1024, 14336, 4096) == parts(1531, 8192, 2048) == 2
    assert parts(640, 14336, 4096) == 2 and parts(777, 8192, 2048) == 2
    assert parts(777, 4096, 4096) == 1
    assert parts(1300, 14336, 4096) == parts(1531, 14336, 4096) == parts(2048, 14336, 4096) == 1
    assert parts(64, 64, 2048) == 1
