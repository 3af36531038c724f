"""The sizes under test on the GPU reach every number of rows that tiles of 256 columns come in."""
import test_gpu_gemm_rows as gpu


def test_every_number_of_rows_is_under_test():
    from flexllm_amd import lib
    for rows, (m, n) in gpu.FLOAT.items():
        for k in gpu.FLOAT_K:
            assert lib().flexllm_linear_float_gemm_rows(m, k, n, 0, 1) == rows
    for (rows, k), (m, n) in gpu.INT.items():
        assert lib().flexllm_linear_i8_gemm_rows(m, k, n, 0) == rows


def test_rows_that_measured_best():
    """Sizes at which another number of rows was 5 to 40 % slower; few rows stay on their tile."""
    from flexllm_amd import lib
    f, i = (lambda *s: lib().flexllm_linear_float_gemm_rows(*s, 0, 1)), (lambda *s: lib().flexllm_linear_i8_gemm_rows(*s, 0))
    assert f(777, 4096, 28672) == f(2528, 2048, 16384) == 224 and f(1531, 2048, 16384) == 192 and f(2596, 2560, 3712) == 160
    assert f(1024, 2048, 16384) == 256 and f(2528, 8192, 2048) == 96 and f(777, 14336, 4096) == 128 and f(1024, 2048, 2048) == 64
    assert i(777, 4096, 28672) == 224 and i(1531, 2048, 16384) == 192 and i(1024, 2048, 16384) == 256
    assert i(2528, 8192, 2048) == lib().flexllm_linear_i8_gemm_rows(2528, 2048, 3072, 1) == 128


def test_few_rows_are_one_pass():
    from flexllm_amd import lib
    import test_gpu_gemm_few as few
    f = lambda m, k, n, parts=1: lib().flexllm_linear_float_gemm_rows(m, k, n, 0, parts)  # noqa: E731
    for m, n in few.FEW:
        rows = 16 if m <= 16 else 32
        assert all(f(m, k, n) == rows for k in few.FILLED[rows])
        # units that k does not fill, and short ones, cost more than the tiles' stages (5 to 50 % more)
        assert all(f(m, k, n) == 64 for k in (64, 448, 1088, 2112, 3008))
    assert f(17, 1024, 16384) == f(32, 1536, 8192) == f(32, 3520, 8192) == 64
    assert f(33, 2048, 16384) == f(9, 4160, 16384) == f(9, 2048, 8188) == f(9, 2048, 16384, 2) == 64


def test_quotients_of_tile_numbers():
    """A workgroup's tile by float quotients put right by the remainder (gemm_walk.h): exact for every number of tiles that a call can
    have, wherever within an ulp the reciprocal lies."""
    import numpy as np
    r = np.random.default_rng(1)
    d = np.concatenate([np.arange(1, 300), np.exp(r.uniform(0, np.log(2.0 ** 21), 4000)).astype(np.int64)])
    q = np.exp(r.uniform(0, np.log(2.0 ** 18), len(d))).astype(np.int64)
    for off in (-1, 0, 1):
        a = np.clip(q * d + off, 0, 2 ** 31 - 1)
        inv = np.float32(1) / d.astype(np.float32)
        for rcp in (inv, np.nextafter(inv, np.float32(0)), np.nextafter(inv, np.float32(2))):
            got = (a.astype(np.float32) * rcp).astype(np.int64)
            rest = a - got * d
            got += (rest >= d).astype(np.int64) - (rest < 0)
            assert np.array_equal(got, a // d)
