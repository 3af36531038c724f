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
    """Outputs on either side of a split between waves, and of one inside a wave's columns."""
    m, n = FLOAT[rows]
    floats.test_gemm_tiles(m, n, {"all": n, "half": n // 512 * 256 + 128, "none": 0, "odd": n // 512 * 256 + 64}[split], glu, k, "bfloat16")


# outputs that do not leave in whole 16-byte pieces: one by one, four at a time, a unit's in both ways, on two sides of a split inside four columns
@pytest.mark.parametrize("cut,split,glu", [(13, None, 0), (4, None, 0), (10, None, 1), (8, None, 2), (6, 3002, 0), (4, 3004, 2), (13, 3001, 0)])
@pytest.mark.parametrize("rows", FLOAT)
def test_rows_bfloat16_in_pieces(rows, cut, split, glu):
    m, n = FLOAT[rows]
    n = (n + 255) // 256 * 256 - cut
    from flexllm_amd import lib
    assert lib().flexllm_linear_float_gemm_rows(m, 320, n, 0, 1) == rows
    floats.test_gemm_tiles(m, n, n if split is None else split, glu, 320, "bfloat16")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("m,n,split,glu", [(129, 771, 771, 0), (129, 770, 770, 1), (70, 515, 258, 0), (300, 2049, 1025, 0), (1300, 331, 331, 0), (33, 70, 35, 0),
                                           (2100, 1030, 1030, 2), (2600, 2053, 2053, 0), (1300, 1924, 964, 2)])
def test_small_tiles_in_pieces(m, n, split, glu, dtype):
    floats.test_gemm_tiles(m, n, split, glu, 320, dtype)


# one row tile, whose weights are read once: one stage, as many as the ring holds and more, the first row
# that takes a second tile
@pytest.mark.parametrize("k", floats.GEMM_K)
@pytest.mark.parametrize("m,n,split,glu", [(33, 132, 132, 0), (64, 2060, 1030, 0), (64, 16380, 16380, 1), (65, 6144, 6144, 2), (100, 2048, 0, 0), (128, 12286, 12286, 0), (129, 6144, 6144, 0)])
def test_one_row_tile(m, n, split, glu, k):
    floats.test_gemm_tiles(m, n, split, glu, k, "bfloat16")


# one row tile and several, tiles of 64 to 256 rows, one stage of k and more than the ring holds
@pytest.mark.parametrize("k", [64, 448, 2048])
@pytest.mark.parametrize("n", [2048, 6144, 16384])
def test_sums_of_a_row_are_the_same_on_every_tile(n, k):
    """bfloat16: k is walked from its beginning everywhere, so that a row's sums are the same bit for bit however many rows there are."""
    import numpy as np
    from flexllm_amd import ops, to_device
    from flexllm_amd.loader import to_bf16
    r = np.random.default_rng(n + k)
    a, w = to_bf16(r.standard_normal((1000, k)).astype(np.float32)), to_device(to_bf16(r.standard_normal((n, k)).astype(np.float32)))
    want = ops.linear_float(to_device(a), w, 0, 0, 3.0)[1].numpy()
    for m in 33, 64, 65, 100, 128, 129, 400:
        assert np.array_equal(ops.linear_float(to_device(a[:m]), w, 0, 0, 3.0)[1].numpy(), want[:m]), m


def test_weights_beyond_the_caches():
    """A product whose weights are more than 256 MiB reads them past the caches where one row tile does: the same bit for bit as its halves, which do not."""
    import numpy as np
    from flexllm_amd import ops, synth, to_device
    from flexllm_amd.loader import to_bf16
    k, half = 2048, 35002
    w = synth.device_uniform_bf16((2 * half, k), 7, -1.0, 1.0)
    parts = [to_device(p) for p in np.split(w.numpy(), 2)]
    a = to_bf16(np.random.default_rng(3).standard_normal((129, k)).astype(np.float32))
    for m in 33, 64, 65, 100, 128, 129:
        x = to_device(a[:m])
        for split, glu in (0, 0), (half, 2):               # all columns float32; gated units
            got = ops.linear_float(x, w, 2 * split, glu, 3.0)[not split].numpy()
            want = np.concatenate([ops.linear_float(x, p, split, glu, 3.0)[not split].numpy() for p in parts], 1)
            assert np.array_equal(got, want), (m, glu)


@pytest.mark.parametrize("rows,m,n", [(r, *FLOAT[r]) for r in FLOAT] + [(0, 129, 772), (0, 1300, 330), (0, 40, 132)])
@pytest.mark.parametrize("cut", [0, 2])
def test_unit_behind_a_bias(rows, m, n, cut):
    import numpy as np
    import lopazen_cases as lc
    from flexllm_amd import ops, to_device
    from flexllm_amd.loader import from_bf16, to_bf16
    from oracle import lopazen_ref
    n, k, r = n - cut, 320, np.random.default_rng(rows + m)
    a, w, bias = lc.round_bf16(r.standard_normal((m, k))), lc.round_bf16(r.standard_normal((n, k))), r.standard_normal(n).astype(np.float32)
    y = from_bf16(ops.linear_float(to_device(to_bf16(a)), to_device(to_bf16(w)), n, 2, bias=to_device(bias))[0].numpy())
    want = a.astype(np.float64) @ w.astype(np.float64).T + bias
    g, u = want[:, 0::2], want[:, 1::2]
    first, d = lopazen_ref.gelu(g) * u, 1e-5 * np.sqrt(k)      # bounds as for the tiles
    assert np.all(np.abs(y - first) <= 5e-3 * np.abs(first) + d * (1.2 * (np.abs(u) + 1) + np.abs(g)))


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


@pytest.mark.parametrize("off", [0, 1, 2])
@pytest.mark.parametrize("rows,k", INT)
def test_units_that_end_inside_16_bytes(fx, rows, k, off):  # noqa: F811
    """A row of the unit's outputs ends in the middle of a lane's 16 bytes, and starts on any word: each row whole, and nothing behind the last."""
    import numpy as np
    m, n = INT[rows, k]
    for n in ((n + 255) // 256 * 256 - 4, (n + 255) // 256 * 256 - 116):
        assert fx.lib().flexllm_linear_i8_gemm_rows(m, k, n, 0) == rows
        r = np.random.default_rng(m + k + n)
        a, w = [fx.to_device(r.integers(-127, 128, s).astype(np.int8)) for s in ((m, k), (n, k))]
        s_x, w_s = [fx.to_device(r.uniform(lo, hi, c).astype(np.float32)) for lo, hi, c in ((.01, .02, m), (1e-3, 1e-2, n))]
        y = fx.ops.linear_i8_gemm_dequant(a, s_x, w, w_s).numpy()
        want = fx.ops.swiglu_f32(*(fx.to_device(np.ascontiguousarray(y[:, i::2])) for i in (0, 1))).numpy()
        size = m * (n // 2)
        buf = fx.to_device(np.full(size + 16, 77.0, np.float32))
        fx.ops.linear_i8_gemm_swiglu(a, s_x, w, w_s, out=buf.view(4 * off, (m, n // 2)))
        got = buf.numpy()
        assert np.array_equal(got[off:off + size].reshape(m, n // 2), want)
        assert (got[:off] == 77.0).all() and (got[off + size:] == 77.0).all()


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
