"""The linear behind the steps of one to eight tokens on its own, against products in float64."""
import numpy as np
import pytest

import lopazen_cases as lc

pytestmark = pytest.mark.gpu
BOTH = pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
# Exact products, and no sum is more than 128 additions deep.
EPS = 128 * 2.0 ** -24


def step(x, w, dtype, **kw):
    from flexllm_amd import ops, to_device
    from flexllm_amd.loader import to_bf16
    rows = np.zeros((len(w), (w.shape[1] + 63) // 64 * 64), np.float32)
    rows[:, :w.shape[1]] = w
    y, y32 = ops.linear_float_step(to_device(x), to_device(rows if dtype == "float32" else to_bf16(rows)), **kw)
    return [a.numpy() if a else None for a in (y, y32)]


def near(got, x, w):
    x, w = x.astype(np.float64), w.astype(np.float64)
    assert np.isfinite(got).all()
    assert np.all(np.abs(got - x @ w.T) <= EPS * (np.abs(x) @ np.abs(w).T))


@BOTH
@pytest.mark.parametrize("tokens", [1, 2, 3, 8])
@pytest.mark.parametrize("k", [100, 2048, 2112, 8200])
def test_values_beyond_bfloat16(k, tokens, dtype):
    """Finite values between the largest bfloat16 and the largest float32."""
    r = np.random.default_rng(k + tokens)
    x = r.standard_normal((tokens, k)).astype(np.float32)
    w = lc.round_bf16(r.uniform(0.5, 1.0, (37, k)) * 2.0 ** -20)
    x[:, [0, 7, k // 2, k - 1]] = [3.4e38, -3.3962e38, np.finfo(np.float32).max, -3.39e38]
    near(step(x, w, dtype)[0], x, w)


@BOTH
@pytest.mark.parametrize("tokens", [1, 2, 3, 8])
@pytest.mark.parametrize("k", [100, 2048, 2112, 8200])
def test_infinite_weights(k, tokens, dtype):
    """An infinite weight gives infinities of the sign that the products have, whichever bits the vector has set; not a number only
    where it meets zero or infinities of both signs meet."""
    r = np.random.default_rng(k + tokens)
    x = (r.standard_normal((tokens, k)) + 0.1).astype(np.float32)
    w = lc.round_bf16(r.standard_normal((37, k)))
    x[:, :4] = [1.0, -1.5, 1.0 + 2.0 ** -9 - 2.0 ** -20, 0.0]        # nothing behind the first bfloat16, the same below zero, parts of both signs
    w[2, 0], w[3, 1], w[5, 2], w[16, k - 1], w[17, 3], w[36, [0, 1]] = np.inf, np.inf, -np.inf, -np.inf, np.inf, np.inf
    with np.errstate(invalid="ignore"):
        want = (x[:, None, :].astype(np.float64) * w[None].astype(np.float64)).sum(-1)
    got = step(x, w, dtype)[0]
    for same in (np.isposinf, np.isneginf, np.isnan):
        assert (same(got) == same(want)).all()
    rows = np.isfinite(want[0])
    near(got[:, rows], x, w[rows])


@BOTH
@pytest.mark.parametrize("tokens", [1, 2, 3, 8])
@pytest.mark.parametrize("k", [64, 192, 2048, 2112, 4160, 8192, 8256])
def test_infinity_in_the_last_piece(k, tokens, dtype):
    """Threads that have no piece of a row add nothing, whatever the vector's last piece holds."""
    r = np.random.default_rng(k + tokens)
    x = r.standard_normal((tokens, k)).astype(np.float32)
    w = lc.round_bf16(r.standard_normal((37, k)))
    x[:, k - 1] = np.inf
    assert np.array_equal(step(x, w, dtype)[0], np.broadcast_to(np.inf * w[:, k - 1], (tokens, 37)))


@BOTH
@pytest.mark.parametrize("tokens", range(1, 9))
@pytest.mark.parametrize("k,n,split", [(1000, 37, 12), (2048, 130, 128), (2112, 131, 0), (4160, 67, 67), (8256, 45, 32)])
def test_columns_of_both_outputs(k, n, split, tokens, dtype):
    """A bias, columns in the first output, in the second, in both; rows that do not fill a group or a tile; every number of tokens per pass."""
    from flexllm_amd import to_device
    r = np.random.default_rng(k + tokens)
    x, bias = r.standard_normal((tokens, k)).astype(np.float32), r.standard_normal(n).astype(np.float32)
    w = lc.round_bf16(r.standard_normal((n, k)))
    y, y32 = step(x, w, dtype, n_split=split, bias=to_device(bias))
    got = np.concatenate([a for a in (y, y32) if a is not None], 1)
    one = lambda a: np.concatenate([a, np.ones((len(a), 1))], 1)      # the bias is one product more
    near(got, one(x), np.concatenate([w, bias[:, None]], 1))


@BOTH
@pytest.mark.parametrize("glu", [1, 2])
@pytest.mark.parametrize("tokens", range(1, 9))
@pytest.mark.parametrize("k,n,split", [(1000, 38, 38), (2048, 131, 128), (4160, 67, 66), (8256, 46, 32)])
def test_gated_unit(k, n, split, tokens, glu, dtype):
    """The unit of neighbouring rows in the epilogue: both rows of a pair lie in one group, whatever the rows' length."""
    from oracle import lopazen_ref, nifunex_ref
    r = np.random.default_rng(k + tokens)
    x = r.standard_normal((tokens, k)).astype(np.float32)
    w = lc.round_bf16(r.standard_normal((n, k)) * k ** -0.5)
    y, y32 = step(x, w, dtype, n_split=split, glu=glu, limit=3.0)
    x, w = x.astype(np.float64), w.astype(np.float64)
    z, d = x @ w.T, EPS * (np.abs(x) @ np.abs(w).T)
    g, u, dg, du = [a[:, i:split:2] for a in (z, d) for i in (0, 1)]
    want = nifunex_ref.clamped_glu(g, u, 3.0) if glu == 1 else lopazen_ref.gelu(g) * u
    # act(g) u has slopes of at most 1.2 (|u| + 1) in g and |g| in u; the function itself is good to 1e-6 of its arguments
    slope_g, slope_u = 1.2 * (np.abs(u) + 1), np.abs(g) + 0.2
    assert np.all(np.abs(y - want) <= slope_g * (dg + 1e-6 * np.abs(g)) + slope_u * (du + 1e-6 * np.abs(u)))
    if split < n:
        assert np.all(np.abs(y32 - z[:, split:]) <= d[:, split:])


@pytest.mark.parametrize("tokens", range(2, 9))
@pytest.mark.parametrize("k,parts", [(2048, 2), (2112, 2), (4160, 3), (8192, 8), (14336, 7), (8200, 5)])
def test_parts_of_k(k, parts, tokens):
    """Sums over parts of k, the last one of any length, add up to the product."""
    r = np.random.default_rng(k + tokens)
    x = r.standard_normal((tokens, k)).astype(np.float32)
    w = lc.round_bf16(r.standard_normal((45, k)))
    near(step(x, w, "bfloat16", n_split=0, parts=parts)[1].astype(np.float64).sum(0), x, w)
