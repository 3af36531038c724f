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
