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


# a workgroup has one tile, or some have a second; a k that fills a unit, that ends inside one, that is no multiple of 4
@pytest.mark.parametrize("tokens", range(2, 9))
@pytest.mark.parametrize("n,parts", [(4096, 1), (4097, 1), (2048, 2), (2064, 2)])
@pytest.mark.parametrize("k", [64, 256, 1021, 1024, 1088, 2048])
def test_one_tile_and_more(k, n, parts, tokens):
    r = np.random.default_rng(k + n + tokens)
    x = r.standard_normal((tokens, k)).astype(np.float32)
    w = lc.round_bf16(r.standard_normal((n, k)).astype(np.float32))
    y, y32 = steps.step(x, w, "bfloat16", n_split=0 if parts > 1 else n, parts=parts)
    steps.near(y if parts == 1 else y32.astype(np.float64).sum(0), x, w)


@pytest.mark.parametrize("tokens", [2, 3, 8])
@pytest.mark.parametrize("k", [100, 1088, 2048])
def test_infinities_behind_a_stream(k, tokens):
    """As test_infinite_weights and test_infinity_in_the_last_piece, where a workgroup has several tiles."""
    r, n = np.random.default_rng(k + tokens), 4200
    x = (r.standard_normal((tokens, k)) + 0.1).astype(np.float32)
    w = lc.round_bf16(r.standard_normal((n, k)))
    x[:, :4] = [1.0, -1.5, 1.0 + 2.0 ** -9 - 2.0 ** -20, 0.0]
    w[2, 0], w[3, 1], w[5, 2], w[16, k - 1], w[4117, 3], w[4190, [0, 1]] = np.inf, np.inf, -np.inf, -np.inf, np.inf, np.inf
    odd = [2, 3, 5, 16, 4117, 4190]
    with np.errstate(invalid="ignore"):
        want = (x[:, None, :].astype(np.float64) * w[odd][None].astype(np.float64)).sum(-1)
    got = steps.step(x, w, "bfloat16")[0]
    for same in (np.isposinf, np.isneginf, np.isnan):
        assert (same(got[:, odd]) == same(want)).all()
    rest = np.delete(np.arange(n), odd)
    steps.near(got[:, rest], x, w[rest])
    x[:, k - 1] = np.inf
    assert np.array_equal(steps.step(x, w[rest], "bfloat16")[0], np.broadcast_to(np.inf * w[rest, k - 1], (tokens, len(rest))))
