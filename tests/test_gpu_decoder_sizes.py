"""The floating-point decoders on the GPU at the sizes where the choice of a kernel changes, against the plain statement of
their equations: edges of tiles, remainders, the smallest and largest of a kernel's range."""
import numpy as np
import pytest

import lopazen_cases as lc
from oracle import lopazen_ref

pytestmark = pytest.mark.gpu
BOTH = pytest.mark.parametrize("dtype", ["float32", "bfloat16"])


def logits(model, toks, cuts, max_pos=512):
    """Logits of every token, fed in portions of the given sizes (the last one repeats)."""
    slot = model.pool.acquire("t")
    out, p, i = [], 0, 0
    while p < len(toks):
        c = min(cuts[min(i, len(cuts) - 1)], len(toks) - p)
        out.append(model.step(slot, toks[p:p + c], range(c)))
        p, i = p + c, i + 1
    model.check()
    model.pool.release("t")
    return np.concatenate(out)


def check_lopazen(cfg, dtype, n, *cuts, max_pos=512):
    from flexllm_amd.lopazen import Lopazen
    w, toks = lc.weights(cfg, 11), lc.tokens(cfg, n)
    want = lopazen_ref.Reference(cfg, w).run(toks)
    m = Lopazen.from_tensors(cfg, w, dtype=dtype, max_pos=max_pos)
    for c in cuts:
        got = logits(m, toks, c)
        assert np.isfinite(got).all(), c
        err = lc.rel_err(got, want)
        assert err.max() < lc.LIMIT[dtype], "portions %s: error %.3g at place %d" % (c, err.max(), err.argmax())
    m.close()


# rows and lengths of the one-token linears: rows per group and pieces per thread change with both
@BOTH
@pytest.mark.parametrize("width,vocab", [(64, 4), (2048, 8191), (2112, 4096), (2112, 4097), (2304, 8301), (4096, 4099), (4160, 515)])
def test_one_token_linears(width, vocab, dtype):
    check_lopazen(lc.config([lc.layer(heads=2, kv_heads=1, dim=32, mlp=lc.dense(97))], width=width, vocab=vocab), dtype, 6, [1], [3])


# splits of the rows in the step kernel: one split, the first two, a last one of one row, more columns than threads, several
# tokens (fewer splits each) ahead of and behind the borders
@BOTH
@pytest.mark.parametrize("heads,kv_heads,dim", [(8, 2, 64), (8, 1, 128), (3, 3, 264), (2, 1, 8)])
def test_few_token_attention_splits(heads, kv_heads, dim, dtype):
    cfg = lc.config([lc.layer(heads=heads, kv_heads=kv_heads, dim=dim, scale=0.8 * dim ** -0.5)])
    check_lopazen(cfg, dtype, 75, [1], [31, 1, 1, 8, 5], [3, 8])
    check_lopazen(cfg, dtype, 1100, [1021, 2, 1, 1, 8, 7, 1], max_pos=1100)
