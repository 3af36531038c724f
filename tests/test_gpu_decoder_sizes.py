"""The floating-point decoders on the GPU at the sizes where the choice of a kernel changes, against the plain statement of
their equations: edges of tiles, remainders, the smallest and largest of a kernel's range."""
import numpy as np
import pytest

import lopazen_cases as lc
import nifunex_cases as nc
from oracle import lopazen_ref, nifunex_ref

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


def check(cls, w, toks, want, cfg, dtype, cuts, max_pos, close=()):
    """close: places where a router's choice may fall either way; they have to be finite, no more."""
    clear = np.setdiff1d(np.arange(len(toks)), close)
    m = cls.from_tensors(cfg, w, dtype=dtype, max_pos=max_pos)
    for c in cuts:
        got = logits(m, toks, c)
        assert np.isfinite(got).all(), c
        err = lc.rel_err(got, want)
        assert err[clear].max() < lc.LIMIT[dtype], "portions %s: error %.3g at %d" % (c, err[clear].max(), clear[err[clear].argmax()])
    m.close()


def check_lopazen(cfg, dtype, n, *cuts, max_pos=512):
    from flexllm_amd.lopazen import Lopazen
    w, toks = lc.weights(cfg, 11), lc.tokens(cfg, n)
    check(Lopazen, w, toks, lopazen_ref.Reference(cfg, w).run(toks), cfg, dtype, cuts, max_pos)


# Router outputs are of size 2 and in bfloat16 off by up to a 100th of that: a choice is clear when the last one taken is further than this
# ahead of the first one left.
CLOSE = 0.04


def check_nifunex(cfg, dtype, n, *cuts, max_pos=512):
    from flexllm_amd.nifunex import Nifunex
    w, toks = nc.weights(cfg, 11), nc.tokens(cfg, n)
    lead, route = [], nifunex_ref.route

    def noted(z, top):
        s = np.sort(z)[::-1]
        lead.append(s[top - 1] - s[top] if top < len(s) else np.inf)
        return route(z, top)

    with pytest.MonkeyPatch.context() as patch:
        patch.setattr(nifunex_ref, "route", noted)
        want = nifunex_ref.Reference(cfg, w).run(toks)
    close = np.nonzero((np.reshape(lead, (-1, n)) < CLOSE).any(0))[0] if dtype == "bfloat16" and lead else ()
    assert len(close) < max(n // 4, 2)
    check(Nifunex, w, toks, want, cfg, dtype, cuts, max_pos, close)


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


# every tile of the GEMM: one k-stage, fewer and more than the ring holds, rows and columns that do not fill the last tile
GEMM_K = [64, 128, 256, 448, 576]
GEMM = [(1024, 16380, 16380, 0), (1021, 16384, 16384, 1), (1100, 16384, 16000, 0), (1000, 4000, 4000, 2), (897, 4096, 0, 0), (1000, 2040, 1024, 0), (961, 2048, 2048, 1),
        (65, 1028, 1028, 0), (1, 64, 0, 0), (1531, 16384, 16384, 1), (1500, 16380, 16000, 0), (3700, 2064, 2064, 2), (3699, 2060, 1000, 0), (2040, 4100, 4100, 0)]


@BOTH
@pytest.mark.parametrize("k", GEMM_K)
@pytest.mark.parametrize("m,n,split,glu", GEMM)
def test_gemm_tiles(m, n, split, glu, k, dtype):
    from flexllm_amd import ops, to_device
    from flexllm_amd.loader import from_bf16, to_bf16
    r = np.random.default_rng(m + n + k)
    a, w = [lc.round_bf16(r.standard_normal(s)) for s in ((m, k), (n, k))]
    dev = to_device if dtype == "float32" else lambda x: to_device(to_bf16(x))
    y, y32 = ops.linear_float(dev(a), dev(w), split, glu, 3.0)
    want = a.astype(np.float64) @ w.astype(np.float64).T
    # A float32 sum of k products of O(1) is within d = 1e-5 sqrt(k).  A unit act(g) u has slopes of at most 1.2 |u| in g and |g| in u
    # (the clamped one: u + 1 with |u| <= 3); a bfloat16 result is besides within 2^-9 of the value.
    d = 1e-5 * np.sqrt(k)
    if split:
        g, u = want[:, 0:split:2], want[:, 1:split:2]
        first = want[:, :split] if not glu else nifunex_ref.clamped_glu(g, u, 3.0) if glu == 1 else lopazen_ref.gelu(g) * u
        got, tol = (y.numpy(), 1e-5) if dtype == "float32" else (from_bf16(y.numpy()), 5e-3)
        slope = 1.2 * (np.abs(u) + 1) + np.abs(g) if glu else 1.0
        assert np.all(np.abs(got - first) <= tol * np.abs(first) + d * slope)
    if split < n:
        assert np.all(np.abs(y32.numpy() - want[:, split:]) <= 1e-5 * np.abs(want[:, split:]) + d)


# both sides of the rows per expert from which on there are tiles of 128 rows, and up to which experts' weights are read once; uneven shares of them
@BOTH
@pytest.mark.parametrize("experts,top,ff,tokens", [(4, 2, 72, 100), (2, 1, 40, 119), (2, 1, 40, 120), (4, 2, 200, 225), (4, 2, 72, 227)])
def test_grouped_tiles_of_few_rows(experts, top, ff, tokens, dtype):
    check_nifunex(nc.config([nc.gla(heads=1, mlp=nc.moe(experts, top, ff, 1.5, 0))], width=192), dtype, tokens, [tokens])


# workgroups that walk several tiles of experts: tiles of 64 and of 128 rows, weights read once and not, a last column tile that is not full, more tiles than a
# workgroup lists at a time, fewer than there are CUs
@pytest.mark.parametrize("experts,top,ff,tokens", [(20, 2, 1024, 470), (12, 2, 1000, 470), (8, 2, 1032, 700), (4, 1, 328, 257), (4, 2, 4096, 4096)])
def test_grouped_tiles_of_one_workgroup(experts, top, ff, tokens):
    check_nifunex(nc.config([nc.gla(heads=1, mlp=nc.moe(experts, top, ff, 1.5, 0))], width=256), "bfloat16", tokens, [tokens], max_pos=max(512, tokens))


def by_experts(mlp, w, pre, h):
    """nifunex_ref.mixture, an expert's rows at a time."""
    out = np.zeros_like(h)
    picks = [nifunex_ref.route(z, mlp["router"]["top"]) for z in h @ w[pre + "router"].T]
    for e in range(mlp["router"]["experts"]):
        rows = [(t, a) for t, (pick, wt) in enumerate(picks) for i, a in zip(pick, wt) if i == e]
        if rows:
            t, a = np.array([r[0] for r in rows]), np.array([r[1] for r in rows])
            out[t] += a[:, None] * nifunex_ref.feed_forward(w, "%se%d." % (pre, e), h[t], mlp["expert"]["limit"])
    return out


# more tiles than CUs, and k of more stages than the ring holds: an odd number of them, so that tiles begin at every place of it, and not.  Where all weights lie in the
# caches (100 MB and less) tiles of 128 rows; beyond them (more than 256 MiB) tiles of 64 and of 128 rows, gate/up and down products with several tiles per workgroup
@pytest.mark.parametrize("experts,top,ff,tokens,width", [(8, 2, 1032, 700, 320), (8, 2, 2056, 700, 448), (6, 2, 2048, 700, 1024),
                                                         (22, 2, 2048, 520, 1024), (21, 2, 2048, 500, 1088), (22, 2, 1088, 900, 2048), (21, 2, 2048, 900, 1088)])
def test_grouped_tiles_of_many_stages(experts, top, ff, tokens, width, monkeypatch):
    monkeypatch.setattr(nifunex_ref, "mixture", by_experts)
    check_nifunex(nc.config([nc.gla(heads=1, mlp=nc.moe(experts, top, ff, 1.5, 0))], width=width), "bfloat16", tokens, [tokens], max_pos=1024)


# weights beyond the caches, which one row tile of 64 and of 128 rows reads past them, and two tiles do not: outputs that leave in whole pieces, and not
@pytest.mark.parametrize("ff", [8192, 1030])
def test_weights_beyond_the_caches(ff):
    check_lopazen(lc.config([lc.layer(heads=2, kv_heads=1, dim=32, mlp=lc.dense(ff))], width=2048, vocab=66000), "bfloat16", 129, [129], [128, 1], [100, 29], [64, 65], [33], max_pos=160)


# tiles of 64 x 64, 64 x 128 and 128 x 128, with more stages of k than the ring holds
@pytest.mark.parametrize("tokens", [40, 50, 100])
def test_experts_in_another_order(tokens):
    """An expert's sums do not hang on its number: with two experts that change places, logits stay the same bit for bit."""
    from flexllm_amd.nifunex import Nifunex
    cfg = nc.config([nc.gla(heads=1, mlp=nc.moe(2, 2, 512, 1.5, 0))], width=1024)
    w, toks = nc.weights(cfg, 11), nc.tokens(cfg, tokens)
    other = {n: w[n.replace(".e0.", ".e#.").replace(".e1.", ".e0.").replace(".e#.", ".e1.")] for n in w}
    other["l0.mlp.router"] = w["l0.mlp.router"][::-1].copy()
    got = []
    for weights in w, other:
        m = Nifunex.from_tensors(cfg, weights, dtype="bfloat16", max_pos=128)
        got.append(logits(m, toks, [tokens]))
        m.close()
    assert np.array_equal(got[0], got[1])


# grouped products of the experts: tiles of 64 rows, narrow and wide ones, and of 128 rows, experts with a tile and a row more, columns that do not fill a tile
@BOTH
@pytest.mark.parametrize("experts,top,ff,tokens", [(2, 1, 40, 200), (3, 2, 100, 194), (4, 4, 72, 129), (8, 1, 130, 70), (4, 2, 100, 130), (2, 1, 40, 130)])
def test_grouped_tiles(experts, top, ff, tokens, dtype):
    cfg = nc.config([nc.gla(heads=1, mlp=nc.moe(experts, top, ff, 1.5, 0))], width=192)
    check_nifunex(cfg, dtype, tokens, [tokens])


# prompts of few rows, whose down and output projections share k out: no row tile filled, one and two of them, parts of uneven lengths,
# with and without a norm behind the sublayer, a mixture's shared expert
@BOTH
@pytest.mark.parametrize("tokens,ff", [(9, 2048), (65, 1100), (130, 4200)])
def test_shared_out_k(tokens, ff, dtype):
    check_lopazen(lc.config([lc.layer(heads=12, kv_heads=3, dim=64, mlp=lc.dense(ff)), lc.layer()], width=192), dtype, tokens, [tokens])
    check_nifunex(nc.config([nc.gla(heads=9, dim=32, vdim=64, mlp=nc.dense(ff)), nc.gla(heads=1, mlp=nc.moe(4, 2, 72, 1.5, ff))], width=192), dtype, tokens, [tokens])


@BOTH
def test_slices_of_a_prompt(dtype):
    """Prompts that go through the step's attention in slices of 64 tokens: whole slices, one token more, one less."""
    for n in (63, 64, 65, 129):
        check_lopazen(lc.config([lc.layer(heads=4, kv_heads=2, dim=264, scale=0.06)]), dtype, n, [n], [9, n])
        check_nifunex(nc.config([nc.latent(heads=2, dim=264, rot_dim=8, vdim=16, kv_rank=48, window=50, scale=0.06)]), dtype, n, [n], [9, n])


# two to eight tokens in one step: every number of tokens per pass over the weights, vectors of one to fifteen pieces per thread, a
# gated unit on vectors so long that its pairs need two rows per group, odd lengths, a mixture
@BOTH
@pytest.mark.parametrize("width,ff", [(160, 88), (160, 1029), (90, 33), (2112, 2050), (64, 4100), (64, 8200), (64, 15360), (8256, 40)])
def test_step_of_several_tokens(width, ff, dtype):
    cfg = lc.config([lc.layer(heads=2, kv_heads=1, dim=32, mlp=lc.dense(ff))], width=width, vocab=131, loop=(0, 1, 2))
    check_lopazen(cfg, dtype, 35, [2, 3, 4, 5, 6, 7, 8])


@BOTH
def test_step_of_several_tokens_nifunex(dtype):
    check_nifunex(nc.mixed(), dtype, 35, [2, 3, 4, 5, 6, 7, 8])


# the experts' down projections of a step: fewer pieces than threads, more than one pass of them, a last pass that is ragged, units that
# are read four at a time and such that are not, no shared expert, rows that do not fill a group
@BOTH
@pytest.mark.parametrize("top,ff,shared,width", [(1, 8, 0, 66), (2, 41, 56, 90), (3, 40, 57, 130), (6, 1024, 2048, 160), (4, 2100, 0, 70), (5, 822, 410, 64)])
def test_experts_down(top, ff, shared, width, dtype):
    cfg = nc.config([nc.gla(heads=1, mlp=nc.moe(top + 1, top, ff, 1.5, shared)), nc.gla(heads=1, mlp=nc.dense(72))], width=width)
    check_nifunex(cfg, dtype, 20, [1], [3])


# gate/up weights that two tokens of a step just still read again, and just not (8191 and 8192; as many as longer rows could be: 5120 and 5121), down products whose
# sums leave whole, and in parts; three and four tokens do not read them again
@pytest.mark.parametrize("ff", [5120, 5121, 8191, 8192])
def test_step_of_several_tokens_reads_weights_once(ff):
    check_lopazen(lc.config([lc.layer(heads=2, kv_heads=1, dim=32, mlp=lc.dense(ff)), lc.layer(heads=2, kv_heads=1, dim=32, mlp=lc.dense(72))], width=2048),
                  "bfloat16", 12, [2], [3], [4])


@BOTH
@pytest.mark.parametrize("ff", [88, 2050])
def test_infinite_units(ff, dtype):
    """A unit beyond float32 leaves infinities of the equations' signs in the residual, and one whose gate is as far below zero leaves
    nothing, however many tokens a step has.  (The gate itself stays small enough for its cube, which gelu forms, to be finite: about 1e12.)"""
    from flexllm_amd.lopazen import Lopazen
    cfg = lc.config([lc.layer(heads=2, kv_heads=1, dim=32, mlp=lc.dense(ff))])
    w, toks = lc.weights(cfg, 11), lc.tokens(cfg, 12)
    for name in w:
        if name.endswith((".gate", ".up")):
            w[name][5] = lc.round_bf16(w[name][5] * np.float32(1e4 if name.endswith("gate") else 1e36))
        if name.endswith(".down"):
            w[name][:, 5] = np.where(w[name][:, 5] < 0, -1.0, 1.0)
    want = []
    lopazen_ref.Reference(cfg, w).run(toks, want)
    want = want[0]
    beyond = np.abs(want) > np.finfo(np.float32).max
    assert beyond.all(1).any() and (np.abs(want).max(1) < 1e30).any()      # tokens of either kind
    m = Lopazen.from_tensors(cfg, w, dtype=dtype, max_pos=64)
    for n in (1, 3, 12):                                  # steps, and a prompt
        slot = m.pool.acquire(n)
        got = np.concatenate([m.step(slot, toks[p:p + n], [n - 1], layers=True)[1] for p in range(0, 12, n)], 1)[0]
        m.pool.release(n)
        assert (np.isposinf(got) == (beyond & (want > 0))).all() and (np.isneginf(got) == (beyond & (want < 0))).all(), n
        assert np.isfinite(got[~beyond]).all(), n
        none = np.abs(want).max(1) < 1e30                 # (units of 1e38 are what is left of sums that cancel)
        assert (np.abs(got[none] - want[none]).max(1) < lc.LIMIT[dtype] * np.abs(want[none]).max(1)).all(), n
    m.close()


def test_splits_of_long_caches():
    """From 12288 rows on these heads have twice the splits: steps on both sides of the border, and decoding across it, whose graph
    is made for the rows that there will be."""
    from flexllm_amd import to_device, zeros
    from flexllm_amd.lopazen import Lopazen
    cfg = lc.config([lc.layer(heads=2, kv_heads=1, dim=16)])
    cuts = [12270, 7, 8, 2, 1, 1, 3, 4, 8, 2]
    check_lopazen(cfg, "float32", sum(cuts), cuts, max_pos=12544)
    check_lopazen(cfg, "bfloat16", sum(cuts), cuts, max_pos=12544)
    w, toks = lc.weights(cfg, 11), lc.tokens(cfg, 12281)
    m = Lopazen.from_tensors(cfg, w, dtype="float32", max_pos=12544, slots=2)
    slots = [m.pool.acquire(n) for n in "ab"]
    for s in slots:
        m.step(s, toks[:-1])
    token, got, want = to_device(np.array(toks[-1:], np.int32)), [], toks[-1:]
    for n in (4, 20, 5):
        out = zeros((n,), np.int32)
        m.decode(slots[0], token, n, out)
        m.check()
        got += out.numpy().tolist()
    for _ in got:
        want.append(int(m.step(slots[1], want[-1:], [0])[0].argmax()))
    m.close()
    assert got == want[1:]


# the last split of the rows repeats in the join of fewer splits than it reads at a time
@BOTH
@pytest.mark.parametrize("rows", [40, 96, 200, 256, 270])
def test_infinite_sums_of_the_splits(rows, dtype):
    """Rows so large that their sum leaves float32 give an infinity in that column, of any number of splits."""
    from flexllm_amd.lopazen import Lopazen
    cfg = lc.config([lc.layer(heads=1, kv_heads=1, dim=8)])
    w, toks = lc.weights(cfg, 11), lc.tokens(cfg, rows + 1)
    w["l0.mix.k.b"][3], w["l0.mix.q.norm"][3] = 2.0 ** 126, 0.0      # this column is in no score
    m = Lopazen.from_tensors(cfg, w, dtype=dtype, max_pos=512)
    slot = m.pool.acquire("t")
    m.step(slot, toks[:rows])
    got = m.step(slot, toks[rows:], layers=True)[1][0, 0]
    m.close()
    assert np.array_equal(got, np.where(w["l0.mix.o"][:, 3] < 0, -np.inf, np.inf))
