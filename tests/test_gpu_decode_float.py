"""Steps of one token as one kernel: models whose sizes it takes, against the plain statement of their equations, token by token and in
loops of several tokens per launch, with one and several splits of the rows."""
import numpy as np
import pytest

import lopazen_cases as lc
import nifunex_cases as nc
from oracle import lopazen_ref
from test_gpu_decoder_sizes import check_lopazen, check_nifunex

pytestmark = pytest.mark.gpu
BOTH = pytest.mark.parametrize("dtype", ["float32", "bfloat16"])


def attention(heads, kv_heads, dim, ff, coef=0.4):
    return lc.layer(heads=heads, kv_heads=kv_heads, dim=dim, scale=dim ** -0.5, coef=coef, mlp=lc.dense(ff) if ff else None)


# rows of one quad and of several, whole numbers of a wave's share and not (14336), the smallest vocabulary, an odd one; heads that share rows
# in fours, in eights, alone, and in threes; no feed-forward; loops
LOPAZEN = {
    "rows of a quad": lc.config([attention(32, 8, 64, 2048), attention(32, 8, 64, 2048)], width=2048, vocab=512),
    "rows of seven quads": lc.config([attention(32, 8, 64, 14336)], width=2048, vocab=517),
    "long heads": lc.config([attention(16, 2, 128, 4096)], width=4096, vocab=600),
    "as many key heads": lc.config([attention(32, 32, 64, 0)], width=2048, vocab=1001),
    "heads in threes": lc.config([attention(48, 16, 128, 2048, coef=0.0)], width=2048, vocab=700),
    "a loop": lc.config([attention(32, 8, 64, 2048), attention(16, 4, 128, 0)], width=2048, vocab=515, loop=(0, 2, 2)),
}


@BOTH
@pytest.mark.parametrize("name", list(LOPAZEN))
def test_token_by_token(name, dtype):
    check_lopazen(LOPAZEN[name], dtype, 40, [1], [23, 1])


# bfloat16: feed-forwards of 12 and of 16 blocks of 512, of which eight waves have one or two each; the longest vector beside many rows of the head
@pytest.mark.parametrize("width,ff,vocab", [(2048, 6144, 514), (2048, 8192, 514), (4096, 14336, 128257)])
def test_long_vectors_in_bfloat16(width, ff, vocab):
    from flexllm_amd._lib import FlexLLMError
    from flexllm_amd.lopazen import Lopazen
    cfg = lc.config([attention(32, 8, 64, ff)], width=width, vocab=vocab)
    check_lopazen(cfg, "bfloat16", 40, [1], [23, 1])
    m = Lopazen.from_tensors(cfg, lc.weights(cfg, 5), dtype="bfloat16", max_pos=64)
    m.set_wait_limit(1)                                    # it is the resident kernel that they take
    with pytest.raises(FlexLLMError, match="timed out"):
        m.step(m.pool.acquire("t"), [1], [0])
    m.close()


def latent(heads, ff, **kw):
    return nc.latent(heads=heads, dim=128, rot_dim=64, vdim=128, kv_rank=512, scale=192 ** -0.5, mlp=nc.dense(ff) if ff else None, **kw)


def gla(heads, ff):
    return nc.gla(heads=heads, dim=128, vdim=128, mlp=nc.dense(ff) if ff else None)


# slices of 8 and of 16 columns, as many heads as there may be and fewer; windows shorter than a split and none; rows of an earlier layer
NIFUNEX = {
    "both kinds": nc.config([latent(16, 2048, window=40), gla(16, 2048), latent(16, 2048, window=40, kv_from=0), gla(16, 0)], width=2048, vocab=512),
    "many heads": nc.config([gla(32, 4096), latent(32, 4096, window=None)], width=4096, vocab=515),
    "rows of seven quads": nc.config([latent(16, 14336, scaling=None)], width=2048, vocab=519),
    "heads that leave workgroups without a slice": nc.config([latent(32, 0), gla(32, 2048)], width=2048, vocab=600),
}


# the experts' rows a half of what a wave asks for at a time, and whole; few experts, one choice, the most choices
MIXTURES = {
    "rows of half a quad in bfloat16": (8, 3, 1024, 2048),
    "rows of half a quad in float32": (5, 1, 512, 1024),
    "rows of a quad": (3, 2, 2048, 4096),
    "all of many": (16, 16, 1024, 2048),
}


@BOTH
@pytest.mark.parametrize("name", list(MIXTURES))
def test_mixtures(name, dtype):
    experts, top, ff, shared = MIXTURES[name]
    moe = dict(mlp=nc.moe(experts, top, ff, 0.75, shared))
    cfg = nc.config([nc.gla(heads=16, dim=128, vdim=128, **moe), nc.latent(heads=16, dim=128, rot_dim=64, vdim=128, kv_rank=512, scale=192 ** -0.5, **moe)], width=2048, vocab=512)
    check_nifunex(cfg, dtype, 40, [1], [30, 1])


@BOTH
@pytest.mark.parametrize("name", list(NIFUNEX))
def test_token_by_token_nifunex(name, dtype):
    check_nifunex(NIFUNEX[name], dtype, 70, [1], [50, 1])


def test_long_sequences_leave_the_resident_kernel():
    """From some number of rows on the chain of kernels is faster: a loop goes on in it where it gets there, steps too."""
    from flexllm_amd import to_device, zeros
    from flexllm_amd._lib import FlexLLMError
    from flexllm_amd.lopazen import Lopazen
    border = 8 * ((384 * 1024 + 160 * 1024) // (128 * 4))  # eight splits of the rows
    cfg = lc.config([attention(32, 8, 128, 0)], width=1024, vocab=512)
    m = Lopazen.from_tensors(cfg, lc.weights(cfg, 5), dtype="float32", max_pos=border + 64, slots=2)
    toks = lc.tokens(cfg, border - 5)
    a, b = [m.pool.acquire(n) for n in "ab"]
    for s in a, b:
        m.step(s, toks[:-1])                               # border - 6 rows
    token, out = to_device(np.array(toks[-1:], np.int32)), zeros((20,), np.int32)
    got = {}
    for s, mode, graph in (a, 0, True), (b, 1, False):
        m.set_decode_mode(mode)
        token.copy_from(np.array(toks[-1:], np.int32))
        m.decode(s, token, 3, out, use_graph=graph)
        first = out.numpy()[:3].tolist()
        m.decode(s, token, 17, out, use_graph=graph)
        got[s] = first + out.numpy()[:17].tolist(), m.step(s, [3], [0])
        m.check()
    assert m.length(a) == border + 15 and got[a][0] == got[b][0]
    assert lc.rel_err(got[a][1], got[b][1]).max() < lc.LIMIT["float32"]
    m.set_decode_mode(0)
    m.set_wait_limit(1)                                    # the resident kernel would give up
    m.step(a, [3], [0])
    m.pool.release("b")
    b = m.pool.acquire("b")
    m.step(b, toks[:-5])
    with pytest.raises(FlexLLMError, match="timed out"):
        m.step(b, [3], [0])
    m.close()


# float32: rows of one quad and of three, which no wave has the same part of in all rows
FLOAT32 = {
    "shared rows of a quad": lc.config([attention(16, 4, 64, 1024)], width=1024, vocab=512),
    "shared rows of three quads": lc.config([attention(48, 16, 64, 3072)], width=3072, vocab=515),
    "both kinds, rows of a quad": nc.config([latent(8, 1024, window=40), gla(8, 1024)], width=1024, vocab=512),
    "both kinds, rows of three quads": nc.config([gla(24, 3072), latent(24, 3072, window=None)], width=3072, vocab=515),
    "mixtures, rows of a quad": nc.config([gla(8, 0) | dict(mlp=nc.moe(5, 2, 512, 0.75, 1024)), latent(8, 0) | dict(mlp=nc.moe(4, 2, 1024, 0.75, 512))], width=1024, vocab=512),
}


@pytest.mark.parametrize("name", list(FLOAT32))
def test_sizes_of_float32_alone(name):
    from flexllm_amd._lib import FlexLLMError
    from flexllm_amd.registry import model_class
    cfg = FLOAT32[name]
    cases, checked = (lc, check_lopazen) if cfg["architecture"] == "Lopazen" else (nc, check_nifunex)
    checked(cfg, "float32", 40, [1], [30, 1])
    m = model_class(cfg["architecture"]).from_tensors(cfg, cases.weights(cfg, 5), dtype="float32", max_pos=64)
    m.set_wait_limit(1)                                    # it is the resident kernel that they take
    with pytest.raises(FlexLLMError, match="timed out"):
        m.step(m.pool.acquire("t"), [1], [0])
    m.close()


@BOTH
@pytest.mark.parametrize("heads,window", [(16, 1024), (16, 300), (32, 700)])
def test_splits_of_latent_rows(heads, window, dtype):
    """One more than a split, the window's edge, and beyond it."""
    cfg = nc.config([latent(heads, 0, window=window)], width=2048, vocab=512)
    check_nifunex(cfg, dtype, window + 90, [62, 1, 1, 1, window - 68, 1, 1, 1, 1, 1, 60, 1], max_pos=1152)


@BOTH
@pytest.mark.parametrize("dim", [64, 128])
def test_splits_of_the_rows(dim, dtype):
    """Around the number of rows from which on there are two splits, three, and where all of them have some."""
    alone = {64: 128, 128: 64}[dim] // (1 if dtype == "bfloat16" else 2)
    for rows in alone, 2 * alone, 16 * alone:
        check_lopazen(lc.config([attention(32, 8, dim, 0)], width=2048, vocab=512), dtype, rows + 5, [rows - 5, 1], max_pos=2112)


@BOTH
@pytest.mark.parametrize("rows_of", [64, 128, "latent"])
def test_splits_inside_a_loop(rows_of, dtype):
    """The second split, and with it the writers and readers of the words, comes in the middle of one launch: as step by step."""
    from flexllm_amd import to_device, zeros
    from flexllm_amd.lopazen import Lopazen
    from flexllm_amd.nifunex import Nifunex
    if rows_of == "latent":
        cfg, alone = nc.config([latent(16, 2048, window=None)] * 2, width=2048, vocab=512), 64
        m = Nifunex.from_tensors(cfg, nc.weights(cfg, 5), dtype=dtype, max_pos=256, slots=2)
    else:
        cfg, alone = lc.config([attention(32, 8, rows_of, 2048)] * 2, width=2048 * rows_of // 64, vocab=512), {64: 128, 128: 64}[rows_of] // (1 if dtype == "bfloat16" else 2)
        m = Lopazen.from_tensors(cfg, lc.weights(cfg, 5), dtype=dtype, max_pos=256, slots=2)
    toks = lc.tokens(cfg, alone - 4)
    a, b = [m.pool.acquire(n) for n in "ab"]
    for s in a, b:
        m.step(s, toks[:-1])
    token, out, one_by_one = to_device(np.array(toks[-1:], np.int32)), zeros((12,), np.int32), toks[-1:]
    m.decode(a, token, 12, out)
    for _ in range(12):
        one_by_one.append(int(m.step(b, one_by_one[-1:], [0])[0].argmax()))
    m.check()
    assert out.numpy().tolist() == one_by_one[1:]
    assert np.array_equal(m.step(a, [3], [0]), m.step(b, [3], [0]))
    m.close()


@BOTH
def test_loop_of_tokens(dtype):
    """70 greedy tokens (two launches) are those of 70 steps, in two slots in turn, continued by a step and by another loop."""
    from flexllm_amd import to_device, zeros
    from flexllm_amd.lopazen import Lopazen
    cfg = LOPAZEN["a loop"]
    w, toks = lc.weights(cfg, 5), lc.tokens(cfg, 30)
    ref = lopazen_ref.Reference(cfg, w)
    m = Lopazen.from_tensors(cfg, w, dtype=dtype, max_pos=256, slots=2)
    slots = [m.pool.acquire(n) for n in "ab"]
    for s in slots:
        m.step(s, toks[:29])
    got, want, token = [], toks[29:], to_device(np.array(toks[29:], np.int32))
    for n in (1, 2, 67):
        out = zeros((n,), np.int32)
        m.decode(slots[0], token, n, out)
        got += out.numpy().tolist()
        assert token.numpy()[0] == got[-1]
        for _ in range(n):
            want.append(int(m.step(slots[1], want[-1:], [0])[0].argmax()))
    m.check()
    assert got == want[1:] and m.length(slots[0]) == m.length(slots[1]) == 99
    last = [m.step(s, got[-1:], [0]) for s in slots]
    assert np.array_equal(last[0], last[1])
    err = lc.rel_err(last[0], ref.run(toks + got)[-1:])
    assert err.max() < lc.LIMIT[dtype]
    m.close()


@pytest.mark.parametrize("name", list(NIFUNEX)[:2])
def test_loops_and_steps_in_turn(name):
    """Steps hand out logits and no candidates: a loop behind one finds none of an earlier loop's."""
    from flexllm_amd import to_device, zeros
    from flexllm_amd.nifunex import Nifunex
    cfg = NIFUNEX[name]
    w, toks = nc.weights(cfg, 5), nc.tokens(cfg, 12)
    m = Nifunex.from_tensors(cfg, w, dtype="float32", max_pos=256)
    seen = []
    for n in (5, 5, 4, 4, 3, 3):
        for _ in range(6):
            slot = m.pool.acquire("t")
            got = [int(m.step(slot, toks, [11])[0].argmax())]
            token, out = to_device(np.array(got, np.int32)), zeros((n,), np.int32)
            m.decode(slot, token, n, out)
            last = m.step(slot, token, [0])
            got += out.numpy().tolist()
            seen.append((got, last))
            m.pool.release("t")
    m.check()
    m.close()
    for got, last in seen:
        assert got == seen[0][0][:len(got)]
    assert all(np.array_equal(a[1], b[1]) for a, b in zip(seen[:6], seen[6:12]))


def test_tokens_outside_the_vocabulary():
    """are reported, and taken as token 0."""
    from flexllm_amd._lib import FlexLLMError
    from flexllm_amd.lopazen import Lopazen
    cfg = LOPAZEN["rows of a quad"]
    m = Lopazen.from_tensors(cfg, lc.weights(cfg, 5), dtype="bfloat16", max_pos=64)
    out = []
    for t in (512, 0):
        s = m.pool.acquire("t")
        out.append(m.step(s, [t], [0]))
        if t:
            with pytest.raises(FlexLLMError, match="vocabulary"):
                m.check()
        m.pool.release("t")
    m.close()
    assert np.array_equal(*out)


def shared_rows(dtype="float32", **kw):
    from flexllm_amd.lopazen import Lopazen
    cfg = LOPAZEN["rows of a quad"]
    return cfg, Lopazen.from_tensors(cfg, lc.weights(cfg, 5), dtype=dtype, max_pos=256, **kw)


def latent_rows_and_gla(dtype="float32", **kw):
    from flexllm_amd.nifunex import Nifunex
    cfg = NIFUNEX["both kinds"]
    return cfg, Nifunex.from_tensors(cfg, nc.weights(cfg, 5), dtype=dtype, max_pos=256, **kw)


def mixture(dtype="float32", **kw):
    from flexllm_amd.nifunex import Nifunex
    moe = dict(mlp=nc.moe(8, 3, 1024, 0.75, 2048))
    cfg = nc.config([nc.gla(heads=16, dim=128, vdim=128, **moe), latent(16, 0, window=None)], width=2048, vocab=512)
    return cfg, Nifunex.from_tensors(cfg, nc.weights(cfg, 5), dtype=dtype, max_pos=256, **kw)


KINDS = pytest.mark.parametrize("make", [shared_rows, latent_rows_and_gla, mixture])


@KINDS
def test_waits_that_time_out(make):
    """are an error of the step, and of whatever comes behind a loop; the model is as before once it has been asked."""
    from flexllm_amd import to_device, zeros
    from flexllm_amd._lib import FlexLLMError
    cfg, m = make()
    toks = [7, 100, 33, 250, 4]
    want = m.generate(toks, 70)
    token, out = to_device(np.array([7], np.int32)), zeros((70,), np.int32)
    slot = m.pool.acquire("t")
    m.set_wait_limit(1)                                    # the first word that is not there yet
    with pytest.raises(FlexLLMError, match="timed out"):
        m.step(slot, toks[:1], [0])
    m.check()
    m.decode(slot, token, 70, out)
    m.stream().sync()
    m.set_wait_limit(0)
    for call in (lambda: m.decode(slot, token, 1, out), lambda: m.step(slot, toks), lambda: m.step(slot, toks[:1], [0])):
        with pytest.raises(FlexLLMError, match="timed out"):
            call()
    with pytest.raises(FlexLLMError, match="timed out"):
        m.check()
    m.pool.release("t")
    assert m.generate(toks, 70) == want
    m.check()
    m.close()


@KINDS
def test_chain_of_kernels_in_its_place(make):
    """Switched off, single tokens and loops, with and without a graph, are a chain of kernels, which waits for nothing; and on again."""
    from flexllm_amd import to_device, zeros
    from flexllm_amd._lib import FlexLLMError
    cfg, m = make()
    toks = [7, 100, 33, 250, 4]
    token, out = to_device(np.array([9], np.int32)), zeros((20,), np.int32)

    def request(use_graph=True):
        slot = m.pool.acquire("t")
        first = m.step(slot, toks, [4])
        token.copy_from(np.array([9], np.int32))
        m.decode(slot, token, 20, out, use_graph=use_graph)
        got = (first, m.step(slot, toks[:1], [0]), out.numpy().tolist())
        m.check()
        m.pool.release("t")
        return got

    want = request()
    m.set_wait_limit(1)                                    # the resident kernel would give up
    m.set_decode_mode(1)
    for use_graph in True, False:
        got = request(use_graph)
        assert np.array_equal(got[0], want[0]) and got[2] == want[2]
        assert lc.rel_err(got[1], want[1]).max() < lc.LIMIT["float32"]
    with pytest.raises(FlexLLMError, match="mode"):
        m.set_decode_mode(2)
    m.set_decode_mode(0)
    with pytest.raises(FlexLLMError, match="timed out"):
        request()
    m.close()


def test_infinities_and_not_a_number():
    """An infinite row of a weight is an infinity (or, against both signs, not a number) in that place alone."""
    from flexllm_amd.lopazen import Lopazen
    cfg = LOPAZEN["as many key heads"]
    w = lc.weights(cfg, 5)
    w["embed"] = w["embed"].copy()
    w["embed"][900, 7] = np.inf                            # the head is the embedding: one logit
    m = Lopazen.from_tensors(cfg, w, dtype="float32", max_pos=64)
    s = m.pool.acquire("t")
    got = m.step(s, lc.tokens(cfg, 1), [0])[0]
    m.check()
    m.close()
    assert np.isinf(got[900]) and np.isfinite(np.delete(got, 900)).all()


# Tokens whose embeddings, and weights whose rows, are not finite: what is not a number goes through every exchange
NOT_FINITE = {
    "shared rows": (LOPAZEN["rows of a quad"], ["l0.mix.k", "l0.mlp.up", "l1.mix.q"]),
    "latent rows and gla": (NIFUNEX["both kinds"], ["l0.mix.dkv", "l1.mix.v", "l1.mlp.gate"]),
    "mixtures": (nc.config([gla(16, 0) | dict(mlp=nc.moe(8, 3, 1024, 0.75, 2048)), latent(16, 0, window=None) | dict(mlp=nc.moe(8, 3, 1024, 0.75, 2048))], width=2048, vocab=512),
                 ["l0.mlp.router", "l0.mlp.shared.up", "l1.mlp.shared.sg"]),
    "rows of 12 blocks": (lc.config([attention(32, 8, 64, 6144)], width=2048, vocab=512), ["l0.mlp.down"]),
}


@BOTH
@pytest.mark.parametrize("name", list(NOT_FINITE))
def test_what_is_not_finite(name, dtype):
    """No wait takes it for a word that is not there; the places are those of the chain of kernels; a sequence in another slot is not
    touched by it.  A loop whose logits are all no numbers finds token 0."""
    from flexllm_amd import to_device, zeros
    from flexllm_amd.registry import model_class
    cfg, infinite = NOT_FINITE[name]
    cases = lc if cfg["architecture"] == "Lopazen" else nc
    base = cases.weights(cfg, 5)
    base["embed"] = base["embed"].copy()
    base["embed"][300, 5], base["embed"][301, 9], base["embed"][302, 5:8] = np.inf, np.nan, [np.inf, -np.inf, np.nan]
    if "head" not in base:                                 # logits of their own, then, are no numbers: 300 to 302 are left out below
        others = np.delete(np.arange(cfg["vocab"]), [300, 301, 302])
    else:
        others = np.arange(cfg["vocab"])
    clean = [7, 100, 33, 250, 4]

    def model(w):
        m = model_class(cfg["architecture"]).from_tensors(cfg, w, dtype=dtype, max_pos=256, slots=2)
        return m, m.pool.acquire("bad"), m.pool.acquire("good")

    def steps(m, slot, toks):
        return np.stack([m.step(slot, [t], [0])[0] for t in toks])

    m, bad, good = model(base)
    want = steps(m, good, clean)
    assert np.isfinite(want[:, others]).all()
    for t in 300, 301, 302:
        m.pool.release("bad")
        bad = m.pool.acquire("bad")
        got = steps(m, bad, [8, t, 9])
        assert np.isfinite(got[0, others]).all() and np.isnan(got[1, others]).all()
        token, out = to_device(np.array([t], np.int32)), zeros((9,), np.int32)
        m.decode(bad, token, 9, out)
        m.check()
        assert out.numpy().tolist() == [0] * 9
        m.pool.release("good")
        good = m.pool.acquire("good")
        assert np.array_equal(steps(m, good, clean)[:, others], want[:, others])
    m.check()
    m.close()
    for t in infinite:
        w = dict(base, **{t: base[t].copy()})
        w[t].reshape(-1)[w[t].size // 2 + 11] = np.inf     # a row in the middle
        m, bad, good = model(w)
        got = steps(m, bad, clean)
        m.check()
        m.set_decode_mode(1)
        chain = steps(m, good, clean)
        m.check()
        m.close()
        for kind in np.isnan, np.isposinf, np.isneginf:
            assert np.array_equal(kind(got), kind(chain)), (t, kind)
        finite = np.isfinite(chain).all(0)
        if finite.any():
            assert cases.rel_err(got[:, finite], chain[:, finite]).max() < cases.LIMIT[dtype]


# an infinite weight in rows of 12 blocks of k and of 28, of which a wave has one or two and three or four, in a wave's first block and in a later one; in rows of four
# blocks, in the query in a workgroup's last group of two rows instead of four; clamped gates and units, which leave finite logits (a gate where it is above zero).
# "units": two hidden values beyond float32 instead, where their gates are above zero.  What is not finite behind a down product is no number in all logits.
LONG_ROWS = [(6144, "l0.mlp.down", 0, 3), (6144, "l0.mlp.down", 1031, 6000), (14336, "l0.mlp.down", 1029, 11000), (6144, "l0.mix.q", 1029, 2000),
             (6144, "l0.mlp.gate", 3071, 5), (6144, "l0.mlp.up", 6143, 2047), (14336, "l0.mlp.up", 77, 1030), (6144, "units", 700, 5000), (14336, "units", 5, 14000)]


@BOTH
@pytest.mark.parametrize("ff,name,row,col", LONG_ROWS)
def test_not_finite_in_long_rows(ff, name, row, col, dtype):
    """The places that are no number, infinite and finite are those of the chain of kernels, and the finite ones agree."""
    from flexllm_amd.registry import model_class
    clamped = name.endswith(("gate", "up"))
    cfg = nc.config([gla(16, ff)], width=2048, vocab=514) if clamped else lc.config([attention(32, 8, 64, ff)], width=2048, vocab=514)
    w = (nc if clamped else lc).weights(cfg, 5)
    if name == "units":
        for unit in row, col:
            w["l0.mlp.gate"][unit] = lc.round_bf16(w["l0.mlp.gate"][unit] * np.float32(1e4))
            w["l0.mlp.up"][unit] = lc.round_bf16(w["l0.mlp.up"][unit] * np.float32(1e36))
            w["l0.mlp.down"][::3, unit] = 0.0              # no number with an infinite unit
    else:
        w[name][row, col] = np.inf
    m = model_class(cfg["architecture"]).from_tensors(cfg, w, dtype=dtype, max_pos=64, slots=2)
    got = []
    for i, mode in enumerate((0, 1)):
        m.set_decode_mode(mode)
        slot = m.pool.acquire(str(i))
        got.append(np.stack([m.step(slot, [t], [0])[0] for t in (7, 100, 33, 250, 4, 19, 60, 301)]))
        m.check()
    m.close()
    for kind in np.isnan, np.isposinf, np.isneginf:
        assert np.array_equal(kind(got[0]), kind(got[1])), kind
    finite = np.isfinite(got[1]).all(1)
    assert finite.all() == name.endswith("up") and (finite.any() or not clamped)
    if clamped:                                            # (the tail of a gelu times a unit of 1e36 is finite and has no digits to agree in)
        assert lc.rel_err(got[0][finite], got[1][finite]).max() < lc.LIMIT[dtype]


# a head of so many rows that its sums leave no room for a vector in three parts: bfloat16 weights meet it as it is, waves meet by counts all the same
@pytest.mark.parametrize("kind", ["shared rows", "latent rows and gla"])
def test_vectors_that_lie_whole(kind):
    from flexllm_amd._lib import FlexLLMError
    from flexllm_amd.lopazen import Lopazen
    from flexllm_amd.nifunex import Nifunex
    vocab = 600064                                         # 2344 rows per workgroup, 8 sums each: 73 KiB beside 24 KiB of the vector
    if kind == "shared rows":
        m = Lopazen.synthetic(lc.config([attention(32, 8, 64, 6144), attention(32, 8, 64, 2048)], width=4096, vocab=vocab), dtype="bfloat16", max_pos=64, slots=2)
    else:
        m = Nifunex.synthetic(nc.config([latent(16, 6144, window=40), gla(16, 2048)], width=4096, vocab=vocab), dtype="bfloat16", max_pos=64, slots=2)
    toks, got = [7, 100, 599999, 250, 4, 300001], []
    for i, mode in enumerate((0, 1)):
        m.set_decode_mode(mode)
        slot = m.pool.acquire(str(i))
        got.append(np.stack([m.step(slot, [t], [0])[0] for t in toks]))
        m.check()
    # Both have float32 activations; what may differ are cached rows, on one side or the other of a bfloat16 step: 2^-8 at worst.
    assert lc.rel_err(got[0], got[1]).max() < 2.0 ** -8
    m.set_decode_mode(0)
    m.set_wait_limit(1)                                    # it is the resident kernel that they take
    m.pool.release("0")
    with pytest.raises(FlexLLMError, match="timed out"):
        m.step(m.pool.acquire("0"), [1], [0])
    m.close()


def test_two_models_on_streams_of_their_own():
    """Each launch needs the whole chip: they run one after the other, whatever streams they are on and threads they come from."""
    import threading
    from flexllm_amd.lopazen import Lopazen
    cfg = LOPAZEN["rows of a quad"]
    w, prompt = lc.weights(cfg, 5), lc.tokens(cfg, 12)
    models = [Lopazen.from_tensors(cfg, w, dtype="bfloat16", max_pos=256) for _ in range(2)]
    want = models[0].generate(prompt, 30)
    got = {}

    def work(i):
        got[i] = [models[i].generate(prompt, 30) for _ in range(10)]

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert got == {i: [want] * 10 for i in range(2)}
    [m.close() for m in models]
