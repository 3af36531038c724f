"""Gated units whose gate lies so far below zero that 1 + exp(-gate) leaves float32: the unit is nothing, wherever it is formed."""
import numpy as np
import pytest

import lopazen_cases as lc
import nifunex_cases as nc
import test_gpu_decode_float as resident
from oracle import lopazen_ref, nifunex_ref

pytestmark = pytest.mark.gpu
BOTH = pytest.mark.parametrize("dtype", ["float32", "bfloat16"])


def gates(n):
    """n gates: far ones from -500 on, where gelu's cube is still finite, among ordinary ones."""
    g = -np.geomspace(500.0, 1e12, n).astype(np.float32)
    named = np.array([-500, -877, -1100, -1300, -2000, -3000, -1e4, -3e7, -4.7e7, -1e8], np.float32)
    g[3:3 + len(named)] = named
    g[::7] = np.linspace(-6, 6, len(g[::7]))
    return g


def weights(n, k):
    """Rows 2i and 2i+1: gate i in two bfloat16 parts, against a vector of ones at the first two k, and an up of 1.5."""
    g, w = gates(n // 2), np.zeros((n, k), np.float32)
    w[0::2, 0] = lc.round_bf16(g)
    w[0::2, 1] = lc.round_bf16(g - w[0::2, 0])
    w[1::2, 0] = 1.5
    return w


def check_units(got, w, glu, tol):
    g = w[0::2, :2].astype(np.float64).sum(1)
    u = np.full_like(g, 1.5)
    want = nifunex_ref.clamped_glu(g, u, 3.0) if glu == 1 else lopazen_ref.gelu(g) * u
    far = g < -400
    # the exponential is capped at 2^126 times a factor that is seldom below a thousandth
    assert np.all(np.abs(got[:, far]) <= 1e-30 * np.abs(g[far]))
    assert np.all(np.abs(got[:, ~far] - want[~far]) <= tol * (np.abs(want[~far]) + 1e-3))


# tiles of 256 columns (every output form of theirs has the unit to itself), of 128 and fewer, up to 32 rows
@BOTH
@pytest.mark.parametrize("glu", [1, 2])
@pytest.mark.parametrize("m,n,k", [(1024, 16384, 320), (961, 2048, 256), (100, 1028, 128), (100, 1030, 128), (9, 8192, 64), (32, 16384, 128)])
def test_products_of_many_rows(m, n, k, glu, dtype):
    from flexllm_amd import ops, to_device
    from flexllm_amd.loader import from_bf16, to_bf16
    w, a = weights(n, k), np.zeros((m, k), np.float32)
    a[:, :2] = 1.0
    dev = to_device if dtype == "float32" else lambda x: to_device(to_bf16(x))
    y = ops.linear_float(dev(a), dev(w), n, glu, 3.0)[0].numpy()
    check_units(y if dtype == "float32" else from_bf16(y), w, glu, 1e-5 if dtype == "float32" else 5e-3)


@BOTH
@pytest.mark.parametrize("glu", [1, 2])
@pytest.mark.parametrize("tokens", [1, 2, 3, 8])
@pytest.mark.parametrize("k", [64, 2112, 4160])
def test_products_of_a_step(k, tokens, glu, dtype):
    from flexllm_amd import ops, to_device
    from flexllm_amd.loader import to_bf16
    w, x = weights(1030, k), np.zeros((tokens, k), np.float32)
    x[:, :2] = 1.0
    y = ops.linear_float_step(to_device(x), to_device(w if dtype == "float32" else to_bf16(w)), glu=glu, limit=3.0)[0].numpy()
    check_units(y, w, glu, 1e-5)


# names of the gates in the models' weights, and how far every eighth of them is moved out (all of them would make steps of the units, over
# which bfloat16 falls one way or the other)
FAR = {".gate": 1e9, "mix.g": 1e9, "shared.sg": 1e10}
MODELS = {
    "gelu": (lc.config([lc.layer(heads=4, kv_heads=2, dim=32, mlp=lc.dense(96)), lc.layer()]), False),
    "gelu, resident": (lc.config([resident.attention(32, 8, 64, 2048)], width=2048, vocab=512), False),
    "every gate": (nc.mixed(), True),
    "clamped units and recurrences, resident": (nc.config([resident.latent(16, 2048), resident.gla(16, 2048)], width=2048, vocab=512), True),
    "experts, resident": (nc.config([nc.gla(heads=16, dim=128, vdim=128, mlp=nc.moe(8, 3, 1024, 1.5, 2048))], width=2048, vocab=512), True),
}


@BOTH
@pytest.mark.parametrize("name", list(MODELS))
def test_whole_models(name, dtype):
    """Steps of one token in the resident kernel (where the sizes allow it) and in the chain, of several tokens, prompts: finite, and
    what the equations say.  gelu's gates go to a few thousand, the others' to 1e9."""
    from flexllm_amd.lopazen import Lopazen
    from flexllm_amd.nifunex import Nifunex
    cfg, nif = MODELS[name]
    cases, cls, ref = (nc, Nifunex, nifunex_ref) if nif else (lc, Lopazen, lopazen_ref)
    w, toks = cases.weights(cfg, 11), cases.tokens(cfg, 37)
    for n in w:
        for end, factor in FAR.items():
            if n.endswith(end):
                w[n][::8] = lc.round_bf16(w[n][::8] * np.float32(factor if nif else 3e3))
    want = ref.Reference(cfg, w).run(toks)
    m = cls.from_tensors(cfg, w, dtype=dtype, max_pos=64)
    for mode, cuts in ((0, [1]), (1, [1]), (0, [3]), (0, [8]), (0, [37])):
        m.set_decode_mode(mode)
        got, slot = [], m.pool.acquire("t")
        for p in range(0, len(toks), cuts[0]):
            got.append(m.step(slot, toks[p:p + cuts[0]], range(min(cuts[0], len(toks) - p))))
        m.check()
        m.pool.release("t")
        got = np.concatenate(got)
        assert np.isfinite(got).all(), (mode, cuts)
        err = lc.rel_err(got, want)
        # a far gate near zero, or a choice of experts, that falls the other way by a rounding to bfloat16 changes a token altogether
        share = 1.0 if dtype == "float32" else 0.75 if any("router" in n for n in w) else 0.9
        assert (err < lc.LIMIT[dtype]).mean() >= share, (mode, cuts, err.max())
    m.close()
