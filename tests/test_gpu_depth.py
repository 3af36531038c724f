"""Depth and length: the full-size model (16 layers, hidden 2048 / 8192, context 4096) against the oracle, layer by
layer with the oracle's own layer input fed to the device ("teacher forcing"), so that each layer is judged on
identical inputs and a rounding tie that falls the other way in one layer is seen there and not amplified by the
layers above; plus one free-running token through all 16 layers, long greedy runs of both decode schedules against
each other, a run that crosses a 128-key chunk boundary inside one launch, and a change of schedule in mid-sequence."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PER_LAYER = ("wq", "wk", "wv", "wo", "wg", "wu", "wd", "sq", "sk", "sv", "so", "sg", "su", "sd")


def token_err(a, ref):
    """per-token maximum error relative to the tensor's scale"""
    a = np.asarray(a, np.float64).reshape(-1, a.shape[-1]); ref = np.asarray(ref, np.float64).reshape(a.shape)
    return np.abs(a - ref).max(axis=1) / np.abs(ref).max()


def layer_views(cfg, w, l, vocab1, device):
    """Weight set of a 1-layer model that is layer l of the deep one: device views / numpy slices, nothing copied.
    gamma rows 2l, 2l+1 become rows 0, 1; row 2 (the final norm of the 1-layer model) is whatever follows."""
    H, qh, kvh = cfg["hidden"], cfg["q_heads"], cfg["kv_heads"]
    out = {n: [w[n][l]] for n in PER_LAYER}
    if device:
        out["gamma"] = w["gamma"].view(2 * l * H * 4, (3, H))
        for n, heads in (("q_s", qh), ("k_s", kvh), ("v_s", kvh), ("a_s", qh)):
            out[n] = w[n].view(l * heads * 4, (1, heads))
        out["embed"] = w["embed"].view(0, (vocab1, H))
    else:
        out["gamma"] = np.ascontiguousarray(w["gamma"][2 * l:2 * l + 3])
        for n in ("q_s", "k_s", "v_s", "a_s"):
            out[n] = np.ascontiguousarray(w[n][l:l + 1])
        out["embed"] = np.ascontiguousarray(w["embed"][:vocab1])
    out["rope_sin"], out["rope_cos"] = w["rope_sin"], w["rope_cos"]
    return out


@pytest.fixture(scope="module")
def full():
    """The benchmark's model on the device and, copied back from there, on the host (bit-identical by construction)."""
    import flexllm_amd as fx
    from flexllm_amd import llama
    from oracle import oracle
    oracle.build()
    cfg = llama.make_config()
    assert cfg["layers"] == 16 and cfg["max_pos"] == 4096
    dev_w = llama.synth_weights(cfg, seed=1, device=True, embed_range=0.03)
    host_w = {}
    for n, v in dev_w.items():
        host_w[n] = [a.numpy() for a in v] if isinstance(v, list) else v.numpy()
    host_w["embed"] = host_w["embed"].view(np.uint16)
    yield fx, llama, oracle, cfg, dev_w, host_w


def test_decode_16_layers_teacher_forced_and_free_running(full):
    """Decode of one token at position 4095 (all 32 key chunks of every KV head in use).
    (1) Layer by layer: the device layer l (a 1-layer model built from layer l's weights and cache) gets the ORACLE's
    layer input and must reproduce the oracle's layer output to fp32 rounding; a layer in which one of its ~150 k
    roundings to int8 / uint8 sat on a tie may differ by the effect of one quantisation step, and such layers are
    counted.  (2) Free-running: the 16-layer persistent kernel from the same token, hidden state and logits against
    the oracle's 16-layer function."""
    fx, llama, oracle, cfg, dev_w, host_w = full
    L, H, P, KV = cfg["layers"], cfg["hidden"], cfg["max_pos"], cfg["kv_hidden"]
    pos = P - 1
    r = np.random.default_rng(41)
    kc = np.zeros((L, P, KV), np.int8); vc = np.zeros((L, P, KV), np.int8)
    kc[:, :pos] = r.integers(-100, 101, (L, pos, KV)); vc[:, :pos] = r.integers(-100, 101, (L, pos, KV))
    x0 = r.standard_normal(H).astype(np.float32)

    om = oracle.OracleModel(cfg, host_w)
    kc_ref, vc_ref = kc.copy(), vc.copy()
    hid_ref, logits_ref = om.decode_token(x0, pos, kc_ref, vc_ref)

    cfg1 = llama.make_config(layers=1, vocab=256)
    x = x0
    errs, cache_diffs = [], 0
    for l in range(L):
        print("layer", l, flush=True)
        om1 = oracle.OracleModel(cfg1, layer_views(cfg, host_w, l, 256, device=False))
        k1, v1 = kc[l:l + 1].copy(), vc[l:l + 1].copy()
        y_ref, _ = om1.decode_token(x, pos, k1, v1, want_logits=False)
        assert np.array_equal(k1[0], kc_ref[l]) and np.array_equal(v1[0], vc_ref[l])     # the chain IS the 16-layer oracle
        m1 = llama.Llama(cfg1, layer_views(cfg, dev_w, l, 256, device=True))
        m1.load_caches_token_major(kc[l:l + 1], vc[l:l + 1])
        y, _ = m1.decode_hidden(fx.to_device(x), pos)
        y = y.numpy()
        m1.check()
        kg, vg = m1.caches_token_major()
        assert np.array_equal(kg[0, :pos], kc[l, :pos]) and np.array_equal(vg[0, :pos], vc[l, :pos])   # history untouched
        d = np.abs(kg[0, pos].astype(int) - k1[0, pos]).max(), np.abs(vg[0, pos].astype(int) - v1[0, pos]).max()
        assert max(d) <= 1
        cache_diffs += int((kg[0, pos] != k1[0, pos]).sum() + (vg[0, pos] != v1[0, pos]).sum())
        errs.append(float(token_err(y[None], y_ref[None])[0]))
        m1.close()
        x = y_ref                                                     # teacher forcing: the oracle's output feeds the next layer
    assert np.array_equal(x, hid_ref)
    errs = np.array(errs)
    print("per-layer errors, teacher-forced:", " ".join("%.1e" % e for e in errs), "| cache bytes off by one:", cache_diffs, flush=True)
    exact = errs <= 2e-5
    assert exact.sum() >= L - 4, "more than four layers differ beyond fp32 rounding: %s" % errs
    assert errs.max() <= 1e-2 and cache_diffs <= 4       # a flipped tie moves one value by one step, never more

    model = llama.Llama(cfg, dev_w)
    model.load_caches_token_major(kc, vc)
    hid, logits = model.decode_hidden(fx.to_device(x0), pos, want_logits=True)
    model.check()
    e_h = float(token_err(hid.numpy()[None], hid_ref[None])[0]); e_l = float(token_err(logits.numpy()[None], logits_ref[None])[0])
    print("free-running 16 layers: hidden %.2e logits %.2e; argmax %d / %d" % (e_h, e_l, int(logits.numpy().argmax()), int(logits_ref.argmax())), flush=True)
    # every flipped tie below is amplified by the layers above it (random weights): the free-running error is reported,
    # and bounded by what the counted flips explain
    assert e_h <= (2e-5 if exact.all() else 0.5)
    kg, vg = model.caches_token_major()
    assert np.array_equal(kg[0, pos], kc_ref[0, pos]) or np.abs(kg[0, pos].astype(int) - kc_ref[0, pos]).max() <= 1
    model.close()


def test_prefill_16_layers_teacher_forced(full):
    """A 64-token prefill, layer by layer on the oracle's layer inputs: per token the device's layer output equals the
    oracle's to fp32 rounding unless a rounding tie of that token fell the other way (counted)."""
    fx, llama, oracle, cfg, dev_w, host_w = full
    L, H = cfg["layers"], cfg["hidden"]
    S = 64
    r = np.random.default_rng(42)
    x = r.standard_normal((S, H)).astype(np.float32)
    cfg1 = llama.make_config(layers=1, vocab=256, max_pos=128)
    beyond, worst, medians = 0, 0.0, []
    for l in range(L):
        print("layer", l, flush=True)
        hw = layer_views(cfg, host_w, l, 256, device=False)
        hw["rope_sin"], hw["rope_cos"] = host_w["rope_sin"][:128], host_w["rope_cos"][:128]
        dw = layer_views(cfg, dev_w, l, 256, device=True)
        dw["rope_sin"] = dev_w["rope_sin"].view(0, (128, 32)); dw["rope_cos"] = dev_w["rope_cos"].view(0, (128, 32))
        om1 = oracle.OracleModel(cfg1, hw)
        k1, v1 = om1.new_caches()
        y_ref = om1.prefill(x, k1, v1)
        m1 = llama.Llama(cfg1, dw)
        y = m1.prefill_hidden(fx.to_device(x)).numpy()
        e = token_err(y, y_ref)
        kg, vg = m1.caches_token_major()
        dk = np.abs(kg[0, :S].astype(int) - k1[0, :S]); dv = np.abs(vg[0, :S].astype(int) - v1[0, :S])
        assert dk.max() <= 1 and dv.max() <= 1
        n_beyond = int((e > 2e-5).sum())
        print("  tokens beyond fp32 rounding: %d, median %.1e, worst %.1e, cache bytes off by one: %d"
              % (n_beyond, np.median(e), e.max(), int((dk != 0).sum() + (dv != 0).sum())), flush=True)
        beyond += n_beyond; worst = max(worst, float(e.max())); medians.append(float(np.median(e)))
        m1.close()
        x = y_ref
    # A layer makes about 1.1 million roundings to int8 / uint8 on 64 tokens; the few that sit on a tie may fall the other
    # way (one step), and a flipped byte of a token's K or V row also touches every later token of that layer through
    # attention, by much less.  So: most tokens exact to fp32 rounding, every layer's typical token exact (at most one
    # layer where an early token's cache byte flipped), nothing beyond the effect of single steps.
    assert beyond <= 0.2 * L * S and worst <= 2e-2, (beyond, worst)
    assert sum(m <= 2e-5 for m in medians) >= L - 1, medians


def test_256_token_greedy_run_both_schedules(full):
    """256 greedy tokens of the full-size model from position 3840 (the context grows to 4096), persistent kernel
    against one kernel per stage, on an embedding table whose logits are of order one so that the generated ids
    keep changing.  Ids and cache bytes must be identical; compared launch by launch, stopping at the first mismatch."""
    fx, llama, oracle, cfg, dev_w, host_w = full
    a, b = llama.Llama(cfg, dev_w), llama.Llama(cfg, dev_w)
    b.set_decode_mode(1)
    lib = fx.lib()
    for m in (a, b):
        fx.check(lib.flexllm_rt_fill_i8(C.c_void_p(m.k_cache.ptr), C.c_size_t(m.k_cache.size), C.c_uint64(911), -100, 100, None))
        fx.check(lib.flexllm_rt_fill_i8(C.c_void_p(m.v_cache.ptr), C.c_size_t(m.v_cache.size), C.c_uint64(912), -100, 100, None))
    steps, pos0, first = 256, 4096 - 256, 777
    stream = fx.Stream()
    outs = []
    for m in (a, b):
        tok = fx.to_device(np.array([first], np.int32)); out = fx.zeros((steps,), np.int32)
        print("greedy run, mode", 0 if m is a else 1, flush=True)
        m.decode_greedy(tok, pos0, steps, out, use_graph=1, stream=stream)
        stream.sync(); m.check()
        outs.append(out.numpy())
        assert int(tok.numpy()[0]) == int(outs[-1][-1])
    ga, gb = outs
    assert len(set(ga.tolist())) > 20, "the run should visit many different ids: %s" % ga[:16]
    mism = np.nonzero(ga != gb)[0]
    assert mism.size == 0, "first mismatch at step %d: %d vs %d" % (mism[0], ga[mism[0]], gb[mism[0]])
    assert np.array_equal(a.k_cache.numpy(), b.k_cache.numpy()) and np.array_equal(a.v_cache.numpy(), b.v_cache.numpy())
    a.close(); b.close()


def test_full_size_runs_are_identical_to_the_byte(full):
    """48 greedy tokens of the full-size model up to the maximum context (every one of the 256 workgroups takes part
    in the attention), thirty times: ids and cache bytes identical each time (see
    test_repeated_runs_are_identical_to_the_byte)."""
    import hashlib
    fx, llama, oracle, cfg, dev_w, host_w = full
    m = llama.Llama(cfg, dev_w)
    lib = fx.lib()
    fx.check(lib.flexllm_rt_fill_i8(C.c_void_p(m.k_cache.ptr), C.c_size_t(m.k_cache.size), C.c_uint64(921), -100, 100, None))
    fx.check(lib.flexllm_rt_fill_i8(C.c_void_p(m.v_cache.ptr), C.c_size_t(m.v_cache.size), C.c_uint64(922), -100, 100, None))
    steps, pos0 = 48, 4096 - 48
    out = fx.zeros((steps,), np.int32)
    seen = set()
    for rep in range(30):
        tok = fx.to_device(np.array([4242], np.int32))
        m.decode_greedy(tok, pos0, steps, out, use_graph=0)
        m.check()
        h = hashlib.md5(out.numpy().tobytes())
        h.update(m.k_cache.numpy().tobytes()); h.update(m.v_cache.numpy().tobytes())
        seen.add(h.hexdigest())
        assert len(seen) == 1, "run %d differs from the runs before it" % rep
    assert len(set(out.numpy().tolist())) > 10
    m.close()


@pytest.fixture(scope="module")
def two_layer():
    import flexllm_amd as fx
    from flexllm_amd import llama
    from oracle import oracle
    oracle.build()
    cfg = llama.make_config(layers=2, vocab=4096, max_pos=256)
    host_w = llama.synth_weights(cfg, seed=21, device=False, embed_range=0.03)
    dev_w = llama.synth_weights(cfg, seed=21, device=True, embed_range=0.03)
    yield fx, llama, oracle, cfg, dev_w, host_w


@pytest.mark.parametrize("top_k", [0, 5], ids=["greedy", "top5"])
def test_run_across_a_key_chunk_boundary(two_layer, top_k):
    """80 tokens from position 100 on the persistent kernel: the first launch (64 tokens) crosses position 127 -> 128,
    where a second workgroup per KV head becomes active and takes over the new token's cache row in mid-launch; the
    run spans two launches.  Checked (a) against the one-kernel-per-stage schedule (ids and cache bytes identical);
    (b) step by step: a third model is fed the run's ids one decode step at a time, which is bit for bit the same forward
    pass - its logits must select the run's next id (arg-max, or the oracle's sampler on those logits with the same
    uniform number), which pins the in-kernel selection, the hand-over of the id and the indexing of the uniform numbers;
    (c) against the oracle, teacher-forced on the same ids and cache bytes: logits to fp32 rounding at the typical
    step and within the tie effect at every step, appended cache rows equal up to single steps."""
    fx, llama, oracle, cfg, dev_w, host_w = two_layer
    steps, pos0, first = 80, 100, 333
    r = np.random.default_rng(5)
    kc = np.zeros((cfg["layers"], cfg["max_pos"], cfg["kv_hidden"]), np.int8); vc = np.zeros_like(kc)
    kc[:, :pos0] = r.integers(-100, 101, (cfg["layers"], pos0, cfg["kv_hidden"]))
    vc[:, :pos0] = r.integers(-100, 101, (cfg["layers"], pos0, cfg["kv_hidden"]))
    rands = r.uniform(0, 1, steps).astype(np.float32)
    res = []
    for mode in (0, 1):
        m = llama.Llama(cfg, dev_w)
        m.set_decode_mode(mode)
        m.load_caches_token_major(kc, vc)
        tok = fx.to_device(np.array([first], np.int32)); out = fx.zeros((steps,), np.int32)
        if top_k:
            m.decode_sample(tok, pos0, steps, fx.to_device(rands), top_k, out)
        else:
            m.decode_greedy(tok, pos0, steps, out, use_graph=0)
        m.check()
        res.append((out.numpy().copy(),) + m.caches_token_major())
        m.close()
    (ga, ka, va), (gb, kb, vb) = res
    mism = np.nonzero(ga != gb)[0]
    assert mism.size == 0, "schedules part at step %d" % mism[0]
    assert np.array_equal(ka, kb) and np.array_equal(va, vb)
    assert len(set(ga.tolist())) > 10
    om = oracle.OracleModel(cfg, host_w)
    kr, vr = kc.copy(), vc.copy()
    step_model = llama.Llama(cfg, dev_w)
    step_model.load_caches_token_major(kc, vc)
    t, errs, skipped, row_flips = first, [], 0, 0
    for i in range(steps):
        x = fx.ops.embed_f16(step_model._embed, fx.to_device(np.array([t], np.int32)))
        _, lg = step_model.decode_hidden(x, pos0 + i, want_logits=True)
        lg = lg.numpy()
        if top_k:
            want, idx, val, prob = oracle.sample_topk(lg, top_k, float(rands[i]), 8)
            if np.abs(np.cumsum(prob.astype(np.float64)) - rands[i]).min() > 1e-5:      # device expf against glibc at a boundary
                assert int(ga[i]) == want, "step %d" % i
            else:
                skipped += 1
        else:
            assert int(ga[i]) == int(np.argmax(lg)), "step %d" % i
        _, logits = om.decode_token(oracle.embed(host_w["embed"], t), pos0 + i, kr, vr)
        errs.append(float(token_err(lg[None], logits[None])[0]))
        # the cache rows this step appended: equal up to a single step where a rounding tie fell the other way; the
        # oracle then continues on the device's bytes, so that each step is judged on identical history
        ks, vs = step_model.caches_token_major()
        for dev, ref in ((ks, kr), (vs, vr)):
            d = np.abs(dev[:, pos0 + i].astype(int) - ref[:, pos0 + i])
            assert d.max() <= 1
            row_flips += int((d != 0).sum())
            ref[:, pos0 + i] = dev[:, pos0 + i]
        t = int(ga[i])
    step_model.check()
    errs = np.array(errs)
    print("logit errors against the oracle: median %.1e, max %.1e, steps beyond 2e-3: %d; cache bytes off by one: %d"
          % (np.median(errs), errs.max(), (errs > 2e-3).sum(), row_flips), flush=True)
    n = pos0 + steps
    assert skipped <= 1 and np.median(errs) <= 1e-4 and errs.max() <= 3e-2 and (errs > 2e-3).mean() <= 0.1
    assert row_flips <= 5e-3 * steps * 2 * cfg["layers"] * cfg["kv_hidden"]       # a flip in layer 0 moves many bytes of layer 1's rows
    ks, vs = step_model.caches_token_major()
    assert np.array_equal(ks, ka) and np.array_equal(vs, va)                             # the same forward passes indeed
    step_model.close()
    assert not ka[:, n:].any() and not va[:, n:].any()


def test_change_of_decode_schedule_in_mid_sequence(two_layer):
    """One kernel per stage for a token, then the persistent kernel for the next: the attention accumulators the first
    schedule leaves behind must not leak into the second (and the other way round).  Compared with a model that never
    changes schedule and with the oracle."""
    fx, llama, oracle, cfg, dev_w, host_w = two_layer
    from flexllm_amd import synth
    sw = llama.Llama(cfg, dev_w)
    steady = llama.Llama(cfg, dev_w)
    om = oracle.OracleModel(cfg, host_w)
    kr, vr = om.new_caches()
    modes = [1, 0, 0, 1, 0]
    for pos, mode in enumerate(modes):
        sw.set_decode_mode(mode)
        x = synth.host_normal_f32((cfg["hidden"],), 700 + pos)
        h_sw, _ = sw.decode_hidden(fx.to_device(x), pos)
        h_st, _ = steady.decode_hidden(fx.to_device(x), pos)
        h_ref, _ = om.decode_token(x, pos, kr, vr, want_logits=False)
        h_sw, h_st = h_sw.numpy(), h_st.numpy()
        assert token_err(h_sw[None], h_st[None])[0] <= 1e-5, "position %d (mode %d)" % (pos, mode)
        assert token_err(h_sw[None], h_ref[None])[0] <= 2e-3
    sw.check(); steady.check()
    for a, b in zip(sw.caches_token_major(), steady.caches_token_major()):
        assert np.array_equal(a, b)
    sw.close(); steady.close()


@pytest.mark.parametrize("top_k", [0, 5], ids=["greedy", "top5"])
def test_repeated_runs_are_identical_to_the_byte(two_layer, top_k):
    """The same 80-token run (two launches, crossing the chunk boundary at position 128) 400 times on one model: token
    ids and every cache byte identical each time, whether the rows the run writes are left in place, reloaded as zeros
    or reloaded with their final values.  All arithmetic of the persistent kernel is order-independent (integer
    accumulation, fixed reduction trees), so any difference is an exchange between workgroups gone wrong: this is the
    check that showed the attention accumulators being cleared before a slow workgroup had read them (about 1 % of
    such runs on some boxes, none on others)."""
    import hashlib
    fx, llama, oracle, cfg, dev_w, host_w = two_layer
    steps, pos0, first = 80, 100, 333
    r = np.random.default_rng(5)
    kc = np.zeros((cfg["layers"], cfg["max_pos"], cfg["kv_hidden"]), np.int8); vc = np.zeros_like(kc)
    kc[:, :pos0] = r.integers(-100, 101, (cfg["layers"], pos0, cfg["kv_hidden"]))
    vc[:, :pos0] = r.integers(-100, 101, (cfg["layers"], pos0, cfg["kv_hidden"]))
    rands = fx.to_device(r.uniform(0, 1, steps).astype(np.float32))
    m = llama.Llama(cfg, dev_w)
    out = fx.zeros((steps,), np.int32)

    def run():
        tok = fx.to_device(np.array([first], np.int32))
        if top_k:
            m.decode_sample(tok, pos0, steps, rands, top_k, out)
        else:
            m.decode_greedy(tok, pos0, steps, out, use_graph=0)
        m.check()
        k, v = m.caches_token_major()
        return out.numpy().copy(), k, v

    m.load_caches_token_major(kc, vc)
    ids0, k0, v0 = run()
    assert len(set(ids0.tolist())) > 10
    want = hashlib.md5(ids0.tobytes() + k0.tobytes() + v0.tobytes()).hexdigest()
    for rep in range(400):
        if rep % 3 == 0:
            m.load_caches_token_major(kc, vc)
        elif rep % 3 == 1:
            m.load_caches_token_major(k0, v0)
        ids, k, v = run()
        if hashlib.md5(ids.tobytes() + k.tobytes() + v.tobytes()).hexdigest() != want:
            step = np.nonzero(ids != ids0)[0]
            rows = np.nonzero((k != k0).any(axis=(0, 2)) | (v != v0).any(axis=(0, 2)))[0]
            raise AssertionError("run %d differs: ids from step %s, cache rows %s" % (rep, step[:1], rows[:4]))
    m.close()


# ---------------------------------------------------------------------------------------------------------------
# The 1024-token prefill of the full-size model: the size at which the launcher picks the 256x256 gate/up tile, the
# 64x128 down tile and the eight-wave attention with four key tiles per wave.

def _stage_chain_with_substitution(fx, oracle, cfg, host_w, dev_w, l, x):
    """Layer l of the full-size model on S rows of input x, stage by stage through the module entry points, next to
    the oracle's stages.  Wherever the two sides may legitimately part - a rounding to int8 / uint8 behind a row
    reduction whose order differs (the two RMSNorms, the softmax) - the differing bytes are counted, required to be
    single steps, and the DEVICE's bytes are fed to the oracle's next stage; behind identical quantised inputs every
    stage must then agree exactly (integer stages, dequantisation, RoPE, static quantisation, Hadamard) or to the
    device's exponential (SiLU, 2e-6).  The two roundings that sit behind a per-row scale which may differ in its last
    bit (static quantisation of q/k/v, the Hadamard quantiser behind SiLU) are also run on the oracle's own inputs and
    the bytes that move are counted.  Returns the chain's output, its caches, and per token the flips that can reach
    it."""
    ops = fx.ops
    S, H, I = x.shape[0], cfg["hidden"], cfg["inter"]
    qh, kvh, hd = cfg["q_heads"], cfg["kv_heads"], cfg["head_dim"]
    KV = kvh * hd
    g0, g1 = host_w["gamma"][2 * l], host_w["gamma"][2 * l + 1]
    dg0 = dev_w["gamma"].view(2 * l * H * 4, (H,)); dg1 = dev_w["gamma"].view((2 * l + 1) * H * 4, (H,))
    sc_host = [host_w[n][l] for n in ("q_s", "k_s", "v_s", "a_s")]
    scales = ops.Scales(*sc_host)
    wqkv = np.concatenate([host_w["wq"][l], host_w["wk"][l], host_w["wv"][l]])
    sqkv = np.concatenate([host_w["sq"][l], host_w["sk"][l], host_w["sv"][l]])
    wgu = np.empty((2 * I, H), np.int8); wgu[0::2] = host_w["wg"][l]; wgu[1::2] = host_w["wu"][l]
    sgu = np.empty(2 * I, np.float32); sgu[0::2] = host_w["sg"][l]; sgu[1::2] = host_w["su"][l]
    sin_t, cos_t = host_w["rope_sin"][:S], host_w["rope_cos"][:S]
    flips = {}

    def rounded_stage(name, dev_q, dev_s, ref_q, ref_s):
        d = np.abs(dev_q.astype(np.int32) - ref_q.astype(np.int32))
        assert d.max() <= 1, "%s: a byte differs by more than one step" % name
        np.testing.assert_allclose(dev_s, ref_s, rtol=1e-6)
        flips[name] = (d != 0).sum(axis=1)

    xd = fx.to_device(x)
    # 1. RMSNorm + per-token quantisation (row sum order differs)
    xq_d, xs_d = ops.rmsnorm_quant_i8(xd, dg0, eps=cfg["eps"])
    xq, xs = xq_d.numpy(), xs_d.numpy()
    xq_o, xs_o = oracle.quant_sym(oracle.rmsnorm_pref(x, g0, cfg["eps"]))
    rounded_stage("norm1", xq, xs, xq_o, xs_o)
    # 2. q/k/v projection, RoPE, static quantisation, cache stores: exact behind identical bytes
    kc, vc = ops.kv_cache(kvh, S)
    q8_d = ops.linear_i8_gemm_qkv_rope_cache(xq_d, xs_d, fx.to_device(wqkv), fx.to_device(sqkv), fx.to_device(sin_t),
                                             fx.to_device(cos_t), scales, kc, vc, qh)
    y = oracle.dequant(oracle.linear_i8(xq, wqkv), xs, sqkv)
    q = oracle.rope(y[:, :H].reshape(S, qh, hd), sin_t, cos_t)
    k = oracle.rope(y[:, H:H + KV].reshape(S, kvh, hd), sin_t, cos_t)
    v = np.ascontiguousarray(y[:, H + KV:]).reshape(S, kvh, hd)
    q8 = oracle.static_quant(q, sc_host[0], factor=float(np.sqrt(np.float32(hd))))
    k8 = oracle.static_quant(k, sc_host[1]); v8 = oracle.static_quant(v, sc_host[2])
    assert np.array_equal(q8_d.numpy(), q8)
    k_tm = kc.numpy().transpose(1, 0, 2)                                           # [pos][kv_head][64]
    v_tm = vc.numpy().transpose(1, 3, 0, 2).reshape(S, kvh, hd)                    # [block][pos in block][kv_head][ch]
    assert np.array_equal(k_tm, k8) and np.array_equal(v_tm, v8)
    # what the oracle gets from ITS OWN norm output (bytes and a scale that may differ in the last bit): the static
    # quantisation behind it can move a byte by one step; counted per token, queries apart from keys / values
    y_f = oracle.dequant(oracle.linear_i8(xq_o, wqkv), xs_o, sqkv)
    q8_f = oracle.static_quant(oracle.rope(y_f[:, :H].reshape(S, qh, hd), sin_t, cos_t), sc_host[0], factor=float(np.sqrt(np.float32(hd))))
    k8_f = oracle.static_quant(oracle.rope(y_f[:, H:H + KV].reshape(S, kvh, hd), sin_t, cos_t), sc_host[1])
    v8_f = oracle.static_quant(np.ascontiguousarray(y_f[:, H + KV:]).reshape(S, kvh, hd), sc_host[2])
    del y_f
    clean = flips["norm1"] == 0                                                    # rows whose int8 input is the same on both sides
    for name, a, b in (("q8", q8, q8_f), ("kv8", np.concatenate([k8, v8], 1), np.concatenate([k8_f, v8_f], 1))):
        d = np.abs(a.astype(np.int32) - b.astype(np.int32)).reshape(S, -1)
        assert d[clean].max() <= 1, "%s: a byte differs by more than one step behind identical int8 input" % name
        flips[name] = (d != 0).sum(axis=1)
    # 3. attention: the probability bytes sit behind the softmax sum; P.V on the device's bytes must be exact
    o_d, p_d = ops.mha_i8_prefill(q8_d, kc, vc, scales, want_p=True)
    p_dev = p_d.numpy(); del p_d
    _, p_ref = oracle.mha_prefill_i8(q8, k8, v8, *sc_host, want_p=True)
    dp = np.abs(p_dev.astype(np.int16) - p_ref.astype(np.int16))
    assert dp.max() <= 1, "a probability byte differs by more than one step"
    flips["softmax"] = (dp != 0).sum(axis=(0, 2))
    del dp, p_ref
    o_sub = oracle.mha_prefill_i8(q8, k8, v8, *sc_host, p8_in=p_dev)
    del p_dev
    att = o_d.numpy()
    assert np.array_equal(att, o_sub), "P.V or its dequantisation differs behind identical probability bytes"
    # 4. quantisation of the attention output, o projection + residual: exact
    aq_d, as_d = ops.quant_sym_i8(o_d.view(0, (S, H), np.float32))
    aq_o, as_o = oracle.quant_sym(att.reshape(S, H))
    assert np.array_equal(aq_d.numpy(), aq_o) and np.array_equal(as_d.numpy(), as_o)
    x2_d = ops.linear_i8_gemm_dequant(aq_d, as_d, dev_w["wo"][l], dev_w["so"][l], residual=xd)
    x2 = x2_d.numpy()
    assert np.array_equal(x2, oracle.residual(oracle.dequant(oracle.linear_i8(aq_o, host_w["wo"][l]), as_o, host_w["so"][l]), x))
    # 5. second RMSNorm + quantisation
    nq_d, ns_d = ops.rmsnorm_quant_i8(x2_d, dg1, eps=cfg["eps"])
    nq, ns = nq_d.numpy(), ns_d.numpy()
    nq_o, ns_o = oracle.quant_sym(oracle.rmsnorm_pref(x2, g1, cfg["eps"]))
    rounded_stage("norm2", nq, ns, nq_o, ns_o)
    # 6. gate/up with SiLU(gate)*up in the epilogue (256x256 tiles at 1024 rows): the device's exponential
    h_d = ops.linear_i8_gemm_swiglu(nq_d, ns_d, fx.to_device(wgu), fx.to_device(sgu))
    h = h_d.numpy()
    gu = oracle.dequant(oracle.linear_i8(nq, wgu), ns, sgu)
    np.testing.assert_allclose(h, oracle.gate(gu[:, 1::2], oracle.swish(gu[:, 0::2])), rtol=2e-6, atol=1e-30)
    # the oracle's own h (from its norm bytes and scale, its exponential) through the Hadamard quantiser: single steps
    gu = oracle.dequant(oracle.linear_i8(nq_o, wgu), ns_o, sgu)
    hq_f, _ = oracle.quant_sym(oracle.fht(oracle.gate(gu[:, 1::2], oracle.swish(gu[:, 0::2])), cfg["fht_scale"]))
    del gu
    # 7. Hadamard + quantisation, down projection + residual: exact behind the device's h
    hq_d, hs_d = ops.fht_quant_i8(h_d, scale=cfg["fht_scale"])
    hq_o, hs_o = oracle.quant_sym(oracle.fht(h, cfg["fht_scale"]))
    assert np.array_equal(hq_d.numpy(), hq_o) and np.array_equal(hs_d.numpy(), hs_o)
    d = np.abs(hq_o.astype(np.int32) - hq_f.astype(np.int32))
    assert d[flips["norm2"] == 0].max() <= 1
    flips["hadamard"] = (d != 0).sum(axis=1)
    x3 = ops.linear_i8_gemm_dequant(hq_d, hs_d, dev_w["wd"][l], dev_w["sd"][l], residual=x2_d).numpy()
    assert np.array_equal(x3, oracle.residual(oracle.dequant(oracle.linear_i8(hq_o, host_w["wd"][l]), hs_o, host_w["sd"][l]), x2))
    # a moved byte of token j's norm output or of its K / V row reaches every later token through attention; moved
    # query, probability, second-norm and Hadamard bytes stay in their own row
    first = np.nonzero((flips["norm1"] > 0) | (flips["kv8"] > 0))[0]
    reach = np.zeros(S, bool)
    if first.size:
        reach[first[0]:] = True
    reach |= (flips["q8"] > 0) | (flips["softmax"] > 0) | (flips["norm2"] > 0) | (flips["hadamard"] > 0)
    return x3, k_tm.reshape(S, KV), v_tm.reshape(S, KV), flips, reach


def test_prefill_1024_tokens_layers_0_and_15_with_causal_tie_attribution(full):
    """Layers 0 and 15 of the full-size model as one-layer views on 1024 rows (layer 15 on the hidden state the
    device's first 15 layers produce, fed to both sides).  (a) The fused prefill graph against the oracle's layer:
    the typical token to fp32 rounding, none beyond the effect of single steps.  (b) The same layer as a chain of module entry points equals the
    fused graph bit for bit (output and caches).  (c) That chain against the oracle stage by stage with the device's
    bytes substituted behind every rounding whose reduction order differs (_stage_chain_with_substitution): all other
    stages exact.  (d) Cause and effect: every token whose fused output differs from the oracle's beyond fp32
    rounding is a token that a counted single-step flip can reach."""
    fx, llama, oracle, cfg, dev_w, host_w = full
    L, H, S = cfg["layers"], cfg["hidden"], 1024
    r = np.random.default_rng(43)
    x0 = r.standard_normal((S, H)).astype(np.float32)
    cfg15 = llama.make_config(layers=L - 1, vocab=256)
    w15 = dict(dev_w); w15["embed"] = dev_w["embed"].view(0, (256, H))
    m15 = llama.Llama(cfg15, w15)
    x15 = m15.prefill_hidden(fx.to_device(x0)).numpy()
    m15.close()
    assert np.isfinite(x15).all()
    cfg1 = llama.make_config(layers=1, vocab=256, max_pos=S)
    for l, x in ((0, x0), (L - 1, x15)):
        print("layer", l, flush=True)
        hw = layer_views(cfg, host_w, l, 256, device=False)
        hw["rope_sin"], hw["rope_cos"] = host_w["rope_sin"][:S], host_w["rope_cos"][:S]
        dw = layer_views(cfg, dev_w, l, 256, device=True)
        dw["rope_sin"] = dev_w["rope_sin"].view(0, (S, 32)); dw["rope_cos"] = dev_w["rope_cos"].view(0, (S, 32))
        om1 = oracle.OracleModel(cfg1, hw)
        k1, v1 = om1.new_caches()
        y_ref = om1.prefill(x, k1, v1)
        m1 = llama.Llama(cfg1, dw)
        y = m1.prefill_hidden(fx.to_device(x)).numpy()
        kg, vg = m1.caches_token_major()
        m1.close()
        e = token_err(y, y_ref)
        dk = np.abs(kg[0].astype(int) - k1[0]); dv = np.abs(vg[0].astype(int) - v1[0])
        assert dk.max() <= 1 and dv.max() <= 1
        beyond = e > 2e-5
        print("  (a) tokens beyond fp32 rounding: %d of %d, median %.1e, worst %.1e, cache bytes off by one: %d"
              % (beyond.sum(), S, np.median(e), e.max(), int((dk != 0).sum() + (dv != 0).sum())), flush=True)
        # (no bound on the count here: at 1024 rows one moved K / V byte of an early token reaches every later row through
        # attention, so the count depends on where the first such byte falls; (d) accounts for every one of them)
        assert np.median(e) <= 2e-5 and e.max() <= 2e-2
        y_chain, k_chain, v_chain, flips, reach = _stage_chain_with_substitution(fx, oracle, cfg, host_w, dev_w, l, x)
        print("  (c) single-step flips, bytes / tokens: " + ", ".join("%s %d / %d" % (n, int(flips[n].sum()), int((flips[n] > 0).sum()))
                                                                      for n in ("norm1", "q8", "kv8", "softmax", "norm2", "hadamard")), flush=True)
        assert np.array_equal(y_chain, y), "(b) the fused graph and the chain of module entry points differ"
        assert np.array_equal(k_chain, kg[0]) and np.array_equal(v_chain, vg[0])
        stray = np.nonzero(beyond & ~reach)[0]
        assert stray.size == 0, "(d) tokens %s differ from the oracle with no counted flip that reaches them" % stray[:8]
        # the flips are rare: a row has 2048 (norms) and 32 x (row + 1) (softmax) roundings
        assert flips["norm1"].sum() + flips["norm2"].sum() <= 1e-4 * 2 * S * H and flips["softmax"].sum() <= 1e-4 * 32 * S * S / 2


def test_prefill_1024_tokens_16_layers_prefix_invariance(full):
    """All 16 layers: the first 512 rows of a 1024-token prefill (256x256 gate/up tiles, eight-wave attention) equal a
    512-token prefill (other tile choices) bit for bit, residual stream and caches; nothing is written past the
    sequence."""
    fx, llama, oracle, cfg, dev_w, host_w = full
    from flexllm_amd import synth
    H, S = cfg["hidden"], 1024
    m = llama.Llama(cfg, dev_w)
    x = synth.device_uniform_f32((S, H), 4300, -1.7, 1.7)
    hid_half = m.prefill_hidden(x.view(0, (S // 2, H), np.float32)).numpy()
    k_half, v_half = m.caches_token_major()
    m.k_cache.zero_(); m.v_cache.zero_()
    hid = m.prefill_hidden(x).numpy()
    k, v = m.caches_token_major()
    m.close()
    assert np.isfinite(hid).all()
    assert np.array_equal(hid[:S // 2], hid_half)
    assert np.array_equal(k[:, :S // 2], k_half[:, :S // 2]) and np.array_equal(v[:, :S // 2], v_half[:, :S // 2])
    assert not k_half[:, S // 2:].any() and not v_half[:, S // 2:].any() and not k[:, S:].any() and not v[:, S:].any()
    assert k[:, S // 2:S].any() and v[:, S // 2:S].any()


def test_generate_from_a_1025_token_prompt_equals_prefill_plus_stepwise_decode(full):
    """flexllm_llama_generate on the full-size model: a 1025-token prompt (1024 prefilled rows), 32 greedy tokens in
    one call, against the same flow done by hand on a second model - embedding rows, prefill_hidden of 1024 rows, then
    one decode launch per token.  Ids and every cache byte identical."""
    fx, llama, oracle, cfg, dev_w, host_w = full
    H, n_p, steps = cfg["hidden"], 1025, 32
    r = np.random.default_rng(44)
    prompt = r.integers(0, cfg["vocab"], n_p).astype(np.int32)
    a, b = llama.Llama(cfg, dev_w), llama.Llama(cfg, dev_w)
    stale = fx.to_device(r.integers(-128, 128, a.k_cache.shape).astype(np.int8))     # stale contents must not matter
    for m in (a, b):
        fx.check(fx.lib().flexllm_rt_memcpy_d2d(C.c_void_p(m.k_cache.ptr), C.c_void_p(stale.ptr), C.c_size_t(stale.nbytes), None))
        m.v_cache.zero_()
    got = a.generate(prompt, steps)
    emb = np.stack([host_w["embed"][int(t)].view(np.float16).astype(np.float32) for t in prompt[:-1]])
    b.prefill_hidden(fx.to_device(emb))
    tok = fx.to_device(prompt[-1:].copy()); out = fx.zeros((1,), np.int32)
    ids = []
    for i in range(steps):
        b.decode_greedy(tok, n_p - 1 + i, 1, out, use_graph=0)
        ids.append(int(out.numpy()[0]))
    b.check()
    assert got == ids
    assert len(set(ids)) > 4, ids
    n = n_p - 1 + steps
    ka, va = a.caches_token_major(); kb, vb = b.caches_token_major()
    assert np.array_equal(ka[:, :n], kb[:, :n]) and np.array_equal(va[:, :n], vb[:, :n])
    a.close(); b.close()
