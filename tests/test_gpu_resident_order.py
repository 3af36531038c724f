"""Kernels that need the whole chip, launched from several streams, threads and models: they run one after the other and each
gives what it gives alone."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

import lopazen_cases as lc
from test_gpu_decode_float import LOPAZEN

pytestmark = pytest.mark.gpu
CFG = LOPAZEN["rows of a quad"]


def hip():
    lib = C.CDLL("libamdhip64.so")

    def call(name, *args):
        rc = getattr(lib, name)(*args)
        assert rc == 0, "%s: %d" % (name, rc)
    return call


class CallersStream:
    """A stream that the library has not made."""

    def __init__(self):
        self.handle = C.c_void_p()
        hip()("hipStreamCreate", C.byref(self.handle))

    def destroy(self):
        hip()("hipStreamDestroy", self.handle)


def lopazen(**kw):
    from flexllm_amd.lopazen import Lopazen
    return Lopazen.from_tensors(CFG, lc.weights(CFG, 5), dtype="bfloat16", max_pos=512, **kw)


class Request:
    """A prompt in a slot of a model of its own, and a greedy loop behind it that is not waited for."""

    def __init__(self, seed, steps):
        from flexllm_amd import to_device, zeros
        self.model = lopazen()
        self.prompt, self.steps = lc.tokens(CFG, 9 + seed), steps
        self.want = self.model.generate(self.prompt, steps)
        self.slot = self.model.pool.acquire("r")
        self.model.step(self.slot, self.prompt[:-1])
        self.token, self.out = to_device(np.array(self.prompt[-1:], np.int32)), zeros((steps,), np.int32)

    def start(self, stream=None):
        self.model.decode(self.slot, self.token, self.steps, self.out, stream=stream)

    def finish(self):
        self.model.check()
        assert self.out.numpy().tolist() == self.want
        self.model.close()


def test_a_capture_begins_behind_a_launch():
    """The stream of the last launch is being captured when the next one, on another stream, has to wait for it: the capture stays
    empty, the launch runs."""
    a, b = Request(1, 300), Request(2, 40)
    call, graph, nodes = hip(), C.c_void_p(), C.c_size_t(99)
    a.start()
    call("hipStreamBeginCapture", a.model.stream().handle, 2)           # relaxed
    b.start()
    call("hipStreamEndCapture", a.model.stream().handle, C.byref(graph))
    call("hipGraphGetNodes", graph, None, C.byref(nodes))
    call("hipGraphDestroy", graph)
    assert nodes.value == 0
    b.finish()
    a.finish()


def test_callers_streams():
    """Streams that the library has not made, one of them gone when the next launch comes, on a stream that may have its handle."""
    a, b, c = Request(1, 200), Request(2, 100), Request(3, 70)
    s = CallersStream()
    a.start(s)
    s.destroy()
    t = CallersStream()
    b.start(t)
    c.start()
    for r in a, b, c:
        r.finish()
    t.destroy()


def test_a_stream_with_half_of_the_chip():
    """The workgroups that have to be there all at once do not fit: its tokens come from the chain of kernels."""
    from flexllm_amd import to_device, zeros
    half, all_of_it = [CallersStream(), CallersStream()]
    for s, word in (half, 0), (all_of_it, 0xFFFFFFFF):
        s.destroy()
        hip()("hipExtStreamCreateWithCUMask", C.byref(s.handle), 8, (C.c_uint32 * 8)(*[0xFFFFFFFF] * 4 + [word] * 4))
    m = lopazen()
    prompt, token, out, got = lc.tokens(CFG, 20), to_device(np.array([0], np.int32)), zeros((30,), np.int32), []
    for mode, s in (1, None), (0, half), (0, all_of_it):
        m.set_decode_mode(mode)
        slot = m.pool.acquire("r")
        m.step(slot, prompt[:-1])
        token.copy_from(np.array(prompt[-1:], np.int32))
        if s is half:
            m.set_wait_limit(1)                            # the resident kernel would give up
        m.decode(slot, token, 30, out, stream=s)
        m.check()
        m.set_wait_limit(0)
        got.append(out.numpy().tolist())
        m.pool.release("r")
    assert got[0] == got[1] and got[0][:3] == got[2][:3]
    m.close()
    half.destroy()
    all_of_it.destroy()


def test_prompts_beside_decoding():
    """Loops of tokens and the prompts of another stream take turns: the prompts do not wait for a gap between loops kernel by kernel."""
    from flexllm_amd import to_device, zeros
    a, b = lopazen(), lopazen()
    prompt, token, out = to_device(np.array(lc.tokens(CFG, 200), np.int32)), to_device(np.array([3], np.int32)), zeros((16,), np.int32)
    done, stop = [], threading.Event()

    def prompts():
        while not stop.is_set():
            s = b.pool.acquire("p")
            b.step(s, prompt)
            b.pool.release("p")
            done.append(1)

    slot = a.pool.acquire("d")
    a.decode(slot, token, 16, out)
    a.stream().sync()
    t = threading.Thread(target=prompts)
    t.start()
    while not done:
        time.sleep(0.01)
    before = len(done)
    for _ in range(25):                                    # 400 tokens
        a.decode(slot, token, 16, out)
        a.stream().sync()
    served = len(done) - before
    stop.set()
    t.join()
    a.check()
    assert served >= 10, served                            # a prompt per loop; kernel by kernel it is one per five
    a.close()
    b.close()


def test_two_designs_and_ordinary_work():
    """Llama's decode kernel, a decoder's, and prompts of a third model, whose kernels hold a part of the chip now and then."""
    from flexllm_amd import llama
    lcfg = llama.make_config(layers=2, vocab=2048, max_pos=256)
    lm = llama.Llama(lcfg, llama.synth_weights(lcfg, seed=5, device=True))
    models, prompt = [lopazen() for _ in range(2)], lc.tokens(CFG, 300)
    lprompt = [5, 77, 1023, 9]

    def prompts():
        m, out = models[1], []
        for _ in range(12):
            s = m.pool.acquire("p")
            out.append(m.step(s, prompt, [len(prompt) - 1])[0])
            m.pool.release("p")
        return out

    from flexllm_amd.device import Stream
    ls = Stream()
    work = {"llama": lambda: [lm.generate(lprompt, 60, stream=ls) for _ in range(8)],
            "tokens": lambda: [models[0].generate(prompt[:20], 70) for _ in range(8)],
            "prompts": prompts}
    want, got = {n: f() for n, f in work.items()}, {}

    def run(name):
        got[name] = work[name]()

    threads = [threading.Thread(target=run, args=(n,)) for n in work]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert got["llama"] == want["llama"] and got["tokens"] == want["tokens"]
    assert all(np.array_equal(g, w) for g, w in zip(got["prompts"], want["prompts"]))
    [m.close() for m in models + [lm]]
