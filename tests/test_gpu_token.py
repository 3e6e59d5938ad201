"""The token kernel (all layers of a decode step in one launch) against the layers' own launches: the same bits."""
import ctypes
import os
import sys
import threading
import time

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llama2.rs_amd"))
from llama2_rs import _lib, ops  # noqa: E402
from llama2_rs.checkpoint import Dims  # noqa: E402

pytestmark = pytest.mark.gpu


def model(dim, hid, heads, kv, group, layers=2, seed=3, max_seq=1100):
    d = Dims(dim=dim, hidden_dim=hid, n_layers=layers, n_heads=heads, n_kv_heads=kv, vocab_size=700, seq_len=64, group_size=group)
    return ops.Model(ops.synth_image(d, seed), d, max_seq=max_seq)


def token_kernel(m, on, missing=0, looks=1 << 17):
    _lib.check(_lib.lib().l2_model_set_token_kernel(m.h, on, missing, looks))


def state_of(m):
    on, gave_up = ctypes.c_int(), ctypes.c_int()
    _lib.check(_lib.lib().l2_model_token_kernel(m.h, ctypes.byref(on), ctypes.byref(gave_up)))
    return on.value, gave_up.value


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


# inputs of one to four waves per row and a part of one, hidden rows of one to fourteen, both associations of the chunk sums, rows behind
# the launches' loops, 1 to 8 query heads per kv head, slices of 16 and of 32 outputs
SHAPES = [(512, 768, 4, 2, 32), (1024, 2816, 8, 2, 64), (1152, 32, 9, 9, 32), (1536, 4480, 12, 12, 128), (2048, 13824, 16, 4, 128),
          (3072, 8192, 24, 3, 64), (4096, 11008, 32, 32, 128), (5120, 5120, 40, 40, 64), (8192, 1024, 64, 8, 32), (2048, 28672, 16, 16, 64)]


@pytest.mark.parametrize("shape", SHAPES)
def test_logits_and_cache_rows_are_those_of_the_launches(shape):
    m = model(*shape)
    rng = np.random.default_rng(7)
    for start, n in ((0, 4), (62, 4), (127, 3), (255, 3), (509, 3), (638, 3), (766, 3), (1023, 2)):
        tokens = rng.integers(0, 700, n)
        got = {}
        for on in (1, 0):
            token_kernel(m, on)
            m.reset()
            if start:
                m.fill_kv_synthetic(0, start, seed=start)
            logits = [m.forward([int(t)], [start + i]).copy() for i, t in enumerate(tokens)]
            got[on] = (logits, [m.read_kv(l, start, n) for l in range(2)])
        assert state_of(m)[1] == 0
        for a, b in zip(got[1][0], got[0][0]):
            assert np.isfinite(b).all() and np.array_equal(bits(a), bits(b)), (shape, start)
        for (ka, va), (kb, vb) in zip(got[1][1], got[0][1]):
            assert np.array_equal(bits(ka), bits(kb)) and np.array_equal(bits(va), bits(vb)), (shape, start)
    m.close()


def test_a_loop_of_steps_and_a_value_that_looks_absent():
    """Greedy tokens over the loop, one call per token, and a step whose residual stream is the NaN that means "absent"."""
    m = model(1024, 2816, 8, 2, 64)
    prompt = np.array([5, 17, 99], np.int32)
    ids = {}
    for on in (1, 0):
        token_kernel(m, on)
        ids[on] = m.generate_greedy(prompt, 120)[0]
        m.reset()
        t, one = 5, []
        for p in range(20):
            t = m.decode_greedy(t, p)
            one.append(t)
        ids[on] = np.concatenate([ids[on], one])
    assert np.array_equal(ids[1], ids[0])
    m.close()
    d = Dims(dim=512, hidden_dim=768, n_layers=2, n_heads=4, n_kv_heads=2, vocab_size=260, seq_len=64, group_size=32)
    img = ops.synth_image(d, 1)
    img[4:].view(np.uint32)[:512] = 0xFFFFFFFF  # the first token's embedding
    m = ops.Model(img, d)
    assert np.isnan(m.forward([0], [0])).all() and state_of(m) == (1, 0)
    m.reset()
    a = m.forward([3], [0]).copy()
    token_kernel(m, 0)
    m.reset()
    assert np.array_equal(bits(a), bits(m.forward([3], [0])))
    m.close()


def test_waits_that_are_given_up():
    """A block is left out, so that the others wait in vain: they leave after 64 looks, and the call does its steps again."""
    m = model(1024, 2816, 8, 2, 64)
    prompt = np.array([5, 17, 99], np.int32)
    token_kernel(m, 0)
    want = m.generate_greedy(prompt, 24)[0]
    m.reset()
    logits = m.forward([9], [0]).copy()
    token_kernel(m, 1, missing=1, looks=64)
    assert np.array_equal(m.generate_greedy(prompt, 24)[0], want) and state_of(m) == (1, 1)
    m.reset()
    assert np.array_equal(bits(m.forward([9], [0])), bits(logits)) and state_of(m) == (1, 2)
    token_kernel(m, 1)  # and with all blocks the kernel is right again
    assert np.array_equal(m.generate_greedy(prompt, 24)[0], want) and state_of(m) == (1, 0)
    token_kernel(m, 1, missing=1, looks=64)
    for i in range(4):  # not asked any more after three calls
        assert np.array_equal(m.generate_greedy(prompt, 8)[0], want[:6]) and state_of(m) == (int(i < 2), min(i + 1, 3))
    m.close()


def test_models_on_threads():
    """Two models decode side by side: one of them at a time has token kernels in flight, and both get their own results."""
    ms = [model(1024, 2816, 8, 2, 64, seed=s) for s in (3, 4)]
    prompt = np.array([5, 17, 99], np.int32)
    want = [m.generate_greedy(prompt, 60)[0] for m in ms]
    bad = []

    def run(i):
        for _ in range(15):
            if not np.array_equal(ms[i].generate_greedy(prompt, 60)[0], want[i]):
                bad.append(i)
    threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad and [state_of(m) for m in ms] == [(1, 0), (1, 0)]
    for m in ms:
        m.close()


# ---- the route that steps take


def takes(shape, timesteps):
    """Whether a step over so many timesteps goes through the token kernel: where attention takes a context whole, but not on the matrix cores."""
    _, _, heads, kv, _ = shape
    if heads == 8 * kv and timesteps <= 256:
        return False
    return timesteps <= ((512 if kv > 32 else 640) if heads <= 2 * kv else 896 if heads < 32 else 1024 if kv <= 4 else 768)


@pytest.mark.parametrize("shape", SHAPES)
def test_the_steps_that_are_compared_take_the_kernel(shape):
    """Steps at the starts of the comparison above, and a loop of them: in one launch where attention takes the context whole, none with the kernel off."""
    m = model(*shape)
    for on in (1, 0):
        token_kernel(m, on)
        for start, n in ((0, 4), (62, 4), (127, 3), (255, 3), (509, 3), (638, 3), (766, 3), (1023, 2)):
            m.reset()
            if start:
                m.fill_kv_synthetic(0, start, seed=start)
            before = m.token_steps()
            for i in range(n):
                m.forward([5 + i], [start + i])
            assert m.token_steps() - before == on * sum(takes(shape, start + i + 1) for i in range(n)), start
        before = m.token_steps()
        m.generate_greedy(np.array([5, 17, 99], np.int32), 120)
        assert m.token_steps() - before == on * sum(takes(shape, p + 1) for p in range(2, 120))  # two positions are the ladder's
    m.close()


def test_loops_ask_about_the_stream_by_the_launches_that_they_make():
    """A step is two launches or 17: 64 or 7 of them between two asks, also behind contexts that the token kernel does not take."""
    def asked(m):
        n = ctypes.c_uint64()
        _lib.check(_lib.lib().l2_model_asked(m.h, ctypes.byref(n)))
        return n.value
    m = model(1024, 2816, 8, 2, 64, layers=3, max_seq=1400)
    m.fill_kv_synthetic(0, 1000, seed=1)
    for on, pos, want, in_one in ((1, 40, 1, 160), (0, 40, 21, 0), (1, 1000, 21, 0), (1, 816, 11, 80)):  # attention takes up to 896 whole
        token_kernel(m, on)
        before, steps = asked(m), m.token_steps()
        m.decode_bench(5, pos, 160)
        assert (asked(m) - before, m.token_steps() - steps) == (want, in_one), pos
    m.close()


def test_a_call_that_comes_through_ends_the_row_of_those_that_did_not():
    m = model(1024, 2816, 8, 2, 64)
    want = m.forward([9], [0]).copy()
    for gave_up in (0, 2, 4):
        for missing, calls in ((1, 2), (0, 1)):
            _lib.check(_lib.lib().l2_model_token_trouble(m.h, missing, 64 if missing else 1 << 17, 0))
            for _ in range(calls):
                steps = m.token_steps()
                m.reset()
                assert np.array_equal(bits(m.forward([9], [0])), bits(want)) and m.token_steps() == steps + 1
        assert state_of(m) == (1, gave_up + 2)
    m.close()


def test_an_error_leaves_nothing_behind():
    """Behind a step that failed: another model gets the device, and the calls that follow, of either, give what they always give."""
    a, b = (model(1024, 2816, 8, 2, 64, seed=s) for s in (3, 4))
    prompt = np.array([5, 17, 99], np.int32)
    want = [m.generate_greedy(prompt, 24)[0] for m in (a, b)]
    calls = [lambda: a.forward([9], [0]), lambda: a.generate_greedy(prompt, 24), lambda: a.decode_greedy(9, 0), lambda: a.decode_bench(9, 0, 12)]
    for i, call in enumerate(calls):
        for missing in (0, 1):  # 1: the step before the one that fails has given up a wait meanwhile
            _lib.check(_lib.lib().l2_model_token_trouble(a.h, missing, 64, 1 if i in (0, 2) else 2))
            with pytest.raises(_lib.L2Error):
                call()
            _lib.check(_lib.lib().l2_model_token_trouble(a.h, 0, 1 << 17, 0))
            for m, ids in ((b, want[1]), (a, want[0])):
                steps = m.token_steps()
                m.reset()
                assert np.array_equal(m.generate_greedy(prompt, 24)[0], ids) and m.token_steps() > steps, (i, missing)
    assert state_of(a)[0] == 1 and state_of(b) == (1, 0)
    for m in (a, b):
        m.close()


def test_steps_beside_other_calls_go_layer_by_layer():
    """While another call is at work on the device, and for a while behind, a model's steps go out as launches that the other's come between; a
    loop that has the device to itself when it starts has only some ms of steps in token kernels ahead when another call comes."""
    a, b = model(1024, 2816, 8, 2, 64, layers=3, seed=3), model(1024, 2816, 8, 2, 64, layers=3, seed=4)
    q = ops.QLinear(*[np.zeros(s, t) for s, t in (((256, 128), np.int32), ((32, 16), np.int32), ((256, 16), np.float32))], np.arange(1024), 64)
    prompt, tokens, x = np.array([5, 17, 99], np.int32), np.arange(64, dtype=np.int32), np.zeros(1024, np.float32)
    want = a.generate_greedy(prompt, 800)[0]

    def steps_of(f):
        n = a.token_steps()
        f()
        return a.token_steps() - n

    def beside(other, f, delay=0.0):
        """f() while another thread calls other() again and again, from `delay` seconds behind its start on."""
        stop, started = threading.Event(), threading.Event()

        def run():
            started.set()
            stop.wait(delay)
            while not stop.is_set():
                other()
        t = threading.Thread(target=run)
        t.start()
        started.wait()
        try:
            return f()
        finally:
            stop.set()
            t.join()

    def check(steps):
        assert np.array_equal(a.generate_greedy(prompt, steps)[0], want[:steps - 2])
    assert steps_of(lambda: check(60)) == 58
    for other in (lambda: b.prefill_chunks(tokens, 0, 64), lambda: b.generate_greedy(prompt, 40), lambda: b.decode_greedy(3, 5), lambda: q.matvec(x)):
        def f():
            check(60)  # the first of these may find the device free
            return steps_of(lambda: [check(60) for _ in range(8)])
        assert beside(other, f) < 58, "of 464"
        time.sleep(0.05)
        assert steps_of(lambda: check(60)) == 58
    assert 20 < beside(lambda: b.prefill_chunks(tokens, 0, 64), lambda: steps_of(lambda: check(800)), delay=0.01) < 600
    q.close()
    a.close()
    b.close()


def test_models_on_threads_take_both_routes():
    """Two models decode on threads, side by side and one at a time as it comes, through the token kernel and as launches: both get their own results."""
    ms = [model(1024, 2816, 8, 2, 64, seed=s) for s in (3, 4)]
    prompt = np.array([5, 17, 99], np.int32)
    want = []
    for m in ms:
        token_kernel(m, 0)
        want.append(m.generate_greedy(prompt, 60)[0])
        token_kernel(m, 1)
    assert [m.token_steps() for m in ms] == [0, 0]
    bad = []

    def run(i, pauses):
        for pause in pauses:
            if not np.array_equal(ms[i].generate_greedy(prompt, 60)[0], want[i]):
                bad.append(i)
            time.sleep(pause)
    rng = np.random.default_rng(0)
    threads = [threading.Thread(target=run, args=(i, [0.0] * 15 + list(rng.uniform(0, 0.03, 25)))) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad and [state_of(m) for m in ms] == [(1, 0), (1, 0)]
    assert all(0 < m.token_steps() < 40 * 58 for m in ms), [m.token_steps() for m in ms]
    for m in ms:
        m.close()
