"""A call that returns results has waited for its work as a whole: nothing of it is left for the next call to wait for."""
import time

import numpy as np
import pytest

from llama2_rs import checkpoint as ck

pytestmark = pytest.mark.gpu


# The reset of a state behind a pass against one behind a call that synchronises in between.  The shortest of 60 each, as
# whatever else the machine does only adds to a time; they differ by some 10 % where nothing is left over and by 2.5 times
# where a pass returns as soon as its results are there.
@pytest.mark.parametrize("call", ["generate", "decode", "prefill", "forward"])
def test_nothing_left_behind_a_pass(call):
    from llama2_rs import ops, _lib
    assert _lib.lib().l2_device_count() >= 1, "no HIP device: the GPU tests cannot run"
    dims = ck.Dims(dim=1024, hidden_dim=2816, n_layers=3, n_heads=8, n_kv_heads=2, vocab_size=2000, seq_len=512, group_size=32)
    m = ops.Model(ops.synth_image(dims, 1), dims)
    prompt = np.arange(33, dtype=np.int32)
    calls = {"generate": lambda: m.generate_greedy(prompt, 40), "decode": lambda: [m.decode_greedy(1, p) for p in range(8)],
             "prefill": lambda: m.prefill_chunks(prompt, 0, 16), "forward": lambda: [m.forward([1], [p]) for p in range(8)]}
    best = {False: 1.0, True: 1.0}
    for _ in range(60):
        for synchronise in best:
            calls[call]()
            if synchronise:
                m.read_kv(0, 0, 1)
            t = time.perf_counter()
            m.reset()
            best[synchronise] = min(best[synchronise], time.perf_counter() - t)
    assert best[False] < 1.7 * best[True], best
    m.close()
