"""fp32 weights in batches (reference: src/model.rs:22-31): K cut into equal slices and a shorter one where whole rounds of blocks leave
compute units idle."""
import ctypes

import numpy as np
import pytest

from llama2_rs import _lib
from llama2_rs import checkpoint as ck


def cut(n_in, out, batch):
    outs, plan = (ctypes.c_int32 * len(out))(*out), (ctypes.c_int32 * 8)()
    _lib.check(_lib.lib().l2_gemm_plan(n_in, outs, len(out), 0, batch, _lib.PREFILL_FP32, plan))
    return plan[2], plan[6], plan[3]  # slices, K steps of the shorter one, blocks


# w1|w3 and q|k|v of 7B's widths, both of up to 128 columns and of more; what fills the units evenly keeps equal slices
@pytest.mark.parametrize("out,batch,want", [((11008, 11008), 100, (2, 14)), ((4096, 4096, 4096), 100, (3, 11)), ((4096, 4096, 4096), 200, (2, 14)),
                                            ((4096,), 100, (8, 0)), ((32768,), 100, (1, 0))])
def test_cut(out, batch, want):
    assert cut(4096, out, batch)[:2] == want


# every cut is of whole K steps, the shorter slice no longer than the others, and a block per row block and slice
def test_cut_over_the_range():
    rng = np.random.default_rng(3)
    for _ in range(300):
        n_in, out, batch = 32 * int(rng.integers(4, 900)), 8 * int(rng.integers(1, 4000)), int(rng.integers(16, 1025))
        slices, last, blocks = cut(n_in, (out,), batch)
        steps, tiles = (n_in + 63) // 64, (out + 127) // 128
        assert 1 <= slices <= 16 and blocks % (tiles * slices) == 0
        if last:
            assert slices > 1 and 2 <= last <= (steps - last) // (slices - 1), (n_in, out, batch, slices, last)


def nrel(a, b):
    return np.abs(a - b).max() / np.sqrt(np.mean(b.astype(np.float64) ** 2))


# a short slice behind one and behind two equal ones; rows that do not fill the last block, one tile of tokens, several and one more;
# then a column with an infinity, which only one slice meets.  The bound is that of sums of K terms in any association for these inputs
@pytest.mark.gpu
@pytest.mark.parametrize("hidden,slices", [(11008, 3), (17888, 2)])
def test_short_slice(hidden, slices):
    from llama2_rs import ops
    import tests.test_oracle_loop as tol
    dims = ck.Dims(dim=2048, hidden_dim=hidden, n_layers=1, n_heads=16, n_kv_heads=1, vocab_size=64, seq_len=32, group_size=0)
    img = ops.synth_image(dims, 6)
    W = tol._split_image(img, dims)["w1"][0].astype(np.float64)
    m, rng = ops.Model(img, dims), np.random.default_rng(hidden)
    for B in (16, 65, 100, 129):
        if B <= 128:
            assert cut(2048, (hidden,), B)[0] == slices and cut(2048, (hidden,), B)[1] > 0
        x = rng.standard_normal((B, 2048)).astype(np.float32)
        if B == 100:
            x[3, -5], x[40, 7] = np.inf, np.nan
        got, fine = m.qmatvec(0, _lib.W1, x), [b for b in range(B) if B != 100 or b not in (3, 40)]
        assert nrel(got[fine], x[fine].astype(np.float64) @ W.T) < 1e-5, B
        if B == 100:
            np.testing.assert_array_equal(got[3], np.sign(W[:, -5]).astype(np.float32) * np.float32(np.inf))
            assert np.all(np.isnan(got[40]))
    m.close()


# chunks one by one and as one pass: the same cut, the same bits
@pytest.mark.gpu
def test_short_slice_by_chunks():
    from llama2_rs import ops
    dims = ck.Dims(dim=2048, hidden_dim=11008, n_layers=1, n_heads=16, n_kv_heads=16, vocab_size=64, seq_len=512, group_size=0)
    img, tokens = ops.synth_image(dims, 7), (np.arange(150) * 7 % 64).astype(np.int32)
    kv = []
    for pieces in ([150], [64, 64, 22]):
        m = ops.Model(img, dims)
        at = 0
        for n in pieces:
            m.prefill_chunks(tokens[at:at + n], at, 64)
            at += n
        kv.append(m.forward([5], [150]))
        m.close()
    np.testing.assert_array_equal(kv[0], kv[1])


# q|k|v in one launch and w1|w3 in one with the gate: each number of loads per lane, with as many rows per wave as it has and with fewer
# (then w1 and w3 are two launches where that is one), rows that do not fill the last wave; one column and three
@pytest.mark.gpu
@pytest.mark.parametrize("dim,hidden", [(1024, 96), (1024, 4128), (2048, 1056), (2048, 2080), (4096, 96), (4096, 1056), (5120, 96)])
def test_projections_in_one_launch(oracle, dim, hidden):
    from llama2_rs import ops
    dims = ck.Dims(dim=dim, hidden_dim=hidden, n_layers=1, n_heads=dim // 128, n_kv_heads=dim // 1024, vocab_size=72, seq_len=32,
                   group_size=0)
    img = ck.synth_weights_image(dims, seed=5)
    m, o = ops.Model(img, dims), oracle.Model(img, dims)
    o.new_state()
    for pos, t in enumerate((1, 60)):
        want, got = o.transformer([t], [pos]), m.forward([t], [pos])
        assert nrel(got, want) < 1e-4, pos
    m.forward([7, 8, 9], [2, 3, 4])
    o.transformer([7, 8, 9], [2, 3, 4])
    for a, b in zip(m.read_kv(0, 0, 5), o.kv_cache()):
        assert nrel(a, b[0, :5]) < 1e-4
    assert nrel(m.forward([3], [5]), o.transformer([3], [5])) < 1e-4
    m.close()
    o.close()
