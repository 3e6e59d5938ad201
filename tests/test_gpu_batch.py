"""Batches in fp32 through the matrix cores (three exact bf16 planes of the activations): the operator at the edges of
its tiles against fp64, and whole prompts against the CPU oracle."""
import numpy as np
import pytest

from llama2_rs import checkpoint as ck
from tests import test_gemm_plan as shapes  # which tiles the shapes of the GEMMs' tests take

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from llama2_rs import ops as o, _lib
    assert _lib.lib().l2_device_count() >= 1, "no HIP device: the GPU tests cannot run"
    return o


def nrel(got, want):
    want = np.asarray(want, np.float64)
    scale = np.maximum(np.abs(want), np.sqrt(np.mean(want ** 2)) + 1e-30)
    return float(np.max(np.abs(np.asarray(got, np.float64) - want) / scale))


# rows: a last row block of 8 rows, of 128 and a whole one; inputs: half a K step at the end, an odd number of groups;
# columns: both sides of the token tiles of 32 and 64, one and several K slices
@pytest.mark.parametrize("n_in,n_out,G,batches", [
    (4128, 4104, 32, (4, 31, 32, 33, 64, 65)), (4160, 4232, 64, (8, 130)), (4224, 8320, 128, (5, 61, 300)),
    (13824, 1160, 128, (16,)), (1056, 29000, 32, (40,))])
def test_batch_operator_vs_fp64(ops, n_in, n_out, G, batches):
    rng = np.random.default_rng(n_in)
    qw, qz, sc, gi = ck.synth_qlinear(rng, n_in, n_out, G, act_order=True)
    W = ck.dequant_bin(qw, qz, sc, gi, G).astype(np.float64)
    q = ops.QLinear(qw, qz, sc, gi, G)
    for B in batches:
        # columns of very different size, so that no column leans on another's range
        x = (rng.standard_normal((B, n_in)) * 10.0 ** rng.uniform(-6, 6, (B, 1))).astype(np.float32)
        want = x.astype(np.float64) @ W.T
        got = q.matvec(x)
        for b in range(B):
            assert nrel(got[b], want[b]) < 1e-5, (B, b)
        np.testing.assert_array_equal(q.matvec(x), got)
    q.close()


# the tiles' other widths: 16, 32 and 64 columns as the only tile and as the last one of a wide block, few blocks (tiles of 32),
# several runs of groups, a slice of one step
@pytest.mark.parametrize("n_in,n_out,G,batches", [
    (4224, 8320, 128, (16, 17, 84, 96, 144)), (1056, 520, 32, (16, 17, 40, 50)), (1088, 264, 64, (15, 33, 80)),
    (28672, 1032, 64, (20, 36)), (2080, 24584, 32, (70, 86)), (64, 8200, 64, (60, 300)), (96, 8200, 32, (300,))])
def test_batch_tiles_vs_fp64(ops, n_in, n_out, G, batches):
    rng = np.random.default_rng(n_out)
    qw, qz, sc, gi = ck.synth_qlinear(rng, n_in, n_out, G, act_order=True)
    W = ck.dequant_bin(qw, qz, sc, gi, G).astype(np.float64)
    q = ops.QLinear(qw, qz, sc, gi, G)
    for B in batches:
        x = rng.standard_normal((B, n_in)).astype(np.float32)
        x[:, n_in // 2] *= 1e6  # one input far above the others
        want, got = x.astype(np.float64) @ W.T, q.matvec(x)
        for b in range(B):
            assert nrel(got[b], want[b]) < 1e-5, (B, b)
    q.close()


# what whole rounds of tiles of 64 and of 80 columns leave over, in tiles of every narrower width, in row blocks of their own and behind whole
# tiles, last tiles that are not full
@pytest.mark.parametrize("n_out,B", [s for s in shapes.FP32_TILES if s not in ((16640, 250), (4104, 61))])
def test_batch_last_round_vs_fp64(ops, n_out, B):
    rng = np.random.default_rng(B)
    qw, qz, sc, gi = ck.synth_qlinear(rng, 256, n_out, 64, act_order=True)
    x = rng.standard_normal((B, 256)).astype(np.float32)
    q = ops.QLinear(qw, qz, sc, gi, 64)
    got = q.matvec(x)
    assert nrel(got, x.astype(np.float64) @ ck.dequant_bin(qw, qz, sc, gi, 64).astype(np.float64).T) < 1e-5
    q.close()


# A column's bits are the same in tiles of every width: rows of weights that repeat every 256 (a block) and columns that repeat every
# seven give the same outputs wherever they stand.  Row blocks with tiles of both widths, tiles of 16 to 80 columns, one round with
# nothing left over.
@pytest.mark.parametrize("n_out,B", list(shapes.FP32_TILES))
def test_batch_bits_whatever_the_tile(ops, n_out, B):
    rng = np.random.default_rng(B)
    qw, qz, sc, gi = ck.synth_qlinear(rng, 256, 256, 64, act_order=True)
    rep = -(-n_out // 256)
    q = ops.QLinear(np.tile(qw, (rep, 1))[:n_out], np.tile(qz, (rep, 1))[:n_out // 8], np.tile(sc, (rep, 1))[:n_out], gi, 64)
    x = rng.standard_normal((7, 256)).astype(np.float32)[np.arange(B) % 7]
    got = q.matvec(x)
    assert nrel(got[:7, :256], x[:7].astype(np.float64) @ ck.dequant_bin(qw, qz, sc, gi, 64).astype(np.float64).T) < 1e-5
    np.testing.assert_array_equal(got, got[:7, :256][np.arange(B) % 7][:, np.arange(n_out) % 256])
    q.close()


# scales and zero points in tiles of 32 rows x 32 groups: a last tile of 8 rows alone, of 24, behind a whole one, and of one group
@pytest.mark.parametrize("n_in,n_out,G,B", [(28672, 8, 32, 300), (28672, 24, 64, 90), (28672, 40, 128, 60), (1056, 2056, 32, 32),
                                            (4160, 520, 64, 33)])
def test_batch_group_tiles_vs_fp64(ops, n_in, n_out, G, B):
    rng = np.random.default_rng(n_out)
    qw, qz, sc, gi = ck.synth_qlinear(rng, n_in, n_out, G, act_order=True)
    x = rng.standard_normal((B, n_in)).astype(np.float32)
    want = x.astype(np.float64) @ ck.dequant_bin(qw, qz, sc, gi, G).astype(np.float64).T
    q = ops.QLinear(qw, qz, sc, gi, G)
    assert nrel(q.matvec(x), want) < 1e-5
    q.close()


@pytest.mark.parametrize("kv,hidden,G,n", [(8, 2816, 32, 70), (4, 2848, 32, 64), (2, 2816, 64, 131), (1, 2816, 128, 97),
                                             (2, 2816, 0, 66), (8, 2848, 0, 135)])
def test_fp32_prompt_vs_oracle(ops, oracle, kv, hidden, G, n):
    dims = ck.Dims(dim=1024, hidden_dim=hidden, n_layers=2, n_heads=8, n_kv_heads=kv, vocab_size=300, seq_len=160, group_size=G)
    img = ck.synth_weights_image(dims, seed=3)
    m, o = ops.Model(img, dims), oracle.Model(img, dims)
    toks = np.random.default_rng(n).integers(0, dims.vocab_size, size=n).astype(np.int32)
    m.prefill_chunks(toks, 0, n)
    o.new_state()
    o.transformer(toks, np.arange(n, dtype=np.int32))
    ko, vo = o.kv_cache()
    for l in range(dims.n_layers):
        k, v = m.read_kv(l, 0, n)
        assert nrel(k, ko[l, :n]) < 1e-4 and nrel(v, vo[l, :n]) < 1e-4
    assert nrel(m.forward([7], [n]), o.transformer([7], [n])) < 1e-4
    if G == 0:  # the dense operator on a batch, at a ragged number of columns
        from llama2_rs import _lib
        import tests.test_oracle_loop as tol
        x = np.random.default_rng(1).standard_normal((33, 1024)).astype(np.float32)
        assert nrel(m.qmatvec(1, _lib.W1, x), x.astype(np.float64) @ tol._split_image(img, dims)["w1"][1].T.astype(np.float64)) < 1e-5
    m.close()
    o.close()


def rms_error(got, want):
    return float(np.sqrt(np.mean(((got - want) / np.sqrt(np.mean(want ** 2, axis=1, keepdims=True))) ** 2)))


# fp32 weights: a batch is no further from the exact sums than its columns one by one.  Rows on both sides of where the
# products summed from zero change (2048, 2560), one K slice (512 columns of 11008 outputs) and eight.  The rms over N > 2e4 values of
# similar size has a standard error of 1 / sqrt(2 N) < 0.5 %, the two of a ratio 0.7 %; three of those
@pytest.mark.parametrize("dim,hidden", [(1024, 11008), (1920, 2528), (2048, 2816)])
def test_dense_batch_error(ops, dim, hidden):
    from llama2_rs import _lib
    import tests.test_oracle_loop as tol
    dims = ck.Dims(dim=dim, hidden_dim=hidden, n_layers=1, n_heads=dim // 128, n_kv_heads=1, vocab_size=64, seq_len=32, group_size=0)
    img = ops.synth_image(dims, 4)
    m, rng = ops.Model(img, dims), np.random.default_rng(dim)
    for name, proj in (("w1", _lib.W1), ("w2", _lib.W2)):
        W = tol._split_image(img, dims)[name][0].astype(np.float64)
        for B in (33, 128, 512):
            x = rng.standard_normal((B, W.shape[1])).astype(np.float32)
            want = x.astype(np.float64) @ W.T
            one = np.stack([m.qmatvec(0, proj, x[b]) for b in range(24)])
            assert rms_error(m.qmatvec(0, proj, x), want) < 1.02 * rms_error(one, want[:24]), (name, B)
    m.close()


# sums in which one or a few terms are all there is, where nothing averages out.  One term: its product is rounded once,
# to 2^-24 of it; what is added before that is below 2^-7 of it, and its at most eight additions err by 2^-23 of that each.
# A few terms, and one far above the others: no further from the exact sums than the columns, as above (N = 2.8e5 values)
@pytest.mark.parametrize("dim,hidden", [(1024, 2816), (2048, 2816)])
def test_dense_batch_few_terms(ops, dim, hidden):
    from llama2_rs import _lib
    import tests.test_oracle_loop as tol
    dims = ck.Dims(dim=dim, hidden_dim=hidden, n_layers=1, n_heads=dim // 128, n_kv_heads=1, vocab_size=64, seq_len=32, group_size=0)
    img = ops.synth_image(dims, 4)
    m, rng, B = ops.Model(img, dims), np.random.default_rng(dim), 100
    W = tol._split_image(img, dims)["w1"][0].astype(np.float64)
    one, few, far = np.zeros((B, dim), np.float32), np.zeros((B, dim), np.float32), rng.standard_normal((B, dim)).astype(np.float32)
    for b in range(B):
        one[b, rng.integers(dim)] = rng.standard_normal()
        few[b, rng.choice(dim, 4, replace=False)] = rng.standard_normal(4)
    far[:, dim // 2] *= 1e6
    want = one.astype(np.float64) @ W.T
    err = np.abs(m.qmatvec(0, _lib.W1, one) - want)
    assert np.all(err <= (2.0 ** -24 + 8 * 2.0 ** -30) * np.abs(want)), np.max(err / np.maximum(np.abs(want), 1e-30))
    for x in (few, far):
        want = x.astype(np.float64) @ W.T
        assert rms_error(m.qmatvec(0, _lib.W1, x), want) < 1.02 * rms_error(np.stack([m.qmatvec(0, _lib.W1, v) for v in x]), want)
    # numbers that bf16 planes do not hold whole: cut at 2^-133, beside the K 2^-24 of the magnitudes that any association stays within
    for e in (-100, -112, -124):
        x = (rng.standard_normal((B, dim)) * 2.0 ** e).astype(np.float32)
        err = np.abs(m.qmatvec(0, _lib.W1, x) - x.astype(np.float64) @ W.T)
        assert np.all(err <= 2.0 ** -133 * np.abs(W).sum(1) + dim * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(W).T) + dim * 2.0 ** -149)
    m.close()


# Every product of a weight and an activation is taken, that of their third planes (up to 2^-32 of the whole) included: pairs of terms
# of which all cancels but the third plane of the weight, up to 2^-17, times the activation.  The matrix unit drops bits of what it
# adds up, the last of them below 2^-32 of the pair's first plane products, and only downwards: a result above the exact one by more
# than the rounding of what is left, 2^-17 2^-24, lacks a negative product
@pytest.mark.parametrize("dim,hidden", [(1024, 2816), (2048, 1344)])
def test_dense_products_are_exact(ops, dim, hidden):
    from llama2_rs import _lib
    import tests.test_oracle_loop as tol
    dims = ck.Dims(dim=dim, hidden_dim=hidden, n_layers=1, n_heads=dim // 128, n_kv_heads=1, vocab_size=64, seq_len=32, group_size=0)
    img, rng = ops.synth_image(dims, 4), np.random.default_rng(hidden)
    at = 1 + 64 * dim + dim + 2 * dim * dim + 2 * 128 * dim + dim  # of w1: in front of it eps, embedding, norm, q, k, v, o, norm
    w1 = img.view(np.float32)[at:at + hidden * dim].reshape(hidden, dim)

    def nearest(v):  # bf16
        b = v.view(np.uint32)
        return ((b + 0x7FFF + (b >> 16 & 1)) & np.uint32(0xFFFF0000)).view(np.float32)

    w = rng.uniform(1, 2, (hidden, dim // 2)).astype(np.float32)
    w[nearest(w - (w - nearest(w) - nearest(w - nearest(w)))) != nearest(w)] = 1.25  # without the third plane the first is another
    third = w - nearest(w) - nearest(w - nearest(w))
    w1[:, 0::2], w1[:, 1::2] = w, third - w
    m = ops.Model(img, dims)
    np.testing.assert_array_equal(tol._split_image(img, dims)["w1"][0], w1)
    for B in (33, 100, 300):
        x, pair = np.zeros((B, dim), np.float32), rng.integers(0, dim // 2, B)
        size = 2.0 ** rng.integers(-20, 20, B)
        of = (size * rng.uniform(1, 2, B) * rng.choice([-1, 1], B)).astype(np.float32)
        x[np.arange(B), 2 * pair] = x[np.arange(B), 2 * pair + 1] = of
        want = of[:, None].astype(np.float64) * third[:, pair].T
        err = (m.qmatvec(0, _lib.W1, x) - want) / size[:, None]
        assert err.max() <= 2.0 ** -39 and err.min() >= -2.0 ** -29, (B, np.log2(np.abs([err.max(), err.min()])))
    m.close()


# tiles of tokens from one to eight and one more block, rows that do not fill a block; then infinities and NaN, which the
# planes of a split number do not carry: a batch has them where its columns one by one have them.  Sums of K terms of either
# association differ by K 2^-24 of the sum of magnitudes at most, which is below sqrt(K) 2 rms for these inputs
@pytest.mark.parametrize("hidden", [2816, 1344])
def test_dense_batch_tiles(ops, hidden):
    from llama2_rs import _lib
    import tests.test_oracle_loop as tol
    dims = ck.Dims(dim=1024, hidden_dim=hidden, n_layers=1, n_heads=8, n_kv_heads=1, vocab_size=64, seq_len=32, group_size=0)
    img = ops.synth_image(dims, 6)
    m, rng = ops.Model(img, dims), np.random.default_rng(hidden)
    for name, proj in (("w1", _lib.W1), ("w2", _lib.W2)):
        W = tol._split_image(img, dims)[name][0].astype(np.float64)
        for B in (16, 17, 33, 48, 64, 65, 81, 97, 112, 113, 128, 129, 177):
            x = rng.standard_normal((B, W.shape[1])).astype(np.float32)
            assert nrel(m.qmatvec(0, proj, x), x.astype(np.float64) @ W.T) < 1e-5, (name, B)
        x = rng.standard_normal((100, W.shape[1])).astype(np.float32)
        x[3, 5], x[40, 100], x[99, 7], x[99, 9], x[70, -1], x[50] = np.inf, -np.inf, np.inf, -np.inf, np.nan, 3e38
        got, one = m.qmatvec(0, proj, x), np.stack([m.qmatvec(0, proj, v) for v in x])
        for b in (3, 40, 70, 99):
            np.testing.assert_array_equal(got[b], one[b])
        fine = [b for b in range(100) if b not in (3, 40, 50, 70, 99)]
        assert nrel(got[fine], x[fine].astype(np.float64) @ W.T) < 1e-5
        x.view(np.uint32)[20, 9] = 0x7F800001  # a NaN by its last bit, as only memory holds one: no arithmetic makes it
        assert np.all(np.isnan(m.qmatvec(0, proj, x)[20])) and np.all(np.isnan(m.qmatvec(0, proj, x[20])))
    m.close()


# rows that end with half a K step: the operator takes the matrix cores as the model does (its bits are not the columns'), and
# what lies behind a row's end, the last weights times zero, adds nothing even where those are infinite
def test_dense_operator_half_step(ops):
    from llama2_rs import _lib
    import tests.test_oracle_loop as tol
    dims = ck.Dims(dim=1024, hidden_dim=2848, n_layers=1, n_heads=8, n_kv_heads=1, vocab_size=64, seq_len=32, group_size=0)
    img = ops.synth_image(dims, 6)
    at = 1 + 64 * 1024 + 1024 + 2 * 1024 * 1024 + 2 * 128 * 1024 + 1024 + 2848 * 1024  # of w2
    w2 = img.view(np.float32)[at:at + 1024 * 2848].reshape(1024, 2848)
    w2[77, -1] = np.inf
    m, rng, W = ops.Model(img, dims), np.random.default_rng(9), w2.astype(np.float64)
    np.testing.assert_array_equal(W, tol._split_image(img, dims)["w2"][0])
    for B in (33, 100, 300):
        x = np.abs(rng.standard_normal((B, 2848))).astype(np.float32) + 0.01
        got, one = m.qmatvec(0, _lib.W2, x), np.stack([m.qmatvec(0, _lib.W2, v) for v in x])
        fine = np.arange(1024) != 77
        assert not np.array_equal(got[:, fine], one[:, fine]) and np.all(got[:, 77] == np.inf)
        assert nrel(got[:, fine], x.astype(np.float64) @ W[fine].T) < 1e-5
    m.close()


# finite operands whose planes or sums are not: every association has an infinity where all terms of a sum have one sign and it is
# above the range, and none where the terms' magnitudes add up to less than the range; a weight that a plane would round to
# infinity; the largest number of all.  Rows beyond the first block, the last tile of tokens, one K slice and several
@pytest.mark.parametrize("dim,hidden", [(1024, 2816), (2048, 1344)])
def test_dense_batch_overflow(ops, dim, hidden):
    from llama2_rs import _lib
    import tests.test_oracle_loop as tol
    dims = ck.Dims(dim=dim, hidden_dim=hidden, n_layers=1, n_heads=dim // 128, n_kv_heads=1, vocab_size=64, seq_len=32, group_size=0)
    img, top = ops.synth_image(dims, 6), np.finfo(np.float32).max
    at = 1 + 64 * dim + dim + 2 * dim * dim + 2 * 128 * dim + dim  # of w1: in front of it eps, embedding, norm, q, k, v, o, norm
    w1 = img.view(np.float32)[at:at + hidden * dim].reshape(hidden, dim)
    w1[300, 7], w1[hidden - 1, 8] = 3.4e38, -top
    m, rng, W = ops.Model(img, dims), np.random.default_rng(dim), w1.astype(np.float64)
    np.testing.assert_array_equal(W, tol._split_image(img, dims)["w1"][0])
    for B in (33, 100, 300):
        x = rng.standard_normal((B, dim)).astype(np.float32)
        x[:, 7:9] = rng.uniform(0.1, 0.3, (B, 2))
        x[5], x[5, 3] = 0, top
        x[B - 1], x[9] = np.sign(w1[2]) * 3e38, -np.sign(w1[hidden - 2]) * 3e38
        got = m.qmatvec(0, _lib.W1, x)
        assert got[B - 1, 2] == np.inf and got[9, hidden - 2] == -np.inf
        want, mag = x.astype(np.float64) @ W.T, np.abs(x).astype(np.float64) @ np.abs(W).T
        held = mag < top  # of the rest of the two rows, associations differ
        assert held[5].all() and np.all(held[[b for b in range(B) if b not in (9, B - 1)]])
        assert np.all(np.abs(got[held] - want[held]) <= dim * 2.0 ** -24 * mag[held])
    m.close()


# the same for quantised weights: several K slices and one, of one run of groups and of several (4128 and 4160 inputs, 512
# columns: three and two; 8320: two), an odd number of K steps and half of one.  The rounding of the matrix unit must not
# lean to one side either: the mean error of 512 columns' 4e6 values is below a thirtieth of their rms
@pytest.mark.parametrize("n_in,n_out,G", [(1024, 2816, 32), (4128, 8456, 32), (4160, 8456, 64), (8320, 8456, 128), (11008, 1024, 32),
                                          (28672, 512, 64)])
def test_batch_error(ops, n_in, n_out, G):
    rng = np.random.default_rng(n_in)
    qw, qz, sc, gi = ck.synth_qlinear(rng, n_in, n_out, G, act_order=True)
    W = ck.dequant_bin(qw, qz, sc, gi, G).astype(np.float64)
    q = ops.QLinear(qw, qz, sc, gi, G)
    for B in (32, 100, 512):
        x = rng.standard_normal((B, n_in)).astype(np.float32)
        want = x.astype(np.float64) @ W.T
        one, got = np.stack([q.matvec(x[b]) for b in range(32)]), q.matvec(x)
        assert rms_error(got, want) < 1.02 * rms_error(one, want[:32]), B
        if B == 512:
            rms = np.sqrt(np.mean(want ** 2, axis=1, keepdims=True))
            assert abs(np.mean((got - want) / rms)) < rms_error(got, want) / 30
    q.close()


# batches that must be the bits of their columns: the operator by both entry points, a projection of a model (quantised
# and not), and the rows that a prompt's first layer leaves, at sizes the default mode gives to the matrix cores
def test_columns_mode(ops):
    from llama2_rs import _lib
    from tests.test_zz_no_alloc import _Hip
    rng = np.random.default_rng(8)
    q = ops.QLinear(*ck.synth_qlinear(rng, 4096, 1160, 32, act_order=True), 32)
    x = rng.standard_normal((61, 4096)).astype(np.float32)
    one = np.stack([q.matvec(c) for c in x])
    assert not np.array_equal(q.matvec(x), one)
    q.set_mode(_lib.PREFILL_COLUMNS)
    np.testing.assert_array_equal(q.matvec(x), one)
    hip = _Hip()
    dx, dy = hip.upload(x), hip.empty(one.nbytes)
    q.matvec_device(dx, 61, dy)
    np.testing.assert_array_equal(hip.download(dy, one.shape), one)
    with pytest.raises(_lib.L2Error):
        q.set_mode(_lib.PREFILL_MFMA)
    q.set_mode(_lib.PREFILL_FP32)
    assert not np.array_equal(q.matvec(x), one)
    q.close()
    hip.close()
    for G in (64, 0):
        dims = ck.Dims(dim=1024, hidden_dim=2816, n_layers=1, n_heads=8, n_kv_heads=2, vocab_size=300, seq_len=128, group_size=G)
        m = ops.Model(ck.synth_weights_image(dims, seed=5), dims)
        x = rng.standard_normal((100, 1024)).astype(np.float32)
        toks = rng.integers(0, 300, size=100).astype(np.int32)
        for t in range(100):
            m.forward([int(toks[t])], [t], want_logits=False)
        rows, one = m.read_kv(0, 0, 100), np.stack([m.qmatvec(0, _lib.W1, c) for c in x])
        for mode in (_lib.PREFILL_FP32, _lib.PREFILL_COLUMNS):
            m.reset()
            m.set_prefill_mode(mode)
            m.prefill_chunks(toks, 0, 100)
            same = [np.array_equal(a, b) for a, b in zip(m.read_kv(0, 0, 100), rows)] + [np.array_equal(m.qmatvec(0, _lib.W1, x), one)]
            assert same == [mode == _lib.PREFILL_COLUMNS] * 3, (G, mode)
        m.close()


# tiles of 80 columns, alone and with what rounds leave over in 16, and of 64 with 16, 32 and 48: last tiles of 1, 49, 70 and 80, one, two and
# three units of K, half a one; a column is the bits it has in a batch of 64
@pytest.mark.parametrize("n_in,n_out,G,batches", [(*s, tuple(by_columns)) for s, by_columns in shapes.FP32_OF_80.items()])
def test_batch_tiles_of_80(ops, n_in, n_out, G, batches):
    rng = np.random.default_rng(n_in + G)
    qw, qz, sc, gi = ck.synth_qlinear(rng, n_in, n_out, G, act_order=True)
    W = ck.dequant_bin(qw, qz, sc, gi, G).astype(np.float64)
    q = ops.QLinear(qw, qz, sc, gi, G)
    x = rng.standard_normal((max(batches), n_in)).astype(np.float32)
    want = x.astype(np.float64) @ W.T
    of_64 = np.concatenate([q.matvec(x[b:b + 64]) for b in range(0, len(x), 64)])
    for B in batches:
        got = q.matvec(x[:B])
        np.testing.assert_array_equal(got[:B // 64 * 64], of_64[:B // 64 * 64])
        for b in range(B):
            assert nrel(got[b], want[b]) < 1e-5, (B, b)
    q.close()


# fp16 prompts: the last tile of tokens in each of its widths, behind tiles of 128 tokens and of 64
@pytest.mark.parametrize("G,batches", [(32, (65, 100)), (64, (65, 257, 300, 340, 370)), (128, (65, 272, 300, 340, 370))])
def test_fp16_operator_last_tile(ops, G, batches):
    from llama2_rs import _lib
    dims = ck.Dims(dim=1024, hidden_dim=2816, n_layers=1, n_heads=8, n_kv_heads=2, vocab_size=300, seq_len=512, group_size=G)
    m = ops.Model(ck.synth_weights_image(dims, seed=5), dims)
    for B in batches:
        x = np.random.default_rng(B).standard_normal((B, 1024)).astype(np.float32)
        m.set_prefill_mode(_lib.PREFILL_FP32)
        want = m.qmatvec(0, _lib.W1, x)
        m.set_prefill_mode(_lib.PREFILL_MFMA)
        got = m.qmatvec(0, _lib.W1, x)
        assert not np.array_equal(got, want)
        for b in range(B):
            assert nrel(got[b], want[b]) < 2e-3, (B, b)
    m.close()


# fp16 prompts in blocks of 256 rows: token tiles of every width, tiles left over in halves, with and without narrow ones
# behind them, one, two and three units of K, a last row block that is not full, rows of one matrix only
@pytest.mark.parametrize("dim,hidden,G,batches", [
    (256, 11008, 64, (890, 788, 800)), (256, 11136, 32, (257, 788)), (128, 22016, 64, (511,)), (384, 11008, 64, (520,)),
    (512, 11264, 128, (890, 430, 224)), (1024, 2816, 32, (300, 511))])
def test_fp16_operator_wide_blocks(ops, dim, hidden, G, batches):
    from llama2_rs import _lib
    dims = ck.Dims(dim=dim, hidden_dim=hidden, n_layers=1, n_heads=dim // 128, n_kv_heads=dim // 128, vocab_size=64, seq_len=1024,
                   group_size=G)
    m = ops.Model(ck.synth_weights_image(dims, seed=9), dims)
    for B in batches:
        # inputs that fp16 holds: with groups of 64 and 128 nothing is rounded but the fp32 sums.  With groups of 32 every weight
        # is, twice to 2^-12 of itself at most: the sum's error is 4e-4 of its rms, and 4e-3 ten times that
        x = np.random.default_rng(B).standard_normal((B, dim)).astype(np.float16).astype(np.float32)
        m.set_prefill_mode(_lib.PREFILL_FP32)
        want = m.qmatvec(0, _lib.W1, x)
        m.set_prefill_mode(_lib.PREFILL_MFMA)
        got = m.qmatvec(0, _lib.W1, x)
        assert not np.array_equal(got, want)
        for b in range(B):
            assert nrel(got[b], want[b]) < (4e-3 if G == 32 else 2e-5), (B, b)
    m.close()


# tiles of 144 tokens and nothing else: one unit of K, two, three, five and six, a last tile of 113, 129 and 144 tokens; the columns are the
# bits of tiles of 128.  (Narrower ones beside and behind them: test_fp16_bits_whatever_the_tile.)
@pytest.mark.parametrize("dim,hidden,G", shapes.FP16_OF_144)
def test_fp16_operator_tiles_of_144(ops, dim, hidden, G):
    from llama2_rs import _lib
    dims = ck.Dims(dim=dim, hidden_dim=hidden, n_layers=1, n_heads=dim // 128, n_kv_heads=dim // 128, vocab_size=64, seq_len=1024,
                   group_size=G)
    m = ops.Model(ck.synth_weights_image(dims, seed=13), dims)
    x = np.random.default_rng(dim).standard_normal((288, dim)).astype(np.float16).astype(np.float32) # as above: only fp32 sums round
    m.set_prefill_mode(_lib.PREFILL_FP32)
    want = m.qmatvec(0, _lib.W1, x)
    m.set_prefill_mode(_lib.PREFILL_MFMA)
    of_128 = m.qmatvec(0, _lib.W1, x[:256])
    for B in (257, 273, 288):
        got = m.qmatvec(0, _lib.W1, x[:B])
        assert np.array_equal(got[:256], of_128), B
        for b in range(B):
            assert nrel(got[b], want[b]) < (4e-3 if G == 32 else 2e-5), (B, b)
    m.close()


# tiles of an odd number of 16 tokens: of 112 with a last one of 88 (200 columns), 80, 48, a last one of 33, blocks of four waves too; the
# columns are the bits of tiles of 32
@pytest.mark.parametrize("dim,hidden,G,batches", [(*s, tuple(by_columns)) for s, by_columns in shapes.FP16_ODD.items()])
def test_fp16_operator_odd_tiles(ops, dim, hidden, G, batches):
    from llama2_rs import _lib
    dims = ck.Dims(dim=dim, hidden_dim=hidden, n_layers=1, n_heads=dim // 128, n_kv_heads=dim // 128, vocab_size=64, seq_len=1024,
                   group_size=G)
    m = ops.Model(ck.synth_weights_image(dims, seed=15), dims)
    x = np.random.default_rng(dim).standard_normal((max(batches), dim)).astype(np.float16).astype(np.float32) # as above: only fp32 sums round
    m.set_prefill_mode(_lib.PREFILL_FP32)
    want = m.qmatvec(0, _lib.W1, x)
    m.set_prefill_mode(_lib.PREFILL_MFMA)
    for B in batches:
        got = m.qmatvec(0, _lib.W1, x[:B])
        for b in range(B):
            assert nrel(got[b], want[b]) < (4e-3 if G == 32 else 2e-5), (B, b)
        if dim < 512:  # one slice of K whatever the batch
            of_32 = np.concatenate([m.qmatvec(0, _lib.W1, x[b:b + 32]) for b in range(0, B // 32 * 32, 32)])
            assert np.array_equal(got[:len(of_32)], of_32), B
    m.close()


# what whole rounds leave over of tiles of 144 columns, a narrow last one (300) and 48 (520), and of 128, 32 behind whole tiles of a row block
# (350) and 96 (590): first and last tiles that are not full, a last row block that is not full, whole tiles that end inside eight row blocks
@pytest.mark.parametrize("B", [300, 350, 520, 590])
def test_fp16_operator_last_round(ops, B):
    from llama2_rs import _lib
    dims = ck.Dims(dim=256, hidden_dim=21888, n_layers=1, n_heads=2, n_kv_heads=2, vocab_size=64, seq_len=1024, group_size=64)
    m = ops.Model(ck.synth_weights_image(dims, seed=11), dims)
    x = np.random.default_rng(B).standard_normal((B, 256)).astype(np.float16).astype(np.float32) # as above: only fp32 sums round
    m.set_prefill_mode(_lib.PREFILL_FP32)
    want = m.qmatvec(0, _lib.W1, x)
    m.set_prefill_mode(_lib.PREFILL_MFMA)
    got = m.qmatvec(0, _lib.W1, x)
    m.close()
    assert not np.array_equal(got, want)
    for b in range(B):
        assert nrel(got[b], want[b]) < 2e-5, b


# as test_batch_bits_whatever_the_tile: tiles of 128 and of 144 tokens with narrower ones of 32 to 128 for what is left, row blocks that have
# both, with and without last tokens of their own; blocks of 128 rows, tiles of 64 tokens with ones of 32
@pytest.mark.parametrize("hidden,B", list(shapes.FP16_TILES))
def test_fp16_bits_whatever_the_tile(ops, hidden, B):
    from llama2_rs import _lib
    dims = ck.Dims(dim=256, hidden_dim=hidden, n_layers=1, n_heads=2, n_kv_heads=2, vocab_size=64, seq_len=1024, group_size=64)
    img = ck.synth_weights_image(dims, seed=11)
    rows, words = np.arange(hidden), img.view(np.int32)
    at = 1 + 64 * 256 + 256 + 4 * (256 * 32 + 32 * 4 + 256 * 4 + 256) + 256  # w1 begins behind q, k, v, o and two norms
    for n, per in ((hidden, 32), (hidden // 8, 4), (hidden, 4)):             # packed weights, zero points, scales
        part = words[at:at + n * per].reshape(n, per)
        part[:] = part[np.arange(n) % (256 * n // hidden)].copy()
        at += n * per
    m = ops.Model(img, dims)
    m.set_prefill_mode(_lib.PREFILL_MFMA)
    x = np.random.default_rng(B).standard_normal((7, 256)).astype(np.float32)[np.arange(B) % 7]
    got = m.qmatvec(0, _lib.W1, x)
    m.set_prefill_mode(_lib.PREFILL_FP32)
    assert nrel(got[:7, :256], m.qmatvec(0, _lib.W1, x)[:7, :256]) < 2e-3
    np.testing.assert_array_equal(got, got[:7, :256][np.arange(B) % 7][:, rows % 256])
    m.close()


# prompt attention with two sets of columns per block (two blocks per compute unit and more), the last block with one
# set, and grids of one to two blocks per unit, whose tiles go in pairs, against passes too short for either
@pytest.mark.parametrize("n_heads,n_kv,n", [(32, 32, 505), (16, 2, 1021), (32, 32, 200), (32, 32, 250), (16, 16, 300)])
def test_prompt_attention_two_sets(ops, n_heads, n_kv, n):
    dims = ck.Dims(dim=128 * n_heads, hidden_dim=256, n_layers=2, n_heads=n_heads, n_kv_heads=n_kv, vocab_size=64,
                   seq_len=1056, group_size=64)
    m = ops.Model(ck.synth_weights_image(dims, seed=9), dims)
    toks = np.random.default_rng(n).integers(0, 64, size=n).astype(np.int32)
    m.prefill_chunks(toks, 0, n)
    k, v = m.read_kv(1, 0, n)
    m.reset()
    for p in range(0, n, 101):
        m.prefill_chunks(toks[p:p + 101], p, 101)
    k2, v2 = m.read_kv(1, 0, n)
    assert nrel(k, k2) < 1e-5 and nrel(v, v2) < 1e-5
    m.close()


# the fp16 mode's attention (three bf16 numbers for each fp32 one): blocks of one set of 16 columns and of two, one to eight query
# heads per kv head, tiles of 16 rows and sets that end anywhere, an odd number of sets, rows of an earlier pass in front, against
# the fp32 mode.  Rows of the second layer: five inputs of products rounded to fp16 on the way, 2^-11 / sqrt(3) each, sqrt(5) of it
@pytest.mark.parametrize("n_heads,n_kv,at,n", [(2, 2, 0, 17), (4, 2, 5, 40), (8, 2, 61, 100), (8, 1, 300, 33), (32, 32, 0, 289), (32, 32, 61, 300),
                                               (16, 8, 0, 701), (32, 8, 3, 260), (64, 8, 33, 255)])
def test_fp16_prompt_attention(ops, n_heads, n_kv, at, n):
    from llama2_rs import _lib
    dims = ck.Dims(dim=128 * n_heads, hidden_dim=256, n_layers=2, n_heads=n_heads, n_kv_heads=n_kv, vocab_size=64,
                   seq_len=1056, group_size=64)
    m = ops.Model(ck.synth_weights_image(dims, seed=9), dims)
    toks = np.random.default_rng(n).integers(0, 64, size=at + n).astype(np.int32)
    rows = []
    for mode in (_lib.PREFILL_MFMA, _lib.PREFILL_FP32):
        m.reset()
        m.set_prefill_mode(mode)
        if at:
            m.prefill_chunks(toks[:at], 0, at)
        m.prefill_chunks(toks[at:], at, n)
        rows.append(m.read_kv(1, at, n))
    for got, want in zip(*rows):
        e = np.sqrt(np.mean((got - want).astype(np.float64) ** 2, axis=(1, 2)) / np.mean(want.astype(np.float64) ** 2, axis=(1, 2)))
        assert e.max() < 6.4e-4
    m.close()


def _planes(v):
    """Three bf16 numbers for each fp32 one, rounded to nearest, in fp64."""
    v, out = v.astype(np.float32), []
    for _ in range(3):
        b = v.view(np.uint32)
        out.append(((b + 0x7FFF + (b >> 16 & 1)) & np.uint32(0xFFFF0000)).view(np.float32))
        v = v - out[-1]
    return [p.astype(np.float64) for p in out]


def _see_through_image(d, rng, qk):
    """Two layers that show attention of the first one in the values of the second: wk is wq (so that a key row is the query), wo and the
    second layer's wv are one, w2 is zero."""
    parts = []

    def put(a, dtype=np.float32):
        parts.append(np.ascontiguousarray(a, dtype).view(np.uint8).reshape(-1))

    def linear(n, scale):  # n: whole numbers -8..7 [out][in]
        g = n.shape[1] // d.group_size
        put(ck.pack_nibbles(n + 8, axis=1), np.int32), put(ck.pack_nibbles(np.full((n.shape[0], g), 7), axis=0), np.int32)
        put(np.full((n.shape[0], g), scale)), put(np.arange(n.shape[1]), np.int32)

    q, one, none = rng.integers(-8, 8, (d.dim, d.dim)), np.eye(d.dim, dtype=np.int64), np.zeros((d.dim, d.dim), np.int64)
    emb = rng.normal(0, 0.02, (d.vocab_size, d.dim)).astype(np.float32)
    put([1e-5]), put(emb), put(np.ones((2, d.dim)))
    for n in (q, q, q, q, none, one, one, none):  # wq, wk, wv and wo of both layers
        linear(n, qk if n is q else 1)
    put(np.ones((2, d.dim)))
    for n_out, n_in in ((d.hidden_dim, d.dim), (d.dim, d.hidden_dim), (d.hidden_dim, d.dim)):
        for _ in range(2):
            linear(np.zeros((n_out, n_in), np.int64), 1)
    put(np.ones(d.dim)), put(np.zeros((2, d.seq_len, 64))), put(emb)
    img = np.concatenate(parts)
    assert img.nbytes == ck.weights_bytes(d)
    return img, emb


# ... and its precision, where it shows behind outputs rounded to fp16: one query, its keys and values made so that much cancels.
#   scores: products of 2e4 rms that add up to what the query has with itself and two more or less.  A partial sum of 2e4 sqrt(128) /
#     sqrt(128) log2(e) = 2.9e4 is rounded to 2^-10, some ten of them: ln 2 sqrt(10) 2^-10 = 2e-3 of a weight; twice that
#   sums: values of 2.4e4 sqrt(100) that add up to one: weights are right to some 2^-23, so 24000 2^-22.5 = 4e-3; five times that
#   bias: scores of 2^18 of products of one sign, keys with all bits of the low planes set in turns with keys without them, whose
#     values are 1 and -1.  A product that lacks 2^-24 of itself on one side takes ln 2 2^-7 = 5e-3 of the weight; the mean of 512 outputs
#     errs by less than 1e-3 if it does not (numbers that were cut instead of rounded: 3e-3 to 9e-3)
# Without any one of the six products an output would be off by more than twice the bound.
@pytest.mark.parametrize("kind,seed", [("scores", 0), ("scores", 1), ("sums", 0), ("sums", 1), ("bias", 0), ("bias", 1), ("bias", 2)])
def test_fp16_prompt_attention_precision(ops, kind, seed):
    from llama2_rs import _lib
    H, at, n, unit, rng = 4, 100, 16, np.log2(np.e) / np.sqrt(128), np.random.default_rng(seed)
    q_rms, bound = {"scores": (8, 4e-3), "sums": (0.1, 2e-2), "bias": (8, 1e-3)}[kind]
    d = ck.Dims(dim=128 * H, hidden_dim=256, n_layers=2, n_heads=H, n_kv_heads=H, vocab_size=64, seq_len=128, group_size=64)
    img, emb = _see_through_image(d, rng, q_rms / (4.6 * np.sqrt(d.dim)))
    m = ops.Model(img, d)
    m.set_prefill_mode(_lib.PREFILL_MFMA)
    toks = rng.integers(0, 64, n).astype(np.int32)
    m.prefill_chunks(toks, at, n)
    k_own, v_own = (a[0] for a in m.read_kv(0, at, 1))
    q = k_own.astype(np.float64)
    own = (q * q).sum(-1) * unit
    score = (2.0 ** 18 if kind == "bias" else own) + rng.uniform(-2, 2, (at, H))
    k = rng.standard_normal((at, H, 128)) * (20000 / q_rms if kind == "scores" else 1)
    if kind == "bias":
        bits = (np.sign(q) * 16000 / np.abs(q) * rng.uniform(0.5, 2, k.shape)).astype(np.float32).view(np.uint32)
        bits[0::2] |= 0x7FFF
        bits[1::2] &= 0xFFFF0000
        k = bits.view(np.float32).astype(np.float64)
        least = np.argmin(np.abs(q), axis=-1)  # takes what is missing from the score
        k[:, np.arange(H), least] += (score / unit - (k * q).sum(-1)) / q[np.arange(H), least]
    else:
        k += q * ((score / unit - (k * q).sum(-1)) / (q * q).sum(-1))[..., None]
    k = k.astype(np.float32)
    s = np.concatenate([(k.astype(np.float64) * q).sum(-1) * unit, own[None]])
    p = np.exp2(s - s.max(0))
    w = p / p.sum(0)
    v = rng.standard_normal((at, H, 128))
    if kind == "sums":
        v *= 24000 * np.sqrt(at)
        for h, j in enumerate(np.argmax(w[:at], axis=0)):
            v[j, h] -= (w[:at, h] @ v[:, h] - rng.standard_normal(128)) / w[j, h]
    if kind == "bias":
        v = np.where(np.arange(at) % 2, -1, 1)[:, None, None] + 0.02 * v
    v = v.astype(np.float32)

    def output(w):
        return np.sum(w[:at, :, None] * v.astype(np.float64), axis=0) + w[at][:, None] * v_own

    out = output(w)
    if kind == "scores":  # without one product of planes
        kp, qp = _planes(k), _planes(k_own)
        for i, j in ((0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0)):
            less = s.copy()
            less[:at] -= (kp[i] * qp[j]).sum(-1) * unit
            less = np.exp2(less - less.max(0))
            assert np.linalg.norm(output(less / less.sum(0)) - out) > 2 * bound * np.linalg.norm(out), (i, j)
    if kind == "sums":
        vp, pp = _planes(v), _planes(p[:at].astype(np.float32))
        for i, j in ((0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0)):
            assert np.linalg.norm(np.sum(pp[j][..., None] * vp[i], axis=0) / p.sum(0)[:, None]) > 2 * bound * np.linalg.norm(out), (i, j)
    m.write_kv(0, 0, k, v)
    m.prefill_chunks(toks, at, n)
    np.testing.assert_array_equal(m.read_kv(0, at, 1)[0][0], k_own)
    x = emb[toks[0]].astype(np.float64) + out.reshape(-1)
    rms = np.sqrt(np.mean(x * x) + 1e-5)
    err = m.read_kv(1, at, 1)[1].reshape(-1) * rms - x
    m.close()
    assert (abs(err.mean()) if kind == "bias" else np.linalg.norm(err) / np.linalg.norm(x)) < bound


# ... and what its planes do not hold: an infinity among the keys, which takes a row's weight to zero or makes the output a NaN, as the
# query's sign has it, and a value near the largest number on the row without weight.  One set of columns and two, both in the
# same places as in the fp32 mode, the other outputs as above
@pytest.mark.parametrize("n_heads,n_kv,at,n", [(4, 4, 40, 40), (8, 4, 5, 100), (32, 32, 61, 300)])
def test_fp16_prompt_attention_not_finite(ops, n_heads, n_kv, at, n):
    from llama2_rs import _lib
    dims = ck.Dims(dim=128 * n_heads, hidden_dim=256, n_layers=2, n_heads=n_heads, n_kv_heads=n_kv, vocab_size=64,
                   seq_len=400, group_size=64)
    m = ops.Model(ck.synth_weights_image(dims, seed=9), dims)
    toks = np.random.default_rng(n).integers(0, 64, size=at + n).astype(np.int32)
    rows = []
    for mode in (_lib.PREFILL_MFMA, _lib.PREFILL_FP32):
        m.reset()
        m.set_prefill_mode(mode)
        m.prefill_chunks(toks[:at], 0, at)
        k, v = m.read_kv(0, 0, at)
        k[3, 0, 70], v[3, 0] = -np.inf, 3.4e38
        m.write_kv(0, 0, k, v)
        m.prefill_chunks(toks[at:], at, n)
        rows.append(m.read_kv(1, at, n))
    for got, want in zip(*rows):
        fine = np.isfinite(want).all(axis=(1, 2))
        np.testing.assert_array_equal(np.isfinite(got).all(axis=(1, 2)), fine)
        assert n / 8 < fine.sum() < n
        e = np.sqrt(np.mean((got - want)[fine].astype(np.float64) ** 2, axis=(1, 2)) / np.mean(want[fine].astype(np.float64) ** 2, axis=(1, 2)))
        assert e.max() < 6.4e-4
    m.close()


# the kernels between the products of a chunk: rows of one, two and four trips of the block (and a consumer's order per
# LDS row, or in turns), few K slices and many, in each kind of plane, against single tokens.  fp16 inputs carry 2^-11 each:
# through the five products in front of the second layer's cache rows some 1e-3, and 4.5 times that at the furthest of
# some 10^6 values, with as much again for rows of small inputs
@pytest.mark.parametrize("n_heads,n_kv,G", [(8, 8, 64), (40, 40, 64), (64, 8, 64), (72, 9, 64), (72, 9, 0)])
def test_between_products(ops, n_heads, n_kv, G):
    from llama2_rs import _lib
    dims = ck.Dims(dim=128 * n_heads, hidden_dim=384, n_layers=2, n_heads=n_heads, n_kv_heads=n_kv, vocab_size=64,
                   seq_len=320, group_size=G)
    m = ops.Model(ck.synth_weights_image(dims, seed=4), dims)
    toks = np.random.default_rng(1).integers(0, 64, size=260).astype(np.int32)
    for n in (33, 70, 260):
        m.reset()
        for t in range(n):
            m.forward([int(toks[t])], [t], want_logits=False)
        want = m.read_kv(1, 0, n)
        for mode, tol in ((_lib.PREFILL_FP32, 1e-4), (_lib.PREFILL_MFMA, 3e-2)):
            if mode == _lib.PREFILL_MFMA and not G:
                continue
            m.reset()
            m.set_prefill_mode(mode)
            m.prefill_chunks(toks[:n], 0, n)
            for got, ref in zip(m.read_kv(1, 0, n), want):
                assert nrel(got, ref) < tol, (n, mode)
    m.close()


# the classifier with whole tiles of rows per wave and with a quarter or half of them, at both sides of where the rule changes, the last
# wave ragged; its running maximum against the logits
@pytest.mark.parametrize("n_heads,vocab", [(8, 1), (8, 2001), (8, 8160), (8, 8163), (16, 4080), (16, 4083), (32, 2033), (32, 2049), (40, 1025)])
def test_classifier_few_rows(ops, n_heads, vocab):
    dim = 128 * n_heads
    dims = ck.Dims(dim=dim, hidden_dim=256, n_layers=1, n_heads=n_heads, n_kv_heads=n_heads, vocab_size=vocab, seq_len=32,
                   group_size=64)
    img = ck.synth_weights_image(dims, seed=vocab)
    m = ops.Model(img, dims)
    W = img[-4 * vocab * dim:].view(np.float32).reshape(vocab, dim).astype(np.float64)
    x = np.random.default_rng(2).standard_normal(dim).astype(np.float32)
    want = W @ x.astype(np.float64)
    # fp32 sums of at most 80 dim / 4096 roundings in a row, and the six of a wave's lanes
    assert np.all(np.abs(m.classifier(x) - want) < 90 * 2.0 ** -24 * (np.abs(W) @ np.abs(x.astype(np.float64))))
    for pos in range(6):
        logits = m.forward([0], [pos])
        assert m.decode_greedy(0, pos) == vocab - 1 - int(np.argmax(logits[::-1]))
    m.close()


# a text whose prompt alone passes `steps`: the prompt's rows are there whatever the next call stages on the host
def test_prompt_past_the_steps(ops):
    import os
    import types
    import llama2_rs
    dims = ck.Dims(dim=1024, hidden_dim=512, n_layers=2, n_heads=8, n_kv_heads=8, vocab_size=32000, seq_len=1024, group_size=64)
    m = ops.Model(ck.synth_weights_image(dims, seed=6), dims)
    tok = llama2_rs.Tokenizer(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "tokenizer.bin"))
    text = "the quick brown fox " * 100
    rows = []
    for follow in (False, True):
        llama2_rs.generate(types.SimpleNamespace(_m=m), tok, text, 2, llama2_rs.Random(1), 0.8)
        if follow:
            m.prefill_chunks(np.full(400, 7, np.int32), 600, 64)
        rows.append(m.read_kv(1, 0, 384))
    for a, b in zip(*rows):
        assert np.any(a[383]) and np.array_equal(a, b)
    m.close()


# two passes of one prompt, the longer chunk cut into more slices of K than the shorter one (5120 inputs, 3 x 5120 rows: 256
# columns in two, 143 in one): the buffers hold either
def test_chunks_cut_into_more_slices_than_the_last(ops):
    from llama2_rs import _lib
    dims = ck.Dims(dim=5120, hidden_dim=384, n_layers=1, n_heads=40, n_kv_heads=40, vocab_size=64, seq_len=512, group_size=64)
    m = ops.Model(ck.synth_weights_image(dims, seed=4), dims)
    m.set_prefill_mode(_lib.PREFILL_MFMA)
    toks = np.random.default_rng(1).integers(0, 64, size=399).astype(np.int32)
    m.prefill_chunks(toks, 0, 256)
    got = m.read_kv(0, 0, 399)
    m.reset()
    for a, b in ((0, 256), (256, 399)):
        m.forward(toks[a:b], np.arange(a, b, dtype=np.int32))
    for x, y in zip(got, m.read_kv(0, 0, 399)):
        np.testing.assert_array_equal(x, y)
    m.close()
