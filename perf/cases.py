"""What this framework is used for, as cases that can be timed: the stand-alone GPTQ 4-bit operator, prompts through
both prefill modes, and the token loop (greedy, sampled, behind a long cache), on the preset geometries.

Weights are random-init in the checkpoint layout and fixed for a shape, as a program loads one checkpoint and then serves
many requests; what a request brings (prompt, text, token, cached rows, activations) comes from the seed.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "llama2.rs_amd"))
from llama2_rs import Random, Tokenizer, _lib, generate, ops  # noqa: E402
from llama2_rs.checkpoint import Dims  # noqa: E402

# dim, hidden_dim, heads, kv heads, vocabulary: the three presets and the small geometry of the parity tests
GEOMETRY = {
    "7B": (4096, 11008, 32, 32, 32000),
    "13B": (5120, 13824, 40, 40, 32000),
    "70B": (8192, 28672, 64, 8, 32000),
    "small": (1024, 2816, 8, 2, 2000),
}


def listed():
    return [
        # One projection called on host arrays, as the reference's CUDA slot is called: the 4096x4096 layer of the
        # benchmark's first configuration.  A single small call: its latency is what counts.
        {"name": "operator_host_one", "kind": "host", "in": 4096, "out": 4096, "group": 128, "batch": 1},
        # The same call for a batch of columns (prefill ladder step of 16) on 13B's w2, the longest ordinary row.
        {"name": "operator_host_batch16", "kind": "host", "in": 13824, "out": 5120, "group": 128, "batch": 16},
        # The operator on device memory for a program with its own loop: one column of 70B's wk at group 64, ...
        {"name": "operator_device_one", "kind": "device", "in": 8192, "out": 1024, "group": 64, "batch": 1},
        # ... and 7B's w1 at group 32 with an odd number of columns.
        {"name": "operator_device_batch61", "kind": "device", "in": 4096, "out": 11008, "group": 32, "batch": 61},
        # A small model, where launches and the host count: a 33-token prompt and 48 positions behind it.
        {"name": "small_generate", "kind": "tokens", "model": "small", "layers": 3, "group": 32, "prompt": 33, "steps": 81},
        # The headline: text in, greedy text out on the whole 7B model (the benchmark's second configuration).
        {"name": "7B_text_greedy", "kind": "text", "model": "7B", "layers": 32, "group": 128, "words": 12, "steps": 96,
         "temperature": 0.0},
        # The same program sampling at a temperature, as interactive use does.
        {"name": "7B_text_sampled", "kind": "text", "model": "7B", "layers": 32, "group": 128, "words": 3, "steps": 48,
         "temperature": 0.8},
        # A longer prompt in the default prefill mode and a short answer: the ladder's ragged end included.
        {"name": "7B_prompt_300_answer_32", "kind": "tokens", "model": "7B", "layers": 32, "group": 128, "prompt": 300,
         "steps": 332},
        # The benchmark's prefill configuration: 512 tokens in chunks of 128 on the matrix cores, then the logits.
        {"name": "7B_prefill_512_mfma", "kind": "prefill", "model": "7B", "layers": 32, "group": 128, "tokens": 512,
         "chunk": 128, "mfma": True},
        # One odd-sized pass over a document on 70B's widths (grouped queries, group 64); eight of its layers.
        {"name": "70B_prefill_777_mfma", "kind": "prefill", "model": "70B", "layers": 8, "group": 64, "tokens": 777,
         "chunk": 1024, "mfma": True},
        # Decode behind a long context on 70B's widths: eight greedy steps behind 4096 cached rows.
        {"name": "70B_decode_behind_4096", "kind": "decode", "model": "70B", "layers": 8, "group": 64, "cached": 4096,
         "tokens": 8},
        # The model without quantisation on 7B's widths: a prompt in chunks of 64 (its only mode), then the logits.
        {"name": "dense_prefill_100", "kind": "prefill", "model": "7B", "layers": 2, "group": 0, "tokens": 100, "chunk": 64,
         "mfma": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("host", "device", "tokens", "text", "prefill", "prefill", "decode"))
    if kind in ("host", "device"):
        n_in = rng.choice((1024, 2816, 4096, 4608, 5120, 8192, 11008, 13824, 28672))
        group = rng.choice([g for g in (32, 64, 128) if n_in % g == 0])
        n_out = 8 * _log(rng, 32, 28672 // 8) if n_in < 16384 else 8 * _log(rng, 32, 1024)
        return {"kind": kind, "in": n_in, "out": n_out, "group": group,
                "batch": min(_log(rng, 1, 130), _max_batch(n_in))}
    # The largest listed cases run the whole 7B model; drawn ones run some layers of every geometry.
    model = rng.choice(tuple(GEOMETRY))
    layers = rng.randint(2, 6)
    case = {"kind": kind, "model": model, "layers": layers, "group": rng.choice((32, 64, 128))}
    if kind == "tokens":
        prompt = _log(rng, 2, 400)
        case.update(prompt=prompt, steps=prompt + rng.randint(8, 64))
    elif kind == "text":
        if model == "small":  # its vocabulary is not the tokenizer's
            case["model"] = "7B"
        words, temperature = _log(rng, 1, 150), rng.choice((0.0, 0.7, 1.0))
        if temperature:  # sampling follows a turn of a dialogue: a few words
            words = min(words, 4)
        case.update(words=words, steps=words + rng.randint(16, 64), temperature=temperature)
    elif kind == "prefill":
        if rng.random() < 0.15:
            case["group"], case["layers"] = 0, 1
        tokens = _log(rng, 16, 900) if case["group"] else _log(rng, 16, 128)
        case.update(tokens=tokens, chunk=rng.choice((64, 128, 256, 1024)), mfma=case["group"] != 0 and rng.random() < 0.6)
    else:
        case.update(cached=_log(rng, 1, 4500), tokens=rng.randint(1, 12))
    return case


def _max_batch(n_in):
    """What l2_qlinear_matvec_device's fixed scratch takes (L2_MATVEC_DEVICE_MAX_ELEMS)."""
    return (1 << 20) // n_in


# ---- what a program has in hand -------------------------------------------------------------------------------


def _dims(case):
    dim, hidden, heads, kv, vocab = GEOMETRY[case["model"]]
    return Dims(dim=dim, hidden_dim=hidden, n_layers=case["layers"], n_heads=heads, n_kv_heads=kv, vocab_size=vocab,
                seq_len=2048, group_size=case["group"])


_models = {}  # loaded checkpoints by shape


def _model(case):
    d = _dims(case)
    max_seq = 4608 if case["kind"] == "decode" else 2048
    key = (case["model"], d.n_layers, d.group_size, max_seq)
    if key not in _models:
        img = ops.synth_image(d, 1)
        # the last norm's weights as trained checkpoints have them, so that the logits have a trained model's spread
        end = img.nbytes - 4 * d.vocab_size * d.dim - 4 * d.seq_len * d.head_size
        img[end - 4 * d.dim:end].view(np.float32)[:] = np.random.default_rng(2).normal(1.8, 0.2, d.dim)
        _models[key] = ops.Model(img, d, max_seq=max_seq)
    return _models[key]


class _Session(ops.Model):
    """One request's state (cache) on a loaded model."""

    def __init__(self, model):
        self.dims, self.h, self.max_seq = model.dims, model.h, model.max_seq
        self.state = type(model.state)()
        _lib.check(_lib.lib().l2_state_new(self.h, ctypes.byref(self.state)))

    def close(self):
        if self.state:
            _lib.lib().l2_state_free(self.state)
            self.state = type(self.state)()
        self.h = None


class _Chat:
    """What generate() takes as its model."""

    def __init__(self, session):
        self._m = session


_tokenizer = []

_WORDS = ("the of and to in is that it was for on are as with his they at be this have from or one had by word but not what "
          "all were we when your can said there use an each which she do how their if will up other about out many then "
          "them these so some her would make like him into time has look two more write go see number no way could people "
          "my than first water been call who oil its now find long down day did get come made may part").split()


def _operator(case, rng):
    n_in, n_out, group = case["in"], case["out"], case["group"]
    groups = n_in // group
    qweight = rng.integers(-2**31, 2**31, (n_out, n_in // 8), dtype=np.int64).astype(np.int32)
    qzeros = rng.integers(-2**31, 2**31, (n_out // 8, groups), dtype=np.int64).astype(np.int32)
    scales = rng.uniform(0.002, 0.02, (n_out, groups)).astype(np.float32)
    g_index = np.argsort(rng.permutation(n_in) // group, kind="stable").astype(np.int32)
    return ops.QLinear(qweight, qzeros, scales, g_index, group)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind in ("host", "device"):
        x = rng.standard_normal((case["batch"], case["in"])).astype(np.float32)
        s = {"kind": kind, "op": _operator(case, rng), "x": x}
        if kind == "device":
            s["x"] = torch.from_numpy(x).cuda()
            s["y"] = torch.empty((case["batch"], case["out"]), device="cuda")
        return s
    m = _Session(_model(case))
    s = {"kind": kind, "m": m}
    vocab = m.dims.vocab_size
    if kind == "tokens":
        s.update(prompt=rng.integers(0, vocab, case["prompt"]).astype(np.int32), steps=case["steps"])
    elif kind == "text":
        if not _tokenizer:
            _tokenizer.append(Tokenizer(os.path.join("tests", "golden", "tokenizer.bin")))
        s.update(model=_Chat(m), text=" ".join(rng.choice(_WORDS, case["words"])), steps=case["steps"],
                 temperature=case["temperature"], seed=int(rng.integers(1, 2**62)))
    elif kind == "prefill":
        s.update(tokens=rng.integers(0, vocab, case["tokens"] - 1).astype(np.int32), last=int(rng.integers(0, vocab)),
                 chunk=case["chunk"], mode=_lib.PREFILL_MFMA if case["mfma"] else _lib.PREFILL_FP32)
    else:
        m.fill_kv_synthetic(0, case["cached"], seed=int(rng.integers(0, 2**31)))
        s.update(token=int(rng.integers(0, vocab)), pos=case["cached"], n=case["tokens"])
    return s


def run(s):
    kind = s["kind"]
    if kind == "host":
        return s["op"].matvec(s["x"])
    if kind == "device":
        x, y = s["x"], s["y"]
        s["op"].matvec_device(x.data_ptr(), x.shape[0], y.data_ptr(), torch.cuda.current_stream().cuda_stream)
        return y
    m = s["m"]
    m.set_prefill_mode(s.get("mode", _lib.PREFILL_FP32))
    if kind == "tokens":
        return m.generate_greedy(s["prompt"], s["steps"])[0]
    if kind == "text":
        _, pieces = generate(s["model"], _tokenizer[0], s["text"], s["steps"], Random(s["seed"]), s["temperature"])
        # the text of each piece, as bytes; prompts of one length may differ by a token or two
        text = np.zeros(s["steps"], "S48")
        text[:len(pieces)] = [p.encode("utf-8") for p in pieces]
        return text.view(np.uint8)
    if kind == "prefill":  # the whole prompt, then the logits of its last token
        tokens = s["tokens"]
        m.prefill_chunks(tokens, 0, s["chunk"])
        return m.forward([s["last"]], [len(tokens)])
    # greedy tokens one at a time, as a streaming server asks for them, and the logits behind them
    token, ids = s["token"], []
    for i in range(s["n"]):
        token = m.decode_greedy(token, s["pos"] + i)
        ids.append(token)
    return {"ids": np.array(ids, np.int32), "logits": m.forward([token], [s["pos"] + s["n"]])}


# ---- what a pass cannot do without ----------------------------------------------------------------------------


def _matrix_bytes(n_in, n_out, group):
    if not group:
        return 4 * n_in * n_out
    groups = n_in // group
    return n_out * n_in // 2 + n_out * groups // 2 + n_out * groups * 4 + n_in * 4


def work(case):
    if case["kind"] in ("host", "device"):
        n_in, n_out, b = case["in"], case["out"], case["batch"]
        return {"bytes": _matrix_bytes(n_in, n_out, case["group"]) + 4 * b * (n_in + n_out), "flops": 2 * b * n_in * n_out}
    d = _dims(case)
    dim, hid, kv, L, g = d.dim, d.hidden_dim, d.kv_dim, d.n_layers, d.group_size
    shapes = [(dim, dim), (dim, kv), (dim, kv), (dim, dim), (dim, hid), (dim, hid), (hid, dim)]
    weights = L * sum(_matrix_bytes(i, o, g) for i, o in shapes)
    params = L * sum(i * o for i, o in shapes)
    head = 4 * dim * d.vocab_size

    def positions(p0, p1):  # rows of K and V that the positions p0..p1-1 read, and their arithmetic
        rows = (p1 * (p1 + 1) - p0 * (p0 + 1)) // 2
        return 8 * L * kv * rows, 4 * L * dim * rows

    if case["kind"] == "prefill":
        p0, n, steps = 0, case["tokens"] - 1, 1
    elif case["kind"] == "decode":
        p0, n, steps = case["cached"], 0, case["tokens"] + 1
    else:
        n = case["prompt"] if case["kind"] == "tokens" else 1 + case["words"]
        n = min(n, case["steps"]) - 1
        p0, steps = 0, case["steps"] - n
    step_bytes, step_flops = positions(p0 + n, p0 + n + steps)
    step_bytes += steps * (weights + head + 4 * dim)
    step_flops += 2 * steps * (params + dim * d.vocab_size)
    fill_bytes = weights + 4 * n * dim + 8 * L * kv * n if n > 0 else 0
    fill_flops = 2 * n * params + positions(0, n)[1] if n > 0 else 0
    return {"bytes": step_bytes + fill_bytes, "flops": step_flops + fill_flops}


def tolerance(case):
    if case["kind"] in ("host", "device"):  # one fp32 sum
        return {"rel": 1e-5, "max": 1e-4}
    if case["kind"] in ("tokens", "text"):  # token ids and text
        return "exact"
    if case["kind"] == "prefill" and case["mfma"]:  # activations rounded to fp16 once per projection, every layer
        return {"rel": 5e-3, "max": 3e-2}
    return {"rel": 5e-5, "max": 5e-4}  # fp32 through the whole stack
