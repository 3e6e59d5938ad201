"""How the token kernel deals a model's rows over its blocks and waves (l2_token_plan): no device needed."""
import ctypes
import os
import re
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llama2.rs_amd"))
from llama2_rs import _lib, ops  # noqa: E402
from llama2_rs.checkpoint import Dims  # noqa: E402


def dims(dim, hid, heads, kv, group):
    return Dims(dim=dim, hidden_dim=hid, n_layers=1, n_heads=heads, n_kv_heads=kv, vocab_size=256, seq_len=64, group_size=group)


def plan(d):
    info = np.zeros(4, np.int32)
    walks = np.zeros(4 * 1024 * 16 * 16, np.int32)
    _lib.check(_lib.lib().l2_token_plan(ctypes.byref(ops.to_cdims(d)), walks.ctypes.data, walks.size, info.ctypes.data))
    return info, walks[:4 * info[1] * info[2] * 16].reshape(4, info[1], info[2], 16)


def rows_behind(n_in, out, group, pair, norm):
    """Rows that stand behind the loop of the launch that does these matrices by itself, read off its kernel and geometry."""
    outs = np.array(out, np.int32)
    name, geo = ctypes.create_string_buffer(200), np.zeros(4, np.int32)
    _lib.check(_lib.lib().l2_q4_plan(n_in, outs.ctypes.data, len(out), group, pair, norm, name, 200, geo.ctypes.data))
    _, _, streams, _, mode, p, _ = re.match(r"q4_stream_kernel<(.*)>", name.value.decode()).group(1).split(", ")
    streams, p, unit = int(streams), int(p), int(geo[2])
    if mode == "3":
        streams, unit = streams // 2, unit // 2

    def behind(o, n_out):
        n = min(unit, n_out - o // unit * unit)
        return o % unit >= (n + streams - 1) // (p * streams) * (p * streams)
    return [np.array([behind(o, n) for o in range(n)]) for n in out]


@pytest.mark.parametrize("shape", [(512, 768, 4, 2, 32), (1024, 2816, 8, 2, 64), (1536, 4480, 12, 12, 128), (2048, 13824, 16, 4, 64),
                                   (3072, 8192, 24, 3, 64), (4096, 11008, 32, 32, 128), (5120, 13824, 40, 40, 128),
                                   (8192, 14336, 64, 8, 64), (4096, 11008, 32, 4, 32), (1152, 32, 9, 9, 32)])
def test_every_row_is_walked_once_and_rounded_as_its_launch_rounds_it(shape):
    dim, hid, heads, kv, group = shape
    info, w = plan(dims(*shape))
    assert info[0] == 1 and info[2] == 16 and info[3] <= 152 * 1024
    kvd = dim // heads * kv
    phases = [(dim, [dim, kvd, kvd], [0, 1, 2], 0, 1), (dim, [dim], [3], 0, 0), (dim, [hid, hid], [4, 5], 1, 1), (hid, [dim], [6], 0, 0)]
    for p, (n_in, outs, mats, pair, norm) in enumerate(phases):
        chunks = n_in // 32
        kslices = (chunks + 63) // 64
        want = rows_behind(n_in, outs, group, pair, norm)
        seen = {(m, k): np.zeros(o, int) for m, o in zip(mats, outs) for k in range(kslices)}
        where = {}
        for b in range(info[1]):
            for v in range(16):
                mat, first, stride, last, steps, r0, n, part_row, kslice, c, groups = w[p, b, v, :11]
                behind, early = int(w[p, b, v, 11]) & 0xFFFFFFFF, w[p, b, v, 12]
                assert c == chunks and groups == n_in // group and steps <= 32 and n <= 1024 and 0 <= kslice < kslices
                assert steps == 0 or (first + (steps - 1) * stride <= last and last == r0 + n - 1 and first >= r0)
                assert part_row == (n if mat == 5 else 0) or steps == 0
                looped = int(max(steps - 1, 0)) // 3 * 3  # kTokenRows
                assert early == (behind & ((1 << looped) - 1) != 0)
                m = mats.index(mat)
                for i in range(steps):
                    o = first + i * stride
                    seen[mat, kslice][o] += 1
                    assert (behind >> i & 1) == want[m][o], (p, mat, o)
                    assert where.setdefault((mat, o), b) == b  # all slices of a row in one block
        assert all((s == 1).all() for s in seen.values())
    # the residual stream of a block's rows stays in it from wo to w2
    assert (w[1, :, 0, 5:7] == w[3, :, 0, 5:7]).all()


def test_models_that_it_does_not_take():
    for shape in [(512, 768, 4, 2, 0),            # fp32 weights
                  (512, 768, 8, 2, 32),           # heads of 64
                  (128 * 65, 1024, 65, 65, 32),   # more slices of heads than blocks, rows of more than 8192 inputs
                  (8192, 28672, 64, 8, 64),       # 56 rows of w1 for a wave
                  (3 * 128 * 4, 1024, 12, 4, 32)]:  # three query heads per kv head
        d = dims(*shape)
        info = np.zeros(4, np.int32)
        rc = _lib.lib().l2_token_plan(ctypes.byref(ops.to_cdims(d)), None, 0, info.ctypes.data)
        assert rc != 0 or info[0] == 0, shape


@pytest.mark.parametrize("shape", [(512, 768, 4, 2, 32), (1024, 2816, 8, 2, 64), (2048, 28672, 16, 16, 64), (4096, 11008, 32, 32, 128)])
def test_a_launch_with_blocks_left_out_stays_within_its_buffers(shape):
    """The kernel reads the plan by its grid, so all blocks are launched: those that stay have their own rows in every phase, the others none,
    and nothing is written behind a vector or behind the LDS."""
    dim, hid, heads, kv, _ = shape
    d = dims(*shape)
    info, w = plan(d)
    out = np.array([dim, dim // heads * kv, dim // heads * kv, dim, hid, hid, dim])
    for missing in (0, 1, 5, int(info[1]) - 1):
        rows = np.zeros(4 * info[1] * 16 * 4, np.int32)
        _lib.check(_lib.lib().l2_token_rows(ctypes.byref(ops.to_cdims(d)), missing, rows.ctypes.data, rows.size))
        r, stay = rows.reshape(4, info[1], 16, 4), info[1] - missing
        assert (r[:, :stay, :, :3] == w[:, :stay][..., [4, 5, 6]]).all() and (r[:, stay:, :, [0, 2]] == 0).all()
        assert (r[..., 1] >= 0).all() and (r[..., 2] >= 0).all()
        reach, here = r[..., 1] + r[..., 2], r[..., 2] > 0
        assert (reach[here] <= out[w[..., 0]][here]).all()
        assert (r[..., 3] <= info[3]).all()
    # all blocks of the plan, whatever is left out
    source = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llama2.rs_amd", "csrc", "host.cpp")
    assert re.findall(r"token_layers_launch\(([^)]*)\)", open(source).read()) == ["a, t.grid, t.lds, t.eight, st"]
