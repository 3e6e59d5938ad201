"""How the matvec launcher cuts one matrix into blocks (no GPU needed: the plan for 256 compute units, nothing is launched)."""
import ctypes as C
import re

import pytest

from llama2_rs import _lib


def _behind_the_loop(out, rows_per_block, streams, in_flight):
    """The rows that stand behind the kernel's loop over whole tiles, as ranges."""
    found = []
    for first in range(0, out, rows_per_block):
        rows = min(rows_per_block, out - first)
        whole = -(-rows // streams) // in_flight * in_flight * streams
        if whole < rows:
            found.append((first + whole, first + rows))
    return tuple(found)


# Rows behind the loop are rounded otherwise than rows in it, and a column's bits may not depend on the columns beside it, nor on
# whether the kernel permutes x itself: the same rows whatever the batch and the form.  One number of inputs for each number of
# waves per row.
@pytest.mark.parametrize("n_in", [32, 2048, 4096, 5120, 8192, 11008, 13824, 16384, 28672])
def test_columns_have_the_same_rows_behind_the_loop(n_in):
    plan = _lib.lib().l2_qlinear_plan
    name, geo = C.create_string_buffer(160), (C.c_int32 * 4)()
    forms = (1, 0) if n_in <= 8192 else (0,)
    known, wrong = {}, []
    for out in list(range(8, 8200, 8)) + list(range(8200, 32769, 328)):
        want = None
        for batch in (1, 2, 3, 5, 8, 13, 16):
            for natural in forms:
                _lib.check(plan(n_in, out, 32, batch, natural, name, 160, geo))
                key = (name.value, geo[2], out)
                if key not in known:
                    m = re.fullmatch(rb"q4_stream_kernel<32, (\d+), (\d+), false, \d, (\d+), (true|false)>", name.value)
                    assert m and m[4] == (b"true" if natural else b"false"), name.value
                    assert geo[1] == 64 * int(m[1]) * int(m[2])
                    known[key] = _behind_the_loop(out, geo[2], int(m[2]), int(m[3]))
                if want is None:
                    want = known[key]
                elif known[key] != want:
                    wrong.append((out, batch, natural))
        known.clear()
    assert not wrong, (len(wrong), wrong[:8])
