"""The operator on host arrays, whose x the host writes into device memory: the bits of the operator on device memory, also where more
calls run at once than there are windows, and with x changing from call to call."""
import ctypes
import os
import sys
import threading

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llama2.rs_amd"))
from llama2_rs import _lib, ops  # noqa: E402

pytestmark = pytest.mark.gpu


def operator(rng, n_in, n_out, group):
    groups = n_in // group
    return ops.QLinear(rng.integers(-2**31, 2**31, (n_out, n_in // 8), dtype=np.int64).astype(np.int32),
                       rng.integers(-2**31, 2**31, (n_out // 8, groups), dtype=np.int64).astype(np.int32),
                       rng.uniform(0.002, 0.02, (n_out, groups)).astype(np.float32),
                       np.argsort(rng.permutation(n_in) // group, kind="stable").astype(np.int32), group)


# one column and several that the matvec permutes itself; rows that a kernel permutes in front; batches, the longest that fits a megabyte,
# and one that does not
@pytest.mark.parametrize("n_in,n_out,group,batch", [(1024, 256, 32, 1), (4096, 512, 128, 1), (8192, 264, 64, 3), (13824, 256, 128, 2),
                                                    (13824, 256, 128, 3), (4096, 512, 128, 61), (8192, 512, 32, 32), (8192, 512, 32, 33)])
def test_host_arrays_give_the_bits_of_device_arrays(n_in, n_out, group, batch):
    import torch
    rng = np.random.default_rng(n_in + batch)
    ops_ = [operator(rng, n_in, n_out, group) for _ in range(6)]
    xs = rng.standard_normal((6, 3, batch, n_in)).astype(np.float32)
    want = np.empty((6, 3, batch, n_out), np.float32)
    if n_in * batch <= 1 << 20:
        y = torch.empty((batch, n_out), device="cuda")
        for i, q in enumerate(ops_):
            for j in range(3):
                x = torch.from_numpy(xs[i, j]).cuda()
                q.matvec_device(x.data_ptr(), batch, y.data_ptr(), torch.cuda.current_stream().cuda_stream)
                want[i, j] = y.cpu().numpy()
    bad = []

    def run(i):
        for r in range(12):
            if not np.array_equal(ops_[i].matvec(xs[i, r % 3]).view(np.uint32), want[i, r % 3].view(np.uint32)):
                bad.append((i, r))
    threads = [threading.Thread(target=run, args=(i,)) for i in range(6)]  # windows: four
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for q in ops_:
        q.close()


@pytest.mark.parametrize("batch", [23, 24])
def test_batches_on_both_sides_of_384_kb(batch):
    test_host_arrays_give_the_bits_of_device_arrays(4096, 512, 128, batch)


def windows_taken():
    n = ctypes.c_uint64()
    _lib.check(_lib.lib().l2_host_windows_taken(ctypes.byref(n)))
    return n.value


def test_windows_are_of_the_handle_s_device():
    """A handle of another device than the calling thread's current one has its x in pinned memory, which all devices read."""
    rng = np.random.default_rng(5)
    for n_in, batch in ((4096, 1), (4096, 2), (8192, 32)):
        q = operator(rng, n_in, 256, 64)
        x = rng.standard_normal((batch, n_in)).astype(np.float32)
        n = windows_taken()
        want = q.matvec(x)
        assert windows_taken() == n + 1
        _lib.check(_lib.lib().l2_qlinear_set_device(q.h, 1))
        assert np.array_equal(q.matvec(x).view(np.uint32), want.view(np.uint32)) and windows_taken() == n + 1
        q.close()
    q = operator(rng, 13824, 256, 128)  # permuted in front, and below the line
    n = windows_taken()
    q.matvec(rng.standard_normal((3, 13824)).astype(np.float32))
    assert windows_taken() == n
    q.close()
