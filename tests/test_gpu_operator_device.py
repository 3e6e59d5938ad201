"""l2_qlinear_matvec_device on buffers as a caller may lay them out, against the same operator on host arrays."""
import ctypes as C

import numpy as np
import pytest

from llama2_rs import checkpoint as ck
from tests.test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from llama2_rs import ops as o, _lib
    assert _lib.lib().l2_device_count() >= 1, "no HIP device: the GPU tests cannot run"
    return o


# y over x: in place, shifted either way, sharing four elements, and touching without sharing any.  One column (which
# takes one launch only where nothing is shared), a few (the matvec kernels) and a batch (the matrix cores).
@pytest.mark.parametrize("n_in,n_out,G", [(1024, 1024, 32), (4096, 4096, 128), (8192, 1024, 64), (2816, 8448, 128)])
@pytest.mark.parametrize("B", [1, 3, 24])
def test_result_over_the_input(ops, n_in, n_out, G, B):
    hip = _Hip()
    rng = np.random.default_rng(n_in + B)
    q = ops.QLinear(*ck.synth_qlinear(rng, n_in, n_out, G, act_order=True), G)
    x = rng.standard_normal((B, n_in)).astype(np.float32)
    want = q.matvec(x)
    nx, ny = B * n_in, B * n_out
    image = np.full(nx + 2 * ny, np.nan, np.float32)
    image[ny:ny + nx] = x.reshape(-1)
    for shift in (0, 4, -4, nx // 2, nx - 4, 4 - ny, nx, -ny):
        buf = hip.upload(image)
        q.matvec_device(buf + 4 * ny, B, buf + 4 * (ny + shift))
        np.testing.assert_array_equal(hip.download(buf + 4 * (ny + shift), (B, n_out)), want, err_msg=f"shift {shift}")
    q.close()
    hip.close()


# x and y at addresses that are multiples of four bytes and of nothing more, and nothing written beside y: one column, a
# few, and batches in one K slice (17160 outputs; 4128 inputs: in several runs of groups) and in several
@pytest.mark.parametrize("n_in,n_out,G,batches", [(1024, 264, 32, (1, 3, 250)), (4096, 4104, 128, (1, 3, 5, 40, 250)),
                                                  (8192, 8192, 64, (1, 2, 100)), (1024, 17160, 32, (250,)), (4128, 17160, 32, (250,))])
def test_any_float_address(ops, n_in, n_out, G, batches):
    hip = _Hip()
    rng = np.random.default_rng(n_in)
    q = ops.QLinear(*ck.synth_qlinear(rng, n_in, n_out, G, act_order=True), G)
    for B in batches:
        x = rng.standard_normal((B, n_in)).astype(np.float32)
        want = q.matvec(x)
        for dx, dy in ((1, 0), (0, 1), (2, 3), (3, 2)):
            px = hip.upload(np.concatenate([np.full(dx, np.nan, np.float32), x.reshape(-1)]))
            py = hip.upload(np.full(dy + want.size + 4, 7.0, np.float32))
            q.matvec_device(px + 4 * dx, B, py + 4 * dy)
            got = hip.download(py, (dy + want.size + 4,))
            np.testing.assert_array_equal(got[dy:dy + want.size].reshape(want.shape), want, err_msg=f"{B} {dx} {dy}")
            assert np.all(got[:dy] == 7.0) and np.all(got[dy + want.size:] == 7.0)
    q.close()
    hip.close()


# The operator on host arrays scatters x from pinned memory where the one on device memory gathers it: the same bits.  Rows that end
# inside a thread's first or second piece and with half a K step (4128), in one part and in two (512 KiB), even and odd; long rows for
# the matvec kernels (12320).
@pytest.mark.parametrize("n_in,n_out,G,batches", [(4128, 4104, 32, (4, 15, 16, 17, 31, 32, 61)), (2048, 4104, 64, (31, 32, 33, 63, 64, 65, 128)),
                                                  (12320, 264, 32, (1, 2, 3)), (28672, 1024, 64, (1, 3, 9))])
def test_host_input_is_the_device_input(ops, n_in, n_out, G, batches):
    hip = _Hip()
    rng = np.random.default_rng(n_in)
    q = ops.QLinear(*ck.synth_qlinear(rng, n_in, n_out, G, act_order=True), G)
    for B in batches:
        x = (rng.standard_normal((B, n_in)) * 10.0 ** rng.integers(-6, 7, (B, n_in))).astype(np.float32)
        px, py = hip.upload(x), hip.empty(4 * B * n_out)
        q.matvec_device(px, B, py)
        np.testing.assert_array_equal(q.matvec(x), hip.download(py, (B, n_out)), err_msg=str(B))
    q.close()
    hip.close()


# The same where the matvec kernel permutes x, which is then copied in one part and in two: every column by itself.
@pytest.mark.parametrize("n_in,G,batches", [(2048, 64, (63, 64, 65)), (8192, 128, (15, 17))])
def test_host_columns_are_the_device_columns(ops, n_in, G, batches):
    from llama2_rs import _lib
    hip = _Hip()
    rng = np.random.default_rng(n_in)
    q = ops.QLinear(*ck.synth_qlinear(rng, n_in, 264, G, act_order=True), G)
    q.set_mode(_lib.PREFILL_COLUMNS)
    for B in batches:
        x = rng.standard_normal((B, n_in)).astype(np.float32)
        px, py = hip.upload(x), hip.empty(4 * B * 264)
        q.matvec_device(px, B, py)
        np.testing.assert_array_equal(q.matvec(x), hip.download(py, (B, 264)), err_msg=str(B))
    q.close()
    hip.close()


# what one column enqueues (captured, not run): one kernel where x and y are apart, a gather in front where they meet
def test_one_launch_only_apart(ops):
    hip = _Hip()
    rt = hip.rt
    q = ops.QLinear(*ck.synth_qlinear(np.random.default_rng(2), 4096, 1024, 128, act_order=True), 128)
    buf, stream = hip.empty(4 * (4096 + 2 * 1024)), C.c_void_p()
    assert rt.hipStreamCreate(C.byref(stream)) == 0
    for shift, nodes in ((0, 2), (-1024, 1), (-1020, 2), (2048, 2), (4092, 2), (4096, 1)):
        graph, n = C.c_void_p(), C.c_size_t()
        assert rt.hipStreamBeginCapture(stream, 0) == 0            # hipStreamCaptureModeGlobal
        try:
            q.matvec_device(buf + 4 * 1024, 1, buf + 4 * (1024 + shift), stream=stream.value)
        finally:
            assert rt.hipStreamEndCapture(stream, C.byref(graph)) == 0
        assert rt.hipGraphGetNodes(graph, None, C.byref(n)) == 0 and n.value == nodes, shift
        assert rt.hipGraphDestroy(graph) == 0
    assert rt.hipStreamDestroy(stream) == 0
    q.close()
    hip.close()
