"""Transfers through pinned host memory that are only queued on a stream, and the error flag that comes with a result."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 4096 * 16 + 3, 300000])
def test_pinned_round_trip_and_error_flag(n):
    from spy_amd import _lib as H
    from tests.gpu_util import dev, dev_empty, call
    H.init(0)
    L = H.load()
    stream, up, down = C.c_void_p(), C.c_void_p(), C.c_void_p()
    call(L.spy_hip_stream_create, C.byref(stream))
    call(L.spy_hip_host_alloc, C.byref(up), n)
    call(L.spy_hip_host_alloc, C.byref(down), n + 64)
    data = np.random.default_rng(n).integers(0, 256, n).astype(np.uint8)
    C.memmove(up, data.ctypes.data, n)
    C.memset(down, 0xEE, n + 64)
    buf = dev_empty(n + 64, 0xFF)
    table, ids, row = dev(np.zeros((2, 4), np.float32)), dev(np.array([2], np.int32)), dev_empty(16)       # row 2 of a table of two
    flag = C.c_int()
    call(L.spy_hip_take_error, C.byref(flag))
    call(L.spy_hip_upload_pinned, buf.ptr, up, n, stream)
    call(L.spy_hip_op_get_row, stream, C.byref(H.tensor(table, H.F32, [4, 2])), C.byref(H.tensor(ids, H.I32, [1])), C.byref(H.tensor(row, H.F32, [4, 1])))
    for want in (1, 0):
        call(L.spy_hip_download_pinned, down.value + 64, buf.ptr, n, down, stream)
        call(L.spy_hip_sync, stream)
        got = np.ctypeslib.as_array((C.c_uint8 * (n + 64)).from_address(down.value)).copy()
        assert got[:4].view(np.int32)[0] == want, "the flag is handed out once"
        assert (got[4:64] == 0xEE).all() and np.array_equal(got[64:], data)
    assert (buf.download(np.uint8)[n:] == 0xFF).all(), "nothing is written beyond the bytes"
    call(L.spy_hip_host_free, up)
    call(L.spy_hip_host_free, down)
    call(L.spy_hip_stream_destroy, stream)
