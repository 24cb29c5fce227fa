"""Operator calls at the edges of what they accept: empty rows, empty contractions, and shapes on either side of a kernel's limit."""
import ctypes as C

import numpy as np
import pytest

from spy_amd import _lib as H
from tests import oracle_lib as O

B = C.byref


@pytest.mark.parametrize("exact", [0, 1])
@pytest.mark.parametrize("ne", [[0, 3], [0, 1], [0, 2, 2, 5]])
def test_norm_rms_of_empty_rows_launches_nothing(exact, ne):
    """NormRMS of rows without elements is accepted and does nothing, in either summation order: it returns before any device call, so the pointers
    here are never used (a launch would fail where there is no device and read before the rows where there is one)."""
    L = H.load()
    prev = L.spy_hip_set_exact_order(exact)
    try:
        assert L.spy_hip_op_norm_rms(None, B(H.tensor(4096, H.F32, ne)), B(H.tensor(8192, H.F32, ne)), 1e-5) == 0
        assert L.spy_hip_op_norm_rms(None, B(H.tensor(4096, H.F32, ne)), B(H.tensor(8192, H.F32, [0, 7])), 1e-5) == H.EINVAL
    finally:
        L.spy_hip_set_exact_order(prev)


@pytest.mark.gpu
@pytest.mark.parametrize("M,T,batch", [(1, 1, 1), (5, 3, 2), (300, 1, 32), (1030, 15, 1)])
def test_fp16_product_with_an_empty_contraction(M, T, batch):
    """fp16 rows of no elements give zeros, one, four and eight outputs per wave; the same with f32 activations is refused."""
    from tests.gpu_util import dev_empty, call
    H.init(0)
    L = H.load()
    prev = L.spy_hip_set_exact_order(0)
    try:
        w, out = dev_empty(256, 0xFF), dev_empty(batch * T * M * 4 + 64, 0xFF)
        tw, to = H.tensor(w, H.F16, [0, M, batch]), H.tensor(out, H.F32, [M, T, batch])
        call(L.spy_hip_op_matmul, None, B(tw), B(H.tensor(w, H.F16, [0, T, batch])), B(to), None, 0)
        got = out.download(np.uint32)
        assert (got[:batch * T * M] == 0).all() and (got[batch * T * M:] == 0xFFFFFFFF).all()
        assert L.spy_hip_op_matmul(None, B(tw), B(H.tensor(w, H.F32, [0, T, batch])), B(to), w.ptr, 256) == H.EINVAL
    finally:
        L.spy_hip_set_exact_order(prev)


@pytest.mark.gpu
def test_fp16_product_of_rows_beyond_32_bit_indices():
    """One output over a contraction of 2^30 + 67 fp16 elements: zeros but for elements at both ends and around 2^30."""
    from tests.gpu_util import dev_empty, call
    H.init(0)
    L = H.load()
    prev = L.spy_hip_set_exact_order(0)
    try:
        K = (1 << 30) + 67
        w, x, out = dev_empty(2 * K, 0), dev_empty(2 * K, 0x3C), dev_empty(64, 0xFF)          # x: 0x3C3C everywhere
        at = [0, 63, 12345, (1 << 30) - 1, 1 << 30, K - 1]
        vals = np.array([1, 2, 4, 8, 16, 32], np.float16)
        for i, v in zip(at, vals):
            b = np.array([v], np.float16)
            call(L.spy_hip_upload, w.ptr + 2 * i, b.ctypes.data, 2, None)
        call(L.spy_hip_op_matmul, None, B(H.tensor(w, H.F16, [K, 1])), B(H.tensor(x, H.F16, [K, 1])), B(H.tensor(out, H.F32, [1, 1])), None, 0)
        got = out.download(np.float32)
        assert got[0] == np.float32(63 * float(np.array([0x3C3C], np.uint16).view(np.float16)[0]))      # exact: 11 bits times 6
        assert (got[1:].view(np.uint32) == 0xFFFFFFFF).all()
    finally:
        L.spy_hip_set_exact_order(prev)


MOST_ROWS = 16 * 65535                       # activation rows that one launch of the packed-activation kernels takes


@pytest.mark.parametrize("order,wtype", [(0, H.Q4_K), (0, H.Q6_K), (1, H.Q4_K), (1, H.Q6_K)])
def test_matmul_scratch_beyond_the_packed_rows(order, wtype):
    """Beyond the rows that the packed-activation kernels take nothing is asked for but the Q8_0 activations of the kernels that run instead."""
    L = H.load()
    prev = L.spy_hip_set_exact_order(order)
    try:
        w = H.tensor(4096, wtype, [256, 4])
        for T in (MOST_ROWS + 1, (1 << 20) - 1, 1 << 20):
            assert L.spy_hip_op_matmul_scratch_size(B(w), B(H.tensor(4096, H.F32, [256, T]))) == T * 8 * 34
        assert L.spy_hip_op_matmul_scratch_size(B(w), B(H.tensor(4096, H.F32, [256, MOST_ROWS]))) > MOST_ROWS * 8 * 34
    finally:
        L.spy_hip_set_exact_order(prev)


@pytest.mark.gpu
@pytest.mark.parametrize("order,wtype", [(1, O.Q4_0), (1, O.Q4_K), (0, O.Q4_K), (0, O.Q6_K)])
@pytest.mark.parametrize("T", [MOST_ROWS, MOST_ROWS + 1, (1 << 20) - 1])
def test_matmul_of_about_a_million_rows(oracle, order, wtype, T):
    """One row more than one launch of the packed-activation kernels takes, and the rest up to 2^20: another kernel, not an error.  The rows repeat, so every
    output is known from the first 64; in the host's order with the oracle's bits."""
    from tests.gpu_util import assert_close, call, dev, dev_empty
    H.init(0)
    L = H.load()
    prev = L.spy_hip_set_exact_order(order)
    try:
        K, M, P = 256, 4, 64
        rng = np.random.default_rng(T + wtype)
        w = O.quantize(oracle, (rng.standard_normal((M, K)) * 0.02).astype(np.float32), wtype)
        x = rng.standard_normal((P, K)).astype(np.float32)
        want = O.matmul(oracle, w, wtype, M, K, x, nthread=4)
        dw, dx, out = dev(w), dev(np.resize(x, (T, K))), dev_empty(T * M * 4 + 64, 0xFF)
        tw, tx = H.tensor(dw, wtype, [K, M]), H.tensor(dx, H.F32, [K, T])
        need = L.spy_hip_op_matmul_scratch_size(B(tw), B(tx))
        scratch = dev_empty(need, 0xEE)
        call(L.spy_hip_op_matmul, None, B(tw), B(tx), B(H.tensor(out, H.F32, [M, T])), scratch.ptr, need)
        got = out.download(np.float32)
        assert (got[T * M:].view(np.uint32) == 0xFFFFFFFF).all()
        got = got[:T * M].reshape(T, M)
        if order == 1:
            assert np.array_equal(got.view(np.uint32), np.resize(want, (T, M)).view(np.uint32))
        else:
            assert_close(got, np.resize(want, (T, M)), "own order, %d rows" % T, tol=1e-5)
    finally:
        L.spy_hip_set_exact_order(prev)


@pytest.mark.gpu
@pytest.mark.parametrize("wtype,M,K,T", [(O.Q4_K, 36, 512, 40), (O.Q4_K, 4096, 512, 400), (O.Q4_K, 260, 11008, 400), (O.Q4_K, 1028, 256, 34), (O.Q4_K, 12288, 256, 129),
                                         (O.Q6_K, 36, 512, 40), (O.Q6_K, 4096, 512, 400), (O.Q6_K, 260, 11008, 400), (O.Q6_K, 1028, 256, 49), (O.Q4_0, 4096, 1024, 400)])
def test_own_order_result_does_not_depend_on_the_scratch_buffer(oracle, wtype, M, K, T):
    """MatMul in this backend's own order with the queried buffer, with room for the activations as Q8_0 blocks only (the packed rows go through it in pieces: one group of
    16, several, a last piece of one row), and from the fixed array of the entry point that allocates nothing: the same bits.  Too little is refused as before."""
    from tests.gpu_util import assert_close, call, dev, dev_empty
    H.init(0)
    L = H.load()
    prev = L.spy_hip_set_exact_order(0)
    try:
        rng = np.random.default_rng(M + K + T)
        w = O.quantize(oracle, (rng.standard_normal((M, K)) * 0.02).astype(np.float32), wtype)
        x = rng.standard_normal((T, K)).astype(np.float32)
        want = O.matmul(oracle, w, wtype, M, K, x, nthread=8)
        tw, tx, out = H.tensor(dev(w), wtype, [K, M]), H.tensor(dev(x), H.F32, [K, T]), dev_empty(T * M * 4 + 64, 0xFF)
        to = H.tensor(out, H.F32, [M, T])
        need, act, group = L.spy_hip_op_matmul_scratch_size(B(tw), B(tx)), T * K // 32 * 34, 36 * K
        assert need == (T + 15) // 16 * group
        scratch = dev_empty(need, 0xEE)
        got = {}
        for room in [need, act, max(act, group + 16), max(act, 2 * group + group // 2), need - 16, None]:
            out.fill(0xFF)
            if room is None: call(L.spy_hip_op_matmul_noalloc, None, B(tw), B(tx), B(to))
            else: call(L.spy_hip_op_matmul, None, B(tw), B(tx), B(to), scratch.ptr, room)
            r = out.download(np.float32)
            assert (r[T * M:].view(np.uint32) == 0xFFFFFFFF).all(), "nothing is written beyond the outputs"
            got[room] = r[:T * M]
        assert_close(got[need].reshape(T, M), want, "own-order matmul type %d %dx%d T=%d" % (wtype, M, K, T), tol=1e-5)
        for room, r in got.items():
            assert np.array_equal(r.view(np.uint32), got[need].view(np.uint32)), (room, need)
        assert L.spy_hip_op_matmul(None, B(tw), B(tx), B(to), scratch.ptr, act - 16) == H.ENOSPACE
    finally:
        L.spy_hip_set_exact_order(prev)
