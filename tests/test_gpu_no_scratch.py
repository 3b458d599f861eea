"""Calls that take scratch from the pool, without it: the quantized linear's
dequantizing loader and attention's rotation of K in its blocks give the bits of
the paths with scratch, eagerly and recorded; calls with no such path fail with
the reason; and an allocation error that is not a lack of memory is reported,
not worked around.  hb_fail_allocs makes the context's allocations fail on the
host; no memory is exhausted."""
import contextlib

import numpy as np
import pytest

from gpu_util import linear_kernel, to_host
from laya_hip import ffi as F
from laya_hip.host import HostTensor

pytestmark = pytest.mark.gpu
OUT_OF_MEMORY, LAUNCH_FAILURE = 2, 719  # hipErrorOutOfMemory, hipErrorLaunchFailure
CODE = {"f16": F.HB_F16, "bf16": F.HB_BF16}


@pytest.fixture(scope="module")
def b():
    from laya_hip.backend import HipBackend
    be = HipBackend(0)
    yield be
    be.destroy()


@contextlib.contextmanager
def failing(b, error):
    b.n.call("fail", "hb_fail_allocs", b.ctx, error)
    try:
        yield
    finally:
        b.n.call("fail", "hb_fail_allocs", b.ctx, 0)


def _up(b, a):
    a = np.ascontiguousarray(a)
    buf = b._malloc(a.nbytes)
    b.n.call("upload", "hb_upload", b.ctx, buf.ptr, a.ctypes.data, a.nbytes)
    return buf


def _bits(b, buf, n):
    out = np.empty(n, np.uint16)
    b.n.call("read", "hb_download", b.ctx, out.ctypes.data, buf.ptr, out.nbytes)
    return out


def _qlinear(b, M, N, K, bits, dtype, geglu=False):
    """A quantized linear through the C ABI: (call, its output's block, its values)."""
    rng = np.random.default_rng(M + N + K + bits)
    rows, G = (2 * N if geglu else N), -(-K // 64)
    x = to_host(rng.standard_normal((M, K)), dtype)
    held = [_up(b, x.data), _up(b, rng.integers(0, 256, (rows, K * bits // 8)).astype(np.uint8)),
            _up(b, (0.002 * (1 + rng.random((rows, G)))).astype(np.float16)),
            _up(b, rng.normal(0, 0.01, (rows, G)).astype(np.float16)), b._malloc(M * N * 2)]
    X, Q, S, Z, Y = held

    def call():
        b.n.call("qlinear", "hb_qlinear", b.ctx, CODE[dtype], X.ptr, K, Q.ptr, S.ptr, Z.ptr, 0, 0, 0, Y.ptr, N, M, N, K,
                 bits, 64, 1 if bits == 4 else 0, F.HB_EPI_GEGLU if geglu else 0)
    return call, Y, M * N, held


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M,N,K,bits,geglu", [(33, 200, 768, 8, False), (130, 768, 1152, 4, False), (130, 264, 768, 4, True),
                                              (2100, 3072, 384, 8, False), (2100, 2304, 320, 4, False)])
def test_quantized_linear_without_scratch(b, M, N, K, bits, geglu, dtype):
    assert not linear_kernel(b, M, N, K, geglu, bits).startswith("codes")  # with scratch: dequantized first
    call, Y, n, _held = _qlinear(b, M, N, K, bits, dtype, geglu)
    call()
    want = _bits(b, Y, n)
    b.n.call("fill", "hb_fill", b.ctx, Y.ptr, 0x7e, 2 * n)
    with failing(b, OUT_OF_MEMORY):
        call()
    np.testing.assert_array_equal(_bits(b, Y, n), want)


def test_recorded_quantized_linear_without_scratch(b):
    call, Y, n, _held = _qlinear(b, 96, 768, 768, 4, "f16")
    call()
    want = _bits(b, Y, n)
    ev = F.U(0)
    b.n.call("begin", "hb_capture_begin", b.ctx)
    with failing(b, OUT_OF_MEMORY):
        call()
        call()
    b.n.call("end", "hb_capture_end", b.ctx, F.C.byref(ev))
    for _ in range(3):
        b.n.call("fill", "hb_fill", b.ctx, Y.ptr, 0x7e, 2 * n)
        b.n.call("run", "hb_graph_launch", b.ctx, ev.value)
        np.testing.assert_array_equal(_bits(b, Y, n), want)
        call()
        np.testing.assert_array_equal(_bits(b, Y, n), want)
    b.n.call("destroy", "hb_graph_destroy", b.ctx, ev.value)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("L", [1025, 1100])
def test_attention_without_scratch(b, L, dtype):
    B, H = 1, 3
    rng = np.random.default_rng(L)
    q, k, v = (b.fromHost(to_host(rng.standard_normal((B, H, L, 64)), dtype)) for _ in range(3))
    out, n = b._malloc(B * H * L * 64 * 2), B * H * L * 64
    st = F.i64s((H * L * 64, L * 64, 64, 1))

    def call():
        b.n.call("sdpa", "hb_sdpa", b.ctx, CODE[dtype], b._ptr(q), st, b._ptr(k), st, b._ptr(v), st, 0,
                 F.i64s((0, 0, 0, 1)), 0, out.ptr, st, B, H, L, L, 64, 0.125, 10000.0, 10000.0)
    call()
    want = _bits(b, out, n)
    b.n.call("fill", "hb_fill", b.ctx, out.ptr, 0x7e, 2 * n)
    with failing(b, OUT_OF_MEMORY):
        call()
    np.testing.assert_array_equal(_bits(b, out, n), want)


def test_calls_that_need_scratch_say_so(b):
    call, _, _, _held = _qlinear(b, 4096, 64, 128, 8, "f16")
    with failing(b, OUT_OF_MEMORY), pytest.raises(F.HipError, match="out of device memory for the dequantized weight"):
        call()
    L = 128
    x, m = b.fromHost(to_host(np.ones((1, 1, L, 64)), "f16")), b.fromHost(HostTensor("bool", (1, L), np.ones((1, L), np.uint8)))
    out, st = b._malloc(L * 128), F.i64s((L * 64, L * 64, 64, 1))
    with failing(b, OUT_OF_MEMORY), pytest.raises(F.HipError, match="out of device memory for the mask summary"):
        b.n.call("sdpa", "hb_sdpa", b.ctx, F.HB_F16, b._ptr(x), st, b._ptr(x), st, b._ptr(x), st, b._ptr(m),
                 F.i64s((L, 0, 0, 1)), 0, out.ptr, st, 1, 1, L, L, 64, 0.125, 0.0, 0.0)
    call()  # memory again


@pytest.mark.parametrize("recording", [False, True])
def test_other_allocation_errors_are_reported(b, recording):
    """An error that is not a lack of memory (an earlier launch's, reported by the
    allocation) reaches the caller, also inside a recording and also where
    earlier calls of the recording left a block to share."""
    call, _, _, _held = _qlinear(b, 33, 200, 768, 8, "f16")
    if recording:
        b.n.call("begin", "hb_capture_begin", b.ctx)
        call()
    with failing(b, LAUNCH_FAILURE), pytest.raises(F.HipError, match="launch failure"):
        call()
    if recording:
        ev = F.U(0)
        b.n.call("end", "hb_capture_end", b.ctx, F.C.byref(ev))
        b.n.call("destroy", "hb_graph_destroy", b.ctx, ev.value)
    call()
