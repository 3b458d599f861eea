"""The small kernels around the layers at their edges: contiguous element-wise
ops in whole 16-byte vectors, softmax of short rows, and dot products of small
outputs in whole 4-element vectors."""
import numpy as np
import pytest

from gpu_util import max_rel, read32, rounded, to_host
from laya_hip.host import HostTensor
from oracle import cpu_ref as cr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def b():
    from laya_hip.backend import HipBackend
    be = HipBackend(0)
    yield be
    be.destroy()


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("n", [8, 2040, 2048, 2056, 70000])
def test_unary_vectors(b, dtype, n):
    """Bit for bit the general kernel's results, which n + 1 values take (not a
    whole number of 16-byte vectors), special values included."""
    rng = np.random.default_rng(n)
    x = rounded(rng.standard_normal(n + 1) * 3, dtype)
    x[:8] = [0.0, -0.0, np.inf, -np.inf, np.nan, 6e-8, 60000.0, -1.0]
    X, XL = b.fromHost(to_host(x[:n], dtype)), b.fromHost(to_host(x, dtype))
    ops = {"relu": b.relu, "gelu": b.gelu, "exp": b.exp, "log": b.log, "neg": b.neg, "abs": b.abs, "sqrt": b.sqrt,
           "rsqrt": b.rsqrt, "tanh": b.tanh, "sigmoid": b.sigmoid, "erf": b.erf, "scale": lambda t: b.scale(t, 0.3)}
    for name, f in ops.items():
        got, want = read32(b, f(X)).reshape(-1), read32(b, f(XL)).reshape(-1)[:n]
        np.testing.assert_array_equal(got, want, err_msg=name)
        np.testing.assert_array_equal(np.signbit(got)[got == 0], np.signbit(want)[want == 0], err_msg=name)


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("rows,n", [(1, 1), (63, 2), (64, 15), (65, 3), (1000, 7)])
def test_softmax_short_rows(b, dtype, rows, n):
    """Against f64: the f32 sum and quotient err by less than 16 roundings of
    2^-24 and the exponent's rounding (|x| < 20: 20 * 2^-23); 16-bit results
    add their own rounding (2^-11, 2^-8)."""
    rng = np.random.default_rng(rows * 16 + n)
    x = rounded(rng.standard_normal((rows, n)) * 3, dtype)
    x[0] = -np.inf if n == 1 else x[0]
    x[-1, n // 2] = -np.inf if n > 1 else 0.0
    got = read32(b, b.softmax(b.fromHost(to_host(x, dtype)), -1)).reshape(x.shape)
    z = x.astype(np.float64)
    with np.errstate(invalid="ignore"):
        e = np.exp(z - z.max(-1, keepdims=True))
        want = e / e.sum(-1, keepdims=True)
    tol = 4e-6 + {"f32": 0.0, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype]
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    assert np.nanmax(np.abs(got - want), initial=0.0) <= tol


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("M,N,K", [(1, 3, 256), (5, 7, 1024), (33, 3, 1028), (16, 257, 772), (2, 1, 2300), (3, 5, 261),
                                   (3, 5, 262)])
def test_dot_vectors(b, dtype, M, N, K):
    """K one vector short of, equal to and past a round of 1024 columns, and K
    that is no whole number of vectors (the scalar kernel).  f32: each output
    within K roundings of 2^-24 of its sum of absolute products; 16-bit: the
    GEMM bounds, and with GeGLU three roundings of 2^-11 (2^-8) and the f32 sums."""
    rng = np.random.default_rng(M + N + K)
    for geglu in (False, True):
        rows = 2 * N if geglu else N
        x = rounded(rng.standard_normal((M, K)), dtype)
        w = rounded(rng.standard_normal((rows, K)) * 0.05, dtype)
        bias = rounded(rng.standard_normal(rows), dtype)
        X, W, B = (b.fromHost(to_host(a, dtype)) for a in (x, w, bias))
        if geglu:
            got, want = read32(b, b.geglu(b.linear(X, W, B))), cr.geglu(cr.linear(x, w, bias))
            assert max_rel(got, want) <= {"f32": 2e-5, "f16": 2e-3, "bf16": 1.6e-2}[dtype]
            continue
        got = read32(b, b.linear(X, W, B)).astype(np.float64)
        if dtype == "f32":
            x6, w6 = x.astype(np.float64), w.astype(np.float64)
            bound = (K + 2) * 2.0 ** -24 * (np.abs(x6) @ np.abs(w6).T + np.abs(bias))
            assert (np.abs(got - (x6 @ w6.T + bias)) <= bound).all()
        else:
            assert max_rel(got, cr.linear(x, w, bias)) <= {"f16": 2e-3, "bf16": 8e-3}[dtype]


def test_bf16_stores_round_to_nearest_even(b):
    """f32 -> bf16 over every upper half and the lower halves around the tie:
    numpy's integer rounding bit for bit, subnormals and infinities included,
    and a NaN (whatever its payload's upper bits) stays a NaN."""
    hi = np.arange(65536, dtype=np.uint32) << 16
    bits = (hi[:, None] | np.array([0, 1, 0x7fff, 0x8000, 0x8001, 0xffff], np.uint32)).reshape(-1)
    got = np.asarray(b.read(b.cast(b.fromHost(HostTensor("f32", bits.shape, bits.view(np.float32))), "bf16")).data)
    got = got.view(np.uint16)
    nan = np.isnan(bits.view(np.float32))
    want = ((bits.astype(np.uint64) + 0x7fff + ((bits >> 16) & 1)) >> 16).astype(np.uint16)
    np.testing.assert_array_equal(got[~nan], want[~nan])
    assert ((got[nan] & 0x7fff) > 0x7f80).all()
