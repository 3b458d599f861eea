"""The GEMM kernels below M = 4096 (16-bit weights): every tile shape of the ring
kernel at its edges, and the 128-row kernel where it takes a call with K % 64 ==
0, against the oracle at the GEMM bounds (max-rel 2e-3 f16, 8e-3 bf16: the
rounding of the stored result, 2^-11 and 2^-8, with room for the f32 sums) and
bit for bit against the other tiles and the large-M kernel, which run the same
MFMA steps in the same order.  hb_linear_kernel names the kernel each shape is
here for (on 256 CUs)."""
import numpy as np
import pytest

from gpu_util import linear_kernel, max_rel, read32, rounded, to_host
from laya_hip import ffi as F
from oracle import cpu_ref as cr

pytestmark = pytest.mark.gpu
TOL = {"f16": 2e-3, "bf16": 8e-3}

# (M, N, K): one 32 x 64 tile and less; a few with row and column remainders;
# K shorter than the ring and long
SHAPES = [(1, 8, 64, "ring 32x64"), (65, 72, 128, "ring 32x64"), (130, 200, 768, "ring 32x64"),
          (70, 136, 2112, "ring 32x64"), (520, 1032, 192, "ring 64x64"), (520, 1032, 2112, "ring 64x64 long"),
          (900, 1304, 192, "ring 128x64"), (1030, 2600, 64, "ring 64x64 three"), (3000, 2952, 64, "ring 64x64 three"),
          (4100, 768, 256, "ring 64x64 three"), (2100, 3080, 768, "ring 128x256"), (1030, 3000, 64, "mfma 128x64"),
          (2100, 2120, 128, "mfma 128x128")]
GEGLU_SHAPES = [(1, 8, 64, "ring 32x64"), (65, 40, 128, "ring 32x64"), (300, 648, 2112, "ring 32x64"),
                (520, 520, 192, "ring 64x64"), (520, 520, 2112, "ring 64x64 long"), (900, 648, 192, "ring 128x64"),
                (1030, 1304, 64, "ring 64x64 three"), (1030, 1504, 64, "mfma 128x64"), (2100, 1064, 128, "mfma 128x128"),
                (4200, 520, 128, "ring 128x256")]


@pytest.fixture(scope="module")
def b():
    from laya_hip.backend import HipBackend
    be = HipBackend(0)
    yield be
    be.destroy()


def _operands(b, rng, M, N, K, dtype, geglu):
    rows = 2 * N if geglu else N
    x = rounded(rng.standard_normal((M, K)), dtype)
    w = rounded(rng.standard_normal((rows, K)) * 0.05, dtype)
    bias = rounded(rng.standard_normal(rows), dtype)
    r = rounded(rng.standard_normal((M, N)), dtype)
    return (x, w, bias, r), [b.fromHost(to_host(a, dtype)) for a in (x, w, bias, r)]


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M,N,K,kernel", SHAPES)
def test_ring_tiles(b, M, N, K, kernel, dtype):
    assert linear_kernel(b, M, N, K) == kernel
    print(f"ring M={M} N={N} K={K} {dtype}", flush=True)
    rng = np.random.default_rng(M + N + K)
    (x, w, bias, r), (X, W, B, R) = _operands(b, rng, M, N, K, dtype, False)
    lin = cr.linear(x, w, bias)
    got = read32(b, b.linear(X, W, B))
    assert max_rel(got, lin) <= TOL[dtype]
    # the residual epilogue adds to the rounded product and rounds once more
    np.testing.assert_array_equal(read32(b, b.add(R, b.linear(X, W, B))), rounded(got + r, dtype))
    # a row's bits do not depend on the call's other rows
    for i in sorted({0, M // 2, M - 1}):
        xi = b.fromHost(to_host(x[i:i + 1], dtype))
        np.testing.assert_array_equal(read32(b, b.linear(xi, W, B))[0], got[i])


@pytest.mark.parametrize("M,N,K,kernel", GEGLU_SHAPES)
def test_ring_geglu(b, M, N, K, kernel):
    assert linear_kernel(b, M, N, K, geglu=True) == kernel
    """Value and gate columns in one tile, in waves of their own: the bits of
    the separate op on the linear's output; N not a multiple of the tile's
    value columns (but of 8: rows of other lengths take the SIMT kernel, whose
    GELU is libm's: N = 650 or 1500 is no call of this kernel)."""
    rng = np.random.default_rng(M + N)
    _, (X, W, B, R) = _operands(b, rng, M, N, K, "f16", True)
    y = b.linear(X, W, B)
    fused = b.geglu(b.linear(X, W, B))
    b.flush(y, fused)
    want = b.geglu(y)
    np.testing.assert_array_equal(read32(b, fused), read32(b, want))


@pytest.mark.parametrize("M,kernel", [(100, "ring 32x64"), (250, "ring 64x64"), (700, "ring 128x64"), (1030, "ring 64x64 three"),
                                      (3000, "ring 128x256"), (2048, "mfma 128x64"), (1536, "mfma 128x64"), (4000, "ring 64x64 three")])
def test_ring_bits_equal_large_m(b, M, kernel):
    """2304 x 768 weights: each tile shape's rows are the large-M kernel's."""
    assert linear_kernel(b, M, 2304, 768) == kernel
    assert linear_kernel(b, 6144, 2304, 768) == "arow 192"
    rng = np.random.default_rng(M)
    (x, w, _, _), (X, W, _, _) = _operands(b, rng, M, 2304, 768, "f16", False)
    big = b.fromHost(to_host(np.resize(x, (6144, 768)), "f16"))
    np.testing.assert_array_equal(read32(b, b.linear(X, W)), read32(b, b.linear(big, W))[:M])


@pytest.mark.parametrize("M,N,K,geglu", [(33, 64, 128, 0), (130, 768, 768, 0), (130, 1152, 768, 1), (4100, 768, 256, 0),
                                         (4100, 48, 128, 1)])
def test_ring_panel_operands(b, M, N, K, geglu):
    """x read from and y written in panel order through the C ABI, bit for bit
    the row-major call."""
    rng = np.random.default_rng(M + N)
    _, (X, W, B, _) = _operands(b, rng, M, N, K, "f16", bool(geglu))
    xp, y, yp, yu = (b._malloc((M + 31) // 32 * 32 * max(K, N) * 2) for _ in range(4))
    fl = F.HB_EPI_BIAS | (F.HB_EPI_GEGLU if geglu else 0)
    b.n.call("pack", "hb_panel_pack", b.ctx, b._ptr(X), K, xp.ptr, M, K)

    def call(xptr, yptr, flags):
        b.n.call("linear", "hb_linear", b.ctx, F.HB_F16, xptr, K, b._ptr(W), b._ptr(B), 0, 0, yptr, N, M, N, K, flags)
        return yptr

    def bits(ptr):
        out = np.empty(M * N, np.uint16)
        b.n.call("read", "hb_download", b.ctx, out.ctypes.data, ptr, out.nbytes)
        return out
    want = bits(call(b._ptr(X), y.ptr, fl))
    np.testing.assert_array_equal(bits(call(xp.ptr, yp.ptr, fl | F.HB_X_PANEL)), want)
    call(xp.ptr, yp.ptr, fl | F.HB_X_PANEL | F.HB_Y_PANEL)
    b.n.call("unpack", "hb_panel_unpack", b.ctx, yp.ptr, yu.ptr, N, M, N)
    np.testing.assert_array_equal(bits(yu.ptr), want)


@pytest.mark.parametrize("M,N,K,geglu", [(3, 48, 128, 0), (33, 128, 64, 0), (35, 32, 192, 1)])
def test_panel_output_of_rows_far_apart(b, M, N, K, geglu):
    """A row-major x with 2^22 or more elements between its rows (past 32-bit byte
    offsets within a tile) and y in panel order: the bits of the dense call."""
    rng = np.random.default_rng(M)
    _, (X, W, B, _) = _operands(b, rng, M, N, K, "f16", bool(geglu))
    ldx = 1 << 22
    far, y, yp, yu = (b._malloc(n) for n in (((M - 1) * ldx + K) * 2, M * N * 2, (M + 31) // 32 * 32 * N * 2, M * N * 2))
    for i in range(M):
        b.n.call("copy", "hb_copy", b.ctx, far.ptr + 2 * i * ldx, b._ptr(X) + 2 * i * K, 2 * K)
    fl = F.HB_EPI_BIAS | (F.HB_EPI_GEGLU if geglu else 0)
    for x, ld, out, flags in ((b._ptr(X), K, y, fl), (far.ptr, ldx, yp, fl | F.HB_Y_PANEL)):
        b.n.call("linear", "hb_linear", b.ctx, F.HB_F16, x, ld, b._ptr(W), b._ptr(B), 0, 0, out.ptr, N, M, N, K, flags)
    b.n.call("unpack", "hb_panel_unpack", b.ctx, yp.ptr, yu.ptr, N, M, N)
    got = [np.empty(M * N, np.uint16) for _ in range(2)]
    for g, t in zip(got, (yu, y)):
        b.n.call("read", "hb_download", b.ctx, g.ctypes.data, t.ptr, g.nbytes)
    np.testing.assert_array_equal(got[0], got[1])
