"""The f32 path (the loaders' default dtype): linear layers and attention on
the f32 matrix cores, and LayerNorm, against the oracle.

Bounds.  A sum of K products in f32, in any order, is off by at most
K * 2^-24 * sum|x||w| (plus the rounding of the value itself): the linear
tests hold each output to that.  Attention adds the softmax: a score off by d
changes a weight by a factor within e^(2d), so an output is off by at most
(2d + (Lk + 8) * 2^-23) * max|v|, d = 70 * 2^-24 * scale * max sum|q||k| (64
products, their scaling and the rotation)."""
import numpy as np
import pytest

from gpu_util import read32, to_host
from laya_hip import compose as C
from laya_hip import ffi as F
from laya_hip.host import HostQuantized, HostTensor, pack_quantized
from laya_hip.modernbert import attentionMasks
from oracle import cpu_ref as cr

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


@pytest.fixture(scope="module")
def b():
    from laya_hip.backend import HipBackend
    be = HipBackend(0)
    yield be
    be.destroy()


def _dev(b, *arrays):
    return [b.fromHost(to_host(a, "f32")) for a in arrays]


def _linear_bound(x, w, bias, resid, K):
    mag = cr.linear(np.abs(x), np.abs(w), None if bias is None else np.abs(bias))
    return (K + 3) * U * mag + (0 if resid is None else 2 * U * (mag + np.abs(resid)))


# tile edges (32 / 64 rows and columns, stages of 32 / 64 / 128), K remainders of 4, the three tile shapes
LINEAR = [(1, 4, 4), (31, 33, 100), (32, 32, 128), (33, 65, 132), (93, 2304, 768), (130, 768, 1152),
          (700, 1000, 260), (1025, 1537, 64), (2050, 2304, 72)]


@pytest.mark.parametrize("M,N,K", LINEAR)
@pytest.mark.parametrize("epi", ["plain", "bias+resid", "geglu"])
def test_linear_f32_tiles(b, M, N, K, epi):
    print(f"f32 linear M={M} N={N} K={K} {epi}", flush=True)
    rng = np.random.default_rng(M + N + K)
    rows = 2 * N if epi == "geglu" else N
    x = rng.standard_normal((M, K)).astype(np.float32)
    w = (rng.standard_normal((rows, K)) * 0.1).astype(np.float32)
    bias = None if epi == "plain" else rng.standard_normal(rows).astype(np.float32)
    r = rng.standard_normal((M, N)).astype(np.float32) if epi == "bias+resid" else None
    X, W = _dev(b, x, w)
    Bt = None if bias is None else _dev(b, bias)[0]
    y = b.linear(X, W, Bt)
    lin = cr.linear(x, w, bias)
    if epi == "geglu":
        # the fused epilogue gives the bits of the separate op on the same product
        fused = read32(b, b.geglu(b.linear(X, W, Bt)))
        b.flush(y)
        np.testing.assert_array_equal(fused, read32(b, b.geglu(y)))
        got, want, bound = read32(b, y), lin, _linear_bound(x, w, bias, None, K)
    elif r is not None:
        got, want, bound = read32(b, b.add(_dev(b, r)[0], y)), lin + r, _linear_bound(x, w, bias, r, K)
    else:
        got, want, bound = read32(b, y), lin, _linear_bound(x, w, None, None, K)
    assert np.all(np.abs(got - want) <= bound + 2 * U * np.abs(want))


@pytest.mark.parametrize("bits,mode", [(8, "symmetric"), (8, "affine"), (4, "symmetric"), (4, "affine")])
@pytest.mark.parametrize("M", [40, 600, 3000])
def test_quantized_linear_f32(b, bits, mode, M):
    """f32 activations on quantized weights, in each tile shape; a group of
    12 columns ends inside K stages."""
    N, K, g = 288, 264, 12
    rng = np.random.default_rng(M + bits)
    lo, hi = {(8, "symmetric"): (-127, 127), (4, "symmetric"): (-7, 7), (8, "affine"): (0, 255),
              (4, "affine"): (0, 15)}[(bits, mode)]
    q = rng.integers(lo, hi + 1, (N, K))
    s = rng.uniform(0.001, 0.01, (N, K // g)).astype(np.float16)
    z = rng.uniform(-0.1, 0.1, (N, K // g)).astype(np.float16) if mode == "affine" else None
    h = HostQuantized((N, K), bits, g, mode, pack_quantized(q, bits), HostTensor("f16", s.shape, s),
                      None if z is None else HostTensor("f16", z.shape, z))
    x = rng.standard_normal((M, K)).astype(np.float32)
    w = q * np.repeat(s.astype(np.float32), g, 1)
    if z is not None:
        w = w + np.repeat(z.astype(np.float32), g, 1)
    w = w.astype(np.float32)
    got = read32(b, C.quantized_linear(b, _dev(b, x)[0], C.upload_quantized(b, h, "f32")))
    want = cr.linear(x, w)
    assert np.all(np.abs(got - want) <= _linear_bound(x, w, None, None, K) + 2 * U * np.abs(want))


def _attention(b, B, H, L, kind, rope, strided=True, seed=0):
    rng = np.random.default_rng(seed + L)
    qkv = rng.standard_normal((B, L, 3, H, 64)).astype(np.float32)
    lens = rng.integers(max(1, L // 3), L + 1, B)
    valid = (np.arange(L)[None] < lens[:, None]).astype(np.uint8)
    mask = None
    if kind is not None:
        full, sliding = attentionMasks(valid, B, L, 128)
        mask = {"full": full, "sliding": sliding}.get(kind)
        if kind == "heads":  # a mask of its own per head
            m = (rng.random((B, H, L, L)) < 0.5).astype(np.uint8)
            m[..., 0] = 1
            mask = HostTensor("bool", m.shape, m)
    t = b.transpose(_dev(b, qkv)[0], [2, 0, 3, 1, 4])  # [3, B, H, L, 64] views, as ModernBert.layer takes them
    q, k, v = [b.reshape(p, [B, H, L, 64]) for p in b.split(t, 3, 0)]
    if rope:
        q, k = b.rope(q, rope), b.rope(k, rope)
    got = read32(b, b.sdpa(q, k, v, None if mask is None else b.fromHost(mask), 0.125))
    hq, hk, hv = [np.ascontiguousarray(p) for p in np.transpose(qkv, (2, 0, 3, 1, 4))]
    if rope:
        hq, hk = cr.rope(hq, rope), cr.rope(hk, rope)
    m = None if mask is None else np.broadcast_to(mask.data.reshape(mask.shape), (B, H, L, L))
    want = cr.sdpa(hq, hk, hv, m, 0.125)
    d = 70 * U * 0.125 * np.max(np.abs(hq).max(-1) * np.abs(hk).sum(-1).max())
    return got, want, (2 * d + (L + 8) * 2 * U) * np.abs(hv).max()


@pytest.mark.parametrize("L", [1, 31, 32, 33, 93, 130, 333, 512])
@pytest.mark.parametrize("kind", [None, "full", "sliding", "heads"])
def test_sdpa_f32(b, L, kind):
    """Key and query tiles of 32 with remainders, more and fewer key tiles
    than waves, with and without RoPE, and masks with and without a summary."""
    print(f"f32 sdpa L={L} {kind}", flush=True)
    got, want, tol = _attention(b, 2, 3, L, kind, 10000.0 if L % 2 else None)
    assert np.isfinite(got).all()
    assert np.max(np.abs(got - want)) <= tol


def test_sdpa_f32_non_finite(b):
    """A hidden key's inf / NaN reaches no query; a visible one reaches
    exactly the queries that see it; a query that sees no key is NaN."""
    B, H, L = 1, 2, 100
    rng = np.random.default_rng(3)
    q, k, v = (rng.standard_normal((B, H, L, 64)).astype(np.float32) for _ in range(3))
    m = np.ones((B, 1, L, L), np.uint8)
    m[0, 0, :, 70] = 0          # hidden from everybody
    m[0, 0, :50, 20] = 0        # hidden from the first half
    m[0, 0, 7] = 0              # sees nothing
    want = cr.sdpa(q, k, v, np.broadcast_to(m, (B, H, L, L)), 0.125)
    v[0, :, 70], k[0, :, 70] = np.nan, np.inf
    v[0, :, 20] = np.inf
    mask = b.fromHost(HostTensor("bool", m.shape, m))
    got = read32(b, b.sdpa(*_dev(b, q, k, v), mask, 0.125))
    assert np.isnan(got[0, :, 7]).all()
    assert not np.isfinite(got[0, :, 50:]).any()
    rows = [i for i in range(50) if i != 7]
    np.testing.assert_allclose(got[0, :, rows], want[0, :, rows], rtol=0, atol=1e-4)


@pytest.mark.parametrize("D", [256, 768, 2048])
@pytest.mark.parametrize("affine", ["none", "w", "w+b"])
def test_layernorm_f32(b, D, affine):
    """Rows of whole 256-value groups, row counts with a part-full last block,
    a strided input; bound: the two sums of D values and the few operations
    behind them, each value at most (D + 8) * 2^-24 of the row's largest."""
    rng = np.random.default_rng(D)
    for rows in (1, 5, 130):
        x = rng.standard_normal((rows, 2 * D)).astype(np.float32)
        w = rng.standard_normal(D).astype(np.float32) if affine != "none" else None
        bias = rng.standard_normal(D).astype(np.float32) if affine == "w+b" else None
        X = b.slice(_dev(b, x)[0], [0, D], [rows, 2 * D])
        got = read32(b, b.layerNorm(X, None if w is None else _dev(b, w)[0], None if bias is None else _dev(b, bias)[0],
                                    1e-5))
        want = cr.layer_norm(x[:, D:], w, bias, 1e-5)
        assert np.max(np.abs(got - want)) <= (D + 8) * U * np.abs(want).max()
