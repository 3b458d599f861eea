"""16-bit attention on either side of 1024 keys (16-query waves up to there,
32-query waves from there): tile remainders, masks whose rows are and are not
16-byte aligned, RoPE on the way to LDS and in a pass of its own, row-major and
panel-order output, through the contract and the C ABI.

Bounds: max-rel 5e-3 (f16) and 2e-2 (bf16) against the oracle on the same
rounded inputs, the bounds of the 16-query kernel's tests (half an ulp of the
weights and of the output, 2^-11 and 2^-8, with room for the sums)."""
import numpy as np
import pytest

from gpu_util import max_rel, read32, rounded, to_host
from laya_hip import ffi as F
from laya_hip.host import HostTensor
from laya_hip.modernbert import attentionMasks
from oracle import cpu_ref as cr

pytestmark = pytest.mark.gpu
TOL = {"f16": 5e-3, "bf16": 2e-2}


@pytest.fixture(scope="module")
def b():
    from laya_hip.backend import HipBackend
    be = HipBackend(0)
    yield be
    be.destroy()


def _views(b, qkv, dtype):
    """q, k, v [B, H, L, 64] views of one [B, L, 3, H, 64] tensor, as ModernBert.layer takes them."""
    B, L, _, H, _ = qkv.shape
    t = b.transpose(b.fromHost(to_host(qkv, dtype)), [2, 0, 3, 1, 4])
    return [b.reshape(p, [B, H, L, 64]) for p in b.split(t, 3, 0)]


def _mask(rng, B, L, kind):
    lens = rng.integers(max(1, L // 3), L + 1, B)
    lens[0] = L
    valid = (np.arange(L)[None] < lens[:, None]).astype(np.uint8)
    full, sliding = attentionMasks(valid, B, L, 128)
    return {"full": full, "sliding": sliding, None: None}[kind]


CASES = [(385, None, 0), (448, "full", 1), (449, "full", 1), (577, "full", 0), (1023, "full", 1), (1024, "full", 1),
         (1025, "sliding", 1), (1040, "sliding", 1), (1027, "sliding", 0), (1090, None, 1), (1025, "full", 0),
         (1088, "full", 1), (1217, "full", 1), (1663, None, 0)]


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("L,kind,rope", CASES)
def test_sdpa_long(b, L, kind, rope, dtype):
    print(f"sdpa L={L} {kind} rope={rope} {dtype}", flush=True)
    B, H = 2, 3
    rng = np.random.default_rng(L)
    qkv = rng.standard_normal((B, L, 3, H, 64)).astype(np.float32)
    mask = _mask(rng, B, L, kind)
    q, k, v = _views(b, qkv, dtype)
    M = None if mask is None else b.fromHost(mask)
    qr, kr = (b.rope(q, 10000.0), b.rope(k, 10000.0)) if rope else (q, k)
    got = read32(b, b.sdpa(qr, kr, v, M, 0.125))
    hq, hk, hv = [rounded(np.ascontiguousarray(p), dtype) for p in np.transpose(qkv, (2, 0, 3, 1, 4))]
    if rope:
        hq, hk = rounded(cr.rope(hq, 10000.0), dtype), rounded(cr.rope(hk, 10000.0), dtype)
    m = None if mask is None else np.broadcast_to(mask.data.reshape(mask.shape), (B, 1, L, L))
    want = cr.sdpa(hq, hk, hv, None if m is None else np.broadcast_to(m, (B, H, L, L)), 0.125)
    assert np.isfinite(got).all()
    assert max_rel(got, want) <= TOL[dtype]
    if rope:
        # rotated beforehand, rounded the same: the same bits
        sep = [b.rope(t, 10000.0) for t in (q, k)]
        for t in sep:
            b.flush(t)
        np.testing.assert_array_equal(got, read32(b, b.sdpa(sep[0], sep[1], v, M, 0.125)))
    # a sequence alone gives the bits it has in the batch
    q1, k1, v1 = _views(b, qkv[1:], dtype)
    if rope:
        q1, k1 = b.rope(q1, 10000.0), b.rope(k1, 10000.0)
    M1 = None if mask is None else b.fromHost(HostTensor("bool", (1,) + mask.shape[1:], mask.data.reshape(mask.shape)[1:]))
    np.testing.assert_array_equal(got[1:], read32(b, b.sdpa(q1, k1, v1, M1, 0.125)))


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("L", [128, 385, 512, 1024, 1025, 1100])
def test_bits_do_not_depend_on_the_form_of_the_mask(b, L, dtype):
    """A padding mask as one row per sequence and spelt out per query, and an
    all-true mask and none, give the same bits: the kernel is chosen by the
    number of keys alone."""
    B, H = 2, 3
    rng = np.random.default_rng(L)
    q, k, v = _views(b, rng.standard_normal((B, L, 3, H, 64)).astype(np.float32), dtype)
    key = np.ones((B, 1, 1, L), np.uint8)
    key[1, ..., L - L // 3:] = 0

    def run(m):
        M = None if m is None else b.fromHost(HostTensor("bool", m.shape, np.ascontiguousarray(m)))
        return read32(b, b.sdpa(b.rope(q, 10000.0), b.rope(k, 10000.0), v, M, 0.125))
    np.testing.assert_array_equal(run(key), run(np.broadcast_to(key, (B, 1, L, L))))
    np.testing.assert_array_equal(run(None), run(np.ones((B, 1, 1, L), np.uint8)))


@pytest.mark.parametrize("L", [449, 1056])
def test_sdpa_long_panel_output(b, L):
    """hb_sdpa_panel: the row-major values in panel order."""
    B, H = 2, 4
    rng = np.random.default_rng(L)
    qkv = b.fromHost(to_host(rng.standard_normal((3, B, H, L, 64)), "f16"))
    mask = b.fromHost(_mask(rng, B, L, "full"))
    p, part = b._ptr(qkv), B * H * L * 64 * 2
    st = F.i64s((H * L * 64, L * 64, 64, 1))
    rows, K = B * L, H * 64
    out, pan, un = (b._malloc((rows + 31) // 32 * 32 * K * 2) for _ in range(3))
    args = (b.ctx, F.HB_F16, p, st, p + part, st, p + 2 * part, st, b._ptr(mask), F.i64s((L, 0, 0, 1)), 0)
    b.n.call("sdpa", "hb_sdpa", *args, out.ptr, F.i64s((L * K, 64, K, 1)), B, H, L, L, 64, 0.125, 1e4, 1e4)
    b.n.call("sdpa", "hb_sdpa_panel", *args, pan.ptr, B, H, L, L, 64, 0.125, 1e4, 1e4)
    b.n.call("unpack", "hb_panel_unpack", b.ctx, pan.ptr, un.ptr, K, rows, K)
    got = [np.empty(rows * K, np.uint16) for _ in range(2)]
    for g, s in zip(got, (out, un)):
        b.n.call("read", "hb_download", b.ctx, g.ctypes.data, s.ptr, g.nbytes)
    np.testing.assert_array_equal(got[0], got[1])


def test_sdpa_long_fully_masked_rows_are_nan(b):
    """A query whose keys are all hidden gives NaN, as on the other kernels."""
    B, H, L = 1, 1, 1100
    rng = np.random.default_rng(0)
    t = [b.fromHost(to_host(rng.standard_normal((B, H, L, 64)), "f16")) for _ in range(3)]
    m = np.ones((B, 1, L, L), np.uint8)
    m[0, 0, 200:240] = 0
    m[0, 0, 600, 1:] = 0
    got = read32(b, b.sdpa(*t, b.fromHost(HostTensor("bool", m.shape, m)), 0.125))[0, 0]
    assert np.isnan(got[200:240]).all()
    assert np.isfinite(np.delete(got, np.s_[200:240], 0)).all()
    np.testing.assert_array_equal(got[600], read32(b, t[2])[0, 0, 0])  # one visible key: its V


@pytest.mark.parametrize("B,H,Lq,copy", [(1, 4, 1100, True), (1, 4, 1, True), (24, 4, 1, False), (24, 4, 150, False),
                                         (24, 4, 1025, True)])
def test_rope_of_k_in_a_pass_where_it_is_shared(B, H, Lq, copy):
    """Fused RoPE takes a rotated copy of K (scratch of the pool) where many
    query tiles or few heads share the pass, and the same bits come out as
    from operands rotated beforehand."""
    from laya_hip.backend import HipBackend
    b, Lk = HipBackend(0), 1100
    try:
        rng = np.random.default_rng(Lq)
        q, k, v = [b.fromHost(to_host(rng.standard_normal((B, H, n, 64)), "f16")) for n in (Lq, Lk, Lk)]
        qr, kr = b.rope(q, 10000.0), b.rope(k, 10000.0)
        b.flush(qr, kr)
        want = read32(b, b.sdpa(qr, kr, v, None, 0.125))
        out = b._malloc(B * H * Lq * 64 * 2)
        st = [F.i64s((H * n * 64, n * 64, 64, 1)) for n in (Lq, Lk)]
        b.pool_stats()  # (returns the blocks that wait for reuse)
        b.n.call("trim", "hb_pool_trim", b.ctx)
        before = b.pool_stats()
        b.n.call("sdpa", "hb_sdpa", b.ctx, F.HB_F16, b._ptr(q), st[0], b._ptr(k), st[1], b._ptr(v), st[1], 0,
                 F.i64s((0, 0, 0, 1)), 0, out.ptr, st[0], B, H, Lq, Lk, 64, 0.125, 10000.0, 10000.0)
        after = b.pool_stats()
        assert (after["cached_bytes"] - before["cached_bytes"] >= B * H * Lk * 64 * 2) == copy
        got = np.empty((B, H, Lq, 64), np.float16)
        b.n.call("read", "hb_download", b.ctx, got.ctypes.data, out.ptr, got.nbytes)
        np.testing.assert_array_equal(got.astype(np.float32), want)
    finally:
        b.destroy()


@pytest.mark.parametrize("Lq,Lk", [(1, 64), (1, 200), (15, 63), (16, 64), (17, 130), (100, 333), (128, 65), (130, 70),
                                   (300, 129)])
def test_mask_classes(b, Lq, Lk):
    """hb_sdpa_mask_info: one byte per 16 queries x 64 keys, 0 nothing visible,
    1 everything, 2 mixed or past the last key; groups without queries are 0."""
    B = 2
    rng = np.random.default_rng(Lq * 7 + Lk)
    nqt, nkt = -(-Lq // 128), -(-Lk // 64)
    for per_query in (True, False):
        m = np.ones((B, Lq if per_query else 1, Lk), np.uint8)
        m[1] = rng.random(m[1].shape) < 0.5
        m[0, :, Lk // 2:] = 0
        M = b.fromHost(HostTensor("bool", m.shape, m))
        info = b._malloc(B * nqt * nkt * 8)
        ms = F.i64s((m.shape[1] * Lk, 0, Lk if per_query else 0, 1))
        b.n.call("fill", "hb_fill", b.ctx, info.ptr, 77, B * nqt * nkt * 8)
        b.n.call("info", "hb_sdpa_mask_info", b.ctx, b._ptr(M), ms, B, Lq, Lk, info.ptr)
        got = np.empty((B, nqt, nkt, 8), np.uint8)
        b.n.call("read", "hb_download", b.ctx, got.ctypes.data, info.ptr, got.nbytes)
        want = np.zeros_like(got)
        full = np.broadcast_to(m, (B, Lq, Lk))
        for i in range(B):
            for q in range(0, Lq, 16):
                for k in range(0, Lk, 64):
                    t = full[i, q:q + 16, k:k + 64]
                    want[i, q // 128, k // 64, q // 16 % 8] = 0 if not t.any() else 1 if t.all() and k + 64 <= Lk else 2
        np.testing.assert_array_equal(got, want)
