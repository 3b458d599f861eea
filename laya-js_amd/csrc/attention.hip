// Scaled dot-product attention (Backend.sdpa) with optional fused RoPE.
//
// sdpa_mfma: flash attention for head dim 64 in fp16 / bf16 on
// v_mfma_f32_16x16x32.  A block owns 128 queries of one (b, h); each of its
// eight waves owns 16 of them.  Per 64-key tile the wave computes
// S^T = K . Q^T, so a lane ends up holding the scores of ONE query for 8
// contiguous keys per 32-key half -- exactly the B-operand layout of
// O^T = V^T . P^T, so P never leaves registers.  The rows of K are fed to the
// MFMA in a permuted order that makes those 8 keys contiguous, which lets the
// lane read its 8 mask bytes with one load and its V^T fragment (V transposed
// in LDS) with one 16-byte read.  K and V^T tiles are double-buffered in LDS,
// loaded into registers two tiles ahead (waves 0-3 fetch K, waves 4-7 V).
// Softmax is online, in f32, in the log2 domain.  A pre-pass over the bool
// mask classes every (b, query tile, key tile, 16-query group) as skipped,
// all visible or masked: tiles no group needs are never staged, and a group
// skips the tiles it cannot see, so the sliding-window layers touch only the
// tiles inside the window (plus the full rows of padded queries, which see
// every valid key).  RoPE, when fused, rotates the Q and K tiles as they are
// staged and rounds them to the storage type, bit-identical to a separate
// Backend.rope.  The output is written row-major or, for the attention output
// projection, in the panel order of the GEMM's X operand.
//
// sdpa32_ring: the same for more than 1024 keys, 32 queries per wave on
// v_mfma_f32_32x32x16.  V goes to LDS by direct loads and is transposed by the LDS read;
// K likewise, or through registers where RoPE rotates it on the way.
//
// sdpa_f32_mfma: the f32 path for head dim 64, on v_mfma_f32_32x32x2_f32.
//
// sdpa_simt: the fallback for other head dims / layouts.
//
// hb_sdpa_noalloc: hb_sdpa without RoPE for callers that cannot allocate; its
// mask summary goes to `scratch`, a file-scope device array.
#include <mutex>
#include <stdexcept>

#include "common.h"

// Scratch of hb_sdpa_noalloc: the mask summary (one byte per 16-query group
// of every 128-query x 64-key tile), for B * ceil(Lq/128) * ceil(Lk/64) <=
// 262144 tiles (B = 32 at Lq = Lk = 8192).  Every GPU the library runs on
// holds its own copy until the process ends.
constexpr size_t kSdpaScratchBytes = (size_t)2 << 20;
static __device__ __align__(256) uint8_t scratch[kSdpaScratchBytes];

namespace hb {

const float* rope_table(uintptr_t ctx, int64_t L, int64_t D, double base);

struct S4 {
  int64_t s[4];
};

static S4 s4(const int64_t* p) {
  S4 r;
  for (int i = 0; i < 4; i++) r.s[i] = p ? p[i] : 0;
  return r;
}

constexpr int kBQ = 128;  // queries per block
constexpr int kQB = 1;    // 16-query blocks per wave
constexpr int kNW = kBQ / (16 * kQB);  // waves per block
constexpr int kNT = kNW * 64;          // threads per block
constexpr int kBK = 64;   // keys per tile
constexpr int kMaxKeyTiles = 1024;  // Lk <= 65536 on the MFMA path
constexpr int kRW = 4;    // sdpa32_ring: waves per block, 32 queries each

// ------------------------------------------------------------------ mask summary

// 4 mask bytes (any nonzero byte is true): bit 7 of each byte set iff the
// byte is nonzero (no carries between bytes)
__device__ __forceinline__ uint32_t mask_nz(uint32_t w) {
  return (((w & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w) & 0x80808080u;
}

// Class of every (batch, 16-query group, 64-key tile) block of a bool mask:
// 0 = no visible key (skipped), 1 = every key visible (no mask reads),
// 2 = mixed or running past Lk (per-element mask).  One byte per group, the
// 8 groups of a 128-query tile together: cls[((b * nqt + qt) * nkt + kt) * 8
// + group].  Computed once per mask tensor and reused by every layer that
// attends with it; the attention kernel skips a key tile for a wave whose
// group has class 0 and stages it only if some group needs it.
// One wave per 16-query group: a lane takes 16 bytes of one of the group's rows
// (unaligned loads, so any row length does), and two ballots give the class.
// Bound by reading the mask once; measured on B = 3, T = 333, where the rows
// are not 16-byte aligned: 11.2 -> 5.2 us against a byte per thread and LDS
// atomics.  Up to 128 queries the block has only the waves whose group has
// rows, and the groups without any are class 0 (16 x 1 x 8192: 4.1 -> 3.4 us).
__global__ __launch_bounds__(kNW * 64) void mask_class_kernel(const uint8_t* __restrict__ mask, S4 ms, int Lq, int Lk,
                                                         int nqt, int nkt, uint8_t* __restrict__ cls) {
  const int kt = blockIdx.x, qt = blockIdx.y, b = blockIdx.z;
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int k0 = kt * kBK, nk = min(kBK, Lk - k0), c = (lane & 3) * 16;
  const int q = qt * kBQ + g * 16 + (lane >> 2);
  bool any = false, all = true;
  if (q < Lq && c < nk) {
    const uint8_t* p = mask + b * ms.s[0] + (int64_t)q * ms.s[2] + (int64_t)(k0 + c) * ms.s[3];
    if (ms.s[3] == 1 && c + 16 <= nk) {
      uint32_t w[4];
      __builtin_memcpy(w, p, 16);
      any = (w[0] | w[1] | w[2] | w[3]) != 0;
      all = (mask_nz(w[0]) & mask_nz(w[1]) & mask_nz(w[2]) & mask_nz(w[3])) == 0x80808080u;
    } else {
      for (int e = 0; e < 16 && c + e < nk; e++) {
        const bool v = p[(int64_t)e * ms.s[3]] != 0;
        any |= v;
        all &= v;
      }
    }
  }
  const bool gany = __ballot(any) != 0, gall = __ballot(!all) == 0;
  uint8_t* out = cls + (((int64_t)b * nqt + qt) * nkt + kt) * kNW;
  const int waves = blockDim.x >> 6;
  if (lane == 0) out[g] = !gany ? 0 : (gall && nk == kBK ? 1 : 2);
  else if (g == 0 && lane >= waves && lane < kNW) out[lane] = 0;
}

static size_t mask_info_bytes(int64_t B, int64_t Lq, int64_t Lk) {
  int64_t nqt = (Lq + kBQ - 1) / kBQ, nkt = (Lk + kBK - 1) / kBK;
  return (size_t)(B * nqt * nkt * kNW);
}

static void launch_mask_info(hipStream_t st, const uint8_t* mask, const S4& ms, int64_t B, int64_t Lq, int64_t Lk,
                             uint8_t* info) {
  int nqt = (int)((Lq + kBQ - 1) / kBQ), nkt = (int)((Lk + kBK - 1) / kBK);
  const int waves = Lq < kBQ ? (int)((Lq + 15) / 16) : kNW;
  mask_class_kernel<<<dim3(nkt, nqt, (unsigned)B), waves * 64, 0, st>>>(mask, ms, (int)Lq, (int)Lk, nqt, nkt, info);
}

// ------------------------------------------------------------------ MFMA kernel (D = 64)

template <bool BF16>
__device__ __forceinline__ float4v mfma16(const uint4v& a, const uint4v& b, float4v c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0,
                                                  0, 0);
}
template <bool BF16>
__device__ __forceinline__ float tof(uint32_t h) {
  return BF16 ? bf16_to_f32((uint16_t)h) : f16_bits_to_f32((uint16_t)h);
}
template <bool BF16>
__device__ __forceinline__ uint32_t fromf(float v) {
  return BF16 ? f32_to_bf16(v) : f32_to_f16_bits(v);
}

// Two f32 values packed as 16-bit (v_cvt_pk_f16_f32 / v_cvt_pk_bf16_f32: RNE).
template <bool BF16>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  typedef float float2v __attribute__((ext_vector_type(2)));
  if constexpr (BF16) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((float2v){a, b}, bf16x2));
  } else {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((float2v){a, b}, half2v));
  }
}

// Cross-lane exchanges for the 4 lanes that hold one query (lane, lane ^ 16,
// lane ^ 32, lane ^ 48): ds_swizzle in bit-mask mode (and 0x1f, xor 0x10)
// reads lane ^ 16 within each half-wave; v_permlane32_swap exchanges the
// two halves, returning (per lane) its own value and the one of lane ^ 32.
__device__ __forceinline__ float from_xor16(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, x), 0x401F));
}
__device__ __forceinline__ float max_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x),
                                                  false, false);
  return fmaxf(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
}
__device__ __forceinline__ float sum_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x),
                                                  false, false);
  return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}

__device__ __forceinline__ int qk_swz(int r, int c) { return r * 64 + ((c ^ (r & 7)) << 3); }
// K tiles: chunk c of row r at c ^ (4 * bit 1 of r + bits 3..4 of r).  A
// 16-lane pass of the S = K.Q^T fragment reads touches rows b + 8a (a, b in
// 0..3), which this spreads over all 64 banks, and the staging stores (rows
// r..r+3, chunks 0..3 or 4..7) hit disjoint banks too.
__device__ __forceinline__ int k_swz(int r, int c) { return r * 64 + ((c ^ ((((r >> 1) & 1) << 2) | ((r >> 3) & 3))) << 3); }
constexpr int kVtLd = 72;  // row stride (elements) of V^T in LDS
// V^T tiles: the 8-key chunk c of row d sits at c ^ (4 * bit 4 of d + 2 * bit 5
// of d), which makes the transposing staging stores (rows 8*vc + i, one
// 32-bit key pair per lane) hit 64 distinct banks; the fragment reads of one
// instruction share bits 4..5 of d, so they stay conflict-free.
__device__ __forceinline__ int vt_swz(int d, int c) {
  return d * kVtLd + ((c ^ ((((d >> 4) & 1) << 2) | (((d >> 5) & 1) << 1))) << 3);
}

// Raw chunks c and c + 4 (d in [8c, 8c+8) and the rotation partners d + 32)
// of one row of a [L, 64] operand; zero when the row is out of range.
__device__ __forceinline__ void load_pair(const uint16_t* __restrict__ src, bool valid, int c, uint4v& lo,
                                          uint4v& hi) {
  lo = uint4v{0, 0, 0, 0};
  hi = uint4v{0, 0, 0, 0};
  if (valid) {
    lo = *(const uint4v*)(src + c * 8);
    hi = *(const uint4v*)(src + 32 + c * 8);
  }
}

// cos / sin of the 8 rotation pairs (d, d + 32), d in [8c, 8c+8), at
// position `pos` of a RoPE table [L][32] (float2).
__device__ __forceinline__ void load_cs(const float2* __restrict__ tab, int pos, int c, float2 (&cs)[8]) {
  const float4v* t = (const float4v*)(tab + pos * 32 + c * 8);
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const float4v v = t[e];
    cs[2 * e] = float2{v[0], v[1]};
    cs[2 * e + 1] = float2{v[2], v[3]};
  }
}

// Rotates a loaded chunk pair by RoPE, rounding to the storage type like a
// separate Backend.rope.
template <bool BF16>
__device__ __forceinline__ void rot_pair(uint4v& lo, uint4v& hi, const float2 (&cs)[8]) {
  uint32_t* l = (uint32_t*)&lo;
  uint32_t* h = (uint32_t*)&hi;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const float2 c0 = cs[2 * e], c1 = cs[2 * e + 1];
    float x0a = tof<BF16>(l[e] & 0xffff), x0b = tof<BF16>(l[e] >> 16);
    float x1a = tof<BF16>(h[e] & 0xffff), x1b = tof<BF16>(h[e] >> 16);
    l[e] = pack2<BF16>(pin_f32(fmaf(-x1a, c0.y, x0a * c0.x)), pin_f32(fmaf(-x1b, c1.y, x0b * c1.x)));
    h[e] = pack2<BF16>(pin_f32(fmaf(x0a, c0.y, x1a * c0.x)), pin_f32(fmaf(x0b, c1.y, x1b * c1.x)));
  }
}

// Rotates a loaded chunk pair by RoPE (when `rot`) with the pairs' cos / sin,
// rounding to the storage type like a separate Backend.rope, and writes it
// to the swizzled [rows][64] LDS tile.
template <bool BF16, bool KSWZ = false>
__device__ __forceinline__ void store_pair(uint4v lo, uint4v hi, bool rot, int c, const float2 (&cs)[8],
                                           uint16_t* lds, int row) {
  if (rot) rot_pair<BF16>(lo, hi, cs);
  *(uint4v*)(lds + (KSWZ ? k_swz(row, c) : qk_swz(row, c))) = lo;
  *(uint4v*)(lds + (KSWZ ? k_swz(row, c + 4) : qk_swz(row, c + 4))) = hi;
}

// Where a block works, of one per (b, h, query tile) on a 1-D grid.  Blocks are
// dealt to the 8 XCDs in turn (block i on XCD i % 8).  The query tiles of one
// (b, h) read the same K / V rows and mask bytes, so they are consecutive blocks
// of one XCD's share and share its L2; the (b, h) pairs are dealt to the XCDs
// in turn, which spreads sequences of different lengths (and work).  Without a
// multiple of 8 pairs the blocks take (b, h, query tile) in order, or, with
// RUNS, in contiguous runs per XCD.
template <bool RUNS>
__device__ __forceinline__ void sdpa_block(int nqt, int nh, int& qt, int& b, int& h) {
  const int nbh = (int)(gridDim.x / nqt);
  int bh;
  if ((nbh & 7) == 0) {
    const int x = blockIdx.x & 7, idx = blockIdx.x >> 3;
    qt = idx % nqt;
    bh = (idx / nqt) * 8 + x;
  } else {
    const uint32_t t = RUNS ? xcd_tile(blockIdx.x, gridDim.x) : blockIdx.x;
    qt = t % nqt;
    bh = t / nqt;
  }
  h = bh % nh;
  b = bh / nh;
}

template <bool BF16>
__global__ __launch_bounds__(kNT) __attribute__((amdgpu_waves_per_eu(4))) void sdpa_mfma(const uint16_t* __restrict__ Q, S4 qs, const uint16_t* __restrict__ K,
                                                 S4 ks, const uint16_t* __restrict__ V, S4 vs,
                                                 const uint8_t* __restrict__ mask, S4 ms, int mask_vec,
                                                 const uint8_t* __restrict__ cls, uint16_t* __restrict__ O, S4 os,
                                                 int Lq, int Lk, float scale_log2, const float2* __restrict__ tabq,
                                                 const float2* __restrict__ tabk, int pK, int nqt, int nh) {
  // Q, and two buffers of K and V^T: tile t + 1 is staged while tile t computes
  __shared__ __attribute__((aligned(16))) uint16_t Qs[kBQ * 64];
  __shared__ __attribute__((aligned(16))) uint16_t Ks[2][kBK * 64];
  __shared__ __attribute__((aligned(16))) uint16_t Vt[2][64 * kVtLd];
  __shared__ uint16_t cls_row[kMaxKeyTiles];  // 2 bits of class per 16-query group

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, li = lane & 15;
  int qt, b, h;
  sdpa_block<false>(nqt, nh, qt, b, h);
  const int nkt = (Lk + kBK - 1) / kBK;
  const int q0 = qt * kBQ;
  const uint16_t* Qb = Q + b * qs.s[0] + h * qs.s[1];
  const uint16_t* Kb = K + b * ks.s[0] + h * ks.s[1];
  const uint16_t* Vb = V + b * vs.s[0] + h * vs.s[1];
  // this block's Q rows (and their RoPE cos / sin) are requested first: they
  // do not depend on the tile classes, so their latency overlaps the class
  // row's
  constexpr int QR = kBQ * 4 / kNT;  // rounds of Q staging (4 threads per row)
  static_assert(QR * kNT == kBQ * 4, "Q staging: whole rounds");
  uint4v qlo[QR], qhi[QR];
  float2 qcs[QR][8];
#pragma unroll
  for (int u = 0; u < QR; u++) {
    const int t = tid + u * kNT, r = t >> 2, c = t & 3, q = q0 + r;
    load_pair(Qb + (int64_t)q * qs.s[2], q < Lq, c, qlo[u], qhi[u]);
    if (tabq != nullptr && q < Lq) load_cs(tabq, q, c, qcs[u]);
  }

  // tile classes of this (b, query tile) for each wave's 16-query group: 0
  // skip, 1 all visible, 2 per-element mask / key bound; staged in LDS once
  // (the host caps nkt at kMaxKeyTiles).  A tile is staged when some group
  // needs it.
  static_assert(kQB == 1 && kNW == 8, "one 16-query group per wave, 8 per tile");
  for (int t = tid; t < nkt; t += kNT) {
    uint32_t c;
    if (cls != nullptr) {
      const uint2v w = *(const uint2v*)(cls + (((int64_t)b * nqt + qt) * nkt + t) * kNW);
      c = 0;
#pragma unroll
      for (int gq = 0; gq < kNW; gq++) c |= (((gq < 4 ? w.x : w.y) >> (8 * (gq & 3))) & 3u) << (2 * gq);
    } else if (mask != nullptr) {
      c = 0xAAAAu;
    } else {
      c = (t + 1) * kBK <= Lk ? 0x5555u : 0xAAAAu;
    }
    cls_row[t] = (uint16_t)c;
  }
  auto tile_needed = [&](int kt) -> bool { return cls_row[kt] != 0; };
  auto wave_class = [&](int kt) -> int { return (cls_row[kt] >> (2 * wave)) & 3; };
  // (the same in every lane: read from the class row in LDS, made
  // wave-uniform so that the tile's address arithmetic is scalar)
  auto next_tile = [&](int kt) -> int {
    kt++;
    while (kt < nkt && !tile_needed(kt)) kt++;
    return __builtin_amdgcn_readfirstlane(kt);
  };
  __syncthreads();  // the class row is complete

  // A K tile is staged by the first 256 threads (row kr, chunk pair kc),
  // the V tile by the other 256 (key pair vj, chunk vc); loaded into
  // registers two tiles ahead and staged into LDS one tile ahead
  static_assert(kNT == 512, "K / V staging: 256 threads each");
  const bool kpart = tid < 256;  // whole waves
  const int kr = (tid & 255) >> 2, kc = tid & 3;
  const int vc = tid & 7, vj = 2 * ((tid & 255) >> 3);
  uint4v pr0, pr1;  // K threads: chunks kc and kc + 4 of row kr; V threads: keys vj and vj + 1
  float2 kcs[8];    // RoPE cos / sin of this thread's K row (fused RoPE)
  // The tile's first row is a scalar address (k0 is wave-uniform); a
  // thread's row within the tile adds a 24-bit product (row < 64, a row
  // stride below 2^24 elements: the host's condition for this kernel).
  auto prefetch = [&](int kt) {
    const int k0 = kt * kBK;
    if (kpart) {
      const uint16_t* kb = Kb + (int64_t)k0 * ks.s[2];
      load_pair(kb + __umul24(kr, (uint32_t)ks.s[2]), k0 + kr < Lk, kc, pr0, pr1);
      if (tabk != nullptr && k0 + kr < Lk) load_cs(tabk + (int64_t)k0 * 32, kr, kc, kcs);
    } else {
      const uint16_t* vb = Vb + (int64_t)k0 * vs.s[2] + vc * 8;
      const uint32_t vo = __umul24(vj, (uint32_t)vs.s[2]);
      pr0 = uint4v{0, 0, 0, 0};
      pr1 = uint4v{0, 0, 0, 0};
      if (k0 + vj < Lk) pr0 = *(const uint4v*)(vb + vo);
      if (k0 + vj + 1 < Lk) pr1 = *(const uint4v*)(vb + vo + (uint32_t)vs.s[2]);
    }
  };

  // this lane's mask bytes of a tile: 8 contiguous keys of its query (one per
  // 16-query block qb) in each 32-key half t
  auto load_mask = [&](int kt, uint2v (&mw)[kQB][2]) {
    const int k0 = kt * kBK;
#pragma unroll
    for (int qb = 0; qb < kQB; qb++) {
      const int q = q0 + wave * 16 * kQB + qb * 16 + li;
      const uint8_t* mrow = mask + b * ms.s[0] + (int64_t)(q < Lq ? q : 0) * ms.s[2];
#pragma unroll
      for (int t = 0; t < 2; t++) {
        const int kbase = k0 + 32 * t + 8 * g;
        if (mask_vec && kbase + 8 <= Lk) {  // (rows of any alignment)
          __builtin_memcpy(&mw[qb][t], mrow + kbase, 8);
        } else {
          uint32_t w0 = 0, w1 = 0;
#pragma unroll
          for (int e = 0; e < 8; e++) {
            uint32_t bit = (kbase + e < Lk) ? (mrow[(int64_t)(kbase + e) * ms.s[3]] != 0) : 0u;
            if (e < 4) w0 |= bit << (8 * e);
            else w1 |= bit << (8 * (e - 4));
          }
          mw[qb][t] = uint2v{w0, w1};
        }
      }
    }
  };

  // K tile `t` (rotated, as a separate Backend.rope would store it) and the
  // transposed V tile from the prefetch registers into LDS buffer `bf`
  auto store_kv = [&](int t, int bf) {
    if (kpart) {
      store_pair<BF16, true>(pr0, pr1, tabk != nullptr && t * kBK + kr < Lk, kc, kcs, Ks[bf], kr);
      return;
    }
    const uint32_t* pa = (const uint32_t*)&pr0;
    const uint32_t* pb = (const uint32_t*)&pr1;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      uint32_t lo = (pa[e] & 0xffff) | (pb[e] << 16);
      uint32_t hi = (pa[e] >> 16) | (pb[e] & 0xffff0000u);
      *(uint32_t*)(Vt[bf] + vt_swz(vc * 8 + 2 * e, vj >> 3) + (vj & 7)) = lo;
      *(uint32_t*)(Vt[bf] + vt_swz(vc * 8 + 2 * e + 1, vj >> 3) + (vj & 7)) = hi;
    }
  };

  // the first K / V tile (and its mask bytes) is requested before Q is
  // staged, so the two loads' latencies overlap
  int kt = next_tile(-1);
  uint2v mw[kQB][2], mwn[kQB][2];
  if (kt < nkt) {
    prefetch(kt);
    if (mask != nullptr && wave_class(kt) == 2) load_mask(kt, mw);
  }

  // ---- stage Q (rotated); this wave's B fragments of Q^T are read below
#pragma unroll
  for (int u = 0; u < QR; u++) {
    const int t = tid + u * kNT, r = t >> 2, c = t & 3, q = q0 + r;
    store_pair<BF16>(qlo[u], qhi[u], tabq != nullptr && q < Lq, c, qcs[u], Qs, r);
  }
  // the first tile into buffer 0; the second tile's loads start
  int nk = nkt;
  if (kt < nkt) {
    store_kv(kt, 0);
    nk = next_tile(kt);
    if (nk < nkt) prefetch(nk);
  }
  __syncthreads();
  uint4v qf[kQB][2];
#pragma unroll
  for (int qb = 0; qb < kQB; qb++)
#pragma unroll
    for (int s = 0; s < 2; s++)
      qf[qb][s] = *(const uint4v*)(Qs + qk_swz(wave * 16 * kQB + qb * 16 + li, s * 4 + g));


  float4v o[kQB][4];
  float m[kQB], l[kQB];
#pragma unroll
  for (int qb = 0; qb < kQB; qb++) {
#pragma unroll
    for (int d = 0; d < 4; d++) o[qb][d] = float4v{0.f, 0.f, 0.f, 0.f};
    m[qb] = -INFINITY;
    l[qb] = 0.f;
  }

  // online softmax of one 64-key tile for query block qb: scores st (raw,
  // -inf where hidden; lane key 32t + 8g + e is st[2t + e/4][e%4]) -> P
  // fragments, running max / sum, O rescale
  uint4v pf[kQB][2];
  auto softmax = [&](int qb, const float4v (&sq)[4], float mx) {
    mx = fmaxf(mx, from_xor16(mx));
    mx = max_xor32(mx);
    const float mnew = fmaxf(m[qb], mx);  // raw (unscaled) row max
    const float mc = mnew == -INFINITY ? 0.f : mnew * scale_log2;
    const float alpha = __builtin_amdgcn_exp2f(m[qb] * scale_log2 - mc);
    m[qb] = mnew;
    float psum = 0.f;
#pragma unroll
    for (int t = 0; t < 2; t++) {
      uint32_t pk[4];
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const float p0 = __builtin_amdgcn_exp2f(fmaf(sq[2 * t + (e >> 2)][e & 3], scale_log2, -mc));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(sq[2 * t + (e >> 2)][(e & 3) + 1], scale_log2, -mc));
        psum += p0 + p1;
        pk[e >> 1] = pack2<BF16>(p0, p1);
      }
      pf[qb][t] = uint4v{pk[0], pk[1], pk[2], pk[3]};
    }
    l[qb] = l[qb] * alpha + psum;
    // rescale O only when some row max of this wave moved
    if (!__all(alpha == 1.0f)) {
#pragma unroll
      for (int d = 0; d < 4; d++) o[qb][d] *= alpha;
    }
  };

  int buf = 0;
  while (kt < nkt) {
    const int k0 = kt * kBK;
    const int cl = wave_class(kt);  // this wave's class of the tile
    const uint16_t* Kc = Ks[buf];
    const uint16_t* Vc = Vt[buf];

    // ---- S^T = K . Q^T over 4 key blocks; block kb row i holds key
    // 32*(kb/2) + 8*(i/4) + (i%4) + 4*(kb%2) so a lane's 8 keys are contiguous
    // (a wave whose queries see no key of the tile skips its MFMAs and softmax)
    float4v st[kQB][4];
#pragma unroll
    for (int kb = 0; kb < 4; kb++) {
      if (cl == 0) break;
      const int krow = 32 * (kb >> 1) + 8 * (li >> 2) + (li & 3) + 4 * (kb & 1);
      uint4v kf0 = *(const uint4v*)(Kc + k_swz(krow, g));
      uint4v kf1 = *(const uint4v*)(Kc + k_swz(krow, 4 + g));
#pragma unroll
      for (int qb = 0; qb < kQB; qb++) {
        float4v z = {0.f, 0.f, 0.f, 0.f};
        z = mfma16<BF16>(kf0, qf[qb][0], z);
        st[qb][kb] = mfma16<BF16>(kf1, qf[qb][1], z);
      }
    }

    // ---- the next tile into the other buffer (its loads were issued one
    // tile ago), the one after it into registers, the next mask bytes
    int nn = nkt;
    if (nk < nkt) {
      store_kv(nk, buf ^ 1);
      nn = next_tile(nk);
      if (nn < nkt) prefetch(nn);
      if (mask != nullptr && wave_class(nk) == 2) load_mask(nk, mwn);
    }

    // ---- mask (only for mixed tiles, in place), online softmax, P fragments
    if (cl != 0) {
#pragma unroll
      for (int qb = 0; qb < kQB; qb++) {
        if (cl == 2) {
#pragma unroll
          for (int t = 0; t < 2; t++) {
            const int kbase = k0 + 32 * t + 8 * g;  // this lane's 8 contiguous keys
            // bit 7 of byte e % 4 of word e / 4: key kbase + e is visible
            // (mask byte nonzero, key < Lk)
            uint32_t vx = 0x80808080u, vy = 0x80808080u;
            if (mask != nullptr) {
              vx = mask_nz(mw[qb][t].x);
              vy = mask_nz(mw[qb][t].y);
            }
            const int left = Lk - kbase;
            if (left < 8) {
              vx &= left >= 4 ? ~0u : (left <= 0 ? 0u : 0xffffffffu >> (8 * (4 - left)));
              vy &= left <= 4 ? 0u : 0xffffffffu >> (8 * (8 - left));
            }
            // a hidden score becomes -inf: the byte's bit 7 sign-extended to
            // a word mask, one bit-field insert per score
#pragma unroll
            for (int e = 0; e < 8; e++) {
              const uint32_t m = (uint32_t)__builtin_amdgcn_sbfe((int)(e < 4 ? vx : vy), 8 * (e & 3) + 7, 1);
              const float sv = st[qb][2 * t + (e >> 2)][e & 3];
              st[qb][2 * t + (e >> 2)][e & 3] = __uint_as_float((__float_as_uint(sv) & m) | (~m & 0xff800000u));
            }
          }
        }
        float mx = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 4; kb++)
#pragma unroll
          for (int e = 0; e < 4; e++) mx = fmaxf(mx, st[qb][kb][e]);
        softmax(qb, st[qb], mx);
      }
    }

    // ---- O^T += V^T . P^T
#pragma unroll
    for (int d = 0; d < 4; d++) {
      if (cl == 0) break;
#pragma unroll
      for (int t = 0; t < 2; t++) {
        uint4v vf = *(const uint4v*)(Vc + vt_swz(d * 16 + li, 4 * t + g));
#pragma unroll
        for (int qb = 0; qb < kQB; qb++) o[qb][d] = mfma16<BF16>(vf, pf[qb][t], o[qb][d]);
      }
    }
#pragma unroll
    for (int qb = 0; qb < kQB; qb++)
#pragma unroll
      for (int t = 0; t < 2; t++) mw[qb][t] = mwn[qb][t];
    // this tile's buffer is free and the next one complete for every wave
    __syncthreads();
    buf ^= 1;
    kt = nk;
    nk = nn;
  }

  // ---- normalise and store (lane: one query, d = 16*dblk + 4g + 0..3)
#pragma unroll
  for (int qb = 0; qb < kQB; qb++) {
    float lt = l[qb];
    lt += from_xor16(lt);
    lt = sum_xor32(lt);
    const float inv = 1.0f / lt;
    const int q = q0 + wave * 16 * kQB + qb * 16 + li;
    if (q >= Lq) continue;
    // strided [B, H, Lq, D], or (pK > 0) panel order of the [B*Lq, pK]
    // matrix whose row b*Lq + q holds the heads side by side: columns
    // 64h + 16d + 4g.. are 16-column block 4h + d, half g/2, offset 4(g%2)
    uint16_t* op;
    int64_t dstep;
    if (pK > 0) {
      const int64_t m = (int64_t)b * Lq + q;
      op = O + ((m >> 5) * (pK >> 4) + 4 * h) * 512 + ((g >> 1) * 32 + (m & 31)) * 8 + 4 * (g & 1);
      dstep = 512;
    } else {
      op = O + b * os.s[0] + h * os.s[1] + (int64_t)q * os.s[2] + 4 * g;
      dstep = 16;
    }
#pragma unroll
    for (int d = 0; d < 4; d++) {
      uint2v w;
      w.x = fromf<BF16>(o[qb][d][0] * inv) | (fromf<BF16>(o[qb][d][1] * inv) << 16);
      w.y = fromf<BF16>(o[qb][d][2] * inv) | (fromf<BF16>(o[qb][d][3] * inv) << 16);
      *(uint2v*)(op + d * dstep) = w;
    }
  }
}

// ------------------------------------------------------------------ 32-query MFMA kernel

typedef short short4t __attribute__((ext_vector_type(4)));
// Transposing LDS read: within 16 lanes, lanes 4r .. 4r + 3 point at 4 x 4
// consecutive values of row r; lane c gets column c's 4 rows.
__device__ __forceinline__ uint2v lds_tr16(const uint16_t* p) {
  const short4t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4t*)p);
  return __builtin_bit_cast(uint2v, v);
}
template <bool BF16>
__device__ __forceinline__ float16v mfma32x16(const uint4v& a, const uint4v& b, float16v c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0,
                                                  0);
}

// chunk c (8 values) of row r of a [64][64] K or V tile sits at c ^ kv_f(r): a
// 16-lane pass of the K fragment reads (16 rows, one chunk) and of the V
// transpose reads (4 rows, 4 chunks) covers all 64 banks
__device__ __forceinline__ int kv_f(int r) { return (((r >> 1) & 1) << 2) | ((r >> 2) & 3); }

// K [B, H, Lk, 64] rotated by RoPE into contiguous [B, H, Lk, 64]: one thread
// per chunk pair (c, c + 4) of a row.  Bandwidth-bound; blocks take 64 rows of
// every (b, h) in turn, so the RoPE table's rows stay in L2.
template <bool BF16>
__global__ __launch_bounds__(256) void rope_k_kernel(const uint16_t* __restrict__ K, S4 ks, uint16_t* __restrict__ Y,
                                                     int Lk, int nh, int nbh, const float2* __restrict__ tab) {
  const int bh = blockIdx.x % nbh, r = (blockIdx.x / nbh) * 64 + (threadIdx.x >> 2), c = threadIdx.x & 3;
  if (r >= Lk) return;
  const uint16_t* kp = K + (bh / nh) * ks.s[0] + (bh % nh) * ks.s[1] + (int64_t)r * ks.s[2];
  uint4v lo, hi;
  float2 cs[8];
  load_pair(kp, true, c, lo, hi);
  load_cs(tab + (int64_t)r * 32, 0, c, cs);
  rot_pair<BF16>(lo, hi, cs);
  uint16_t* yp = Y + ((int64_t)bh * Lk + r) * 64;
  *(uint4v*)(yp + 8 * c) = lo;
  *(uint4v*)(yp + 8 * (c + 4)) = hi;
}

// One wave's state: 32 queries (lane l holds query l % 32; the lane halves
// split its columns of Q and O and its keys).
struct Wave32 {
  uint4v qf[4];   // chunk 2 s + lg of the query (columns 16 s + 8 lg ..) per MFMA step s
  float16v o[2];  // O^T: columns 32 d + 8 (r / 4) + 4 lg + r % 4
  float m, l;     // raw (unscaled) row max, sum of the lane's weights
};

// Loads the wave's queries and, with a table, rotates them, rounded as a
// separate Backend.rope stores them.
template <bool BF16>
__device__ __forceinline__ void wave32_init(Wave32& w, const uint16_t* qrow, const float2* tab, int pos, int lg) {
#pragma unroll
  for (int s = 0; s < 4; s++) w.qf[s] = *(const uint4v*)(qrow + 8 * lg + 16 * s);
  if (tab != nullptr) {
    const float4v* tp = (const float4v*)(tab + (int64_t)pos * 32 + 8 * lg);
#pragma unroll
    for (int s = 0; s < 2; s++) {
      float2 cs[8];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float4v v = tp[8 * s + e];
        cs[2 * e] = float2{v[0], v[1]};
        cs[2 * e + 1] = float2{v[2], v[3]};
      }
      rot_pair<BF16>(w.qf[s], w.qf[s + 2], cs);
    }
  }
#pragma unroll
  for (int d = 0; d < 2; d++)
#pragma unroll
    for (int r = 0; r < 16; r++) w.o[d][r] = 0.f;
  w.m = -INFINITY;
  w.l = 0.f;
}

// LDS element offsets of a lane's fragment reads within a [64][64] tile: K
// chunk 2 s + lg of row l32 (+ 2048 for the second 32 keys); V transpose
// read of keys 16 t + 8 u + 4 lg .., columns 32 d .. (+ 1024 t).
struct Frag32 {
  int ka[4], va[2][2];
};
__device__ __forceinline__ Frag32 frag32(int lane) {
  Frag32 f;
  const int l32 = lane & 31, lg = lane >> 5, j16 = lane & 15, vrow = 4 * lg + (j16 >> 2);
#pragma unroll
  for (int s = 0; s < 4; s++) f.ka[s] = l32 * 64 + (((2 * s + lg) ^ kv_f(l32)) << 3);
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int d = 0; d < 2; d++) {
      const int r = 8 * u + vrow, c = 4 * d + 2 * ((lane >> 4) & 1) + ((j16 & 3) >> 1);
      f.va[u][d] = r * 64 + ((c ^ kv_f(r)) << 3) + 4 * (j16 & 1);
    }
  return f;
}

// One 64-key tile (keys k0 ..) for the wave's queries: scores, mask (`mixed`),
// online softmax, O += P . V.  mrow: the lane's mask row, or null (only the
// bound Lk hides keys); mask_vec: its rows are contiguous and 16-byte aligned,
// and lane half lg fetches the 32 bytes of key block lg, the halves swapping
// words afterwards; otherwise a lane's own words (keys 32 kb + 8 j + 4 lg ..).
template <bool BF16>
__device__ __forceinline__ void wave32_tile(Wave32& w, const Frag32& f, const uint16_t* Kc, const uint16_t* Vc, int k0,
                                            int Lk, bool mixed, const uint8_t* mrow, int64_t ms3, int mask_vec,
                                            float scale_log2, int lg) {
  const bool vec = mask_vec && k0 + kBK <= Lk;
  uint32_t mw[8];
  if (mixed && mrow != nullptr) {
    if (vec) {
      const uint4v a = *(const uint4v*)(mrow + k0 + 32 * lg), c = *(const uint4v*)(mrow + k0 + 32 * lg + 16);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        mw[e] = a[e];
        mw[4 + e] = c[e];
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int key = k0 + 32 * (i >> 2) + 8 * (i & 3) + 4 * lg;
        uint32_t v = 0;
        if (ms3 == 1 && key + 4 <= Lk) {
          __builtin_memcpy(&v, mrow + key, 4);
        } else {
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (key + e < Lk && mrow[(int64_t)(key + e) * ms3] != 0) v |= 1u << (8 * e);
        }
        mw[i] = v;
      }
    }
  }
  float16v st[2];
#pragma unroll
  for (int kb = 0; kb < 2; kb++) {
#pragma unroll
    for (int r = 0; r < 16; r++) st[kb][r] = 0.f;
#pragma unroll
    for (int s = 0; s < 4; s++) st[kb] = mfma32x16<BF16>(*(const uint4v*)(Kc + f.ka[s] + kb * 2048), w.qf[s], st[kb]);
  }
  if (mixed) {
    uint32_t x[8];
    if (mrow == nullptr) {
#pragma unroll
      for (int i = 0; i < 8; i++) x[i] = 0x01010101u;
    } else if (vec) {
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const auto y = __builtin_amdgcn_permlane32_swap(mw[2 * j], mw[2 * j + 1], false, false);
        x[j] = (uint32_t)y[0];
        x[4 + j] = (uint32_t)y[1];
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; i++) x[i] = mw[i];
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
      // bit 7 of byte e: key visible; a hidden score becomes -inf
      uint32_t vis = mask_nz(x[i]);
      const int left = Lk - (k0 + 32 * (i >> 2) + 8 * (i & 3) + 4 * lg);
      vis &= left >= 4 ? ~0u : (left <= 0 ? 0u : 0xffffffffu >> (8 * (4 - left)));
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const uint32_t mk = (uint32_t)__builtin_amdgcn_sbfe((int)vis, 8 * e + 7, 1);
        const float sv = st[i >> 2][4 * (i & 3) + e];
        st[i >> 2][4 * (i & 3) + e] = __uint_as_float((__float_as_uint(sv) & mk) | (~mk & 0xff800000u));
      }
    }
  }
  float mx = -INFINITY;
#pragma unroll
  for (int kb = 0; kb < 2; kb++)
#pragma unroll
    for (int r = 0; r < 16; r++) mx = fmaxf(mx, st[kb][r]);
  mx = max_xor32(mx);
  const float mnew = fmaxf(w.m, mx);
  const float mc = mnew == -INFINITY ? 0.f : mnew * scale_log2;
  const float alpha = __builtin_amdgcn_exp2f(w.m * scale_log2 - mc);
  w.m = mnew;
  float psum = 0.f;
  uint4v pf[4];
#pragma unroll
  for (int t = 0; t < 4; t++) {
    uint32_t pk[4];
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const float p0 = __builtin_amdgcn_exp2f(fmaf(st[t >> 1][8 * (t & 1) + e], scale_log2, -mc));
      const float p1 = __builtin_amdgcn_exp2f(fmaf(st[t >> 1][8 * (t & 1) + e + 1], scale_log2, -mc));
      psum += p0 + p1;
      pk[e >> 1] = pack2<BF16>(p0, p1);
    }
    pf[t] = uint4v{pk[0], pk[1], pk[2], pk[3]};
  }
  w.l = w.l * alpha + psum;
  if (!__all(alpha == 1.0f)) {  // rescale O only when some row max of this wave moved
#pragma unroll
    for (int d = 0; d < 2; d++)
#pragma unroll
      for (int r = 0; r < 16; r++) w.o[d][r] *= alpha;
  }
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int d = 0; d < 2; d++) {
      const uint2v v0 = lds_tr16(Vc + f.va[0][d] + t * 1024), v1 = lds_tr16(Vc + f.va[1][d] + t * 1024);
      w.o[d] = mfma32x16<BF16>(uint4v{v0.x, v0.y, v1.x, v1.y}, pf[t], w.o[d]);
    }
}

// Normalises and stores query q: 4 consecutive columns 32 d + 8 j + 4 lg per 8
// bytes, strided [B, H, Lq, D], or (pK > 0) in panel order of the [B*Lq, pK]
// matrix whose rows hold the heads side by side: 16-column block 4 h + 2 d +
// j / 2, half j % 2.
template <bool BF16>
__device__ __forceinline__ void wave32_store(const Wave32& w, uint16_t* O, const S4& os, int pK, int b, int h, int q,
                                             int Lq, int lg) {
  const float inv = 1.0f / sum_xor32(w.l);
  if (q >= Lq) return;
  const int64_t mrw = (int64_t)b * Lq + q;
  uint16_t* op = pK > 0 ? O + ((mrw >> 5) * (pK >> 4) + 4 * h) * 512 + (mrw & 31) * 8 + 4 * lg
                        : O + b * os.s[0] + h * os.s[1] + (int64_t)q * os.s[2] + 4 * lg;
#pragma unroll
  for (int d = 0; d < 2; d++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      uint2v x;
      x.x = pack2<BF16>(pin_f32(w.o[d][4 * j] * inv), pin_f32(w.o[d][4 * j + 1] * inv));
      x.y = pack2<BF16>(pin_f32(w.o[d][4 * j + 2] * inv), pin_f32(w.o[d][4 * j + 3] * inv));
      *(uint2v*)(op + (pK > 0 ? (2 * d + (j >> 1)) * 512 + (j & 1) * 256 : 32 * d + 8 * j)) = x;
    }
}

// Classes of up to 64 key tiles: lane i gets the class of tile base + i for the
// wave's own 32 queries qw .. (0 skip, 1 all visible, 2 mixed) in *mine;
// returns the tiles some wave of the block (queries q0 ..) needs.  cls: the
// mask's summary, or null for no mask.
__device__ __forceinline__ uint64_t tile_classes(const uint8_t* cls, int b, int q0, int wave, int Lq, int Lk, int nkt,
                                                 int base, int lane, uint32_t* mine) {
  const int kt = base + lane, qw = q0 + 32 * wave;
  uint32_t any = 0, c = 0;
  if (kt < nkt) {
    if (cls != nullptr) {
      const int nqt128 = (Lq + kBQ - 1) / kBQ;
#pragma unroll
      for (int i = 0; i < kRW; i++) {
        const int qq = q0 + 32 * i;
        if (qq >= Lq) break;
        const uint32_t x =
            *(const uint16_t*)(cls + (((int64_t)b * nqt128 + qq / kBQ) * nkt + kt) * kNW + ((qq >> 4) & 7));
        any |= x;
        if (i == wave) c = x;
      }
      const uint32_t c0 = c & 255u, c1 = qw + 16 < Lq ? c >> 8 : c0;  // (groups past Lq have class 0)
      c = c0 == c1 ? c0 : 2u;
    } else {
      c = qw >= Lq ? 0u : (kt + 1) * kBK <= Lk ? 1u : 2u;
      any = 1;
    }
  }
  *mine = c;
  return __ballot(any != 0);
}

// A K or V tile by direct-to-LDS loads: 8 pieces of 1 KB (8 rows); a piece's
// lane l fills slot l % 8 of row l / 8, so it fetches chunk (l % 8) ^
// kv_f(row).  Rows past Lk become zeros (an offset past the buffer's records).
// The caller waits for the loads (vmcnt(0)).
__device__ __forceinline__ void dma_piece(const uint16_t* base, int64_t stride, int k0, int piece, int Lk, uint16_t* dst,
                                          int lane) {
  const uint64_t a = (uint64_t)(base + (int64_t)k0 * stride);
  const uint4v rs = {(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)a),
                     (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu), 0x80000000u, 0x00020000u};
  const int r = piece * 8 + (lane >> 3);
  const uint32_t off = __umul24(r, (uint32_t)stride) * 2u + (((lane & 7) ^ kv_f(r)) << 4);
  const uint32_t lds = (uint32_t)__builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t*)(dst + piece * 512));
  buffer_lds16(rs, k0 + r < Lk ? off : 0xfffffff0u, lds);
}

struct KPair {  // a K row's chunks c and c + 4 and their rotation
  uint4v lo, hi;
  float2 cs[8];
};
// (rows past Lk repeat the last one: their scores are hidden)
__device__ __forceinline__ void kpair_load(KPair& p, const uint16_t* Kb, int64_t stride, const float2* tab, int k0, int r,
                                           int c, int Lk) {
  const int rr = k0 + r < Lk ? r : Lk - 1 - k0;
  load_pair(Kb + (int64_t)k0 * stride + __umul24(rr, (uint32_t)stride), true, c, p.lo, p.hi);
  load_cs(tab + (int64_t)k0 * 32, rr, c, p.cs);
}
template <bool BF16>
__device__ __forceinline__ void kpair_store(KPair& p, uint16_t* tile, int r, int c) {
  rot_pair<BF16>(p.lo, p.hi, p.cs);
  *(uint4v*)(tile + r * 64 + ((c ^ kv_f(r)) << 3)) = p.lo;
  *(uint4v*)(tile + r * 64 + (((c + 4) ^ kv_f(r)) << 3)) = p.hi;
}

// K and V tiles in a two-buffer LDS ring, one barrier per tile, four waves of
// 32 queries.  What bounds it: a wave's tile is ~200 VALU instructions (32 exp2,
// fma, add and 16 packed conversions of scores among them) and 16 MFMAs; at
// T = 2048 the SIMDs issue VALU 58% and MFMA 30% of the time, and the two
// overlap little.  Against the 16-query kernel a staged tile and its fragment
// reads serve twice the queries, and nothing of V passes through registers.
// Three blocks per CU (168 VGPRs); four, at 128 VGPRs, measured the same, eight
// waves a block slower (T 512 B 32 50 -> 58 us).  T = 2048, B = 16, 16 heads:
// 566 -> 434 us (635 TFLOP/s), T = 8192, B = 1, 12 heads 460 -> 322 us.
template <bool BF16, bool ROPEK>
__global__ __launch_bounds__(kRW * 64) __attribute__((amdgpu_waves_per_eu(3))) void sdpa32_ring(
    const uint16_t* __restrict__ Q, S4 qs, const uint16_t* __restrict__ K, S4 ks, const uint16_t* __restrict__ V, S4 vs,
    const uint8_t* __restrict__ mask, S4 ms, int mask_vec, const uint8_t* __restrict__ cls, uint16_t* __restrict__ O,
    S4 os, int Lq, int Lk, float scale_log2, const float2* __restrict__ tabq, const float2* __restrict__ tabk, int pK,
    int nqt, int nh) {
  static_assert(kRW == 4, "K staging: one chunk pair per thread");
  __shared__ __attribute__((aligned(16))) uint16_t Ks[2][kBK * 64];
  __shared__ __attribute__((aligned(16))) uint16_t Vs[2][kBK * 64];
  const int tid = threadIdx.x, lane = tid & 63, lg = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int qt, b, h;
  sdpa_block<true>(nqt, nh, qt, b, h);
  const int q0 = qt * 32 * kRW, q = q0 + 32 * wave + (lane & 31), qc = q < Lq ? q : Lq - 1;
  const int nkt = (Lk + kBK - 1) / kBK;
  const uint16_t* Kb = K + b * ks.s[0] + h * ks.s[1];
  const uint16_t* Vb = V + b * vs.s[0] + h * vs.s[1];
  const uint8_t* mrow = mask == nullptr ? nullptr : mask + b * ms.s[0] + (int64_t)qc * ms.s[2];

  int base = 0;
  uint32_t mine;
  uint64_t need = tile_classes(cls, b, q0, wave, Lq, Lk, nkt, 0, lane, &mine);
  // the next tile some wave needs (nkt: none) and its class for this wave
  auto next_tile = [&](uint32_t* c) -> int {
    while (need == 0) {
      base += 64;
      if (base >= nkt) return nkt;
      need = tile_classes(cls, b, q0, wave, Lq, Lk, nkt, base, lane, &mine);
    }
    const int i = __builtin_ctzll(need);
    need &= need - 1;
    *c = (uint32_t)__builtin_amdgcn_readlane((int)mine, i);
    return base + i;
  };
  Wave32 w;
  wave32_init<BF16>(w, Q + b * qs.s[0] + h * qs.s[1] + (int64_t)qc * qs.s[2], tabq, qc, lg);

  KPair kp;
  const int kr = tid >> 2, kc = tid & 3;
  auto fetch = [&](int kt, int bf) __attribute__((always_inline)) {
    const int k0 = kt * kBK;
#pragma unroll
    for (int i = 0; i < 8 / kRW; i++) dma_piece(Vb, vs.s[2], k0, wave * (8 / kRW) + i, Lk, Vs[bf], lane);
    if constexpr (ROPEK) {
      kpair_load(kp, Kb, ks.s[2], tabk, k0, kr, kc, Lk);
    } else {
#pragma unroll
      for (int i = 0; i < 8 / kRW; i++) dma_piece(Kb, ks.s[2], k0, wave * (8 / kRW) + i, Lk, Ks[bf], lane);
    }
  };
  // everything requested has landed (before the barrier that publishes it)
  auto landed = [&](int bf) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if constexpr (ROPEK) kpair_store<BF16>(kp, Ks[bf], kr, kc);
  };
  uint32_t cl = 0;
  int kt = next_tile(&cl), bf = 0;
  if (kt < nkt) {
    fetch(kt, 0);
    landed(0);
  }
  const Frag32 f = frag32(lane);
  __syncthreads();
  while (kt < nkt) {
    // the next tile into the other buffer (free since the last barrier)
    uint32_t ncl = 0;
    const int nk = next_tile(&ncl);
    if (nk < nkt) fetch(nk, bf ^ 1);
    if (cl != 0)
      wave32_tile<BF16>(w, f, Ks[bf], Vs[bf], kt * kBK, Lk, cl == 2, mrow, ms.s[3], mask_vec, scale_log2, lg);
    if (nk < nkt) landed(bf ^ 1);
    kt = nk;
    cl = ncl;
    bf ^= 1;
    __syncthreads();
  }
  wave32_store<BF16>(w, O, os, pK, b, h, q, Lq, lg);
}

// ------------------------------------------------------------------ f32 MFMA kernel (D = 64)

// Flash attention in f32 on v_mfma_f32_32x32x2_f32.  A block owns 32 queries
// of one (b, h); its four waves take the 32-key tiles those queries can see in
// turn, each with its own running max, sum and output, and merge them in LDS
// at the end, so a short sequence still runs its key tiles side by side and no
// wave waits for another in between.  What bounds it is the f32 matrix rate:
// a tile is 64 MFMAs of 64 cycles against 16 KB of K and V, so K goes through
// a wave-private LDS tile (rotated by RoPE on the way when fused) and V
// straight into operand registers, a whole 128-byte line per 32 lanes.
// S^T = K . Q^T leaves lane l with the scores of query l % 32 for keys
// 8 * (r / 4) + 4 * (l / 32) + r % 4, which are the columns the B operand of
// O^T += V^T . P^T takes when MFMA step r multiplies keys 8 * (r / 4) + r % 4
// and + 4: P stays in registers.
// Scores, probabilities and sums are f32; exp is the library's expf.
// Measured (12 heads): B = 8, T = 512, padded, sliding window 5820 -> 96 us
// (sdpa_simt before, one query per wave and every key rotated per query),
// B = 1, T = 93 104 -> 12 us, B = 1, T = 8192 without a window 88 TFLOP/s.
constexpr int kFQ = 32;  // queries per block
constexpr int kFK = 32;  // keys per tile
constexpr int kFW = 4;   // waves per block

__global__ __launch_bounds__(kFW * 64) __attribute__((amdgpu_waves_per_eu(2))) void sdpa_f32_mfma(
    const float* __restrict__ Q, S4 qs, const float* __restrict__ K, S4 ks, const float* __restrict__ V, S4 vs,
    const uint8_t* __restrict__ mask, S4 ms, const uint8_t* __restrict__ cls, float* __restrict__ O, S4 os, int Lq,
    int Lk, float scale, const float2* __restrict__ tabq, const float2* __restrict__ tabk, int nqt, int nh) {
  __shared__ __attribute__((aligned(16))) float buf[kFW][kFK * 64];  // K tiles; the partial outputs at the end
  __shared__ uint16_t todo[2 * kMaxKeyTiles];  // key tiles to visit: 2 * tile + mixed (Lk < 40960: sdpa_takes_f32)
  __shared__ int ntodo;
  __shared__ float part_m[kFW][kFQ], part_l[kFW][kFQ];

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, lg = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the query tiles of one (b, h) share K and V: consecutive blocks of one XCD
  const int t = xcd_tile(blockIdx.x, gridDim.x);
  const int qt = t % nqt, bh = t / nqt, h = bh % nh, b = bh / nh;
  const int q0 = qt * kFQ, q = q0 + l32;
  const int nkt = (Lk + kFK - 1) / kFK;
  const float* Kb = K + b * ks.s[0] + h * ks.s[1];
  const float* Vb = V + b * vs.s[0] + h * vs.s[1];

  // This lane's query: element e of qf[i] is column 8 * i + 4 * lg + e, the
  // columns its half supplies to MFMA steps e of chunk pair i
  float4v qf[8];
  {
    const float* qp = Q + b * qs.s[0] + h * qs.s[1] + (int64_t)(q < Lq ? q : Lq - 1) * qs.s[2] + 4 * lg;
#pragma unroll
    for (int i = 0; i < 8; i++) qf[i] = *(const float4v*)(qp + 8 * i);
    if (tabq != nullptr) {
      const float2* tp = tabq + (int64_t)(q < Lq ? q : Lq - 1) * 32 + 4 * lg;
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float2 cs = tp[8 * i + e];
          const float x0 = qf[i][e], x1 = qf[i + 4][e];
          qf[i][e] = fmaf(-x1, cs.y, x0 * cs.x);
          qf[i + 4][e] = fmaf(x0, cs.y, x1 * cs.x);
        }
    }
  }

  // The key tiles some query of the block sees, in order, from the mask
  // summary (classes of 16 queries x 64 keys) where there is one; wave 0
  // packs 64 tiles at a time.
  if (wave == 0) {
    int n = 0;
    for (int base = 0; base < nkt; base += 64) {
      const int kt = base + lane;
      int c = 0;  // 0 skip, 1 all visible, 2 mixed
      if (kt < nkt) {
        if (mask == nullptr) {
          c = (kt + 1) * kFK <= Lk ? 1 : 2;
        } else if (cls == nullptr) {
          c = 2;
        } else {
          const int g = (q0 >> 4) & 7, nkt64 = (Lk + kBK - 1) / kBK, nqt128 = (Lq + kBQ - 1) / kBQ;
          const uint8_t* p = cls + (((int64_t)b * nqt128 + q0 / kBQ) * nkt64 + (kt >> 1)) * kNW + g;
          // (a group past Lq has class 0: its queries are not stored)
          const int c0 = p[0], c1 = q0 + 16 < Lq ? p[1] : p[0];
          c = c0 == c1 ? c0 : 2;
        }
      }
      const uint64_t m = __ballot(c != 0);
      if (c != 0) todo[n + __popcll(m & ((1ull << lane) - 1))] = (uint16_t)(2 * kt + (c == 2));
      n += __popcll(m);
    }
    if (lane == 0) ntodo = n;
  }
  __syncthreads();
  const int nt = ntodo;

  // K tile staging: 8 lanes per row; lane c8 of a row holds its chunks c8 and
  // c8 + 8 (columns 4 * c8 .. and their rotation partners + 32)
  const int kr = lane >> 3, c8 = lane & 7;
  float4v klo[4], khi[4];
  auto load_k = [&](int kt) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int key = kt * kFK + i * 8 + kr;
      const float* p = Kb + (int64_t)(key < Lk ? key : Lk - 1) * ks.s[2] + 4 * c8;
      klo[i] = *(const float4v*)p;
      khi[i] = *(const float4v*)(p + 32);
    }
  };
  // chunk c of row r at c ^ (r & 15): a 16-lane pass of the fragment reads
  // (16 rows, one chunk) covers all 64 banks
  auto kslot = [](int r, int c) { return r * 64 + ((c ^ (r & 15)) << 2); };
  float* kb = buf[wave];
  auto store_k = [&](int kt) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int r = i * 8 + kr, key = kt * kFK + r;
      float4v lo = klo[i], hi = khi[i];
      if (tabk != nullptr) {
        const float4v* tp = (const float4v*)(tabk + (int64_t)(key < Lk ? key : Lk - 1) * 32 + 4 * c8);
        const float4v t0 = tp[0], t1 = tp[1];
        const float cc[4] = {t0[0], t0[2], t1[0], t1[2]}, ss[4] = {t0[1], t0[3], t1[1], t1[3]};
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float x0 = lo[e], x1 = hi[e];
          lo[e] = fmaf(-x1, ss[e], x0 * cc[e]);
          hi[e] = fmaf(x0, ss[e], x1 * cc[e]);
        }
      }
      *(float4v*)(kb + kslot(r, c8)) = lo;
      *(float4v*)(kb + kslot(r, c8 + 8)) = hi;
    }
  };

  float16v o[2];
#pragma unroll
  for (int d = 0; d < 2; d++)
#pragma unroll
    for (int r = 0; r < 16; r++) o[d][r] = 0.f;
  float m = -INFINITY, l = 0.f;

  int i0 = wave;
  if (i0 < nt) load_k(todo[i0] >> 1);
  for (; i0 < nt; i0 += kFW) {
    const int ent = __builtin_amdgcn_readfirstlane((int)todo[i0]), kt = ent >> 1, k0 = kt * kFK;
    store_k(kt);
    // the tile is this wave's own: its LDS stores and loads only need to stay
    // in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // V of the tile, the next tile's K
    float v[2][16];
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int key = k0 + 8 * (r >> 2) + 4 * lg + (r & 3);
      const float* p = Vb + (int64_t)(key < Lk ? key : Lk - 1) * vs.s[2] + l32;
      v[0][r] = p[0];
      v[1][r] = p[32];
    }
    if (i0 + kFW < nt) load_k(todo[i0 + kFW] >> 1);

    float16v s;
#pragma unroll
    for (int r = 0; r < 16; r++) s[r] = 0.f;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float4v kf = *(const float4v*)(kb + kslot(l32, 2 * i + lg));
#pragma unroll
      for (int e = 0; e < 4; e++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[e], qf[i][e], s, 0, 0, 0);
    }
    // (the next store_k must not overtake these reads)
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_wave_barrier();

    const bool mixed = ent & 1;
    const uint8_t* mrow = mask == nullptr ? nullptr
                                          : mask + b * ms.s[0] + h * ms.s[1] + (int64_t)(q < Lq ? q : Lq - 1) * ms.s[2];
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      s[r] *= scale;
      if (mixed) {
        const int key = k0 + 8 * (r >> 2) + 4 * lg + (r & 3);
        const bool vis = key < Lk && (mrow == nullptr || mrow[(int64_t)key * ms.s[3]] != 0);
        s[r] = vis ? s[r] : -INFINITY;
      }
      mx = fmaxf(mx, s[r]);
    }
    mx = max_xor32(mx);
    const float mnew = fmaxf(m, mx);
    const float mc = mnew == -INFINITY ? 0.f : mnew;  // no visible key yet: every weight is exp(-inf) = 0
    const float alpha = expf(m - mc);
    m = mnew;
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      s[r] = expf(s[r] - mc);
      sum += s[r];
    }
    l = l * alpha + sum;
    if (!__all(alpha == 1.0f)) {
#pragma unroll
      for (int d = 0; d < 2; d++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[d][r] *= alpha;
    }
    // A non-finite V must not reach a query whose weight for that key is 0
    // (hidden, or exp underflowed), as 0 * inf in the product would: such a
    // tile is added key by key, zero weights skipped.
    float fin = 0.f;
#pragma unroll
    for (int r = 0; r < 16; r++) fin += v[0][r] * 0.f + v[1][r] * 0.f;
    if (__any(fin != 0.f)) {  // 0 * finite = 0, 0 * (inf or NaN) = NaN
#pragma unroll
      for (int r = 0; r < 16; r++) kb[(8 * (r >> 2) + 4 * lg + (r & 3)) * 32 + l32] = s[r];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll 1
      for (int j = 0; j < kFK; j++) {
        const float p = kb[j * 32 + l32];
        if (p == 0.f) continue;  // keys past Lk among them
        const float* vp = Vb + (int64_t)(k0 + j) * vs.s[2] + 4 * lg;
#pragma unroll
        for (int d = 0; d < 2; d++)
#pragma unroll
          for (int r = 0; r < 16; r++) o[d][r] = fmaf(p, vp[32 * d + 8 * (r >> 2) + (r & 3)], o[d][r]);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      continue;
    }
#pragma unroll
    for (int r = 0; r < 16; r++)
#pragma unroll
      for (int d = 0; d < 2; d++) o[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[d][r], s[r], o[d], 0, 0, 0);
  }

  // merge the waves' outputs: weights exp(m_w - max); wave w finishes
  // registers [8 w, 8 w + 8) of the 32
  l = sum_xor32(l);
  if (lg == 0) {
    part_m[wave][l32] = m;
    part_l[wave][l32] = l;
  }
  __syncthreads();  // every wave is done with its K tile
#pragma unroll
  for (int d = 0; d < 2; d++)
#pragma unroll
    for (int r = 0; r < 16; r++) buf[wave][(d * 16 + r) * 64 + lane] = o[d][r];
  __syncthreads();
  float mt = -INFINITY;
#pragma unroll
  for (int w = 0; w < kFW; w++) mt = fmaxf(mt, part_m[w][l32]);
  const float mc = mt == -INFINITY ? 0.f : mt;
  float wt[kFW], lt = 0.f;
#pragma unroll
  for (int w = 0; w < kFW; w++) {
    wt[w] = expf(part_m[w][l32] - mc);
    lt += part_l[w][l32] * wt[w];
  }
  const float inv = 1.0f / lt;
  if (q >= Lq) return;
  float* op = O + b * os.s[0] + h * os.s[1] + (int64_t)q * os.s[2];
#pragma unroll
  for (int r4 = 0; r4 < 2; r4++) {
    const int x = wave * 8 + r4 * 4;  // register x: column 32 * (x / 16) + 8 * (x % 16 / 4) + 4 * lg
    float4v ov;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      float a = 0.f;
#pragma unroll
      for (int w = 0; w < kFW; w++) a += buf[w][(x + e) * 64 + lane] * wt[w];
      ov[e] = a * inv;
    }
    *(float4v*)(op + 32 * (x >> 4) + 8 * ((x & 15) >> 2) + 4 * lg) = ov;
  }
}

// ------------------------------------------------------------------ SIMT kernel (any dtype / D)

// One wave per query row: scores for every key into LDS, softmax in f32,
// then each lane accumulates its own output dims.
__device__ __forceinline__ float roped(int dt, const void* base, int64_t row, int64_t sd, int d, int D,
                                       const float2* tab, int pos) {
  float x = load_f(base, row + d * sd, dt);
  if (tab == nullptr) return x;
  int half = D / 2;
  int j = d < half ? d : d - half;
  float2 cs = tab[pos * half + j];
  float p = load_f(base, row + (d < half ? d + half : d - half) * sd, dt);
  // rotation rounded to the storage dtype, as a separate Backend.rope stores it
  float r = d < half ? fmaf(-p, cs.y, x * cs.x) : fmaf(p, cs.y, x * cs.x);
  return round_to(r, dt);
}

__global__ __launch_bounds__(64) void sdpa_simt(int dt, const void* __restrict__ Q, S4 qs,
                                                const void* __restrict__ K, S4 ks, const void* __restrict__ V, S4 vs,
                                                const uint8_t* __restrict__ mask, S4 ms, void* __restrict__ O, S4 os,
                                                int H, int Lq, int Lk, int D, float scale,
                                                const float2* __restrict__ tabq, const float2* __restrict__ tabk) {
  extern __shared__ float sc[];  // [Lk] scores, then [D] roped query
  float* qv = sc + Lk;
  const int lane = threadIdx.x;
  const int q = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int64_t qrow = b * qs.s[0] + h * qs.s[1] + (int64_t)q * qs.s[2];
  for (int d = lane; d < D; d += 64) qv[d] = roped(dt, Q, qrow, qs.s[3], d, D, tabq, q);
  __syncthreads();
  float mx = -INFINITY;
  for (int j = lane; j < Lk; j += 64) {
    bool vis = mask == nullptr || mask[b * ms.s[0] + h * ms.s[1] + (int64_t)q * ms.s[2] + (int64_t)j * ms.s[3]];
    float s = -INFINITY;
    if (vis) {
      const int64_t krow = b * ks.s[0] + h * ks.s[1] + (int64_t)j * ks.s[2];
      float acc = 0.f;
      for (int d = 0; d < D; d++) acc = fmaf(qv[d], roped(dt, K, krow, ks.s[3], d, D, tabk, j), acc);
      s = acc * scale;
    }
    sc[j] = s;
    mx = fmaxf(mx, s);
  }
  mx = wave_max(mx);
  float sum = 0.f;
  for (int j = lane; j < Lk; j += 64) {
    float p = sc[j] == -INFINITY ? 0.f : expf(sc[j] - mx);
    sc[j] = p;
    sum += p;
  }
  sum = wave_sum(sum);
  __syncthreads();
  const float inv = 1.0f / sum;
  for (int d = lane; d < D; d += 64) {
    float acc = 0.f;
    for (int j = 0; j < Lk; j++) {
      float p = sc[j];
      if (p != 0.f) acc = fmaf(p, load_f(V, b * vs.s[0] + h * vs.s[1] + (int64_t)j * vs.s[2] + d * vs.s[3], dt), acc);
    }
    store_f(O, b * os.s[0] + h * os.s[1] + (int64_t)q * os.s[2] + d * os.s[3], dt, acc * inv);
  }
}

}  // namespace hb

using namespace hb;

extern "C" int hb_sdpa_mask_info_bytes(int64_t B, int64_t Lq, int64_t Lk, size_t* bytes) {
  HB_API_BEGIN
  HB_REQUIRE(bytes && B >= 0 && Lq >= 0 && Lk >= 0, "hb_sdpa_mask_info_bytes: bad arguments");
  *bytes = mask_info_bytes(B, Lq, Lk);
  HB_API_END
}

extern "C" int hb_sdpa_mask_info(uintptr_t ctx, uintptr_t mask, const int64_t* ms, int64_t B, int64_t Lq, int64_t Lk,
                                 uintptr_t info) {
  HB_API_BEGIN
  HB_REQUIRE(mask && ms && info, "hb_sdpa_mask_info: null argument");
  HB_REQUIRE(B >= 0 && Lq >= 0 && Lk >= 0 && B < 65536 && Lq < (1 << 30) && Lk < (1 << 30),
             "hb_sdpa_mask_info: bad shape");
  if (B == 0 || Lq == 0 || Lk == 0) return 0;
  launch_mask_info(stream_of(ctx), (const uint8_t*)mask, s4(ms), B, Lq, Lk, (uint8_t*)info);
  check_launch("hb_sdpa_mask_info");
  HB_API_END
}

// The MFMA kernel's conditions on a call (else sdpa_simt): 16-bit data,
// D = 64, unit inner strides, 16-byte aligned rows and 8-element strides, a
// mask that does not vary over heads, at most kMaxKeyTiles key tiles, and K /
// V row strides in [0, 2^24) (the kernel adds them as unsigned 24-bit
// products).  Lk == 0 takes the generic kernel: every row is fully masked,
// which it gives as 0/0 = NaN, as both kernels do for a row whose keys are
// all masked, and it needs no mask summary.
static bool sdpa_takes_mfma(int dt, uintptr_t q, const int64_t* qs, uintptr_t k, const int64_t* ks, uintptr_t v,
                            const int64_t* vs, uintptr_t mask, const int64_t* ms, uintptr_t o, const int64_t* os,
                            int64_t Lk, int64_t D) {
  return Lk > 0 && (dt == HB_F16 || dt == HB_BF16) && D == 64 && qs[3] == 1 && ks[3] == 1 && vs[3] == 1 &&
         os[3] == 1 && q % 16 == 0 && k % 16 == 0 && v % 16 == 0 && o % 8 == 0 && qs[2] % 8 == 0 &&
         ks[2] % 8 == 0 && vs[2] % 8 == 0 && qs[0] % 8 == 0 && qs[1] % 8 == 0 && ks[0] % 8 == 0 &&
         ks[1] % 8 == 0 && vs[0] % 8 == 0 && vs[1] % 8 == 0 && os[0] % 4 == 0 && os[1] % 4 == 0 &&
         os[2] % 4 == 0 && (mask == 0 || ms[1] == 0) && (Lk + kBK - 1) / kBK <= kMaxKeyTiles && ks[2] >= 0 &&
         ks[2] < (1 << 24) && vs[2] >= 0 && vs[2] < (1 << 24);
}

// The f32 MFMA kernel's conditions: D = 64, unit inner strides, 16-byte
// aligned rows, and no more keys than sdpa_simt takes.  Any mask goes: one
// without a summary (it varies over heads) is read for every tile.
static bool sdpa_takes_f32(int dt, uintptr_t q, const int64_t* qs, uintptr_t k, const int64_t* ks, uintptr_t v,
                           const int64_t* vs, uintptr_t o, const int64_t* os, int64_t Lk, int64_t D) {
  auto rows16 = [](uintptr_t p, const int64_t* s) {
    return p % 16 == 0 && s[3] == 1 && s[0] % 4 == 0 && s[1] % 4 == 0 && s[2] % 4 == 0;
  };
  return dt == HB_F32 && D == 64 && Lk > 0 && rows16(q, qs) && rows16(k, ks) && v % 4 == 0 && vs[3] == 1 &&
         rows16(o, os) && (Lk + D) * 4 <= 160 * 1024;
}

// The argument checks every sdpa entry point makes before it launches
// anything.
static void sdpa_check(int dt, const int64_t* qs, const int64_t* ks, const int64_t* vs, uintptr_t mask,
                       const int64_t* ms, const int64_t* os, int64_t B, int64_t H, int64_t Lq, int64_t Lk, int64_t D) {
  HB_REQUIRE(dt == HB_F32 || dt == HB_F16 || dt == HB_BF16, "hb_sdpa: dtype must be f32, f16 or bf16");
  HB_REQUIRE(qs && ks && vs && os, "hb_sdpa: null strides");
  HB_REQUIRE(!mask || ms, "hb_sdpa: mask without strides");
  HB_REQUIRE(B >= 0 && H >= 0 && Lq >= 0 && Lk >= 0 && D > 0, "hb_sdpa: bad shape");
  HB_REQUIRE(B < 65536 && H < 65536 && Lq < (1 << 30) && Lk < (1 << 30), "hb_sdpa: shape too large");
}

// pK > 0: o is the panel-order [B*Lq, pK] matrix (pK = H*D), MFMA path only.
// A masked call on the MFMA path without a summary (mask_info == 0) builds
// one into a pool block, unless `noalloc`, where that is an error.
static void sdpa_impl(uintptr_t ctx, int dt, uintptr_t q, const int64_t* qs, uintptr_t k, const int64_t* ks,
                      uintptr_t v, const int64_t* vs, uintptr_t mask, const int64_t* ms, uintptr_t mask_info,
                      uintptr_t o, const int64_t* os, int64_t B, int64_t H, int64_t Lq, int64_t Lk, int64_t D,
                      float scale, double rope_q, double rope_k, int pK, bool noalloc = false) {
  sdpa_check(dt, qs, ks, vs, mask, ms, os, B, H, Lq, Lk, D);
  if (B == 0 || H == 0 || Lq == 0) return;
  HB_REQUIRE((rope_q <= 0 && rope_k <= 0) || D % 2 == 0, "hb_sdpa: rope needs an even head dim");
  HB_REQUIRE(!noalloc || (rope_q <= 0 && rope_k <= 0), "hb_sdpa_noalloc: no RoPE tables");
  hipStream_t st = stream_of(ctx);
  const float2* tq = rope_q > 0 ? (const float2*)rope_table(ctx, Lq, D, rope_q) : nullptr;
  const float2* tk = rope_k > 0 ? (const float2*)rope_table(ctx, Lk, D, rope_k) : nullptr;
  S4 Qs = s4(qs), Ks = s4(ks), Vs = s4(vs), Ms = s4(ms), Os = s4(os);
  const bool fast = sdpa_takes_mfma(dt, q, qs, k, ks, v, vs, mask, ms, o, os, Lk, D);
  if (pK > 0)
    HB_REQUIRE(fast && o % 16 == 0 && pK == H * D,
               "hb_sdpa_panel: needs the MFMA path (f16/bf16, D = 64, aligned operands, mask not varying over heads)");
  if (fast) {
    int nqt = (int)((Lq + kBQ - 1) / kBQ);
    uint8_t* info = (uint8_t*)mask_info;
    CallScratch tmp(ctx);
    if (mask) {
      if (!info) {
        HB_REQUIRE(!noalloc, "hb_sdpa_noalloc: no mask summary");
        HB_REQUIRE(tmp.take(mask_info_bytes(B, Lq, Lk)), "hb_sdpa: out of device memory for the mask summary");
        info = (uint8_t*)tmp.p;
        launch_mask_info(st, (const uint8_t*)mask, Ms, B, Lq, Lk, info);
        check_launch("hb_sdpa(mask info)");
      }
    } else {
      info = nullptr;
    }
    const float sl2 = scale * 1.4426950408889634f;
    const int64_t nblk = (int64_t)nqt * H * B;
    HB_REQUIRE(nblk < ((int64_t)1 << 31), "hb_sdpa: too many (batch, head, query tile) blocks");
    // Which kernel: by the number of keys only, so that a sequence's bits depend
    // neither on its batch nor on how its mask is given (none, one row for every
    // query, or a row per query: the two kernels sum in different orders).  Up to
    // 1024 keys the 16-query kernel has the shorter chain per block, and with a
    // windowed mask it is the faster one: us, 16 / 32 queries a wave, 12 heads
    // (16 from T = 1024), padded below T = 1024, RoPE on both operands:
    //   every key:  T 128 B 1 9.0 / 9.6, T 384 B 8 18.9 / 19.3, T 512 B 4 19.0 /
    //               18.3, T 512 B 32 55.4 / 50.2, T 2048 B 16 566 / 465
    //   windowed:   T 512 B 8 23.4 / 26.3, T 512 B 32 53.0 / 53.2, T 1024 B 8
    //               59.1 / 61.3, T 2048 B 16 125 / 121
    const bool all_keys = !mask || ms[2] == 0;
    const bool wide = Lk > 1024;
    if (wide) {
      // Where every query tile reads every key, K is rotated once in a pass of
      // its own instead of by every block that stages it (T 2048 B 16 465 -> 434,
      // T 8192 B 1 367 -> 322 us, the pass included), if that is shared by eight
      // query tiles, or the pass is small against the chain of tiles whose
      // rotations it takes out.  us, in the blocks / in a pass, 12 heads:
      //   queries x keys  1024 x 2048 B 16 183 / 163, 512 x 2048 B 16 padded 75 /
      //   78, 128 x 4096 B 16 98 / 141, 1 x 2048 B 64 90 / 191; few (b, h):
      //   1 x 2048 B 1 41 / 38, 256 x 4096 B 4 95 / 80, 1 x 8192 B 4 176 / 146
      // (Without memory for the rotated copy the blocks rotate what they stage.)
      CallScratch rotated(ctx);
      const int64_t kblk = (Lk + 63) / 64 * B * H;
      const bool pass = tk && all_keys && (nqt >= 8 || B * H <= 64);
      if (pass && kblk < ((int64_t)1 << 31) && rotated.take((size_t)(B * H * Lk * 64 * 2))) {
        auto kern = dt == HB_F16 ? rope_k_kernel<false> : rope_k_kernel<true>;
        kern<<<(unsigned)kblk, 256, 0, st>>>((const uint16_t*)k, Ks, (uint16_t*)rotated.p, (int)Lk, (int)H, (int)(B * H),
                                             tk);
        check_launch("hb_sdpa (rotate K)");
        k = (uintptr_t)rotated.p;
        Ks = S4{{H * Lk * 64, Lk * 64, 64, 1}};
        tk = nullptr;
      }
      const int mask_vec = mask && ms[3] == 1 && mask % 16 == 0 && ms[0] % 16 == 0 && ms[2] % 16 == 0;
      auto kern = dt == HB_F16 ? (tk ? sdpa32_ring<false, true> : sdpa32_ring<false, false>)
                               : (tk ? sdpa32_ring<true, true> : sdpa32_ring<true, false>);
      kern<<<(unsigned)nblk, 256, 0, st>>>((const uint16_t*)q, Qs, (const uint16_t*)k, Ks, (const uint16_t*)v, Vs,
                                           (const uint8_t*)mask, Ms, mask_vec, info, (uint16_t*)o, Os, (int)Lq, (int)Lk,
                                           sl2, tq, tk, pK, nqt, (int)H);
    } else {
      // 8 contiguous mask bytes per lane and load, of any alignment
      const int mask_vec = mask && ms[3] == 1;
      auto kern = dt == HB_F16 ? sdpa_mfma<false> : sdpa_mfma<true>;
      kern<<<(unsigned)nblk, kNT, 0, st>>>((const uint16_t*)q, Qs, (const uint16_t*)k, Ks, (const uint16_t*)v, Vs,
                                           (const uint8_t*)mask, Ms, mask_vec, info, (uint16_t*)o, Os, (int)Lq, (int)Lk,
                                           sl2, tq, tk, pK, nqt, (int)H);
    }
    check_launch("hb_sdpa");
  } else if (sdpa_takes_f32(dt, q, qs, k, ks, v, vs, o, os, Lk, D)) {
    const int nqt = (int)((Lq + kFQ - 1) / kFQ);
    const int64_t nblk = (int64_t)nqt * H * B;
    HB_REQUIRE(nblk < ((int64_t)1 << 31), "hb_sdpa: too many (batch, head, query tile) blocks");
    // (a caller's summary only describes a mask that does not vary over heads)
    const uint8_t* info = mask && ms[1] == 0 ? (const uint8_t*)mask_info : nullptr;
    sdpa_f32_mfma<<<(unsigned)nblk, kFW * 64, 0, st>>>((const float*)q, Qs, (const float*)k, Ks, (const float*)v, Vs,
                                                       (const uint8_t*)mask, Ms, info, (float*)o, Os, (int)Lq, (int)Lk,
                                                       scale, tq, tk, nqt, (int)H);
    check_launch("hb_sdpa(f32)");
  } else {
    size_t lds = sizeof(float) * (size_t)(Lk + D);
    HB_REQUIRE(lds <= 160 * 1024, "hb_sdpa: sequence too long for the generic kernel");
    if (lds > 64 * 1024)
      HB_CHECK_HIP(hipFuncSetAttribute((const void*)sdpa_simt, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    dim3 grid((unsigned)Lq, (unsigned)H, (unsigned)B);
    sdpa_simt<<<grid, 64, lds, st>>>(dt, (const void*)q, Qs, (const void*)k, Ks, (const void*)v, Vs,
                                     (const uint8_t*)mask, Ms, (void*)o, Os, (int)H, (int)Lq, (int)Lk, (int)D, scale,
                                     tq, tk);
    check_launch("hb_sdpa(generic)");
  }
}

// The device address of `scratch` on each device, found once per device at
// hb_init (with that device current).  Host code passes these addresses to
// kernels; the array's name is only a host-side stand-in.
static std::mutex g_scratch_mu;
static void* g_scratch[64];

namespace hb {
void sdpa_scratch_init(int device) {
  HB_REQUIRE(device >= 0 && device < 64, "sdpa scratch: device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch[device]) return;
  void* p = nullptr;
  HB_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  HB_REQUIRE(p != nullptr, "sdpa scratch: no device address");
  g_scratch[device] = p;
}
}  // namespace hb

extern "C" int hb_sdpa_noalloc(uintptr_t ctx, int dt, uintptr_t q, const int64_t* qs, uintptr_t k, const int64_t* ks,
                               uintptr_t v, const int64_t* vs, uintptr_t mask, const int64_t* ms, uintptr_t o,
                               const int64_t* os, int64_t B, int64_t H, int64_t Lq, int64_t Lk, int64_t D,
                               float scale) {
  HB_API_BEGIN
  sdpa_check(dt, qs, ks, vs, mask, ms, os, B, H, Lq, Lk, D);
  uintptr_t info = 0;
  // Only a masked call on the MFMA path reads a summary; the others launch
  // the generic kernel alone and have no size limit here.
  if (mask && B > 0 && H > 0 && Lq > 0 && sdpa_takes_mfma(dt, q, qs, k, ks, v, vs, mask, ms, o, os, Lk, D)) {
    const size_t need = mask_info_bytes(B, Lq, Lk);
    HB_REQUIRE(need <= kSdpaScratchBytes,
               "hb_sdpa_noalloc: the mask summary needs " + std::to_string(need) + " bytes, more than the " +
                   std::to_string(kSdpaScratchBytes) + "-byte scratch (B * ceil(Lq/128) * ceil(Lk/64) * 8); "
                   "use hb_sdpa for this shape");
    void* p;
    {
      std::lock_guard<std::mutex> lock(g_scratch_mu);
      p = g_scratch[device_of(ctx) & 63];
    }
    HB_REQUIRE(p, "hb_sdpa_noalloc: scratch not set up for this device (hb_init does it)");
    // every byte the attention kernel reads is written here: nothing to clear
    launch_mask_info(stream_of(ctx), (const uint8_t*)mask, s4(ms), B, Lq, Lk, (uint8_t*)p);
    check_launch("hb_sdpa_noalloc(mask info)");
    info = (uintptr_t)p;
  }
  sdpa_impl(ctx, dt, q, qs, k, ks, v, vs, mask, ms, info, o, os, B, H, Lq, Lk, D, scale, 0.0, 0.0, 0, true);
  HB_API_END
}

extern "C" int hb_sdpa(uintptr_t ctx, int dt, uintptr_t q, const int64_t* qs, uintptr_t k, const int64_t* ks,
                       uintptr_t v, const int64_t* vs, uintptr_t mask, const int64_t* ms, uintptr_t mask_info,
                       uintptr_t o, const int64_t* os, int64_t B, int64_t H, int64_t Lq, int64_t Lk, int64_t D,
                       float scale, double rope_q, double rope_k) {
  HB_API_BEGIN
  sdpa_impl(ctx, dt, q, qs, k, ks, v, vs, mask, ms, mask_info, o, os, B, H, Lq, Lk, D, scale, rope_q, rope_k, 0);
  HB_API_END
}

extern "C" int hb_sdpa_panel(uintptr_t ctx, int dt, uintptr_t q, const int64_t* qs, uintptr_t k, const int64_t* ks,
                             uintptr_t v, const int64_t* vs, uintptr_t mask, const int64_t* ms, uintptr_t mask_info,
                             uintptr_t o, int64_t B, int64_t H, int64_t Lq, int64_t Lk, int64_t D, float scale,
                             double rope_q, double rope_k) {
  HB_API_BEGIN
  const int64_t os[4] = {0, 0, 0, 1};  // unused: the output is addressed in panel order
  sdpa_impl(ctx, dt, q, qs, k, ks, v, vs, mask, ms, mask_info, o, os, B, H, Lq, Lk, D, scale, rope_q, rope_k,
            (int)(H * D));
  HB_API_END
}
