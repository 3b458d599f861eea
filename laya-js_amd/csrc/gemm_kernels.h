// MFMA GEMM kernels and their launchers (templates), shared by the
// translation units that instantiate them by weight format: gemm_f16.hip
// (16-bit weights), gemm_q8.hip and gemm_q4.hip (laya's quantized format);
// gemm.hip holds the entry points, the SIMT kernels and the dispatch.
#pragma once
#include <math.h>

#include <atomic>
#include <stdexcept>
#include <type_traits>

#include "common.h"

namespace hb {


// ------------------------------------------------------------------ helpers


template <bool BF16>
__device__ __forceinline__ float16v mfma32(const uint4v& a, const uint4v& b, float16v c) {
  if constexpr (BF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0,
                                                  0, 0);
  }
}

template <bool BF16>
__device__ __forceinline__ float to_f(uint32_t h) {
  return BF16 ? bf16_to_f32((uint16_t)h) : f16_bits_to_f32((uint16_t)h);
}
template <bool BF16>
__device__ __forceinline__ uint16_t from_f(float v) {
  return BF16 ? f32_to_bf16(v) : f32_to_f16_bits(v);
}

// LDS element offset of 16-byte chunk c of row r in a [rows][64] u16 tile.
__device__ __forceinline__ int swz(int r, int c) { return r * 64 + ((c ^ (r & 7)) << 3); }

// One 16-byte global -> LDS copy per lane (global_load_lds_dwordx4): lane l
// fills LDS bytes [lds + 16 l, lds + 16 l + 16), `lds` being the wave's
// (wave-uniform) LDS byte address.  Issued from inline asm, so the compiler
// neither orders later LDS accesses behind it nor counts it in its own load
// waits (an extra load in flight only makes those waits stronger); the
// caller waits for it (vmcnt) before anything reads the destination.
__device__ __forceinline__ void lds_copy16(const void* g, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds) : "memory", "m0");
}

// Quantized code e (0..7) of a chunk: q8 codes are bytes of (w0, w1), q4
// codes nibbles of w0 (even column in the low nibble).
template <int QB, bool AFF>
__device__ __forceinline__ int qcode(uint32_t w0, uint32_t w1, int e) {
  if constexpr (QB == 8) {
    uint32_t w = e < 4 ? w0 : w1;
    int sh = 8 * (e & 3);
    return AFF ? (int)((w >> sh) & 0xff) : (int)(int8_t)((w >> sh) & 0xff);
  } else {
    int v = (int)((w0 >> (4 * e)) & 0xf);
    return AFF ? v : ((v ^ 8) - 8);
  }
}

// 8 dequantized weights as 16-bit values.  f16 with f16 scales: one f16 fma
// (q is exact in f16), so the weight is fl16(q*s + z) rounded once.  Other
// combinations compute in f32 and round once to the storage type.
template <int QB, bool AFF, bool SF32, bool BF16>
__device__ __forceinline__ uint4v dequant8(uint32_t w0, uint32_t w1, uint32_t sbits, uint32_t zbits, float sf,
                                           float zf) {
  uint32_t out[4];
  if constexpr (!SF32 && !BF16) {
    // Two codes per 32-bit word, each as the f16 1024 + c (c in 0..255 or
    // 0..15 is the low mantissa bits under the exponent of 1024, exact), then
    // one packed subtraction gives the code as f16 exactly and one packed
    // multiply (symmetric) or fma (affine) rounds q*s (+ z) once.
    const half2v s2 = __builtin_bit_cast(half2v, (sbits & 0xffffu) * 0x10001u);
    const half2v z2 = __builtin_bit_cast(half2v, (zbits & 0xffffu) * 0x10001u);
    uint32_t pr[4];  // value pairs (2e, 2e + 1) in the low bits of each half
    if constexpr (QB == 8) {
      // byte b of w0:w1 -> half (b & 1) of pair b / 2
      pr[0] = __builtin_amdgcn_perm(0u, w0, 0x0c010c00u);
      pr[1] = __builtin_amdgcn_perm(0u, w0, 0x0c030c02u);
      pr[2] = __builtin_amdgcn_perm(0u, w1, 0x0c010c00u);
      pr[3] = __builtin_amdgcn_perm(0u, w1, 0x0c030c02u);
    } else {
      // nibble e of w0 (e even: low nibble of byte e / 2)
      const uint32_t lo = w0 & 0x0f0f0f0fu, hi = (w0 >> 4) & 0x0f0f0f0fu;
#pragma unroll
      for (int p = 0; p < 4; p++) pr[p] = __builtin_amdgcn_perm(hi, lo, 0x0c040c00u + 0x00010001u * p);
    }
    // signed codes are stored offset by 2^(QB-1): q + 2^(QB-1) = c ^ 2^(QB-1)
    constexpr uint32_t flip = AFF ? 0u : (QB == 8 ? 0x00800080u : 0x00080008u);
    constexpr _Float16 base = AFF ? (_Float16)1024 : (_Float16)(1024 + (1 << (QB - 1)));
#pragma unroll
    for (int p = 0; p < 4; p++) {
      const half2v q2 = __builtin_bit_cast(half2v, (pr[p] ^ flip) | 0x64006400u) - half2v{base, base};
      const half2v r2 = AFF ? __builtin_elementwise_fma(q2, s2, z2) : q2 * s2;
      out[p] = __builtin_bit_cast(uint32_t, r2);
    }
  } else {
    const float s = SF32 ? sf : f16_bits_to_f32((uint16_t)sbits);
    const float z = SF32 ? zf : f16_bits_to_f32((uint16_t)zbits);
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      float q0 = (float)qcode<QB, AFF>(w0, w1, e), q1 = (float)qcode<QB, AFF>(w0, w1, e + 1);
      float r0 = AFF ? fmaf(q0, s, z) : q0 * s;
      float r1 = AFF ? fmaf(q1, s, z) : q1 * s;
      out[e >> 1] = (uint32_t)from_f<BF16>(r0) | ((uint32_t)from_f<BF16>(r1) << 16);
    }
  }
  return uint4v{out[0], out[1], out[2], out[3]};
}

struct QW {  // quantized weight operand
  const uint8_t* q;
  const void* scales;
  const void* zeros;
  int G;      // groups per row
  int group;  // values per group
};

// The fused-projection epilogue (QKV): y = x . W^T with W the
// stacked [3 * H * 64, K] q / k / v projection, written head-major as
// [3][B][H][L][64] (B = M / L) with RoPE applied to the q and k parts.
struct QK {
  const float2* tab;  // RoPE cos / sin [L][32], or null: no rotation
  int L;              // sequence length (M = B * L)
  int H;              // heads (N = 3 * H * 64)
};

// Copies a [BM][BNO] 16-bit tile staged in LDS to Y with 16-byte coalesced
// stores; with a residual, y = round(tile + resid) (linear, then add).
template <bool BF16, int BM, int BNO, int NT>
__device__ __forceinline__ void write_tile(const uint16_t* Cs, int m0, int n0, int M, int N,
                                           const uint16_t* __restrict__ R, int64_t ldr, uint16_t* __restrict__ Y,
                                           int64_t ldy) {
  constexpr int CPR = BNO / 8;  // chunks per row
  for (int q = threadIdx.x; q < BM * CPR; q += NT) {
    const int r = q / CPR, c = q % CPR;
    const int gm = m0 + r, gn = n0 + c * 8;
    if (gm >= M || gn >= N) continue;
    uint4v v = *(const uint4v*)(Cs + r * BNO + c * 8);
    if (gn + 8 <= N) {
      if (R != nullptr) {
        uint4v rv = *(const uint4v*)(R + (int64_t)gm * ldr + gn);
        uint32_t vv[4] = {v.x, v.y, v.z, v.w};
        uint32_t rr[4] = {rv.x, rv.y, rv.z, rv.w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
          uint16_t lo = from_f<BF16>(to_f<BF16>(vv[e] & 0xffff) + to_f<BF16>(rr[e] & 0xffff));
          uint16_t hi = from_f<BF16>(to_f<BF16>(vv[e] >> 16) + to_f<BF16>(rr[e] >> 16));
          vv[e] = (uint32_t)lo | ((uint32_t)hi << 16);
        }
        v = uint4v{vv[0], vv[1], vv[2], vv[3]};
      }
      *(uint4v*)(Y + (int64_t)gm * ldy + gn) = v;
    } else {
      uint16_t vs[8];
      __builtin_memcpy(vs, &v, 16);
      for (int e = 0; e < 8 && gn + e < N; e++) {
        uint16_t o = vs[e];
        if (R != nullptr) o = from_f<BF16>(to_f<BF16>(o) + to_f<BF16>(R[(int64_t)gm * ldr + gn + e]));
        Y[(int64_t)gm * ldy + gn + e] = o;
      }
    }
  }
}

// ------------------------------------------------------------------ MFMA kernel

template <int BM, int BN, int WM, int WN, bool BF16, bool GEGLU, int QB, bool AFF, bool SF32>
__global__ __launch_bounds__(WM* WN * 64) void gemm_mfma(const uint16_t* __restrict__ X, int64_t ldx,
                                                         const uint16_t* __restrict__ W, QW qw,
                                                         const uint16_t* __restrict__ bias,
                                                         const uint16_t* __restrict__ R, int64_t ldr,
                                                         uint16_t* __restrict__ Y, int64_t ldy, int M, int N, int K,
                                                         int tiles_n) {
  constexpr int NT = WM * WN * 64;
  constexpr int BK = 64;
  constexpr int WTM = BM / WM, WTN = BN / WN;  // wave tile
  constexpr int TM = WTM / 32, TN = WTN / 32;  // 32x32 blocks per wave
  constexpr int A_LD = BM * 8 / NT, B_LD = BN * 8 / NT;
  constexpr int BNO = GEGLU ? BN / 2 : BN;  // output columns per tile
  static_assert(A_LD * NT == BM * 8 && B_LD * NT == BN * 8, "tile/threads mismatch");
  static_assert(!GEGLU || (TN % 2 == 0), "GEGLU needs an even number of column blocks per wave");

  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  uint16_t* As = smem;                // [2][BM*64]
  uint16_t* Bs = smem + 2 * BM * BK;  // [2][BN*64]

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int m0 = (tile / tiles_n) * BM;
  const int n0 = (tile % tiles_n) * BNO;  // first output column (pair index for GEGLU)

  // B tile row r -> W row (GEGLU: first half value rows, second half gate
  // rows).  wlane: byte offsets of the lane's W pieces from the tile's first
  // row of their half; load i holds rows 32i + tid/8, gate rows from
  // i = B_LD / 2 on.
  static_assert(!GEGLU || (B_LD % 2 == 0 && (B_LD / 2) * (NT / 8) == BN / 2), "GEGLU halves of the W loads");
  uint32_t wlane[B_LD];
#pragma unroll
  for (int i = 0; i < B_LD; i++) {
    const int q = tid + i * NT, r = q >> 3, c = q & 7;
    const int rr = GEGLU && r >= BN / 2 ? r - BN / 2 : r;
    wlane[i] = (uint32_t)(((int64_t)rr * K + c * 8) * 2);
  }
  auto w_row = [&](int r) -> int {
    if constexpr (GEGLU) return r < BN / 2 ? n0 + r : N + n0 + (r - BN / 2);
    else return n0 + r;
  };
  auto w_valid = [&](int r) -> bool {
    if constexpr (GEGLU) return n0 + (r < BN / 2 ? r : r - BN / 2) < N;
    else return n0 + r < N;
  };

  // One K stage in registers on its way to LDS.  16-bit weights: one set, a
  // stage loaded one stage before it is computed.  Quantized weights: two sets
  // rotate, a stage loaded two stages ahead, so the loads and the
  // dequantization behind them have two stages to complete (M = 512, q4:
  // 29 -> 23 us for Wqkv; the 16-bit kernel measured 1 us slower that way)
  struct RegSet {
    uint4v ra[A_LD], rb[B_LD];
    uint32_t rs[QB ? B_LD : 1], rz[QB ? B_LD : 1];
    float rsf[QB && SF32 ? B_LD : 1], rzf[QB && SF32 ? B_LD : 1];
  };
  auto load_regs = [&](RegSet& R, int k0) __attribute__((always_inline)) {
    uint4v(&ra)[A_LD] = R.ra;
    uint4v(&rb)[B_LD] = R.rb;
    auto& rs = R.rs;
    auto& rz = R.rz;
    auto& rsf = R.rsf;
    auto& rzf = R.rzf;
#pragma unroll
    for (int i = 0; i < A_LD; i++) {
      int q = tid + i * NT, r = q >> 3, c = q & 7;
      int k = k0 + c * 8;
      if (m0 + r < M && k < K) ra[i] = *(const uint4v*)(X + (int64_t)(m0 + r) * ldx + k);
      else ra[i] = uint4v{0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < B_LD; i++) {
      int q = tid + i * NT, r = q >> 3, c = q & 7;
      int k = k0 + c * 8;
      bool ok = w_valid(r) && k < K;
      if constexpr (QB == 0) {
        rb[i] = ok ? *(const uint4v*)(W + (int64_t)w_row(r) * K + k) : uint4v{0, 0, 0, 0};
      } else {
        rb[i] = uint4v{0, 0, 0, 0};
        rs[i] = rz[i] = 0;
        if constexpr (SF32) rsf[i] = rzf[i] = 0.f;
        if (ok) {
          int64_t row = w_row(r);
          if constexpr (QB == 8) {
            uint2v w = *(const uint2v*)(qw.q + row * K + k);
            rb[i].x = w.x;
            rb[i].y = w.y;
          } else {
            rb[i].x = *(const uint32_t*)(qw.q + row * (K / 2) + k / 2);
          }
          int64_t gi = row * qw.G + k / qw.group;
          if constexpr (SF32) {
            rsf[i] = ((const float*)qw.scales)[gi];
            if constexpr (AFF) rzf[i] = ((const float*)qw.zeros)[gi];
          } else {
            rs[i] = ((const uint16_t*)qw.scales)[gi];
            if constexpr (AFF) rz[i] = ((const uint16_t*)qw.zeros)[gi];
          }
        }
      }
    }
  };
  auto store_lds = [&](int buf, const RegSet& R) __attribute__((always_inline)) {
    const uint4v(&ra)[A_LD] = R.ra;
    const uint4v(&rb)[B_LD] = R.rb;
    const auto& rs = R.rs;
    const auto& rz = R.rz;
    const auto& rsf = R.rsf;
    const auto& rzf = R.rzf;
    uint16_t* a = As + buf * BM * BK;
    uint16_t* b = Bs + buf * BN * BK;
#pragma unroll
    for (int i = 0; i < A_LD; i++) {
      int q = tid + i * NT, r = q >> 3, c = q & 7;
      *(uint4v*)(a + swz(r, c)) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < B_LD; i++) {
      int q = tid + i * NT, r = q >> 3, c = q & 7;
      if constexpr (QB == 0) {
        *(uint4v*)(b + swz(r, c)) = rb[i];
      } else {
        float sf = 0.f, zf = 0.f;
        if constexpr (SF32) {
          sf = rsf[i];
          zf = rzf[i];
        }
        *(uint4v*)(b + swz(r, c)) = dequant8<QB, AFF, SF32, BF16>(rb[i].x, rb[i].y, rs[i], rz[i], sf, zf);
      }
    }
  };

  // column block tn of this wave -> tile column (B tile row)
  auto bcol = [&](int tn) -> int {
    if constexpr (GEGLU) {
      constexpr int H = TN / 2;
      return tn < H ? wn * (WTN / 2) + tn * 32 : BN / 2 + wn * (WTN / 2) + (tn - H) * 32;
    } else {
      return wn * WTN + tn * 32;
    }
  };

  float16v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
  const int l32 = lane & 31, lg = lane >> 5;

  const int KT = (K + BK - 1) / BK;
  constexpr int AHEAD = QB ? 2 : 1;  // register sets, stages loaded ahead
  RegSet R0, R1;
  load_regs(R0, 0);
  if (AHEAD == 2 && KT > 1) load_regs(R1, BK);
  store_lds(0, R0);
  __syncthreads();
  // stage kt: loads stage kt + AHEAD into `rfree` (AHEAD = 2: its previous
  // stage is in LDS already; AHEAD = 1: rfree is rnext), computes stage kt
  // from LDS, stages kt + 1 (held in `rnext`) into the other LDS buffer
  auto stage = [&](int kt, RegSet& rnext, RegSet& rfree) __attribute__((always_inline)) {
    const int buf = kt & 1;
    if (kt + AHEAD < KT) load_regs(rfree, (kt + AHEAD) * BK);
    const uint16_t* a = As + buf * BM * BK;
    const uint16_t* b = Bs + buf * BN * BK;
    // k16 substeps in increasing k; W rows as the A operand and X rows as
    // the B operand, the order the large-M kernel uses, so both kernels
    // produce the same bits for a row whatever M is
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int c = 2 * s + lg;
      uint4v af[TM], bf[TN];
#pragma unroll
      for (int i = 0; i < TM; i++) af[i] = *(const uint4v*)(a + swz(wm * WTM + i * 32 + l32, c));
#pragma unroll
      for (int j = 0; j < TN; j++) bf[j] = *(const uint4v*)(b + swz(bcol(j) + l32, c));
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = mfma32<BF16>(bf[j], af[i], acc[i][j]);
    }
    if (kt + 1 < KT) store_lds(buf ^ 1, rnext);
    __syncthreads();
  };
  if constexpr (AHEAD == 2) {
    for (int kt = 0; kt < KT; kt += 2) {
      stage(kt, R1, R0);
      if (kt + 1 < KT) stage(kt + 1, R0, R1);
    }
  } else {
    for (int kt = 0; kt < KT; kt++) stage(kt, R0, R0);
  }

  // ---- epilogue: bias, one rounding, GeGLU, stage in LDS as [BM][BNO];
  // lane l holds row l % 32 and columns 8*(r/4) + 4*(l/32) + {0..3}
  uint16_t* Cs = smem;
  constexpr int OUT_TN = GEGLU ? TN / 2 : TN;
  constexpr int WTNO = GEGLU ? WTN / 2 : WTN;
#pragma unroll
  for (int i = 0; i < TM; i++) {
    const int orow = wm * WTM + i * 32 + l32;
#pragma unroll
    for (int j = 0; j < OUT_TN; j++) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int ocol = wn * WTNO + j * 32 + 8 * g + 4 * lg;  // tile output column of element 0
        uint16_t o[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int gcol = n0 + ocol + e;
          float bv = 0.f, bg = 0.f;
          if (bias != nullptr && gcol < N) {
            bv = to_f<BF16>(bias[gcol]);
            if constexpr (GEGLU) bg = to_f<BF16>(bias[N + gcol]);
          }
          float v = to_f<BF16>(from_f<BF16>(acc[i][j][4 * g + e] + bv));
          if constexpr (GEGLU) {
            const float gt = to_f<BF16>(from_f<BF16>(acc[i][j + TN / 2][4 * g + e] + bg));
            v = pin_f32(gelu_fast(v) * gt);  // the f32 product, then one rounding to the storage type
          }
          o[e] = from_f<BF16>(v);
        }
        *(uint2v*)(Cs + orow * BNO + ocol) =
            uint2v{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
      }
    }
  }
  __syncthreads();

  write_tile<BF16, BM, BNO, NT>(Cs, m0, n0, M, N, R, ldr, Y, ldy);
}

// ------------------------------------------------------------------ ring MFMA kernel

// GEMM for 16-bit weights and K % 64 == 0 in calls of few tiles (ring_tile says
// how few).  Both operands go to an LDS ring of NST 64-wide K
// stages by direct loads (no registers, so requests run stages ahead whatever the
// wave is doing), with one barrier per stage; waves of 32 x 32 outputs (32 x 64 in
// the widest tile) read each k16 step's fragments one step ahead.
// What bounds it: up to one 64 x 64 tile per CU the chain of K stages, 0.17 us
// each (four waves share the ring's requests and fragment reads: two took 0.26),
// behind about 4 us of launch, first load and write-out; at several tiles per CU
// LDS, which a wave of 32 x 32 reads 2 KB of per 32-clock MFMA.  The kernels
// before it waited for each stage's loads (gemm_mfma: 0.8 us a stage) or loaded X
// fragments of 32 rows x 32 bytes from global memory (a slab kernel).  Measured
// (us, f16, before -> after): 128 x 2304 x 768 9.3 -> 5.6, 128 x 2304 x 768 GeGLU
// 15.1 -> 5.9, 128 x 768 x 3072 32.7 -> 11.3, 2048 x 768 x 1152 15.6 -> 9.1, 2048
// x 2304 x 768 21.9 -> 17.6 (413 TFLOP/s).
// Same MFMA, operand order (W rows as the A operand, X rows as the B operand) and
// ascending k16 steps as the other kernels: a row's bits do not depend on M or on
// the tile.
template <int N>
__device__ __forceinline__ void ring_wait_barrier() {
  // this wave's loads up to the stage about to be read have landed, its LDS
  // reads of the last stage are done; then everybody's
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// ... with at most `later` (up to MOST) stages of PW loads each still in flight
template <int PW, int MOST>
__device__ __forceinline__ void ring_wait_stages(int later) {
  if constexpr (MOST <= 0) {
    ring_wait_barrier<0>();
  } else {
    if (later >= MOST) ring_wait_barrier<MOST * PW>();
    else ring_wait_stages<PW, MOST - 1>(later);
  }
}

template <int BM, int BN, int WM, int WN, int NST, bool BF16, bool GEGLU>
__global__ __launch_bounds__(WM* WN * 64) void gemm_ring(const uint16_t* __restrict__ X, int64_t ldx,
                                                         const uint16_t* __restrict__ W,
                                                         const uint16_t* __restrict__ bias,
                                                         const uint16_t* __restrict__ R, int64_t ldr,
                                                         uint16_t* __restrict__ Y, int64_t ldy, int M, int N, int K,
                                                         int tiles_n, int xpan, int ypan) {
  constexpr int NW = WM * WN, NT = NW * 64;
  constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / 32, TN = WTN / 32;
  constexpr int PCS = (BM + BN) / 8, PW = PCS / NW;  // 1 KB pieces (8 rows x 64 k) per stage, per wave
  constexpr int STAGE = (BM + BN) * 64;              // u16 per stage
  constexpr int BNO = GEGLU ? BN / 2 : BN;
  static_assert(PW * NW == PCS, "whole rounds of pieces");
  static_assert(!GEGLU || (BN / 2) % 32 == 0, "value blocks, then gate blocks");
  static_assert(NST >= 3, "a stage is published one stage ahead");
  static_assert(PW * (NST - 2) <= 63, "vmcnt immediate");
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, lg = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int m0 = (tile / tiles_n) * BM, n0 = (tile % tiles_n) * BNO;

  // A stage is 1 KB pieces: X rows, then W rows (GeGLU: value rows, then gate
  // rows).  Row-major piece p is tile rows 8 p .. 8 p + 7: lane l fills slot
  // l % 8 of row l / 8, so it fetches chunk (l % 8) ^ f(row), f(r) = (r / 2) % 8,
  // and the 16 lanes of a fragment-read pass (16 rows, one chunk) cover all 64
  // banks.  With X in panel order (xpan) piece p is k16 block p % 4 of 32-row
  // group p / 4, already a fragment.  Rows past the operand are clamped (their
  // outputs are never stored).
  const uint64_t xa = (uint64_t)(xpan ? X + (int64_t)(m0 >> 5) * 32 * K : X + (int64_t)m0 * ldx);
  uint32_t off[PW], step[PW];  // byte offsets of the lane's 16 bytes, and per stage
  uint4v rsrc[PW];             // W: the base is the piece's first row
#pragma unroll
  for (int i = 0; i < PW; i++) {
    const int p = wave * PW + i, r = p * 8 + (lane >> 3);
    const uint32_t c = ((lane & 7) ^ ((r >> 1) & 7)) * 16;
    uint64_t base;
    step[i] = 128;
    if (p * 8 < BM) {
      base = xa;
      if (xpan) {
        const int last = ((M + 31) >> 5) - 1 - (m0 >> 5), grp = min(p >> 2, last);
        off[i] = (uint32_t)grp * (uint32_t)K * 64u + (uint32_t)(p & 3) * 1024u + (uint32_t)lane * 16u;
        step[i] = 4096;
      } else {
        off[i] = (uint32_t)(m0 + r < M ? r : M - 1 - m0) * (uint32_t)ldx * 2u + c;
      }
    } else {
      const int wr = r - BM, wr0 = p * 8 - BM;  // (a piece never straddles the halves)
      const bool gate = GEGLU && wr0 >= BN / 2;
      const int n = n0 + (gate ? wr - BN / 2 : wr), nb = n0 + (gate ? wr0 - BN / 2 : wr0);
      const int nc = n < N ? n : N - 1, nbc = nb < N ? nb : N - 1;
      base = (uint64_t)(W + (int64_t)(nbc + (gate ? N : 0)) * K);
      off[i] = (uint32_t)(nc - nbc) * (uint32_t)K * 2u + c;
    }
    rsrc[i] = uint4v{(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)base),
                     (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(base >> 32) & 0xffffu), 0x80000000u, 0x00020000u};
  }
  const uint32_t lds0 = (uint32_t)__builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t*)smem);
  auto issue = [&](int kt, int slot, int i0, int i1) __attribute__((always_inline)) {
#pragma unroll
    for (int i = i0; i < i1; i++)
      buffer_lds16(rsrc[i], off[i], (uint32_t)kt * step[i], lds0 + (uint32_t)(slot * STAGE * 2 + (wave * PW + i) * 1024));
  };

  float16v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
  // fragment chunk 2 s + lg of row l32 (f depends on l32 alone: blocks start at multiples of 32 rows)
  int fo[4];
#pragma unroll
  for (int s = 0; s < 4; s++) fo[s] = l32 * 64 + (((2 * s + lg) ^ ((l32 >> 1) & 7)) << 3);
  int xo[4];  // X's, the same unless it is in panel order
#pragma unroll
  for (int s = 0; s < 4; s++) xo[s] = xpan ? s * 512 + lane * 8 : fo[s];
  // Fragments of a k16 step are read one step ahead of its MFMAs, across stages
  // too: a stage is published one stage before it is multiplied.
  uint4v xf[2][TM], wf[2][TN];
  auto read = [&](int slot, int s, int d) __attribute__((always_inline)) {
    const uint16_t* b = smem + slot * STAGE;
#pragma unroll
    for (int i = 0; i < TM; i++) xf[d][i] = *(const uint4v*)(b + xo[s] + (wm * WTM + i * 32) * 64);
#pragma unroll
    for (int j = 0; j < TN; j++) wf[d][j] = *(const uint4v*)(b + fo[s] + (BM + wn * WTN + j * 32) * 64);
  };
  // req >= 0: stage `req` is requested into slot `rs` between the MFMAs
  auto compute = [&](int slot, int next, bool more, int req, int rs) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 4; s++) {  // k16 steps in order, W rows as A, X rows as B: the other kernels' bits
      if (s < 3) read(slot, s + 1, (s + 1) & 1);
      else if (more) read(next, 0, 0);
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = mfma32<BF16>(wf[s & 1][j], xf[s & 1][i], acc[i][j]);
      if (req >= 0) issue(req, rs, s * PW / 4, (s + 1) * PW / 4);
    }
  };

  const int KT = K >> 6;
  // stages 0 .. NST - 2 in flight; stage 0 landed
#pragma unroll
  for (int s = 0; s < NST - 1; s++)
    if (s < KT) issue(s, s, 0, PW);
  ring_wait_stages<PW, NST - 2>(KT - 1);
  read(0, 0, 0);
  int slot = 0, kt = 0;
  auto succ = [](int v) { return v == NST - 1 ? 0 : v + 1; };
  // stage kt: stage kt + 1 has landed and everybody is done with stage kt - 1,
  // whose slot takes stage kt + NST - 1
  for (; kt + NST - 1 < KT; kt++) {
    ring_wait_barrier<(NST - 3) * PW>();
    compute(slot, succ(slot), true, kt + NST - 1, slot == 0 ? NST - 1 : slot - 1);
    slot = succ(slot);
  }
  for (; kt < KT; kt++) {  // nothing more to request
    ring_wait_stages<PW, NST - 3>(KT - 2 - kt);
    compute(slot, succ(slot), kt + 1 < KT, -1, 0);
    slot = succ(slot);
  }
  __syncthreads();

  // ---- epilogue, as gemm_mfma's: bias, one rounding, staged in LDS as [BM][BN];
  // GeGLU then pairs each value column with its gate on the way out
  uint16_t* Cs = smem;
#pragma unroll
  for (int i = 0; i < TM; i++) {
    const int orow = wm * WTM + i * 32 + l32;
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const int tc = wn * WTN + j * 32;  // tile column of the block
      const bool gate = GEGLU && tc >= BN / 2;
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int c = 8 * g + 4 * lg;
        uint16_t o[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int gcol = n0 + tc + c + e - (gate ? BN / 2 : 0);
          float bv = 0.f;
          if (bias != nullptr && gcol < N) bv = to_f<BF16>(bias[gcol + (gate ? N : 0)]);
          o[e] = from_f<BF16>(acc[i][j][4 * g + e] + bv);
        }
        *(uint2v*)(Cs + orow * BN + tc + c) =
            uint2v{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
      }
    }
  }
  __syncthreads();
  if constexpr (!GEGLU) {
    if (!ypan) {
      write_tile<BF16, BM, BN, NT>(Cs, m0, n0, M, N, R, ldr, Y, ldy);
      return;
    }
  }
  // GeGLU, or panel order (N % 16 == 0, no residual: 32 rows of a 16-byte
  // column are 512 contiguous bytes, so the lanes go down the rows)
  constexpr int CPR = BNO / 8;
  for (int q = tid; q < BM * CPR; q += NT) {
    const int r = ypan ? q % BM : q / CPR, c = (ypan ? q / BM : q % CPR) * 8, gm = m0 + r, gn = n0 + c;
    if (gm >= M || gn >= N) continue;
    uint4v o = *(const uint4v*)(Cs + r * BN + c);
    if constexpr (GEGLU) {
      const uint4v g = *(const uint4v*)(Cs + r * BN + BNO + c);
      uint32_t res[4] = {0, 0, 0, 0};
      if (R != nullptr) {
        if (gn + 8 <= N) {
          const uint4v rv = *(const uint4v*)(R + (int64_t)gm * ldr + gn);
#pragma unroll
          for (int e = 0; e < 4; e++) res[e] = rv[e];
        } else {
          for (int e = 0; gn + e < N; e++) res[e >> 1] |= (uint32_t)R[(int64_t)gm * ldr + gn + e] << (16 * (e & 1));
        }
      }
#pragma unroll
      for (int e = 0; e < 4; e++) {
        uint32_t h[2];
#pragma unroll
        for (int k = 0; k < 2; k++) {
          const float val = to_f<BF16>((o[e] >> (16 * k)) & 0xffff), gt = to_f<BF16>((g[e] >> (16 * k)) & 0xffff);
          h[k] = from_f<BF16>(pin_f32(gelu_fast(val) * gt));  // the f32 product, then one rounding
          if (R != nullptr) h[k] = from_f<BF16>(to_f<BF16>(h[k]) + to_f<BF16>((res[e] >> (16 * k)) & 0xffff));
        }
        o[e] = h[0] | (h[1] << 16);
      }
    }
    uint16_t* yp = ypan ? Y + ((int64_t)(gm >> 5) * (N >> 4) + (gn >> 4)) * 512 + (((gn >> 3) & 1) * 32 + (gm & 31)) * 8
                        : Y + (int64_t)gm * ldy + gn;
    if (gn + 8 <= N) {
      *(uint4v*)yp = o;
    } else {
      for (int e = 0; e < 8 && gn + e < N; e++) yp[e] = (uint16_t)(o[e >> 1] >> (16 * (e & 1)));
    }
  }
}

// ------------------------------------------------------------------ large-M MFMA kernel


// Persistent GEMM over 256 x BN output tiles.  Four waves are stacked along
// M: each wave owns 64 rows and every column of the tile as 2 x (BN/32)
// blocks of v_mfma_f32_32x32x16 (on gfx950 the 32x32 MFMA runs at twice the
// rate of the 16x16x32 one, and reaches it from a single wave per SIMD).
// A wave's A rows are private, so they go from global memory straight into
// MFMA operand registers; only the weight tile is shared, through
// double-buffered LDS.
//
// One block per CU walks a list of tiles as one continuous stream of
// 64-wide K stages: loads run two stages ahead (three A and two W register
// sets rotating by name, issued between the MFMAs) and cross tile
// boundaries, so the next tile's first stages arrive while the current tile
// finishes.  Blocks on one XCD (block b runs on XCD b % 8) take consecutive
// tiles, which share A rows in that XCD's L2.
//
// The MFMA computes the transposed product (W rows as the A operand, X rows
// as the B operand): lane l then holds output row l % 32 and the four
// consecutive columns 8*(r/4) + 4*(l/32) + {0..3} of each accumulator, so the
// epilogue writes 8-byte pieces of Y straight from registers.
//
// QKV (16-bit weights, no GeGLU, no bias, no residual): the epilogue of the fused
// q / k / v projection (struct QK): each 64-column head of the tile is a pair
// of column blocks whose lanes hold the rotation partners d and d + 32 at the
// same register, so RoPE is applied in registers, and the tile leaves
// head-major.
template <int BN, bool BF16, bool GEGLU, bool KTAIL, bool QKV = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm_mfma_arow(
    const uint16_t* __restrict__ X, int64_t ldx, const uint16_t* __restrict__ W, const uint16_t* __restrict__ bias,
    const uint16_t* __restrict__ R, int64_t ldr, uint16_t* __restrict__ Y, int64_t ldy, int M, int N, int K,
    int tiles_n, int tiles, int xpan, int ypan, QK qk) {
  static_assert(!QKV || (!GEGLU && BN % 64 == 0), "QKV: no GeGLU, whole heads per tile");
  constexpr int NT = 256, BM = 256, BK = 64;
  constexpr int TM = 2, TN = BN / 32;  // 32x32 blocks per wave
  constexpr int KS = BK / 16;          // k16 substeps per stage
  constexpr int B_LD = BN * 8 / NT;
  constexpr int BNO = GEGLU ? BN / 2 : BN;
  static_assert(B_LD * NT == BN * 8 && BN % 32 == 0, "BN must be a multiple of 32");
  static_assert(!GEGLU || (TN % 2 == 0), "GEGLU needs an even number of column blocks");
  static_assert((BM * (BNO / 8)) % NT == 0, "write-out assumes whole rounds of chunks");

  constexpr int CPR = BNO / 8;           // 16-byte chunks per output row
  constexpr int RG = (CPR + 7) / 8;      // C tile: groups of 8 chunks per row
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  uint16_t* Bs = smem;               // [2][BN*64] W tiles
  uint16_t* Cs = smem + 2 * BN * BK;  // [RG][BM][8] 16-byte chunks: residual in, output out

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, lg = lane >> 5;

  // This block's tiles (gridDim.x % 8 == 0).  XCD x owns the row panels
  // [mb0, mb1) with every column tile, and its blocks take the panel's tiles
  // column-tile-major: local tile l = slot + i * nx is row panel mb0 + l % mx,
  // column tile l / mx.  The tiles one XCD computes at a time then share a
  // few column tiles of W and cycle over the XCD's own rows of X, which stay
  // in its L2 from one column tile to the next.
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, nx = gridDim.x >> 3;
  const int tiles_m = tiles / tiles_n;
  const int mb0 = xcd * tiles_m / 8, mx = (xcd + 1) * tiles_m / 8 - mb0;
  const int nloc = mx * tiles_n;
  const int ntile = nloc > slot ? (nloc - slot + nx - 1) / nx : 0;
  if (ntile == 0) return;
  const int KT = (K + BK - 1) / BK;
  const int S = ntile * KT;  // stages in this block's stream
  auto tile_m0 = [&](int i) { return (mb0 + (slot + i * nx) % mx) * BM; };
  auto tile_n0 = [&](int i) { return ((slot + i * nx) / mx) * BNO; };

  // X is row-major (x[row * ldx + k]) or in panel order (xpan; 32-row x
  // 16-column blocks of 1 KB in MFMA operand order, rows padded to a multiple
  // of 32).  For k % 8 == 0 both are x[xs_hi * (row / 32) + xs_lo * (row % 32)
  // + xk * k]; in panel order one fragment load then reads one whole block.
  const int64_t xs_hi = xpan ? (int64_t)32 * K : (int64_t)32 * ldx;
  const int64_t xs_lo = xpan ? 8 : ldx;
  const int xk = xpan ? 32 : 1;
  const int mlim = xpan ? ((M + 31) & ~31) : M;
  // Loads are branch-free: addresses are clamped into the operand.  Rows past
  // M (A) or N (W) only feed outputs that are never stored, so they need no
  // zeroing; a K tail (K % 64 != 0, KTAIL, row-major X only) is zeroed.
  //
  // Without a K tail the loads are buffer loads: the resource's base is the
  // first row of the tile (wave-uniform, 64-bit), the lanes' offsets from it
  // are kernel constants and the K position is the scalar offset, so a stage
  // spends no vector instructions on addresses.  Rows past the operand lie
  // outside the resource's range and read 0.
  constexpr bool BUFX = !KTAIL, BUFW = !KTAIL;
  constexpr int BUF_FLAGS = 0x00020000;  // resource word 3: 32-bit raw data
  uint32_t xlane[TM];                    // byte offsets of the lane's rows in a tile
#pragma unroll
  for (int rb = 0; rb < TM; rb++) {
    const int lr = wave * 64 + rb * 32 + l32;
    xlane[rb] = (uint32_t)(((lr >> 5) * xs_hi + (lr & 31) * xs_lo + xk * lg * 8) * 2);
  }
  const int64_t x_elems = xpan ? (int64_t)mlim * K : (int64_t)(M - 1) * ldx + K;
  auto load_a = [&](int m0, int k0, uint4v (&a)[TM][KS]) {
    if constexpr (BUFX) {
      const int64_t base = xpan ? (int64_t)(m0 >> 5) * xs_hi : (int64_t)m0 * ldx;
      const int64_t left = (x_elems - base) * 2;
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(X + base), (short)0, (int)(left < 0x7ffffff0 ? left : 0x7ffffff0), BUF_FLAGS);
#pragma unroll
      for (int rb = 0; rb < TM; rb++)
#pragma unroll
        for (int s = 0; s < KS; s++)
          a[rb][s] = __builtin_amdgcn_raw_buffer_load_b128(rs, xlane[rb], (k0 + s * 16) * xk * 2, 0);
      return;
    }
    const int arow = m0 + wave * 64 + l32;
#pragma unroll
    for (int rb = 0; rb < TM; rb++)
#pragma unroll
      for (int s = 0; s < KS; s++) {
        const int row = arow + rb * 32, k = k0 + s * 16 + lg * 8;
        const int rc = row < mlim ? row : mlim - 1;
        const uint4v v = *(const uint4v*)(X + (int64_t)(rc >> 5) * xs_hi + (int64_t)(rc & 31) * xs_lo +
                                          (int64_t)xk * (KTAIL && k >= K ? 0 : k));
        a[rb][s] = (KTAIL && k >= K) ? uint4v{0, 0, 0, 0} : v;
      }
  };

  struct BRegs {
    uint4v v[B_LD];
  };
  // B tile row r -> W row (GEGLU: first half value rows, second half gate
  // rows).  wlane: byte offsets of the lane's 16-byte W pieces from the
  // tile's first row of their half; load i holds rows 32i + tid/8, gate rows
  // from i = B_LD / 2 on.
  static_assert(!GEGLU || (B_LD % 2 == 0 && (B_LD / 2) * (NT / 8) == BN / 2), "GEGLU halves of the W loads");
  const int64_t wrow_b = (int64_t)K * 2;  // bytes per W row
  uint32_t wlane[B_LD];
#pragma unroll
  for (int i = 0; i < B_LD; i++) {
    const int q = tid + i * NT, r = q >> 3, c = q & 7;
    const int rr = GEGLU && r >= BN / 2 ? r - BN / 2 : r;
    wlane[i] = (uint32_t)(rr * wrow_b + c * 16);
  }
  auto load_b = [&](int n0, int k0, BRegs& br) {
    if constexpr (BUFW) {
      // value rows from W row n0, gate rows (GEGLU) from W row N + n0; each
      // resource ends with row N - 1 of its half
      const uint8_t* wb = (const uint8_t*)W;
      const int64_t left = (int64_t)(N - n0) * wrow_b;
      const int nrec = (int)(left < 0x7ffffff0 ? left : 0x7ffffff0);
      const __amdgpu_buffer_rsrc_t rv =
          __builtin_amdgcn_make_buffer_rsrc((void*)(wb + (int64_t)n0 * wrow_b), (short)0, nrec, BUF_FLAGS);
      const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(wb + (int64_t)((GEGLU ? N : 0) + n0) * wrow_b), (short)0, nrec, BUF_FLAGS);
#pragma unroll
      for (int i = 0; i < B_LD; i++) {
        const __amdgpu_buffer_rsrc_t rs = GEGLU && i >= B_LD / 2 ? rg : rv;
        br.v[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, wlane[i], k0 * 2, 0);
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < B_LD; i++) {
      const int q = tid + i * NT, r = q >> 3, c = q & 7;
      const int k = k0 + c * 8;
      const int nn = GEGLU ? n0 + (r < BN / 2 ? r : r - BN / 2) : n0 + r;
      const bool rv = nn < N;
      const int wr = GEGLU && r >= BN / 2 ? N + nn : nn;
      const uint4v v = *(const uint4v*)(W + (int64_t)(rv ? wr : 0) * K + (KTAIL && k >= K ? 0 : k));
      br.v[i] = (KTAIL && k >= K) ? uint4v{0, 0, 0, 0} : v;
    }
  };
  auto store_b = [&](int buf, const BRegs& br) {
    uint16_t* b = Bs + buf * BN * BK;
#pragma unroll
    for (int i = 0; i < B_LD; i++) {
      int q = tid + i * NT, r = q >> 3, c = q & 7;
      *(uint4v*)(b + swz(r, c)) = br.v[i];
    }
  };

  // column block j of the tile -> W tile row (GEGLU: value blocks, then gate blocks)
  auto bcol = [&](int j) -> int {
    if constexpr (GEGLU) return j < TN / 2 ? j * 32 : BN / 2 + (j - TN / 2) * 32;
    else return j * 32;
  };

  // The C tile in LDS: 16-byte chunk c of tile row r sits in slot
  // (c/8)*BM*8 + r*8 + ((c%8) ^ (r%8)).  The epilogue's 8-byte accesses of 32
  // consecutive rows then spread over the banks, and 8 consecutive chunks of
  // a row are 8 distinct slots of one 128-byte span.  With a residual the
  // tile is first filled with R straight from global memory
  // (global_load_lds_dwordx4, issued at the tile's first K stage); the
  // epilogue adds the rounded linear output in place, and the whole tile
  // leaves with coalesced 16-byte stores (whole rows per instruction: partial
  // lines written from registers cost HBM write-backs twice over).
  auto r_slot = [&](int r, int c) { return (c >> 3) * (BM * 8) + r * 8 + ((c & 7) ^ (r & 7)); };
  // DMA instruction i of wave w fills slots (4i + w)*64 + lane, i.e. row
  // 32*(i%8) + 8w + lane/8, chunk 8*(i/8) + ((lane%8) ^ (lane/8)).  Every lane
  // writes its own slot, so slots outside the operand load a clamped,
  // in-bounds address (ldr % 8 == 0: a chunk starting below N lies inside the
  // row) and are never stored.
  // The copies are issued from inline asm (lds_copy16): the compiler then
  // does not take the fragment reads and W stores of the following stages for
  // possible readers of the C tile, each of which it would otherwise precede
  // with a wait for every load in flight.  The epilogue waits for them.
  //
  // They go out in six pieces (DMA_P instructions each), piece p at the end
  // of stage dma0 + p, after that stage's wait for its W tile.  The compiler
  // does not count them, so the first load wait issued after a piece also
  // waits for the piece: one stage later it has landed, whereas copies issued
  // at the start of a stage would hold that stage's own wait for the whole
  // residual tile.
  constexpr int DMA_N = RG * 8, DMA_P = (DMA_N + 5) / 6;
  auto dma_piece = [&](int m0, int n0, auto P_) __attribute__((always_inline)) {
    constexpr int P = decltype(P_)::value;
    int ln = lane, wv = wave;
    asm volatile("" : "+v"(ln), "+v"(wv));  // per-tile address math, not hoisted (see the epilogue)
    const int r_cx = (ln & 7) ^ (ln >> 3);
    const int rbase = m0 + wv * 8 + (ln >> 3), cbase = n0 + r_cx * 8;
    const uint32_t cs0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t*)Cs +
                         (uint32_t)__builtin_amdgcn_readfirstlane(wave) * 1024u;
#pragma unroll
    for (int i = P * DMA_P; i < (P + 1) * DMA_P && i < DMA_N; i++) {
      const int row = rbase + (i & 7) * 32, col = cbase + (i >> 3) * 64;
      const bool cok = (i >> 3) * 8 + r_cx < CPR && col < N;
      lds_copy16(R + (int64_t)(row < M ? row : M - 1) * ldr + (cok ? col : 0), cs0 + (uint32_t)i * 4096u);
    }
  };

  float16v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

  // ---- epilogue: bias, one rounding to the storage type, GeGLU (value
  // block j and gate block j + TN/2 hold the same output columns), then the
  // residual add, y = round(round(x.w^T + b) + r), into the C tile
  constexpr int OUT_TN = GEGLU ? TN / 2 : TN;
  // The lane indices are re-read through an empty asm inside the epilogue,
  // the write-out and the residual DMA: the compiler then computes their
  // per-lane addresses there, once per tile, instead of hoisting all of them
  // out of the tile loop and spilling them to scratch (an HBM write per
  // spilled register).
  auto epilogue = [&](int n0, auto has_bias, auto has_r) {
    constexpr bool HB = decltype(has_bias)::value, HR = decltype(has_r)::value;
    int l32 = lane & 31, lg = lane >> 5, wv = wave;
    asm volatile("" : "+v"(l32), "+v"(lg), "+v"(wv));
#pragma unroll
    for (int j = 0; j < OUT_TN; j++) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int col = j * 32 + 8 * g + 4 * lg;  // tile output column of element 0
        float bv[4] = {0.f, 0.f, 0.f, 0.f}, bg[4] = {0.f, 0.f, 0.f, 0.f};
        if constexpr (HB) {
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (n0 + col + e < N) {
              bv[e] = to_f<BF16>(bias[n0 + col + e]);
              if constexpr (GEGLU) bg[e] = to_f<BF16>(bias[N + n0 + col + e]);
            }
        }
#pragma unroll
        for (int i = 0; i < TM; i++) {
          uint16_t o[4];
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float a = HB ? acc[i][j][4 * g + e] + bv[e] : acc[i][j][4 * g + e];
            if constexpr (GEGLU) {
              const float ag = HB ? acc[i][j + TN / 2][4 * g + e] + bg[e] : acc[i][j + TN / 2][4 * g + e];
              o[e] = from_f<BF16>(pin_f32(gelu_fast(to_f<BF16>(from_f<BF16>(a))) * to_f<BF16>(from_f<BF16>(ag))));
            } else {
              o[e] = from_f<BF16>(a);
            }
          }
          uint2v* cp = (uint2v*)(Cs + r_slot(wv * 64 + i * 32 + l32, col >> 3) * 8 + (col & 7));
          if constexpr (HR) {
            const uint2v rv = *cp;
            const uint16_t rr[4] = {(uint16_t)(rv.x & 0xffff), (uint16_t)(rv.x >> 16), (uint16_t)(rv.y & 0xffff),
                                    (uint16_t)(rv.y >> 16)};
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = from_f<BF16>(to_f<BF16>(o[e]) + to_f<BF16>(rr[e]));
          }
          *cp = uint2v{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
        }
      }
    }
  };
  // the C tile -> Y: thread t takes chunks t, t + 256, ...; consecutive
  // threads cover consecutive 16-byte pieces of a row (row-major Y) or of a
  // 1 KB block (panel-order Y, ypan: chunk q is row 32 * rb + q % 32, column
  // chunk 2 * nb + (q / 32) % 2 with (rb, nb) = divmod(q / 64, CPR / 2))
  static_assert(CPR % 2 == 0, "panel-order output needs whole 16-column blocks");
  const int yblk = (N + 15) >> 4;  // 16-column blocks per panel-order row block
  auto panel_chunk = [&](int q, int& r, int& c) -> int64_t {
    const int r32 = q & 31, h = (q >> 5) & 1, rest = q >> 6, rb = rest / (CPR / 2), nb = rest - rb * (CPR / 2);
    r = rb * 32 + r32;
    c = nb * 2 + h;
    return ((int64_t)rb * yblk + nb) * 512 + (h * 32 + r32) * 8;  // relative to the tile's first block
  };
  // output chunk c of C tile row r
  auto out_chunk = [&](int r, int c) __attribute__((always_inline)) -> uint4v {
    return *(const uint4v*)(Cs + r_slot(r, c) * 8);
  };
  auto write_out = [&](int m0, int n0) {
    int t0 = tid;
    asm volatile("" : "+v"(t0));
    if (ypan) {
      uint16_t* yb = Y + ((int64_t)(m0 >> 5) * yblk + (n0 >> 4)) * 512;
      const int rbl = ((M + 31) >> 5) - (m0 >> 5);  // row blocks of the padded output left from m0
      for (int q = t0; q < BM * CPR; q += NT) {
        int r, c;
        const int64_t o = panel_chunk(q, r, c);
        if ((r >> 5) >= rbl || n0 + c * 8 >= N) continue;
        *(uint4v*)(yb + o) = out_chunk(r, c);
      }
      return;
    }
    if (m0 + BM <= M && n0 + BNO <= N) {  // interior tile: no bounds checks
      // TPR threads per row, chunks c = t % TPR + TPR * j: a pass covers
      // NT / TPR rows (a multiple of 8, so a thread's C-tile slots differ
      // only by the pass: immediate LDS offsets), and every address is a
      // per-thread row pointer plus constants.  Two passes' LDS reads are
      // issued before their stores.
      constexpr int TPR = CPR % 8 == 0 ? 8 : 4, CPT = CPR / TPR, RPP = NT / TPR, NP = BM / RPP;
      static_assert(CPR % TPR == 0 && RPP % 8 == 0 && NP % 2 == 0, "interior write-out layout");
      const int tc = t0 % TPR, tr = t0 / TPR;
      uint16_t* yr = Y + (int64_t)(m0 + tr) * ldy + n0 + tc * 8;
      const int64_t ystep = (int64_t)RPP * ldy;
#pragma unroll
      for (int p = 0; p < NP; p += 2) {
        uint4v v[2][CPT];
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
          for (int j = 0; j < CPT; j++) v[h][j] = out_chunk(tr + (p + h) * RPP, tc + TPR * j);
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
          for (int j = 0; j < CPT; j++) *(uint4v*)(yr + h * ystep + TPR * 8 * j) = v[h][j];
        yr += 2 * ystep;
      }
      return;
    }
    for (int q = t0; q < BM * CPR; q += NT) {
      const int r = q / CPR, c = q - r * CPR;
      const int gm = m0 + r, gn = n0 + c * 8;
      if (gm >= M || gn >= N) continue;
      const uint4v v = out_chunk(r, c);
      uint16_t* yp = Y + (int64_t)gm * ldy + gn;
      if (gn + 8 <= N) {
        *(uint4v*)yp = v;
      } else {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        for (int e = 0; gn + e < N; e++) yp[e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
      }
    }
  };

  // ---- spread write-out.  With several tiles per block, an interior tile
  // leaves the C tile during the next tile's first six stages instead of in
  // one burst: stage s stores chunks WO_PS * s .. WO_PS * s + WO_PS - 1 of
  // each thread's WO_N (those below WO_N), as buffer stores issued after the
  // stage's loads.
  // The wait counter counts loads and stores in issue order, so after a
  // burst the next tile's first load wait also waits for every store of the
  // tile, which all CUs issue at once; spread, a stage's stores are younger
  // than every load waited for until two stages later.  Those six stages are
  // a copy of the stage code of their own (the other stages carry no store
  // instructions); the resource's record count bounds every store to the
  // tile.
  //
  // Thread t's chunk q: row-major Y as in the interior burst below (WTPR
  // threads per row, chunk t % WTPR + WTPR * (q % WCPT) of row
  // t / WTPR + WRPP * (q / WCPT)); panel-order Y chunk t + NT q as in
  // panel_chunk, whose row block and block column are wave-uniform (lane
  // offset 16 * lane, scalar block offset).
  constexpr int WO_N = BM * CPR / NT, WO_PS = (WO_N + 5) / 6;
  constexpr int WTPR = CPR % 8 == 0 ? 8 : 4, WCPT = CPR / WTPR, WRPP = NT / WTPR;
  // The layout is a compile-time one, panel order for GeGLU (whose output
  // feeds the next linear) and row-major otherwise; an output in the other
  // layout leaves in a burst.
  constexpr bool YP = GEGLU;
  const bool spread = !QKV && ntile > 1 && KT >= 12 && (ypan != 0) == YP;
  // the pending output: its first element (row-major) or block (panel
  // order), and the bytes up to its last chunk (0: nothing pending)
  uint16_t* wo_base = Y;
  int wo_rec = 0;
  // Every address below is recomputed per stage from values re-read through
  // an empty asm: hoisted out of the stage loop, the addresses of the
  // chunks would each hold a register for the whole kernel.
  auto wo_part = [&](auto S_) __attribute__((always_inline)) {
    constexpr int S = decltype(S_)::value;
    int t0 = tid, wv = __builtin_amdgcn_readfirstlane(wave), ld2 = (int)ldy * 2, yb = yblk;
    asm volatile("" : "+v"(t0), "+s"(wv), "+s"(ld2), "+s"(yb));
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)wo_base, (short)0, wo_rec, BUF_FLAGS);
    if constexpr (YP) {
      // chunk t + NT q: row block rb, block column nb of the tile (scalars)
      const int ln = t0 & 63, r32 = ln & 31, lx = (ln >> 5) ^ (r32 & 7);
#pragma unroll
      for (int u = 0; u < WO_PS; u++) {
        if (S * WO_PS + u >= WO_N) break;
        const int rest = wv + (NT / 64) * (S * WO_PS + u);
        const int rb = rest / (CPR / 2), nb = rest - rb * (CPR / 2);
        const int slot = (nb >> 2) * (BM * 8) + (rb * 32 + r32) * 8 + (((nb & 3) * 2) ^ lx);
        const uint4v v = *(const uint4v*)(Cs + slot * 8);
        __builtin_amdgcn_raw_buffer_store_b128(v, rs, ln * 16, (rb * yb + nb) * 1024, 0);
      }
    } else {
      // tile row wtr + WRPP pass, chunk wtc + WTPR j
      const int wtc = t0 % WTPR, wtr = t0 / WTPR;
      const int voff = (wtr * ld2) + wtc * 16;
#pragma unroll
      for (int u = 0; u < WO_PS; u++) {
        if (S * WO_PS + u >= WO_N) break;
        const int q = S * WO_PS + u, pass = q / WCPT, j = q % WCPT;
        const int cr = wtc + WTPR * j;
        const int slot = (cr >> 3) * (BM * 8) + (wtr + WRPP * pass) * 8 + ((cr & 7) ^ (wtr & 7));
        const uint4v v = *(const uint4v*)(Cs + slot * 8);
        __builtin_amdgcn_raw_buffer_store_b128(v, rs, voff, WRPP * pass * ld2 + WTPR * 16 * j, 0);
      }
    }
  };
  // sets the pending output to tile (m0, n0)
  auto wo_set = [&](int m0, int n0) {
    int64_t bytes;
    if constexpr (YP) {
      wo_base = Y + ((int64_t)(m0 >> 5) * yblk + (n0 >> 4)) * 512;
      bytes = ((int64_t)(BM / 32 - 1) * yblk + CPR / 2) * 1024;
    } else {
      wo_base = Y + (int64_t)m0 * ldy + n0;
      bytes = ((int64_t)(BM - 1) * ldy + BNO) * 2;
    }
    wo_rec = (int)(bytes < 0x7ffffff0 ? bytes : 0x7ffffff0);
  };

  // ---- QKV epilogue: one rounding to the storage type (the linear
  // output), then, for a head of q or k, the split-half rotation of that
  // rounded value in f32 and a second rounding (a separate Backend.rope),
  // into the C tile.  Head pair hp of the tile is column blocks 2hp (dims
  // 0..31) and 2hp + 1 (dims 32..63); a lane holds dims 8g + 4lg + e of both.
  auto epilogue_qkv = [&](int m0, int n0) {
    int l32 = lane & 31, lg = lane >> 5, wv = wave;
    asm volatile("" : "+v"(l32), "+v"(lg), "+v"(wv));
    // the QK fields are re-read here (through an empty asm), so what is
    // derived from them is computed per tile, not held across the K loop
    int L = qk.L, H = qk.H;
    const float2* tab = qk.tab;
    asm volatile("" : "+s"(L), "+s"(H), "+s"(tab));
    const int HD = H * 64;
#pragma unroll
    for (int i = 0; i < TM; i++) {
      const int row = wv * 64 + i * 32 + l32;
      const int pos = (m0 + row < M ? m0 + row : M - 1) % L;
      // cos / sin of dims 8g + 4lg + 0..3 at this row's position
      float4v cs[4][2];
      if (tab != nullptr && n0 < 2 * HD) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const float4v* t = (const float4v*)(tab + (int64_t)pos * 32 + 8 * g + 4 * lg);
          cs[g][0] = t[0];
          cs[g][1] = t[1];
        }
      }
#pragma unroll
      for (int hp = 0; hp < TN / 2; hp++) {
        const int c0 = 64 * hp;                                   // tile column of the head's dim 0
        const bool rot = tab != nullptr && n0 + c0 < 2 * HD;     // a head of q or k
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const int col = c0 + 8 * g + 4 * lg;  // tile column of dim 8g + 4lg
          uint16_t o0[4], o1[4];
#pragma unroll
          for (int e = 0; e < 4; e++) {
            o0[e] = from_f<BF16>(acc[i][2 * hp][4 * g + e]);
            o1[e] = from_f<BF16>(acc[i][2 * hp + 1][4 * g + e]);
          }
          if (rot) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
              const float c = cs[g][e >> 1][2 * (e & 1)], sn = cs[g][e >> 1][2 * (e & 1) + 1];
              const float x0 = to_f<BF16>(o0[e]), x1 = to_f<BF16>(o1[e]);
              o0[e] = from_f<BF16>(pin_f32(fmaf(-x1, sn, x0 * c)));
              o1[e] = from_f<BF16>(pin_f32(fmaf(x0, sn, x1 * c)));
            }
          }
          *(uint2v*)(Cs + r_slot(row, col >> 3) * 8 + (col & 7)) =
              uint2v{(uint32_t)o0[0] | ((uint32_t)o0[1] << 16), (uint32_t)o0[2] | ((uint32_t)o0[3] << 16)};
          *(uint2v*)(Cs + r_slot(row, (col + 32) >> 3) * 8 + (col & 7)) =
              uint2v{(uint32_t)o1[0] | ((uint32_t)o1[1] << 16), (uint32_t)o1[2] | ((uint32_t)o1[3] << 16)};
        }
      }
    }
  };
  // ---- QKV write-out: 8 threads per tile row, thread t8 takes the 16-byte
  // chunk t8 of each head (dims 8 t8 .. 8 t8 + 7), so 8 threads write one
  // head row of 128 bytes and a wave 8 consecutive rows of one head
  auto write_out_qkv = [&](int m0, int n0) {
    int t0 = tid, L = qk.L, H = qk.H;
    asm volatile("" : "+v"(t0), "+s"(L), "+s"(H));
    const int t8 = t0 & 7, HD = H * 64, Bn = M / L;
#pragma unroll 1
    for (int r = t0 >> 3; r < BM; r += NT / 8) {
      const int gm = m0 + r;
      if (gm >= M) break;
      const int bb = gm / L, tt = gm - bb * L;
#pragma unroll
      for (int hp = 0; hp < BNO / 64; hp++) {
        const int gn = n0 + 64 * hp;  // the head's first column
        if (gn >= N) break;
        const int part = gn / HD, hh = (gn - part * HD) >> 6;
        uint16_t* dst = Y + ((((int64_t)part * Bn + bb) * H + hh) * L + tt) * 64 + 8 * t8;
        *(uint4v*)dst = out_chunk(r, 8 * hp + t8);
      }
    }
  };

  uint4v A0[TM][KS], A1[TM][KS], A2[TM][KS];
  BRegs B0, B1;
  // step g: MFMAs on `ac` and LDS buffer g&1; loads stage g+2 of the stream
  // into (al, bl); stages the W tile of g+1 (held in bs) into the other buffer.
  //
  // Origins of the block's current tile and of the tile after it, set per
  // tile, so that a stage finds the tile of the stage it loads with scalar
  // selects (for the last tile nxt = cur, nxt_kb = (KT - 1) * BK and
  // nxt_ks = 0: loads past the end of the stream repeat its last stage).
  int cur_m0 = 0, cur_n0 = 0, nxt_m0 = 0, nxt_n0 = 0, nxt_kb = 0, nxt_ks = 0;
  // The residual's pieces go out from stage dma0 on, once the C tile is free
  // (with a spread write-out pending it is read until stage 5), one per
  // stage up to stage dma0 + dpl, which sends the rest: the last piece then
  // has one more stage to land before the epilogue, if the tile has it.
  const int dma0 = spread ? 6 : 0;
  const int dpl = KT - 2 - dma0 < 0 ? 0 : (KT - 2 - dma0 < 5 ? KT - 2 - dma0 : 5);
  // S_: the stage's place in its group of six (a compile-time constant)
  // WO_: whether the stage stores its share of a pending write-out
  auto step = [&](auto S_, auto WO_, int g, int kin, uint4v (&ac)[TM][KS], uint4v (&al)[TM][KS], BRegs& bl,
                  BRegs& bs) __attribute__((always_inline)) {
    constexpr int SP = decltype(S_)::value;
    constexpr bool WO = decltype(WO_)::value && !QKV;
    // stage g + 2 of the stream: stage kin + 2 of this tile, or stage
    // kin + 2 - KT of the next (a block with several tiles has KT >= 6)
    const int k2 = __builtin_amdgcn_readfirstlane(kin + 2);
    const int wrap = __builtin_amdgcn_readfirstlane(k2 >= KT ? 1 : 0);
    const int m2 = __builtin_amdgcn_readfirstlane(wrap ? nxt_m0 : cur_m0);
    const int n2 = __builtin_amdgcn_readfirstlane(wrap ? nxt_n0 : cur_n0);
    const int k2b = __builtin_amdgcn_readfirstlane(wrap ? nxt_kb + (k2 - KT) * nxt_ks : k2 * BK);
    load_a(m2, k2b, al);
    load_b(n2, k2b, bl);
    const uint16_t* b = Bs + (g & 1) * BN * BK;
    uint4v bf[KS][TN];
#pragma unroll
    for (int s = 0; s < KS; s++)
#pragma unroll
      for (int j = 0; j < TN; j++) bf[s][j] = *(const uint4v*)(b + swz(bcol(j) + l32, 2 * s + lg));
#pragma unroll
    for (int s = 0; s < KS; s++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int i = 0; i < TM; i++) acc[i][j] = mfma32<BF16>(bf[s][j], ac[i][s], acc[i][j]);
    if constexpr (WO) wo_part(S_);
    // schedule: substep-0 fragment reads, then MFMA pairs, each preceded by
    // one global load (while any remain) and one fragment read of the next
    // substep; the write-out's C-tile reads ride with the last loads, its
    // stores follow every load; the W staging for the next stage goes last
    constexpr int NVMEM = TM * KS + B_LD, NPAIR = KS * TN, WOS = WO ? WO_PS : 0;
    // the stores two pairs after the last load, or as late as they fit
    constexpr int WST = NVMEM + 2 + WOS <= NPAIR ? NVMEM + 2 : NPAIR - WOS;
    static_assert(NVMEM <= NPAIR && WST > NVMEM - WOS && WST + WOS <= NPAIR, "write-out stores after their reads");
    __builtin_amdgcn_sched_group_barrier(0x100, TN, 0);
#pragma unroll
    for (int p = 0; p < NPAIR; p++) {
      if (p < NVMEM) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      if (p < (KS - 1) * TN) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (p >= NVMEM - WOS && p < NVMEM) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (p >= WST && p < WST + WOS) __builtin_amdgcn_sched_group_barrier(0x040, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, TM, 0);
    }
    store_b((g + 1) & 1, bs);
    __builtin_amdgcn_sched_group_barrier(0x200, B_LD, 0);
    // the residual tile arrives in the C tile while the tile computes: piece
    // p at stage dma0 + min(p, dpl), the last ones together
    if (R != nullptr && kin - SP == dma0 && SP <= dpl) {
      dma_piece(cur_m0, cur_n0, S_);
      if (SP == dpl) {
        if constexpr (SP < 1) dma_piece(cur_m0, cur_n0, std::integral_constant<int, 1>{});
        if constexpr (SP < 2) dma_piece(cur_m0, cur_n0, std::integral_constant<int, 2>{});
        if constexpr (SP < 3) dma_piece(cur_m0, cur_n0, std::integral_constant<int, 3>{});
        if constexpr (SP < 4) dma_piece(cur_m0, cur_n0, std::integral_constant<int, 4>{});
        if constexpr (SP < 5) dma_piece(cur_m0, cur_n0, std::integral_constant<int, 5>{});
      }
    }
    __syncthreads();
  };

  {
    const int m0 = tile_m0(0), n0 = tile_n0(0);
    const int g1 = S > 1 ? 1 : 0, i1 = g1 / KT, k1 = (g1 - i1 * KT) * BK;
    load_a(m0, 0, A0);
    load_b(n0, 0, B0);
    store_b(0, B0);
    load_a(tile_m0(i1), k1, A1);
    load_b(tile_n0(i1), k1, B1);
    __syncthreads();
  }
  // The register rotation has period 6; a tile whose KT is not a multiple of
  // 6 ends with a tail that moves the next tile's registers back to phase 0.
  for (int it = 0; it < ntile; it++) {
    const int g0 = it * KT;
    cur_m0 = tile_m0(it);
    cur_n0 = tile_n0(it);
    const bool has_next = it + 1 < ntile;
    nxt_m0 = has_next ? tile_m0(it + 1) : cur_m0;
    nxt_n0 = has_next ? tile_n0(it + 1) : cur_n0;
    nxt_kb = has_next ? 0 : (KT - 1) * BK;
    nxt_ks = has_next ? BK : 0;
    // Six stages at a time (the register rotation's period), with no branch
    // between them: the compiler places its load waits by tracking which
    // registers have loads in flight, and where paths that ran different
    // numbers of stages join it must assume the union of their loads, which
    // makes a stage wait for the loads issued one stage earlier (for the
    // stage after next) and halves the latency the stream hides.
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    using I4 = std::integral_constant<int, 4>;
    using I5 = std::integral_constant<int, 5>;
    using T = std::true_type;
    using F = std::false_type;
    int kt = 0;
    // a pending write-out leaves in the tile's first six stages (KT >= 12):
    // their own copy of the stage code, so that the other stages carry no
    // store instructions
    if (wo_rec != 0) {
      step(I0{}, T{}, g0, 0, A0, A2, B0, B1);
      step(I1{}, T{}, g0 + 1, 1, A1, A0, B1, B0);
      step(I2{}, T{}, g0 + 2, 2, A2, A1, B0, B1);
      step(I3{}, T{}, g0 + 3, 3, A0, A2, B1, B0);
      step(I4{}, T{}, g0 + 4, 4, A1, A0, B0, B1);
      step(I5{}, T{}, g0 + 5, 5, A2, A1, B1, B0);
      wo_rec = 0;
      kt = 6;
    }
    for (; kt + 6 <= KT; kt += 6) {
      step(I0{}, F{}, g0 + kt, kt, A0, A2, B0, B1);
      step(I1{}, F{}, g0 + kt + 1, kt + 1, A1, A0, B1, B0);
      step(I2{}, F{}, g0 + kt + 2, kt + 2, A2, A1, B0, B1);
      step(I3{}, F{}, g0 + kt + 3, kt + 3, A0, A2, B1, B0);
      step(I4{}, F{}, g0 + kt + 4, kt + 4, A1, A0, B0, B1);
      step(I5{}, F{}, g0 + kt + 5, kt + 5, A2, A1, B1, B0);
    }
    // The last q = KT % 6 stages.  Every load is drained after them, so the
    // join after this tail leaves the compiler's view of the loads in flight
    // exactly that of the loop above.  The next tile's first two stages are
    // then in registers named by phase q (its stage-0 X rows in set q % 3,
    // its stage-1 X rows in set (q + 1) % 3, its stage-1 W in set
    // (q + 1) % 2): they are moved to the names the tile loop starts from
    // (A0, A1, B1), so that every tile starts at phase 0 whatever KT is.
    if (kt < KT) {
      const int q = KT - kt;
      step(I0{}, F{}, g0 + kt, kt, A0, A2, B0, B1);
      if (q > 1) step(I1{}, F{}, g0 + kt + 1, kt + 1, A1, A0, B1, B0);
      if (q > 2) step(I2{}, F{}, g0 + kt + 2, kt + 2, A2, A1, B0, B1);
      if (q > 3) step(I3{}, F{}, g0 + kt + 3, kt + 3, A0, A2, B1, B0);
      if (q > 4) step(I4{}, F{}, g0 + kt + 4, kt + 4, A1, A0, B0, B1);
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
      if (has_next) {
        if (q % 3 == 1) {  // stage 0 in A1, stage 1 in A2 (A0 is free)
#pragma unroll
          for (int i = 0; i < TM; i++)
#pragma unroll
            for (int s = 0; s < KS; s++) {
              A0[i][s] = A1[i][s];
              A1[i][s] = A2[i][s];
            }
        } else if (q % 3 == 2) {  // stage 0 in A2, stage 1 in A0 (A1 is free)
#pragma unroll
          for (int i = 0; i < TM; i++)
#pragma unroll
            for (int s = 0; s < KS; s++) {
              A1[i][s] = A0[i][s];
              A0[i][s] = A2[i][s];
            }
        }
        if (q & 1) B1 = B0;  // stage-1 W in B0
      }
    }
    // The residual's last pieces went out at the end of stage dma0 + dpl, and
    // memory operations complete in issue order: they have landed once at
    // most the loads and stores of one later stage are outstanding (or none,
    // when they went out with the last stage).  The
    // barrier makes every wave's part of the C tile visible (and, without R,
    // keeps the previous tile's write-out reads ahead of this epilogue's
    // writes).
    constexpr int VM1 = TM * KS + B_LD;  // the loads of one stage (stages after the pieces store nothing)
    static_assert(VM1 <= 63, "vmcnt immediate");
    if (R != nullptr) {
      if (dma0 + dpl >= KT - 1) __builtin_amdgcn_s_waitcnt(0x0F70);
      else __builtin_amdgcn_s_waitcnt(0x0F70 | (VM1 & 15) | ((VM1 >> 4) << 14));
    }
    __syncthreads();
    {
      const int n0 = cur_n0;
      if constexpr (QKV) {
        epilogue_qkv(cur_m0, n0);
      } else if (bias == nullptr) {
        if (R == nullptr) epilogue(n0, F{}, F{});
        else epilogue(n0, F{}, T{});
      } else {
        if (R == nullptr) epilogue(n0, T{}, F{});
        else epilogue(n0, T{}, T{});
      }
    }
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
    __syncthreads();
    if constexpr (QKV) {
      write_out_qkv(cur_m0, cur_n0);
    } else if (spread && has_next && cur_m0 + BM <= M && cur_n0 + BNO <= N) {
      wo_set(cur_m0, cur_n0);  // leaves during the next tile's first six stages
    } else {
      write_out(cur_m0, cur_n0);
      if (R != nullptr) __syncthreads();  // the next tile's residual DMA refills the C tile
    }
  }
}

// ------------------------------------------------------------------ launchers

template <int BM, int BN, int WM, int WN, bool BF16, bool GEGLU, int QB, bool AFF, bool SF32>
void launch_mfma(hipStream_t st, const uint16_t* x, int64_t ldx, const uint16_t* w, QW qw,
                        const uint16_t* bias, const uint16_t* r, int64_t ldr, uint16_t* y, int64_t ldy, int M, int N,
                        int K) {
  constexpr int BNO = GEGLU ? BN / 2 : BN;
  int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BNO - 1) / BNO;
  size_t stage = (size_t)2 * (BM + BN) * 64 * sizeof(uint16_t);
  size_t ctile = (size_t)BM * BNO * sizeof(uint16_t);
  size_t lds = stage > ctile ? stage : ctile;
  auto kern = gemm_mfma<BM, BN, WM, WN, BF16, GEGLU, QB, AFF, SF32>;
  static std::atomic<uint64_t> attr{0};
  once_per_device(attr, [&] {
    HB_CHECK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  });
  kern<<<tiles_m * tiles_n, WM * WN * 64, lds, st>>>(x, ldx, w, qw, bias, r, ldr, y, ldy, M, N, K, tiles_n);
}

// Blocks per XCD of the large-M kernel, and the tiles the busiest one walks:
// an XCD owns whole row panels, so it may hold more than an eighth of the tiles.
inline int64_t arow_tiles_per_xcd(int64_t M, int64_t tiles_n) { return ((M + 255) / 256 + 7) / 8 * tiles_n; }
inline int64_t arow_rounds(int64_t M, int64_t tiles_n, int cus) {
  return (arow_tiles_per_xcd(M, tiles_n) + cus / 8 - 1) / (cus / 8);
}

template <int BN, bool BF16, bool GEGLU, bool KTAIL, bool QKV = false>
void launch_arow(hipStream_t st, int cus, unsigned pan, const uint16_t* x, int64_t ldx, const uint16_t* w,
                 const uint16_t* bias, const uint16_t* r, int64_t ldr, uint16_t* y, int64_t ldy, int M, int N, int K,
                 QK qk = QK{nullptr, 1, 1}) {
  constexpr int BNO = GEGLU ? BN / 2 : BN;
  const int tiles_m = (M + 255) / 256, tiles_n = (N + BNO - 1) / BNO, tiles = tiles_m * tiles_n;
  // one persistent block per CU, a multiple of 8 (one per XCD), streaming
  // its tiles when they have a multiple of 6 or at least 12 K stages (the
  // shapes measured and tested).  Otherwise one tile per block: every XCD
  // gets as many blocks as the largest XCD share of tiles (ceil(tiles_m / 8)
  // row panels).
  const int KT = (K + 63) / 64;
  const bool stream = KT % 6 == 0 || KT >= 12;
  // (streaming: never fewer blocks than the busiest XCD has tiles to run side by
  // side: 5120 x 768 x 768, 20 row panels, 38 -> 23 us)
  const int64_t per_xcd = arow_tiles_per_xcd(M, tiles_n);
  const int grid = (int)(8 * (stream && per_xcd > cus / 8 ? cus / 8 : per_xcd));
  HB_REQUIRE(grid >= 8, "hb_linear: large-M GEMM needs at least 8 tiles");
  constexpr int RG = (BNO / 8 + 7) / 8;
  // W tiles and the C tile
  const size_t lds = ((size_t)2 * BN * 64 + (size_t)RG * 256 * 64) * sizeof(uint16_t);
  auto kern = gemm_mfma_arow<BN, BF16, GEGLU, KTAIL, QKV>;
  static std::atomic<uint64_t> attr{0};
  once_per_device(attr, [&] {
    HB_CHECK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  });
  kern<<<grid, 256, lds, st>>>(x, ldx, w, bias, r, ldr, y, ldy, M, N, K, tiles_n, tiles, (pan & HB_X_PANEL) ? 1 : 0,
                               (pan & HB_Y_PANEL) ? 1 : 0, qk);
}

template <int BM, int BN, int WM, int WN, int NST, bool BF16, bool GEGLU>
void launch_ring_t(hipStream_t st, unsigned pan, const uint16_t* x, int64_t ldx, const uint16_t* w, const uint16_t* bias,
                   const uint16_t* r, int64_t ldr, uint16_t* y, int64_t ldy, int M, int N, int K) {
  constexpr int BNO = GEGLU ? BN / 2 : BN;
  constexpr int lds = NST * (BM + BN) * 128;
  static_assert(lds >= BM * BN * 2 && lds <= 160 * 1024, "the C tile reuses the ring");
  auto kern = gemm_ring<BM, BN, WM, WN, NST, BF16, GEGLU>;
  static std::atomic<uint64_t> attr{0};
  once_per_device(attr, [&] {
    HB_CHECK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  });
  const int64_t tiles_m = (M + BM - 1) / BM, tiles_n = (N + BNO - 1) / BNO;
  HB_REQUIRE(tiles_m * tiles_n < (1ll << 31), "hb_linear: too many tiles");
  kern<<<(unsigned)(tiles_m * tiles_n), WM * WN * 64, lds, st>>>(x, ldx, w, bias, r, ldr, y, ldy, M, N, K, (int)tiles_n,
                                                                  (pan & HB_X_PANEL) ? 1 : 0, (pan & HB_Y_PANEL) ? 1 : 0);
}

// Operands that the ring kernel's and the large-M kernel's 32-bit offsets reach
// (the last row of a tile is at most 255 strides away).
inline bool ring_ok(int64_t ldx, int64_t K) { return K % 64 == 0 && K < (1 << 22) && ldx < (1 << 22); }

// The kernels of a linear layer with 16-bit weights (and, the mfma ones, with
// codes that their loader dequantizes).
enum class LinearKernel {
  kRing32x64,     // six stages
  kRing64x64,     // four stages
  kRing64x64k,    // five: K chains of 32 and more stages wait for memory
  kRing64x64x3,   // three, so that three blocks share a CU
  kRing128x64,
  kRing128x256,
  kMfma128x64,
  kMfma128x128,
  kArow192,
  kArow192Tail,   // any K, 64-bit addresses
  kArow128,
  kArow128Tail,
};
inline bool is_ring(LinearKernel k) { return k <= LinearKernel::kRing128x256; }
inline const char* linear_kernel_name(LinearKernel k) {
  static const char* const names[] = {"ring 32x64",  "ring 64x64",   "ring 64x64 long", "ring 64x64 three",
                                      "ring 128x64", "ring 128x256", "mfma 128x64",     "mfma 128x128",
                                      "arow 192",    "arow 192 tail", "arow 128",       "arow 128 tail"};
  return names[(int)k];
}

// The ring's tile, by how many of each shape the call has (wrows: weight rows;
// us, f16, back to back; 64 x 64 / 128 x 64 / 64 x 64 with three stages, and the
// 128-row kernel):
// - 32 x 64, six stages, while they fit one per CU: with weights that come from
//   HBM (a model's layers in turn), where the bytes a launch has in flight count,
//   128 x 2304 x 768 7.9 -> 6.7, 128 x 2304 x 768 GeGLU 8.2 -> 7.0 against 64 x 64;
// - 64 x 64, four stages, while those fit: 128 x 768 x 768 (24 tiles)
//   5.8 / 7.4 / 6.3 (9.7), 256 x 2304 x 768 (144) 5.9 / 7.4 / 6.6 (11.5); from
//   K = 2048 five stages: 512 x 768 x 3072 16.1 -> 13.7 (32.5);
// - 128 x 64 while those fit: 512 x 3072 x 768 (192) 10.7 / 8.3 / 11.3 (12.1),
//   768 x 2304 x 768 (216) 8.7 / 8.4 / 9.3 (12.3);
// - 64 x 64 with three stages while three fit a CU: 1024 x 3072 x 768 15.4 /
//   15.7 / 12.6 (16.4), 4096 x 768 x 768 12.1 / 14.0 / 11.1;
// - 128 x 256, one round of them: where the 128-row kernel does not take the call
//   (`wide`) if it fills half the CUs: 4200 x 1536 x 384 14.3, 64 x 64 with three
//   stages 16.5, 5500 x 768 x 3072 52.2 / 57.6.  Against the 128-row kernel from
//   three quarters of the CUs on, or half for a weight just written (`cached`),
//   for K of 512 to 1536 (beyond that the three stages wait for weights from HBM:
//   2048 x 2304 x 3072 69 against 58 us) and without GeGLU (whose epilogue costs
//   the single block of a CU more: 2048 x 1152 x 768 21.5 / 19.7); weights in the
//   caches / from HBM: 2048 x 2304 x 768 (144 tiles) 18.3 and 20.5 / 23.1 and 20.6,
//   2048 x 3072 x 768 (192) 20.9 and 22.4 / 23.8 and 23.1, 3072 x 2304 x 768 (216)
//   20.4 and 22.5 / 23.7 and 23.5; a 2048-token f16 forward takes 1.98 ms without
//   them at 144 tiles, 2.05 with, a q4 one, whose weights are copies just
//   dequantized, 2.19 and 2.17;
// - 64 x 64 with three stages in up to three rounds where the 128-row kernel's
//   128 x 128 tiles begin a second round (two fit a CU), unless the weight is
//   the wider side: 4095 x 2304 x 768 30 / 36, 3072 x 3072 x 1024 38 / 44, 1792 x
//   5248 x 1024 46 / 44;
// - else none below M = 4096 (not `wide`): the 128-row kernel reads half as
//   much LDS per product as a 64 x 64 tile.  1536 x 2304 x 768 18.0 / 16.0 us,
//   2048 x 2624 x 1024 GeGLU 56.8 / 43.4, 3840 x 4096 x 1024 68.1 / 51.9.
inline bool ring_tile(int cus, int64_t M, int64_t wrows, int64_t K, bool geglu, bool wide, bool cached,
                      LinearKernel* tile) {
  auto tiles = [&](int bm, int bn) { return ((M + (int64_t)bm - 1) / bm) * ((wrows + bn - 1) / bn); };
  const int64_t t64 = tiles(64, 64), t256 = tiles(128, 256);
  if (tiles(32, 64) <= cus) *tile = LinearKernel::kRing32x64;
  else if (t64 <= cus) *tile = K < 2048 ? LinearKernel::kRing64x64 : LinearKernel::kRing64x64k;
  else if (tiles(128, 64) <= cus) *tile = LinearKernel::kRing128x64;
  else if (t64 <= 3 * (int64_t)cus) *tile = LinearKernel::kRing64x64x3;
  else if (t256 > (cached || wide ? cus / 2 : cus * 3 / 4 - 1) && t256 <= cus &&
           (wide || (!geglu && K >= 512 && K <= 1536)))
    *tile = LinearKernel::kRing128x256;
  else if (wide || (t64 <= 9 * (int64_t)cus && tiles(128, 128) > 2 * (int64_t)cus && M >= wrows))
    *tile = LinearKernel::kRing64x64x3;
  else return false;
  return true;
}

// From M = 4096, the ring kernel still beats the large-M one where its 256 x 192
// tiles are few (N = 768 at M = 4096: 64 tiles): both as measured, in us: the
// large-M kernel a fixed 7.5 and 3 + 0.016 K a round, the ring 4 and 3.4 per
// 64 x 64 tile and CU at K = 768.  Both sides (large-M with panel-order X /
// ring): 4096 x 768 x 768 22.8 / 15.4, 6144 x 768 x 1152 28.5 / 26.7, 8192 x 768
// x 768 23.5 / 23.6, 4096 x 2304 x 768 25.3 / 33.6, 6144 x 768 x 3072 55.6 / 58.2.
// Checked as a choice on 160 calls of M = 4200 to 20000 (128-column tiles, K of 200
// to 4096, GeGLU and quantized ones among them): none slower than the large-M
// kernel alone, by 2% or more.
inline bool ring_beats_arow(int64_t M, int64_t N_out, int64_t K, bool geglu, int bn, int cus) {
  const int64_t wrows = geglu ? 2 * N_out : N_out, bno = geglu ? bn / 2 : bn;
  const double per_cu = (double)(((M + 63) / 64) * ((wrows + 63) / 64)) / cus;
  const double ring = 4 + 3.4 * (K / 768.0) * (per_cu > 1 ? per_cu : 1);
  const double arow = 7.5 + (double)arow_rounds(M, (N_out + bno - 1) / bno, cus) * (3 + 0.016 * K) * (bn / 192.0);
  return ring < arow;
}

// Calls below M = 4096 that take panel-order operands: 16-bit weights within the
// bounds that laya_hip.h gives its callers.  They are the interface's and not
// gemm_ring's, which takes panel order at any size with K % 64 == 0.
inline bool small_panel_path(int64_t M, int64_t N_out, int64_t K, bool geglu, int cus) {
  const int64_t tiles_n = (N_out + 31) / 32, chunks = (M + 127) / 128;
  return K % 64 == 0 && K * 32 * (geglu ? 2 : 1) * 2 <= 160 * 1024 && tiles_n * chunks <= cus;
}

// Calls of the large-M kernel's size (the ring kernel takes those it beats it
// at); both take panel-order operands.
inline bool arow_path(int64_t M) { return M >= 4096; }

// 128 x 64 tiles of the 128-row kernel (instead of 128 x 128) where 128 x 128
// tiles would leave the GPU short of blocks: the K stages of a block run one
// after another, so a launch with few blocks is bound by that chain.
// N_out: output columns (GeGLU: value / gate pairs).
inline bool thin_tiles(int64_t M, int64_t N_out, bool geglu, int cus) {
  const int64_t t128 = ((M + 127) / 128) * ((N_out + (geglu ? 63 : 127)) / (geglu ? 64 : 128));
  return t128 <= cus + cus / 8;
}

// The 128-row kernel, which reads codes too.
inline LinearKernel code_kernel(int cus, int64_t M, int64_t N_out, bool geglu) {
  return thin_tiles(M, N_out, geglu, cus) ? LinearKernel::kMfma128x64 : LinearKernel::kMfma128x128;
}

// The kernel a call with 16-bit weights takes.  `ldx`: X's row stride, K in
// panel order; `panel`: X or Y in panel order, which the 128-row kernel does
// not take; `cached`: the weight is a copy that a kernel just wrote.  Every output keeps its MFMA sequence and epilogue, so the bits do
// not depend on the choice.
inline LinearKernel linear_kernel(int cus, int64_t M, int64_t N_out, int64_t K, int64_t ldx, bool geglu, bool panel,
                                  bool cached) {
  // 128-column tiles of the large-M kernel where N is a multiple of 128 and
  // not of 192 (N = 1024: 8 whole tiles instead of 5 1/3 of 192 columns)
  const bool n128 = !geglu && N_out % 192 != 0 && N_out % 128 == 0;
  const bool ring = ring_ok(ldx, K), large = arow_path(M);
  LinearKernel tile;
  if (ring && (!large || ring_beats_arow(M, N_out, K, geglu, n128 ? 128 : 192, cus)) &&
      ring_tile(cus, M, geglu ? 2 * N_out : N_out, K, geglu, large || panel, cached, &tile))
    return tile;
  if (large || panel) {
    // (X rows too far apart for 32-bit offsets: the tail variant's are 64-bit)
    if (ring) return n128 ? LinearKernel::kArow128 : LinearKernel::kArow192;
    return n128 ? LinearKernel::kArow128Tail : LinearKernel::kArow192Tail;
  }
  return code_kernel(cus, M, N_out, geglu);
}

// Whether a quantized weight is dequantized once per call, into a 16-bit copy
// for the kernel above, instead of in the 128-row kernel's loader in every row
// tile.  The pass costs a launch and its traffic (5 bytes a weight and more, 1
// us per million weights once they leave the caches); the loader about 0.6 us
// a K stage over the ring, whatever the width while its tiles run side by
// side.  So the ring takes the call where the weight is small against its K
// chain.  us, pass + ring / loader, q8 to f16: 128 x 2304 x 768 12.5 / 13.9, 512
// x 768 x 1152 11 / 18.8, 128 x 768 x 3072 19.8 / 41, 256 x 5248 x 1024 15.8 /
// 17.6; 768 x 48 x 64 6.4 / 5.3, 256 x 16384 x 768 30.8 / 18.8, 1 x 50368 x 768
// 40 / 25, 1 x 256000 x 1024 261 / 116.  From M = 1024, where the 128-row kernel
// would run 128 x 128 tiles, its loader repeats the work too often (3072 x 2304
// x 768 23.9 / 27.8).
inline bool dequantizes_first(int cus, int64_t M, int64_t N_out, int64_t K, int64_t ldx, bool geglu) {
  if (arow_path(M) || (M >= 1024 && !thin_tiles(M, N_out, geglu, cus))) return true;
  return is_ring(linear_kernel(cus, M, N_out, K, ldx, geglu, false, true)) &&
         (geglu ? 2 : 1) * N_out * K <= (K / 64 - 4) * 500000;
}

template <bool BF16, bool GEGLU, int QB, bool AFF, bool SF32>
void mfma_dispatch(hipStream_t st, int cus, unsigned pan, const uint16_t* x, int64_t ldx, const uint16_t* w,
                          QW qw, const uint16_t* bias, const uint16_t* r, int64_t ldr, uint16_t* y, int64_t ldy, int M,
                          int N, int K) {
  // (codes are read by the 128-row kernel alone: hb_qlinear dequantizes them
  // beforehand for the others, and passes them along with the copy)
  HB_REQUIRE(QB == 0 || !arow_path(M), "hb_qlinear: large-M quantized weights are dequantized before the GEMM");
  const LinearKernel kern = QB == 0 ? linear_kernel(cus, M, N, K, (pan & HB_X_PANEL) ? K : ldx, GEGLU, pan != 0, qw.q != nullptr)
                                    : code_kernel(cus, M, N, GEGLU);
  if constexpr (QB == 0) {
    auto args = [&](auto launch) { launch(st, pan, x, ldx, w, bias, r, ldr, y, ldy, M, N, K); };
    auto arow = [&](auto launch) { launch(st, cus, pan, x, ldx, w, bias, r, ldr, y, ldy, M, N, K, QK{nullptr, 1, 1}); };
    switch (kern) {
      case LinearKernel::kRing32x64: return args(launch_ring_t<32, 64, 1, 2, 6, BF16, GEGLU>);
      case LinearKernel::kRing64x64: return args(launch_ring_t<64, 64, 2, 2, 4, BF16, GEGLU>);
      case LinearKernel::kRing64x64k: return args(launch_ring_t<64, 64, 2, 2, 5, BF16, GEGLU>);
      case LinearKernel::kRing64x64x3: return args(launch_ring_t<64, 64, 2, 2, 3, BF16, GEGLU>);
      case LinearKernel::kRing128x64: return args(launch_ring_t<128, 64, 4, 2, 4, BF16, GEGLU>);
      case LinearKernel::kRing128x256: return args(launch_ring_t<128, 256, 4, 4, 3, BF16, GEGLU>);
      case LinearKernel::kArow192: return arow(launch_arow<192, BF16, GEGLU, false>);
      case LinearKernel::kArow192Tail: return arow(launch_arow<192, BF16, GEGLU, true>);
      case LinearKernel::kArow128:
        if constexpr (!GEGLU) return arow(launch_arow<128, BF16, false, false>);
        break;
      case LinearKernel::kArow128Tail:
        if constexpr (!GEGLU) return arow(launch_arow<128, BF16, false, true>);
        break;
      default: break;
    }
  }
  HB_REQUIRE(pan == 0, "hb_linear: panel-order operands on a kernel that does not take them");
  if (kern == LinearKernel::kMfma128x64)
    launch_mfma<128, 64, 4, 1, BF16, GEGLU, QB, AFF, SF32>(st, x, ldx, w, qw, bias, r, ldr, y, ldy, M, N, K);
  else
    launch_mfma<128, 128, 2, 2, BF16, GEGLU, QB, AFF, SF32>(st, x, ldx, w, qw, bias, r, ldr, y, ldy, M, N, K);
}

template <int QB, bool AFF, bool SF32>
void mfma_dtype(int dt, bool geglu, hipStream_t st, int cus, unsigned pan, const uint16_t* x, int64_t ldx,
                       const uint16_t* w, QW qw, const uint16_t* bias, const uint16_t* r, int64_t ldr, uint16_t* y,
                       int64_t ldy, int M, int N, int K) {
  if (dt == HB_F16) {
    if (geglu) mfma_dispatch<false, true, QB, AFF, SF32>(st, cus, pan, x, ldx, w, qw, bias, r, ldr, y, ldy, M, N, K);
    else mfma_dispatch<false, false, QB, AFF, SF32>(st, cus, pan, x, ldx, w, qw, bias, r, ldr, y, ldy, M, N, K);
  } else {
    if (geglu) mfma_dispatch<true, true, QB, AFF, SF32>(st, cus, pan, x, ldx, w, qw, bias, r, ldr, y, ldy, M, N, K);
    else mfma_dispatch<true, false, QB, AFF, SF32>(st, cus, pan, x, ldx, w, qw, bias, r, ldr, y, ldy, M, N, K);
  }
}

// The fused q / k / v projection (16-bit weights, M >= 4096, K % 64 == 0):
// the large-M kernel with the QKV epilogue.
template <bool BF16>
void launch_qkv(hipStream_t st, int cus, unsigned pan, const uint16_t* x, int64_t ldx, const uint16_t* w,
                uint16_t* y, int M, int N, int K, QK qk) {
  launch_arow<192, BF16, false, false, true>(st, cus, pan, x, ldx, w, nullptr, nullptr, 0, y, 0, M, N, K, qk);
}

// Instantiated by gemm_f16.hip (QB = 0), gemm_q8.hip and gemm_q4.hip.
extern template void launch_qkv<false>(hipStream_t, int, unsigned, const uint16_t*, int64_t, const uint16_t*,
                                       uint16_t*, int, int, int, QK);
extern template void launch_qkv<true>(hipStream_t, int, unsigned, const uint16_t*, int64_t, const uint16_t*,
                                      uint16_t*, int, int, int, QK);
extern template void mfma_dtype<0, false, false>(int, bool, hipStream_t, int, unsigned, const uint16_t*, int64_t,
                                                 const uint16_t*, QW, const uint16_t*, const uint16_t*, int64_t,
                                                 uint16_t*, int64_t, int, int, int);
extern template void mfma_dtype<8, false, false>(int, bool, hipStream_t, int, unsigned, const uint16_t*, int64_t,
                                                 const uint16_t*, QW, const uint16_t*, const uint16_t*, int64_t,
                                                 uint16_t*, int64_t, int, int, int);
extern template void mfma_dtype<8, true, false>(int, bool, hipStream_t, int, unsigned, const uint16_t*, int64_t,
                                                const uint16_t*, QW, const uint16_t*, const uint16_t*, int64_t,
                                                uint16_t*, int64_t, int, int, int);
extern template void mfma_dtype<4, false, false>(int, bool, hipStream_t, int, unsigned, const uint16_t*, int64_t,
                                                 const uint16_t*, QW, const uint16_t*, const uint16_t*, int64_t,
                                                 uint16_t*, int64_t, int, int, int);
extern template void mfma_dtype<4, true, false>(int, bool, hipStream_t, int, unsigned, const uint16_t*, int64_t,
                                                const uint16_t*, QW, const uint16_t*, const uint16_t*, int64_t,
                                                uint16_t*, int64_t, int, int, int);

}  // namespace hb
