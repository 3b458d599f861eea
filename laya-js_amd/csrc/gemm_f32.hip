// f32 linear layers on the matrix cores: y = x . w^T with
// v_mfma_f32_32x32x2_f32 (f32 operands, f32 accumulation), for f32 or
// quantized weights.  gemm.hip's hb_linear / hb_qlinear call it; the SIMT
// kernels there keep the operands this one's 16-byte loads cannot take.
//
// What bounds it: the f32 matrix rate (256 flop per clock and CU, 152 TFLOP/s
// measured with an 8192^3 library product) where tiles fill the chip, the
// latency of one chain of K stages where they do not.  An f32 MFMA takes 64
// cycles for 2 KB of operands, so neither LDS (16-32 bytes per clock of 128)
// nor L2 is near its limit and small tiles cost nothing:
// - 32 x 32 tiles for few rows, each K stage of 128 split over the block's 8
//   waves (16 columns each; the partial sums are added in LDS in wave order),
//   so that 93 rows of a 768-wide layer still run 72 blocks of 8 waves and
//   the chain over K = 768 is 6 stages, loaded two ahead;
// - 32 x 64 tiles, stages of 64 split four ways, in between: a CU's last tile
//   is half the work of a 64 x 64 one;
// - 64 x 64 tiles, stages of 32 split two ways, for many rows: half the L2
//   traffic per product.
// Measured, 768 wide: 93 rows x 2304 columns 450 -> 7.8 us (gemm_simt before),
// 4096 x 2304 1360 -> 129 us (112 TFLOP/s).  The sums are shorter than one
// chain over K and their error against 64 bits smaller: 2.9e-7 relative at 93
// x 2304 x 768 with one chain, 1.5e-7 split eight ways.
#include <stdexcept>

#include "common.h"

namespace hb {

struct F32Weight {  // f32 rows, or codes with f16 scales (and zeros)
  const float* w;
  const uint8_t* q;
  const uint16_t* scales;
  const uint16_t* zeros;
  int G, group;
};

// Tile: BM rows x BN weight rows (GEGLU: BN/2 value rows, then their gate
// rows), WM x WN x WK waves of TM x TN 32 x 32 blocks; wave group wk of WK
// multiplies columns [KW * wk, KW * (wk + 1)) of each stage.  LDS rows hold
// one stage of a row in 16-byte chunks, XOR-swizzled so that the 16 lanes of
// a fragment-read pass (16 rows, one chunk column) and of a staging store
// cover all 64 banks.
template <int BM, int BN, int WM, int WN, int WK, int KW, int AHEAD, bool GEGLU, int QB, bool AFF>
__global__ __launch_bounds__(WM* WN* WK * 64) void gemm_f32_kernel(const float* __restrict__ X, int64_t ldx, F32Weight W,
                                                                   const float* __restrict__ bias,
                                                                   const float* __restrict__ R, int64_t ldr,
                                                                   float* __restrict__ Y, int64_t ldy, int M, int N,
                                                                   int K, int tiles_m, int tiles_n) {
  constexpr int NT = WM * WN * WK * 64, BK = KW * WK, CH = BK / 4;
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  constexpr int WAVES = WM * WN * WK, NJ = TN * WN;  // column blocks of the tile
  constexpr int NOUT = GEGLU ? NJ / 2 : NJ;           // output column blocks
  constexpr int XL = BM * CH / NT, WL = BN * CH / NT;  // staged chunks per thread
  constexpr int STAGE = (BM + BN) * BK;                // floats per LDS buffer
  static_assert(XL * NT == BM * CH && WL * NT == BN * CH, "whole rounds of staging");
  static_assert(!GEGLU || NJ % 2 == 0, "value and gate blocks");
  static_assert(CH == 8 || CH % 16 == 0, "swizzle");
  constexpr bool VIA_LDS = WK > 1 || GEGLU;  // sums, or a column's value and gate, meet in LDS
  static_assert(!VIA_LDS || WAVES * TM * TN * 1024 <= 2 * STAGE, "the tile's partial sums fit the stage buffers");
  extern __shared__ __attribute__((aligned(16))) float smem_f32[];

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, lg = lane >> 5;
  // the same in every lane: keeps the wave's addressing scalar
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave / (WM * WN), wm = (wave / WN) % WM, wn = wave % WN;
  // Tiles go to XCDs in contiguous runs, in groups of 8 row tiles walked
  // column by column: the blocks an XCD runs together share 8 row panels and
  // a few weight tiles, which fit its 4 MB L2 (the whole weight, 7 MB at
  // 2304 x 768, does not).
  const int t = xcd_tile(blockIdx.x, gridDim.x);
  const int per = 8 * tiles_n, grp = t / per, gm = min(8, tiles_m - grp * 8);
  const int m0 = (grp * 8 + (t - grp * per) % gm) * BM;
  const int n0 = ((t - grp * per) / gm) * (GEGLU ? BN / 2 : BN);

  // a tile's weight row r; rows past the matrix are clamped (never stored)
  auto wrow = [&](int r) -> int {
    const bool gate = GEGLU && r >= BN / 2;
    const int n = n0 + (gate ? r - BN / 2 : r);
    return (n < N ? n : N - 1) + (gate ? N : 0);
  };
  auto slot = [](int r, int c) { return CH == 8 ? c ^ ((r >> 1) & 7) : c ^ (r & 15); };

  struct Regs {
    float4v x[XL], w[WL];  // quantized weights: w.x = 4 codes, w.y / w.z = scale / zero (f16 bits)
  };
  auto load = [&](Regs& g, int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XL; i++) {
      const int q = tid + i * NT, r = q / CH, k = k0 + (q % CH) * 4;
      const int row = m0 + r < M ? m0 + r : M - 1;
      g.x[i] = k < K ? *(const float4v*)(X + (int64_t)row * ldx + k) : float4v{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int i = 0; i < WL; i++) {
      const int q = tid + i * NT, r = q / CH, k = k0 + (q % CH) * 4;
      g.w[i] = float4v{0.f, 0.f, 0.f, 0.f};
      if (k >= K) continue;
      const int64_t row = wrow(r);
      if constexpr (QB == 0) {
        g.w[i] = *(const float4v*)(W.w + row * K + k);
      } else {
        const uint32_t code = QB == 8 ? *(const uint32_t*)(W.q + row * K + k)
                                      : (uint32_t) * (const uint16_t*)(W.q + ((row * K + k) >> 1));
        const int64_t gi = row * W.G + k / W.group;
        g.w[i].x = __uint_as_float(code);
        g.w[i].y = __uint_as_float((uint32_t)W.scales[gi]);
        if constexpr (AFF) g.w[i].z = __uint_as_float((uint32_t)W.zeros[gi]);
      }
    }
  };
  // 4 dequantized weights, each q*s (+ z) rounded once to f32 (q*s is exact)
  auto value = [](float4v v) -> float4v {
    if constexpr (QB == 0) {
      return v;
    } else {
      const uint32_t code = __float_as_uint(v.x);
      const float s = f16_bits_to_f32((uint16_t)__float_as_uint(v.y));
      const float z = AFF ? f16_bits_to_f32((uint16_t)__float_as_uint(v.z)) : 0.f;
      float4v o;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const uint32_t u = (code >> (QB * e)) & (QB == 8 ? 255u : 15u);
        const int c = AFF ? (int)u : (QB == 8 ? (int)(int8_t)u : ((int)u ^ 8) - 8);
        o[e] = AFF ? (float)c * s + z : (float)c * s;
      }
      return o;
    }
  };
  auto stage_in = [&](const Regs& g, float* buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XL; i++) {
      const int q = tid + i * NT, r = q / CH;
      *(float4v*)(buf + r * BK + slot(r, q % CH) * 4) = g.x[i];
    }
#pragma unroll
    for (int i = 0; i < WL; i++) {
      const int q = tid + i * NT, r = BM + q / CH;
      *(float4v*)(buf + r * BK + slot(r, q % CH) * 4) = value(g.w[i]);
    }
  };

  float16v acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

  // One stage: registers -> LDS, the stage AHEAD of it -> the freed
  // registers, one barrier, then the products.  The buffer written here was
  // last read two stages ago, before the barrier of the stage in between.
  // A chunk's 4 values are 4 MFMA steps; the two lane halves hold the two
  // columns of a step (k and k + 4), the same for both operands.
  const int S = (K + BK - 1) / BK;
  Regs regs[AHEAD];
#pragma unroll
  for (int a = 0; a < AHEAD; a++)
    if (a < S) load(regs[a], a * BK);
  auto stage = [&](int s, Regs& g) __attribute__((always_inline)) {
    float* buf = smem_f32 + (s & 1) * STAGE;
    stage_in(g, buf);
    if (s + AHEAD < S) load(g, (s + AHEAD) * BK);
    __syncthreads();
#pragma unroll
    for (int c8 = 0; c8 < KW / 8; c8++) {
      const int c = wk * (KW / 4) + 2 * c8 + lg;
      float4v a[TM], b[TN];
#pragma unroll
      for (int i = 0; i < TM; i++) {
        const int r = (wm * TM + i) * 32 + l32;
        a[i] = *(const float4v*)(buf + r * BK + slot(r, c) * 4);
      }
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const int r = BM + (wn * TN + j) * 32 + l32;
        b[j] = *(const float4v*)(buf + r * BK + slot(r, c) * 4);
      }
#pragma unroll
      for (int e = 0; e < 4; e++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < TN; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][e], b[j][e], acc[i][j], 0, 0, 0);
    }
  };
  for (int s = 0; s < S; s += AHEAD) {
#pragma unroll
    for (int a = 0; a < AHEAD; a++)
      if (s + a < S) stage(s + a, regs[a]);
  }

  // register r of a block is row 8 * (r / 4) + 4 * lg + r % 4, column l32: a
  // store instruction writes two whole 128-byte lines
  auto emit = [&](int i, int j, int r, float v, float g) __attribute__((always_inline)) {
    const int row = m0 + i * 32 + 8 * (r >> 2) + 4 * lg + (r & 3), col = n0 + j * 32 + l32;
    if (row >= M || col >= N) return;
    if (bias != nullptr) v += bias[col];
    if constexpr (GEGLU) {
      if (bias != nullptr) g += bias[N + col];
      v = gelu_erf(v) * g;
    }
    if (R != nullptr) v += R[(int64_t)row * ldr + col];
    Y[(int64_t)row * ldy + col] = v;
  };
  if constexpr (!VIA_LDS) {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) emit(wm * TM + i, wn * TN + j, r, acc[i][j][r], 0.f);
  } else {
    // every wave leaves its blocks in LDS as [wk][row block][column block][r]
    // [lane]; the waves then share out the tile's registers: the WK partial
    // sums of a value are added in wave order, its gate's likewise
    __syncthreads();
    constexpr int MI = TM * WM;
    auto at = [&](int u, int i, int j, int r) -> float& {
      return smem_f32[(((u * MI + i) * NJ + j) * 16 + r) * 64 + lane];
    };
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) at(wk, wm * TM + i, wn * TN + j, r) = acc[i][j][r];
    __syncthreads();
    constexpr int TOTAL = MI * NOUT * 16;
    static_assert(TOTAL % WAVES == 0, "whole rounds of the epilogue");
#pragma unroll 4
    for (int p = 0; p < TOTAL / WAVES; p++) {
      const int o = p * WAVES + wave, r = o & 15, j = (o >> 4) % NOUT, i = (o >> 4) / NOUT;
      float v = 0.f, g = 0.f;
#pragma unroll
      for (int u = 0; u < WK; u++) {
        v += at(u, i, j, r);
        if constexpr (GEGLU) g += at(u, i, j + NOUT, r);
      }
      emit(i, j, r, v, g);
    }
  }
}

template <int BM, int BN, int WM, int WN, int WK, int KW, int AHEAD, bool GEGLU, int QB, bool AFF>
static void launch_f32_tile(hipStream_t st, const float* x, int64_t ldx, const F32Weight& w, const float* bias,
                            const float* r, int64_t ldr, float* y, int64_t ldy, int M, int N, int K) {
  constexpr int lds = 2 * (BM + BN) * KW * WK * (int)sizeof(float), BNO = GEGLU ? BN / 2 : BN;
  auto kern = gemm_f32_kernel<BM, BN, WM, WN, WK, KW, AHEAD, GEGLU, QB, AFF>;
  if constexpr (lds > 64 * 1024) {
    static std::atomic<uint64_t> attr{0};
    once_per_device(attr, [&] {
      HB_CHECK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    });
  }
  const int tm = (M + BM - 1) / BM, tn = (N + BNO - 1) / BNO;
  HB_REQUIRE((int64_t)tm * tn < (1ll << 31) && 8ll * tn < (1ll << 31), "f32 linear: too many tiles");
  kern<<<(unsigned)((int64_t)tm * tn), WM * WN * WK * 64, lds, st>>>(x, ldx, w, bias, r, ldr, y, ldy, M, N, K, tm, tn);
}

template <bool GEGLU, int QB, bool AFF>
static void launch_f32(hipStream_t st, int cus, const float* x, int64_t ldx, const F32Weight& w, const float* bias,
                       const float* r, int64_t ldr, float* y, int64_t ldy, int M, int N, int K) {
  const int64_t wrows = GEGLU ? 2 * (int64_t)N : N;
  // By the number of 32 x 32 tiles, and not by GEGLU: the fused and the
  // separate GeGLU take the same sums.  The tiles split K eight, four and two
  // ways, so (unlike a 16-bit row's) an f32 row's last bits depend on the call's
  // row count.  Both sides of each line, us at K = 768
  // (small / middle / large):
  // - up to two tiles per CU: 93 x 2304 (216 tiles) 7.8 / 11.7 / 19, 512 x 768
  //   (384) 11.6 / 11.6 / 18.8, 256 x 2304 (576) 17.4 / 19.4 / 19.7, and with
  //   GeGLU 93 rows 11.2 / 11.5 / 19.2, 256 rows (576) 21.2 / 19.2 / 19.5;
  // - up to 20 per CU: 1024 x 2304 (2304 tiles) 44.7 / 41.6 / 46.9, 2048 x 768
  //   (1536) 29.9 / 26.4 / 31.6, 2048 x 2304 (4608) 85 / 72.3 / 73.8, and
  //   2048 x 3072 at K = 1024 (6144) 143 / 121.5 / 114.9.
  const int64_t t32 = (int64_t)((M + 31) / 32) * ((wrows + 31) / 32);
  const int c = t32 <= 2 * cus ? 0 : t32 <= 20 * cus ? 1 : 2;
  if (c == 0)
    launch_f32_tile<32, GEGLU ? 64 : 32, 1, GEGLU ? 2 : 1, 8, 16, 2, GEGLU, QB, AFF>(st, x, ldx, w, bias, r, ldr, y, ldy,
                                                                                    M, N, K);
  else if (c == 1)
    launch_f32_tile<32, 64, 1, 2, 4, 16, 2, GEGLU, QB, AFF>(st, x, ldx, w, bias, r, ldr, y, ldy, M, N, K);
  else
    launch_f32_tile<64, 64, 2, 2, 2, 16, 2, GEGLU, QB, AFF>(st, x, ldx, w, bias, r, ldr, y, ldy, M, N, K);
}

// f32 linear layer; bits = 0: f32 weights `w`, else codes with f16 scales
// (and, `aff`, zeros).  The caller has checked f32_linear_ok.
void f32_linear(hipStream_t st, int cus, const float* x, int64_t ldx, const float* w, const uint8_t* q, const uint16_t* scales,
                const uint16_t* zeros, int bits, int group, int aff, const float* bias, const float* r, int64_t ldr,
                float* y, int64_t ldy, int M, int N, int K, bool geglu) {
  const F32Weight W{w, q, scales, zeros, bits ? (K + group - 1) / group : 0, group};
  auto go = [&](auto qb, auto af) {
    constexpr int QB = decltype(qb)::value;
    constexpr bool AF = decltype(af)::value;
    if (geglu) launch_f32<true, QB, AF>(st, cus, x, ldx, W, bias, r, ldr, y, ldy, M, N, K);
    else launch_f32<false, QB, AF>(st, cus, x, ldx, W, bias, r, ldr, y, ldy, M, N, K);
  };
  using std::integral_constant;
  if (bits == 0) go(integral_constant<int, 0>{}, std::false_type{});
  else if (bits == 8 && !aff) go(integral_constant<int, 8>{}, std::false_type{});
  else if (bits == 8) go(integral_constant<int, 8>{}, std::true_type{});
  else if (!aff) go(integral_constant<int, 4>{}, std::false_type{});
  else go(integral_constant<int, 4>{}, std::true_type{});
}

// 16-byte loads of X and of f32 weights, 4-code loads of quantized ones that
// stay inside one group.
bool f32_linear_ok(uintptr_t x, int64_t ldx, uintptr_t w, int64_t K, int bits, int group) {
  return K > 0 && K % 4 == 0 && ldx % 4 == 0 && x % 16 == 0 && (bits == 0 ? w % 16 == 0 : (w % 4 == 0 && group % 4 == 0));
}

}  // namespace hb
