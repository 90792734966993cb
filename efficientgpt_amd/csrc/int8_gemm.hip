// Int8-weight GEMM for prefill (more than 16 activation rows) on gfx950 MFMA.
//
//   y[m, n] = bf16( fp32( bf16( sum_k x[m, k] * w[n, k] ) ) * scale[n] )
//
// The reference's prefill formula (research/realmodel/int8_linear.py:96-97): a bf16
// GEMM of x with the exact bf16 image of the int8 weights (fp32 accumulation,
// rounded once to bf16), then the per-row scale in fp32 and a second bf16
// rounding. The reference materialises w.to(bfloat16) and calls the library
// GEMM; here the weights are converted on the chip, so they cross HBM once, as int8.
//
// Design:
//   * Aligned shapes run v_mfma_f32_16x16x32_bf16 tiles with their operands loaded straight into LDS, the weights as int8:
//     128 x 128 to 256 x 256 for large products (int8_gemm_dma_kernel: eight wavefronts whose two halves take turns
//     at the matrix cores), 32 x 64 to 128 x 128 for the others (int8_gemm_ring_kernel: more and shorter blocks).
//     All of these sum an output in the same order, so its bits do not depend on the tile.
//   * int8 -> bf16 is exact: every value in [-127, 127] is a bf16.
//   * Rows past M or N read a valid row and are never stored.
//   * Split-K (short M, long K: too few output tiles to give every CU a block):
//     block (split, tile) sums its K slice and stores the fp32 tile to a caller's
//     workspace [splits][M][N]; a second kernel adds the slices in split order and
//     applies the two roundings. The fp32 sum is the same product in another
//     order, as any GEMM blocking is.
// Operand layouts of v_mfma_f32_16x16x32_bf16 (checked on the MI355X): lane l holds A[l % 16][8 (l / 16) + e]
// and B[8 (l / 16) + e][l % 16], e = 0..7; accumulator register r of lane l is C[4 (l / 16) + r][l % 16].
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace egpt {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kBK = 64;        // K must be a multiple of it
constexpr int kBKSplit = 128;  // K slices of a split are multiples of it

// 8 int8 (one LDS fragment) -> 8 bf16, exact.
__device__ __forceinline__ bf16x8 int8x8_to_bf16(const uint32_t w0, const uint32_t w1) {
  const uint32_t w[2] = {w0, w1};
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float f0 = (float)(int)(int8_t)(w[i] & 0xffu);
    const float f1 = (float)(int)(int8_t)((w[i] >> 8) & 0xffu);
    const float f2 = (float)(int)(int8_t)((w[i] >> 16) & 0xffu);
    const float f3 = (float)(int)(int8_t)(w[i] >> 24);
    // the upper halves of two floats in one v_perm_b32 (bytes 2, 3 of f0, then of f1)
    o[2 * i] = __builtin_amdgcn_perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
    o[2 * i + 1] = __builtin_amdgcn_perm(__float_as_uint(f3), __float_as_uint(f2), 0x07060302u);
  }
  return __builtin_bit_cast(bf16x8, u32x4{o[0], o[1], o[2], o[3]});
}

struct GemmArgs {
  const uint16_t* x;
  int64_t ldx;
  const int8_t* w;
  int64_t ldw;
  const float* scale;
  uint16_t* y;
  int64_t ldy;
  int M, N, K;
  int tiles_m, tiles_n;
  int splits, kchunk;  // K slices (1: no split) of kchunk columns each, the last one shorter
  float* part;         // splits > 1: fp32 partial tiles [splits][M][N]
  int inter;           // SwiGLU form: features (w holds inter gate rows, then inter up rows; N = 2 inter)
};

constexpr int kXcds = 8;        // MI355X: 8 XCDs, each with its own L2
constexpr int kGroupM = 8;      // M tiles per group of the tile order

// Block -> output tile. Blocks are dispatched round-robin to the XCDs (block b on
// XCD b % 8), so XCD x is given the contiguous range of tile numbers
// [start_x, start_x + count_x); within a range, tiles go in groups of kGroupM
// M-tiles sweeping N. The blocks that run together on one XCD then share their x
// and weight slices in that XCD's L2 instead of each streaming its own from HBM.
// Both steps are bijections of [0, tiles), so every tile is computed once whatever
// the dispatch order.
__device__ __forceinline__ void gemm_tile(int b, int tiles_m, int tiles_n, int& pid_m, int& pid_n) {
  const int tiles = tiles_m * tiles_n;
  const int base = tiles / kXcds, extra = tiles % kXcds;
  const int x = b % kXcds, j = b / kXcds;
  const int t = x * base + min(x, extra) + j;
  const int group = kGroupM * tiles_n;
  const int first_m = (t / group) * kGroupM;
  const int gm = min(tiles_m - first_m, kGroupM);
  pid_m = first_m + (t % group) % gm;
  pid_n = (t % group) / gm;
}

// The large tiles: 32 TM x 64 TN of y per block, eight wavefronts as 2 (M) x 4 (N) of 16 TM x 16 TN each.
//
// v_mfma_f32_16x16x32_bf16, not 32x32x16: over random operands in registers the chip sustains 1.90 PFLOP/s of the
// former and 1.37 of the latter (on zeros 2.45 and 1.65). The weights are the A operand, so an accumulator's four
// registers are four consecutive columns of one x row, and the weight rows of a wavefront's tiles are dealt so that
// lane l ends with the 4 TN consecutive columns from 4 TN (l / 16): each row is stored in 16-byte pieces.
//
// Operands go straight into LDS (global_load_lds_dwordx4), x rows as bf16 and weight rows as int8, through three
// stages of 64 K columns, the loads of step k + 2 issued as step k starts. Each 16-byte weight read feeds two MFMAs:
// the MFMA k index 8 h + e of half u stands for the step's column 16 h + 8 u + e in both operands.
//
// What bounded the kernel was each SIMD's two wavefronts reading LDS, converting and multiplying in the same phase
// (MFMA busy 51% of the time). Here they take turns: wavefronts 4-7 run one barrier behind 0-3, so that on every SIMD
// one wavefront reads and converts a whole step's fragments while the other, at raised issue priority, does nothing
// but the 2 TM TN MFMAs of its own. Conversions moved among the MFMAs instead cost 8% (256 x 256 tile), 32-column
// phases 1-2%. MFMA busy 68%, at a clock of 1.92 GHz: the chip's power is the next bound.
// Measured on the MI355X (us, the former 32x32x16 kernel with all wavefronts in one phase -> this): 8192 x 4096 ->
// 24576 1476-1491 -> 1203 (1.37 PFLOP/s), 8192 x 4096 -> 6144 374 -> 296, 6001 x 12288 -> 4096 608 -> 484, 1000 x
// 4096 -> 24576 233 -> 175 and -> 6144 72 -> 60, 300 x 2048 -> 12288 36.6 -> 28.3.
constexpr int kDmaBK = 64;
constexpr int kDmaWaves = 8;
constexpr int kDmaStages = 3;

// LDS positions of the 16-byte chunks: chunk c of x row r sits at c ^ dma_aswz(r), chunk c of weight row n (t = the
// row's group of 4 TN within its wavefront's 16 TN rows) at c ^ dma_bswz(t). A 16-byte LDS read serves 16 lanes
// together ({0-3, 12-15, 20-23, 24-27} or {4-7, 8-11, 16-19, 28-31} of a half wavefront, measured on the MI355X);
// with these both operands' fragment reads put them on distinct banks.
__device__ __forceinline__ int dma_aswz(int r) { return ((r >> 1) & 1) | (((r >> 3) & 1) << 2); }
__device__ __forceinline__ int dma_bswz(int t) { return ((t & 1) << 1) ^ (3 * ((t >> 1) & 1)); }

typedef uint32_t u32x2_h __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t u32_h __attribute__((aligned(2)));
typedef float f32x4_w __attribute__((ext_vector_type(4), aligned(4)));

// C consecutive outputs of row m from column c0, rounded to bf16: 16- and 8-byte stores at any element alignment, or one
// by one where the row ends among them.
template <int C>
__device__ __forceinline__ void store_row(const GemmArgs& a, int64_t m, int64_t c0, int64_t cols, const float (&o)[C]) {
  if (m >= a.M) return;
  uint16_t* p = a.y + m * a.ldy + c0;
  if (c0 + C <= cols) {
    uint32_t w[C / 2];
#pragma unroll
    for (int i = 0; i < C / 2; ++i) w[i] = pack2_bf16(o[2 * i], o[2 * i + 1]);
#pragma unroll
    for (int i = 0; i + 4 <= C / 2; i += 4)
      *(global_ptr<u32x4_h>)(p + 2 * i) = u32x4{w[i], w[i + 1], w[i + 2], w[i + 3]};
    if constexpr (C % 8 == 4) *(global_ptr<u32x2_h>)(p + C - 4) = u32x2{w[C / 2 - 2], w[C / 2 - 1]};
    if constexpr (C % 8 == 2) *(global_ptr<u32_h>)(p + C - 2) = w[C / 2 - 1];
  } else {
#pragma unroll
    for (int i = 0; i < C; ++i)
      if (c0 + i < cols) gstore(p + i, f32_to_bf16(o[i]));
  }
}

// The store of a wavefront's accumulators in the 16x16x32 layout: lane l holds, for rows m, m + 16, ..., the 4 TN
// consecutive columns from c0; y = bf16(bf16(acc) * scale), the reference's two roundings, or with SWIGLU the activation
// of the 2 TN features from c0 (their gate columns, then their up columns).
template <int TM, int TN, bool SWIGLU>
__device__ __forceinline__ void gemm_store_rows(const GemmArgs& a, const f32x4 (&acc)[TM][TN], int64_t m, int64_t c0) {
  if constexpr (SWIGLU) {
    float gs[2 * TN], us[2 * TN];
#pragma unroll
    for (int e = 0; e < 2 * TN; ++e) {
      const int64_t f = min(c0 + e, (int64_t)a.inter - 1);
      gs[e] = a.scale[f];
      us[e] = a.scale[a.inter + f];
    }
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
      float o[2 * TN];
#pragma unroll
      for (int e = 0; e < 2 * TN; ++e) {
        const int v = 2 * TN + e;
        const float g = bf16_to_f32(f32_to_bf16(bf16_to_f32(f32_to_bf16(acc[tm][e / 4][e % 4])) * gs[e]));
        const float u = bf16_to_f32(f32_to_bf16(bf16_to_f32(f32_to_bf16(acc[tm][v / 4][v % 4])) * us[e]));
        o[e] = bf16_to_f32(f32_to_bf16(g / (1.0f + expf(-g)))) * u;
      }
      store_row<2 * TN>(a, m + 16 * tm, c0, a.inter, o);
    }
  } else {
    float sc[4 * TN];
#pragma unroll
    for (int e = 0; e < 4 * TN; ++e) sc[e] = a.scale[min(c0 + e, (int64_t)a.N - 1)];
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
      float o[4 * TN];
#pragma unroll
      for (int e = 0; e < 4 * TN; ++e) o[e] = bf16_to_f32(f32_to_bf16(acc[tm][e / 4][e % 4])) * sc[e];
      store_row<4 * TN>(a, m + 16 * tm, c0, a.N, o);
    }
  }
}

template <int TM, int TN, bool SWIGLU>
__global__ __launch_bounds__(kDmaWaves * kWave, 1) void int8_gemm_dma_kernel(const GemmArgs a) {
  constexpr int WN = 4, BM = 32 * TM, BN = 64 * TN;
  constexpr int kARow = kDmaBK * 2, kBRow = kDmaBK;  // bytes per x row / weight row of a stage
  constexpr int kAStage = BM * kARow, kStage = kAStage + BN * kBRow;
  constexpr int kALoads = kAStage / (kDmaWaves * 1024);             // 1 KiB loads per wavefront and step
  constexpr int kBBlocks = BN * kBRow / 1024;                       // 1 KiB weight loads per step, over the block
  constexpr int kBLoads = (kBBlocks + kDmaWaves - 1) / kDmaWaves;   // per wavefront, the last one maybe not
  constexpr bool kBEven = kBBlocks % kDmaWaves == 0;
  static_assert(TM % 2 == 0 && (!SWIGLU || TN % 2 == 0), "");
  __shared__ __align__(16) char smem[kDmaStages * kStage];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm0 = (wave / WN) * (16 * TM);
  const int wn0 = (wave % WN) * (16 * TN);
  int pid_m, pid_n;
  gemm_tile((int)blockIdx.x, a.tiles_m, a.tiles_n, pid_m, pid_n);
  const int64_t m0 = (int64_t)pid_m * BM;
  const int64_t n0 = (int64_t)pid_n * BN;

  // 32-bit byte offsets from the operands' bases (the host checks that both span < 2 GiB); rows past M or N read the
  // last one.
  uint32_t xo[kALoads], wo[kBLoads];
#pragma unroll
  for (int q = 0; q < kALoads; ++q) {
    const int row = (wave * kALoads + q) * 8 + lane / 8;
    const int c = (lane % 8) ^ dma_aswz(row);
    xo[q] = (uint32_t)((min(m0 + row, (int64_t)a.M - 1) * a.ldx + 8 * c) * 2);
  }
  // Tile column j -> weight row. SwiGLU: each lane's 4 TN columns are 2 TN features' gate rows, then their up rows.
#pragma unroll
  for (int q = 0; q < kBLoads; ++q) {
    const int row = (q * kDmaWaves + wave) * 16 + lane / 4;
    const int c = (lane % 4) ^ dma_bswz((row / (4 * TN)) % 4);
    int64_t wrow;
    if constexpr (SWIGLU) {
      const int o = row % (4 * TN);
      const int64_t f = min((int64_t)pid_n * (BN / 2) + row / (4 * TN) * (2 * TN) + o % (2 * TN), (int64_t)a.inter - 1);
      wrow = o < 2 * TN ? f : a.inter + f;
    } else {
      wrow = min(n0 + row, (int64_t)a.N - 1);
    }
    wo[q] = (uint32_t)(wrow * a.ldw + 16 * c);
  }
  const uint32_t sbase = lds_addr(smem);
  auto issue = [&](int kt, int stage) {
    const uint32_t abase = sbase + (uint32_t)(stage * kStage);
    const char* xb = (const char*)a.x + (int64_t)kt * kARow;
    const char* wb = (const char*)a.w + (int64_t)kt * kBRow;
#pragma unroll
    for (int q = 0; q < kALoads; ++q) lds_load16_at(abase + (uint32_t)((wave * kALoads + q) * 1024), xb, xo[q]);
#pragma unroll
    for (int q = 0; q < kBLoads; ++q)
      if (kBEven || q * kDmaWaves + wave < kBBlocks)
        lds_load16_at(abase + (uint32_t)(kAStage + (q * kDmaWaves + wave) * 1024), wb, wo[q]);
  };
  // Wait until at most the loads of S steps are in flight.
  auto wait_steps = [&](auto S) {
    if (kBEven || wave < kBBlocks % kDmaWaves)
      EGPT_WAIT_VMCNT(decltype(S)::value * (kALoads + kBLoads));
    else
      EGPT_WAIT_VMCNT(decltype(S)::value * (kALoads + kBLoads - 1));
  };
  using One = std::integral_constant<int, 1>;

  const int r16 = lane % 16, h = lane / 16;
  // Weight row of tile tn's slot i: 4 TN (i / 4) + 4 tn + i % 4, so that lane l's accumulators hold, for x row l % 16
  // of tile tm, the 4 TN consecutive columns from 4 TN (l / 16).
  const int aoff[2] = {(wm0 + r16) * kARow + 16 * ((2 * h) ^ dma_aswz(r16)),
                       (wm0 + r16) * kARow + 16 * ((2 * h + 1) ^ dma_aswz(r16))};
  const int boff = kAStage + (wn0 + 4 * TN * (r16 / 4) + r16 % 4) * kBRow + 16 * (h ^ dma_bswz(r16 / 4));

  f32x4 acc[TM][TN];
#pragma unroll
  for (int tm = 0; tm < TM; ++tm)
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) acc[tm][tn] = f32x4{};

  bf16x8 af[2][TM], bf[2][TN];
  auto load_fragments = [&](const char* sm) {
    u32x4 raw[TN];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) raw[tn] = *(const u32x4*)(sm + boff + tn * 4 * kBRow);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) af[u][tm] = *(const bf16x8*)(sm + aoff[u] + tm * 16 * kARow);
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      bf[0][tn] = int8x8_to_bf16(raw[tn].x, raw[tn].y);
      bf[1][tn] = int8x8_to_bf16(raw[tn].z, raw[tn].w);
    }
  };
  auto mma = [&]() {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int u = 1; u >= 0; --u)
#pragma unroll
      for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
          acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[u][tn], af[u][tm], acc[tm][tn], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
  };
  auto phase_end = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  const int nk = a.K / kDmaBK;
  const bool second = wave >= kDmaWaves / 2;
  issue(0, 0);
  if (nk > 1) {
    issue(1, 1);
    wait_steps(One{});
  } else {
    EGPT_WAIT_VMCNT(0);
  }
  lds_barrier();
  if (second) lds_barrier();
  int stage = 0;
  for (int kt = 0; kt < nk; ++kt) {
    const char* sm = smem + stage * kStage;
    auto wait_next = [&]() {
      if (kt + 2 < nk)
        wait_steps(One{});
      else
        EGPT_WAIT_VMCNT(0);
    };
    if (kt + 2 < nk) issue(kt + 2, stage == 0 ? 2 : stage - 1);
    load_fragments(sm);
    if (second) wait_next();
    phase_end();
    mma();
    if (!second) wait_next();
    phase_end();
    stage = stage == kDmaStages - 1 ? 0 : stage + 1;
  }
  if (!second) lds_barrier();

  gemm_store_rows<TM, TN, SWIGLU>(a, acc, m0 + wm0 + r16, (int64_t)pid_n * (SWIGLU ? BN / 2 : BN) +
                                  (wave % WN) * (SWIGLU ? 8 * TN : 16 * TN) + (SWIGLU ? 2 : 4) * TN * h);
}

// The small tiles: BM x BN of y per block (16 TM x 16 TN per wavefront, WM x WN wavefronts), for products with too few
// large tiles to fill the chip. Operands go straight into LDS as in int8_gemm_dma_kernel, 128 K columns a step through a
// ring of STAGES; a wavefront reads a step's fragments into registers while it multiplies the step before, one barrier a
// step. Each output is summed in the order of the large tiles (two MFMAs per 64 columns, the second half's first).
//
// What bounds it is LDS: at 300 x 12288 -> 4096 (96 x 64 tiles, one round of 256 blocks, 96 steps) the loads alone take
// 43 us, the reads, conversions and MFMAs alone 29, together 64; the loads' distance (2 to 4 steps) and row slices of
// 256 columns made no difference. Each x row is read from LDS by WN wavefronts and each weight row by WM, so eight
// wavefronts as 2 x 4 did better than 4 x 2 (6-8%) or four (8-15%, too few to hide a barrier). It replaced 64 x 64 and
// 128 x 64 tiles staged through registers, on the MI355X with the weights out of cache (us): 20 x 4096 -> 24576 SwiGLU
// 36 -> 26, 77 x 2048 -> 12288 SwiGLU 20.4 -> 14.2, 200 x 4096 -> 6144 31.6 -> 26.7, 300 x 12288 -> 4096 97 -> 64, 300 x
// 4096 -> 6144 42.5 -> 30, 600 x 2048 -> 2048 18.8 -> 13.1, 600 x 6144 -> 2048 51 -> 32.5; split slices 20 x 12288 ->
// 4096 18.5 -> 16.5. As 128 x 128 it also replaces int8_gemm_dma_kernel's where the blocks are one round: 1000 x 12288 ->
// 4096 126 -> 111 us, 2048 x 6144 -> 2048 66 -> 58, 512 x 2048 -> 6144 24.4 -> 21.6 (a block is all a CU holds; that
// kernel's fits twice and stays for two rounds).
constexpr int kRingBK = 128;

// LDS positions of a stage's 16-byte chunks: chunk c of x row r (16 a row) sits at c ^ (r & 15), chunk c of the weight
// row that is slot i of its MFMA operand (8 a row) at c ^ (i >> 1): the 16 lanes that a 16-byte LDS read serves together
// (see dma_bswz) fall on distinct banks.
template <int TN>
__device__ __forceinline__ int ring_slot(int row) { return (row / (4 * TN)) % 4 * 4 + row % 4; }

template <int BM, int BN, int WM, int WN, int STAGES, bool SPLIT, bool SWIGLU>
__global__ __launch_bounds__(WM * WN * kWave) void int8_gemm_ring_kernel(const GemmArgs a) {
  constexpr int NW = WM * WN, TM = BM / (16 * WM), TN = BN / (16 * WN);
  constexpr int kARow = kRingBK * 2, kBRow = kRingBK;  // bytes per x row / weight row of a stage
  constexpr int kAStage = BM * kARow, kStage = kAStage + BN * kBRow;
  constexpr int kALoads = kAStage / (NW * 1024), kBLoads = BN * kBRow / (NW * 1024);  // 1 KiB loads per wavefront
  constexpr int kLoads = kALoads + kBLoads;
  static_assert(kALoads * NW * 1024 == kAStage && kBLoads * NW * 1024 == BN * kBRow && TM >= 1 && TN >= 1, "");
  static_assert(!(SPLIT && SWIGLU) && STAGES >= 2 && (STAGES - 1) * kLoads < 64, "");
  __shared__ __align__(16) char smem[STAGES * kStage];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm0 = (wave / WN) * (16 * TM);
  const int wn0 = (wave % WN) * (16 * TN);
  const int tiles = a.tiles_m * a.tiles_n;
  const int split = SPLIT ? (int)blockIdx.x / tiles : 0;
  int pid_m, pid_n;
  gemm_tile((int)blockIdx.x - split * tiles, a.tiles_m, a.tiles_n, pid_m, pid_n);
  const int64_t m0 = (int64_t)pid_m * BM;
  const int64_t n0 = (int64_t)pid_n * BN;
  const int kbeg = SPLIT ? split * a.kchunk : 0;
  const int klen = SPLIT ? min(a.kchunk, a.K - kbeg) : a.K;  // a multiple of 64
  const int nk = (klen + kRingBK - 1) / kRingBK;

  // 32-bit byte offsets from the operands' bases (the host checks that both span < 2 GiB); rows past M or N read the
  // last one, columns past the slice (a last step of 64) its last 16 bytes.
  constexpr int kAC = kRingBK / 8, kBC = kRingBK / 16;  // chunks per row
  uint32_t xr[kALoads], xc[kALoads], wr[kBLoads], wc[kBLoads];  // row offset, column offset in a step
#pragma unroll
  for (int q = 0; q < kALoads; ++q) {
    const int row = (wave * kALoads + q) * (64 / kAC) + lane / kAC;
    xc[q] = 16 * ((lane % kAC) ^ (row & 15));
    xr[q] = (uint32_t)((min(m0 + row, (int64_t)a.M - 1) * a.ldx + kbeg) * 2);
  }
#pragma unroll
  for (int q = 0; q < kBLoads; ++q) {
    const int row = (wave * kBLoads + q) * (64 / kBC) + lane / kBC;
    wc[q] = 16 * ((lane % kBC) ^ (ring_slot<TN>(row) >> 1));
    int64_t wrow;
    if constexpr (SWIGLU) {  // each lane's 4 TN columns are 2 TN features' gate rows, then their up rows
      const int o = row % (4 * TN);
      const int64_t f = min((int64_t)pid_n * (BN / 2) + row / (4 * TN) * (2 * TN) + o % (2 * TN), (int64_t)a.inter - 1);
      wrow = o < 2 * TN ? f : a.inter + f;
    } else {
      wrow = min(n0 + row, (int64_t)a.N - 1);
    }
    wr[q] = (uint32_t)(wrow * a.ldw + kbeg);
  }
  const uint32_t sbase = lds_addr(smem);
  const uint32_t xlim = (uint32_t)(2 * klen - 16), wlim = (uint32_t)(klen - 16);
  auto issue = [&](int kt, int stage) {
    const uint32_t abase = sbase + (uint32_t)(stage * kStage);
#pragma unroll
    for (int q = 0; q < kBLoads; ++q)
      lds_load16_at(abase + (uint32_t)(kAStage + (wave * kBLoads + q) * 1024), a.w,
                    wr[q] + min(wc[q] + (uint32_t)(kt * kBRow), wlim));
#pragma unroll
    for (int q = 0; q < kALoads; ++q)
      lds_load16_at(abase + (uint32_t)((wave * kALoads + q) * 1024), a.x,
                    xr[q] + min(xc[q] + (uint32_t)(kt * kARow), xlim));
  };

  const int r16 = lane % 16, h = lane / 16;
  const int arow = (wm0 + r16) * kARow;
  const int brow = kAStage + (wn0 + 4 * TN * (r16 / 4) + r16 % 4) * kBRow;
  f32x4 acc[TM][TN];
#pragma unroll
  for (int tm = 0; tm < TM; ++tm)
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) acc[tm][tn] = f32x4{};
  struct Frags {
    u32x4 w[kRingBK / 64][TN];
    bf16x8 x[kRingBK / 64][2][TM];
  };
  auto read = [&](Frags& f, const char* sm) {
#pragma unroll
    for (int s = 0; s < kRingBK / 64; ++s) {
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
        f.w[s][tn] = *(const u32x4*)(sm + brow + tn * 4 * kBRow + 16 * ((4 * s + h) ^ (r16 >> 1)));
#pragma unroll
      for (int u = 1; u >= 0; --u)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
          f.x[s][u][tm] = *(const bf16x8*)(sm + arow + tm * 16 * kARow + 16 * ((8 * s + 2 * h + u) ^ r16));
    }
  };
  auto mma = [&](const Frags& f, int s) {  // 64 columns
    bf16x8 w[2][TN];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      w[1][tn] = int8x8_to_bf16(f.w[s][tn].z, f.w[s][tn].w);
      w[0][tn] = int8x8_to_bf16(f.w[s][tn].x, f.w[s][tn].y);
    }
#pragma unroll
    for (int u = 1; u >= 0; --u)
#pragma unroll
      for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
          acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][tn], f.x[s][u][tm], acc[tm][tn], 0, 0, 0);
  };
  // Wait until no more than the loads of `later` steps are in flight, then publish what has arrived.
  auto arrive = [&](int later) {
    if (later >= STAGES - 1)
      EGPT_WAIT_VMCNT((STAGES - 1) * kLoads);
    else if (later == STAGES - 2)
      EGPT_WAIT_VMCNT((STAGES - 2) * kLoads);
    else if (STAGES > 3 && later == STAGES - 3)
      EGPT_WAIT_VMCNT((STAGES > 3 ? STAGES - 3 : 0) * kLoads);
    else
      EGPT_WAIT_VMCNT(0);
    lds_barrier();
  };
  // Step kt: the fragments of step kt + 1 are read while those of step kt, in registers, are multiplied. The barrier
  // publishes stage kt + 1 and tells that every wavefront has read stage kt, whose buffer takes step kt + STAGES.
  int stage = 0;
  auto step = [&](int kt, const Frags& cur, Frags& next) {
    const int ahead = stage == STAGES - 1 ? 0 : stage + 1;
    if (kt + 1 < nk) {
      arrive(min(STAGES - 2, nk - 2 - kt));
      read(next, smem + ahead * kStage);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (kt + STAGES < nk) issue(kt + STAGES, stage);
    __builtin_amdgcn_sched_barrier(0);
    mma(cur, 0);
    if (kt * kRingBK + 64 < klen) mma(cur, 1);
    __builtin_amdgcn_sched_barrier(0);
    stage = ahead;
  };

#pragma unroll
  for (int s = 0; s < STAGES; ++s)
    if (s < nk) issue(s, s);
  Frags f0, f1;
  arrive(min(STAGES - 1, nk - 1));
  read(f0, smem);
  for (int kt = 0; kt < nk; kt += 2) {
    step(kt, f0, f1);
    if (kt + 1 < nk) step(kt + 1, f1, f0);
  }

  if constexpr (SPLIT) {  // the fp32 tile of this K slice; the reduce kernel rounds
    float* part = a.part + (int64_t)split * a.M * a.N;
    const int64_t c0 = n0 + wn0 + 4 * TN * h;
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
      const int64_t m = m0 + wm0 + 16 * tm + r16;
      if (m >= a.M) continue;
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) {
        float* p = part + m * a.N + c0 + 4 * tn;
        if (c0 + 4 * tn + 4 <= a.N) {
          *(global_ptr<f32x4_w>)p = acc[tm][tn];
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (c0 + 4 * tn + r < a.N) gstore(p + r, (float)acc[tm][tn][r]);
        }
      }
    }
  } else {
    gemm_store_rows<TM, TN, SWIGLU>(a, acc, m0 + wm0 + r16, (int64_t)pid_n * (SWIGLU ? BN / 2 : BN) +
                                    (wave % WN) * (SWIGLU ? 8 * TN : 16 * TN) + (SWIGLU ? 2 : 4) * TN * h);
  }
}

// Split-K reduce: y[m, n] = bf16(bf16(sum_s part[s][m][n]) * scale[n]), splits added in order. The split
// count is a template argument so that every slice's load is issued before the first addition.
constexpr int kReduceThreads = 256;

template <int S>
__global__ __launch_bounds__(kReduceThreads) void int8_gemm_reduce_kernel(const float* __restrict__ part,
                                                                          const float* __restrict__ scale,
                                                                          uint16_t* __restrict__ y, int64_t ldy, int M,
                                                                          int N) {
  const int64_t mn = (int64_t)M * N;
  for (int64_t i = (int64_t)blockIdx.x * kReduceThreads + threadIdx.x; i < mn;
       i += (int64_t)gridDim.x * kReduceThreads) {
    float v[S];
#pragma unroll
    for (int sp = 0; sp < S; ++sp) v[sp] = part[sp * mn + i];
    float acc = v[0];
#pragma unroll
    for (int sp = 1; sp < S; ++sp) acc += v[sp];
    const int64_t m = i / N, n = i - m * N;
    y[m * ldy + n] = f32_to_bf16(bf16_to_f32(f32_to_bf16(acc)) * scale[n]);
  }
}

constexpr int kMaxSplits = 16;

// The reduce for a.splits (2 ... S) slices; false for a count outside that range.
template <int S>
bool launch_reduce(const GemmArgs& a, unsigned blocks, hipStream_t st) {
  if constexpr (S < 2) {
    return false;
  } else {
    if (a.splits != S) return launch_reduce<S - 1>(a, blocks, st);
    hipLaunchKernelGGL(int8_gemm_reduce_kernel<S>, dim3(blocks), dim3(kReduceThreads), 0, st, a.part, a.scale, a.y,
                       a.ldy, a.M, a.N);
    return true;
  }
}

template <int BM, int BN, int WM, int WN, int STAGES, bool SPLIT, bool SWIGLU>
int launch_ring(GemmArgs a, hipStream_t st) {
  a.tiles_m = (int)(((int64_t)a.M + BM - 1) / BM);
  a.tiles_n = SWIGLU ? (int)(((int64_t)a.inter + BN / 2 - 1) / (BN / 2)) : (int)(((int64_t)a.N + BN - 1) / BN);
  const unsigned blocks = (unsigned)a.tiles_m * (unsigned)a.tiles_n * (unsigned)(SPLIT ? a.splits : 1);
  hipLaunchKernelGGL((int8_gemm_ring_kernel<BM, BN, WM, WN, STAGES, SPLIT, SWIGLU>), dim3(blocks),
                     dim3(WM * WN * kWave), 0, st, a);
  return EGPT_LAUNCH_STATUS();
}

// The split slices' fp32 tiles into a.part (a.splits > 1); no reduce. Tiles of 32 rows for up to 32 rows and where the
// 64-row ones are more than one round of 256 blocks (three of the smaller fit on a CU): 64 x 2048 -> 6144 (384 blocks) 12.7
// -> 12.0 us, 192 x 2048 -> 2048 9.5 -> 8.9, 128 x 2048 -> 6144 16.1 -> 15.6; at 256 blocks 64 x 4096 -> 4096 12.0 ->
// 12.2; 33 x 4096 -> 6144 14.2 -> 14.8.
int launch_split_partials(const GemmArgs& a, hipStream_t st) {
  const int64_t blocks = ((int64_t)a.M + 63) / 64 * (((int64_t)a.N + 63) / 64) * a.splits;
  const int last = (a.M - 1) % 64 + 1;  // rows of the last 64; a second 32 of a few rows is not worth its blocks
  if (a.M <= 32 || (blocks > 256 && (last <= 32 || last >= 40))) return launch_ring<32, 64, 1, 4, 3, true, false>(a, st);
  return launch_ring<64, 64, 2, 4, 3, true, false>(a, st);
}

int launch_split(const GemmArgs& a, hipStream_t st) {
  if (launch_split_partials(a, st) != EGPT_OK) return EGPT_ERR_LAUNCH;
  const int64_t mn = (int64_t)a.M * a.N;
  const unsigned blocks = (unsigned)std::min<int64_t>((mn + kReduceThreads - 1) / kReduceThreads, 4096);
  if (!launch_reduce<kMaxSplits>(a, blocks, st)) return EGPT_ERR_INVALID;
  return EGPT_LAUNCH_STATUS();
}

// The LDS-direct large tiles; with SWIGLU each block covers 32 TN features.
template <int TM, int TN, bool SWIGLU>
int launch_dma(GemmArgs a, hipStream_t st) {
  constexpr int BM = 32 * TM, BN = 64 * TN;
  a.tiles_m = (int)(((int64_t)a.M + BM - 1) / BM);
  a.tiles_n = SWIGLU ? (int)(((int64_t)a.inter + BN / 2 - 1) / (BN / 2)) : (int)(((int64_t)a.N + BN - 1) / BN);
  hipLaunchKernelGGL((int8_gemm_dma_kernel<TM, TN, SWIGLU>), dim3((unsigned)a.tiles_m * (unsigned)a.tiles_n),
                     dim3(kDmaWaves * kWave), 0, st, a);
  return EGPT_LAUNCH_STATUS();
}

// Which tile: the least time of the launch's rounds of 256 blocks (one per CU; where two blocks fit on a CU, a pair of
// them takes less than two rounds). The costs are the us of one full round over K = 4096, launch excluded, measured on
// the MI355X (the 128 x 128 ring tile's from its ratio to the other kernel's, 0.89-0.91 over K 2048 to 12288); their
// ratios hold for other K.
struct GemmTile {
  int bm, bn;
  float round;  // 256 blocks
  float pair;   // 512 blocks, where two fit on a CU
  bool ring;    // int8_gemm_ring_kernel, else int8_gemm_dma_kernel
  bool swiglu;  // has the SwiGLU form
  int (*launch)(GemmArgs, hipStream_t);
  int (*launch_swiglu)(GemmArgs, hipStream_t);
};
template <int TM, int TN>
constexpr GemmTile dma_tile(float round, float pair = 0.f) {
  if constexpr (TN % 2 == 0)
    return {32 * TM, 64 * TN, round, pair, false, true, launch_dma<TM, TN, false>, launch_dma<TM, TN, true>};
  else
    return {32 * TM, 64 * TN, round, pair, false, false, launch_dma<TM, TN, false>, nullptr};
}
template <int BM, int BN, int WM, int WN, int STAGES>
constexpr GemmTile ring_tile(float round, float pair = 0.f) {
  return {BM, BN, round, pair, true, true, launch_ring<BM, BN, WM, WN, STAGES, false, false>,
          launch_ring<BM, BN, WM, WN, STAGES, false, true>};
}
constexpr GemmTile kGemmTiles[] = {
    dma_tile<8, 4>(95.0f), dma_tile<6, 4>(79.5f), dma_tile<8, 3>(79.5f), dma_tile<6, 3>(65.3f), dma_tile<4, 4>(61.7f),
    dma_tile<8, 2>(59.5f), dma_tile<4, 3>(53.8f), dma_tile<6, 2>(50.0f), dma_tile<4, 2>(39.7f, 64.0f),
    ring_tile<128, 128, 2, 4, 3>(36.0f), ring_tile<64, 128, 2, 4, 4>(26.5f), ring_tile<128, 64, 2, 4, 3>(23.6f),
    ring_tile<96, 64, 2, 4, 3>(21.3f), ring_tile<64, 64, 2, 4, 3>(17.3f, 27.0f),
    ring_tile<32, 64, 1, 4, 3>(14.0f, 24.0f)};

float tile_cost(const GemmTile& t, int64_t M, int64_t N) {
  const int64_t tiles = ((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
  if (t.pair == 0.f) return t.round * (float)((tiles + 255) / 256);
  const int64_t rest = tiles % 512;
  return t.pair * (float)(tiles / 512) + (rest == 0 ? 0.f : rest <= 256 ? t.round : t.pair);
}

// N counts a SwiGLU product's gate and up columns.
const GemmTile& best_tile(int64_t M, int64_t N, bool swiglu) {
  const GemmTile* best = nullptr;
  for (const GemmTile& t : kGemmTiles)
    if ((t.swiglu || !swiglu) && (!best || tile_cost(t, M, N) < tile_cost(*best, M, N))) best = &t;
  return *best;
}

int launch_best_tile(const GemmArgs& a, bool swiglu, hipStream_t st) {
  const GemmTile& t = best_tile(a.M, a.N, swiglu);
  return swiglu ? t.launch_swiglu(a, st) : t.launch(a, st);
}

// Any K, alignment and size: 64 x 64 of y per block, four wavefronts as 2 x 2. The tiles above need 16-byte aligned rows
// for their loads into LDS and K in whole steps; here both operands go through registers with loads of any alignment,
// BK (64 or 128) K columns a step and two steps ahead, and into LDS as bf16 (rows padded by 16 bytes against bank
// conflicts). Rows past M or N read the last one. Against the vector kernel below, us: 300 x 4001 -> 4096 1749 -> 47, 500 x
// 7001 -> 8000 19055 -> 146, 40 x 7001 -> 8000 955 -> 64.
constexpr int64_t rag_column(int kt, int BK) { return (int64_t)kt * BK; }  // a step's first, for any int K
static_assert(rag_column(INT32_MAX / 64 + 2, 64) > INT32_MAX, "");

template <int BK>
__global__ __launch_bounds__(256) void int8_gemm_ragged_kernel(const GemmArgs a) {
  constexpr int TM = 2, TN = 2, BM = 64, BN = 64;
  constexpr int kRow = BK + 8;                            // bf16 elements per row in LDS
  constexpr int kXT = BK / 8, kWT = BK / 16;              // threads per x row, per weight row
  constexpr int kXL = BM * kXT / 256, kWL = BN * kWT / 256;  // 16-byte loads per thread and step
  __shared__ __align__(16) uint16_t As[2][BM * kRow];
  __shared__ __align__(16) uint16_t Bs[2][BN * kRow];
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  const int wm0 = (wave / 2) * 32, wn0 = (wave % 2) * 32;
  int pid_m, pid_n;
  gemm_tile((int)blockIdx.x, a.tiles_m, a.tiles_n, pid_m, pid_n);
  const int64_t m0 = (int64_t)pid_m * BM, n0 = (int64_t)pid_n * BN;

  // this thread's chunks of a step: 8 columns of x rows tid / kXT + j 256 / kXT, 16 columns of weight rows likewise
  const int xc = 8 * (tid % kXT), wc = 16 * (tid % kWT);
  const uint16_t* xp[kXL];
  const int8_t* wp[kWL];
#pragma unroll
  for (int j = 0; j < kXL; ++j)
    xp[j] = a.x + min(m0 + 256 / kXT * j + tid / kXT, (int64_t)a.M - 1) * a.ldx + xc;
#pragma unroll
  for (int j = 0; j < kWL; ++j) wp[j] = a.w + min(n0 + 256 / kWT * j + tid / kWT, (int64_t)a.N - 1) * a.ldw + wc;
  const int nk = a.K / BK;  // whole steps
  struct Regs {
    u32x4 x[kXL], w[kWL];
  };
  auto load = [&](Regs& r, int64_t k0) {
#pragma unroll
    for (int j = 0; j < kXL; ++j) r.x[j] = ld16_any(xp[j] + k0);
#pragma unroll
    for (int j = 0; j < kWL; ++j) r.w[j] = ld16_any(wp[j] + k0);
  };
  auto store = [&](const Regs& r, int buf) {
#pragma unroll
    for (int j = 0; j < kXL; ++j) *(u32x4*)&As[buf][(256 / kXT * j + tid / kXT) * kRow + xc] = r.x[j];
#pragma unroll
    for (int j = 0; j < kWL; ++j) {
      bf16x8* b = (bf16x8*)&Bs[buf][(256 / kWT * j + tid / kWT) * kRow + wc];
      b[0] = int8x8_to_bf16(r.w[j].x, r.w[j].y);
      b[1] = int8x8_to_bf16(r.w[j].z, r.w[j].w);
    }
  };

  const int r16 = lane % 16, h = lane / 16;
  const int arow = (wm0 + r16) * kRow + 8 * h;
  const int brow = (wn0 + 4 * TN * (r16 / 4) + r16 % 4) * kRow + 8 * h;
  f32x4 acc[TM][TN];
#pragma unroll
  for (int tm = 0; tm < TM; ++tm)
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) acc[tm][tn] = f32x4{};
  auto mma = [&](int buf) {
#pragma unroll
    for (int k2 = 0; k2 < BK / 64; ++k2) {
      bf16x8 xf[2][TM], wf[2][TN];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
          xf[ks][tm] = *(const bf16x8*)&As[buf][arow + tm * 16 * kRow + 64 * k2 + 32 * ks];
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
          wf[ks][tn] = *(const bf16x8*)&Bs[buf][brow + tn * 4 * kRow + 64 * k2 + 32 * ks];
      }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
          for (int tn = 0; tn < TN; ++tn)
            acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[ks][tn], xf[ks][tm], acc[tm][tn], 0, 0, 0);
    }
  };
  // Step kt from LDS buffer and register set kt % 2: its loads' successors go out first, then its MFMAs, then the next
  // step's data into the other buffer.
  Regs r0, r1;
  auto step = [&](int kt, int cur, Regs& mine, const Regs& next) {
    if (kt + 2 < nk) load(mine, rag_column(kt + 2, BK));
    __builtin_amdgcn_sched_barrier(0);
    mma(cur);
    if (kt + 1 < nk) store(next, 1 - cur);
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
  };
  if (nk > 0) {
    load(r0, 0);
    if (nk > 1) load(r1, BK);
    store(r0, 0);
    lds_barrier();
    for (int kt = 0; kt < nk; kt += 2) {
      step(kt, 0, r0, r1);
      if (kt + 1 < nk) step(kt + 1, 1, r1, r0);
    }
  }
  const int left = a.K % BK;
  if (left) {  // the columns past the last whole step
    Regs r;
    if (nk > 0) {
      // the BK columns before K, with zeros for the activations already added
      load(r, (int64_t)a.K - BK);
      u32x4 mask;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        mask[i] = (xc + 2 * i >= BK - left ? 0xffffu : 0u) | (xc + 2 * i + 1 >= BK - left ? 0xffff0000u : 0u);
#pragma unroll
      for (int j = 0; j < kXL; ++j) r.x[j] &= mask;
    } else {  // a row shorter than a step: element by element, zeros after it
#pragma unroll
      for (int j = 0; j < kXL; ++j) {
        uint32_t d[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (xc + e < left) d[e / 2] |= (uint32_t)gload(xp[j] + e) << (16 * (e % 2));
        r.x[j] = u32x4{d[0], d[1], d[2], d[3]};
      }
#pragma unroll
      for (int j = 0; j < kWL; ++j) {
        uint32_t d[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (wc + e < left) d[e / 4] |= (uint32_t)(uint8_t)gload(wp[j] + e) << (8 * (e % 4));
        r.w[j] = u32x4{d[0], d[1], d[2], d[3]};
      }
    }
    store(r, 0);
    lds_barrier();
    mma(0);
  }
  gemm_store_rows<TM, TN, false>(a, acc, m0 + wm0 + r16, n0 + wn0 + 4 * TN * h);
}

// The same for short rows and small outputs: one wavefront per feature n and group of kVectorRows rows, lanes striding K
// one element at a time, fp32 sums reduced across the wavefront in a fixed order.
constexpr int kVectorRows = 4;
constexpr int kVectorWaves = 4;

__global__ __launch_bounds__(kVectorWaves * kWave) void int8_gemm_vector_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, const int8_t* __restrict__ w, int64_t ldw,
    const float* __restrict__ scale, uint16_t* __restrict__ y, int64_t ldy, int M, int N, int K) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t mgroups = ((int64_t)M + kVectorRows - 1) / kVectorRows;
  const int64_t wv = (int64_t)blockIdx.x * kVectorWaves + threadIdx.x / kWave;
  if (wv >= mgroups * N) return;   // wave-uniform
  const int64_t n = wv / mgroups;  // neighbouring wavefronts share a weight row
  const int64_t m0 = (wv - n * mgroups) * kVectorRows;
  const int8_t* wr = w + n * ldw;
  float acc[kVectorRows] = {};
  for (int64_t k = lane; k < K; k += kWave) {
    const float wk = (float)gload(wr + k);
#pragma unroll
    for (int r = 0; r < kVectorRows; ++r)
      if (m0 + r < M) acc[r] = fmaf(bf16_to_f32(gload(x + (m0 + r) * ldx + k)), wk, acc[r]);
  }
#pragma unroll
  for (int r = 0; r < kVectorRows; ++r) {
    const float sum = wave_sum(acc[r]);
    if (lane == r && m0 + r < M) gstore(y + (m0 + r) * ldy + n, f32_to_bf16(bf16_to_f32(f32_to_bf16(sum)) * scale[n]));
  }
}

// Outputs up to which the vector kernel is the faster one. Measured on the MI355X, us, vector / tiles: K below one step,
// which the tiles load element by element, 64 x 20 -> 300 4.5 / 5.6, 128 x 20 -> 300 5.8 / 5.7; short rows, 32 x 257 -> 64
// 5.2 / 5.7, 128 x 257 -> 128 5.9 / 5.8; 64 x 520 -> 64 7.2 / 6.4.
constexpr int64_t vector_outputs(int K) { return K < 64 ? 32768 : K < 512 ? 10240 : 0; }

// Steps of 128 columns where the tiles are at most two a CU (70 KiB of LDS each) and a row is several steps long: 17 x
// 8191 -> 1000 70 -> 57 us, 200 x 8191 -> 8192 96 -> 91; 17 x 520 -> 300 6.5 -> 6.8; 1024 tiles, 512 x 8191 -> 8192, 5% slower.
constexpr int64_t kRagWideTiles = 512;
constexpr int kRagWideK = 768;

int launch_ragged(GemmArgs a, hipStream_t st) {
  if ((int64_t)a.M * a.N <= vector_outputs(a.K)) {
    const int64_t waves = ((int64_t)a.M + kVectorRows - 1) / kVectorRows * a.N;
    hipLaunchKernelGGL(int8_gemm_vector_kernel, dim3((unsigned)((waves + kVectorWaves - 1) / kVectorWaves)),
                       dim3(kVectorWaves * kWave), 0, st, a.x, a.ldx, a.w, a.ldw, a.scale, a.y, a.ldy, a.M, a.N, a.K);
    return EGPT_LAUNCH_STATUS();
  }
  const int64_t tm = ((int64_t)a.M + 63) / 64, tn = ((int64_t)a.N + 63) / 64;
  if (tm * tn > (int64_t)INT32_MAX) return EGPT_ERR_UNSUPPORTED;
  a.tiles_m = (int)tm;
  a.tiles_n = (int)tn;
  if (tm * tn <= kRagWideTiles && a.K >= kRagWideK)
    hipLaunchKernelGGL(int8_gemm_ragged_kernel<128>, dim3((unsigned)(tm * tn)), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL(int8_gemm_ragged_kernel<64>, dim3((unsigned)(tm * tn)), dim3(256), 0, st, a);
  return EGPT_LAUNCH_STATUS();
}

// K slices for a short-M GEMM (at most 256 rows) whose 64 x 64 tiles leave CUs
// idle: the fewest (a power of two, at most 16) that give every CU a block, each
// slice a multiple of kBKSplit and at least 256 wide. 1 when the tiles already fill
// the chip, or K is short or not a multiple of kBKSplit. The rule was chosen on tiles
// that are gone; with the present ones, us, split (slices and reduce) / one pass: where
// K is long it gains, 128 x 12288 -> 4096 31.0 / 41.3, 128 x 6144 -> 2048 12.4 / 21.8,
// 64 x 2048 -> 2048 6.7 / 8.9; where two slices do, 32 x 64 tiles would fill the chip
// in one pass and it loses, 128 x 2048 -> 4096 11.3 / 9.1, 64 x 2048 -> 12288 16.2 /
// 12.8, 200 x 2048 -> 2048 9.6 / 9.0.
constexpr int kMinSliceSteps = 4;
constexpr int kSplitTargetBlocks = 256;

void gemm_split(int64_t M, int64_t N, int64_t K, int& splits, int& kchunk) {
  const int64_t tiles = ((M + 63) / 64) * ((N + 63) / 64);
  splits = 1;
  kchunk = (int)K;
  if (M > 256 || K % kBKSplit) return;  // taller blocks take the larger tiles below
  // Past 128 rows only grids that fill at most half the CUs split.
  if (M > 128 && tiles > kSplitTargetBlocks / 2) return;
  while (tiles * splits < kSplitTargetBlocks && splits < kMaxSplits && K / (2 * splits) >= kMinSliceSteps * kBK) splits *= 2;
  if (splits == 1) return;
  kchunk = (int)(((K + splits - 1) / splits + kBKSplit - 1) / kBKSplit * kBKSplit);
  splits = (int)((K + kchunk - 1) / kchunk);
}

}  // namespace
}  // namespace egpt

using namespace egpt;

extern "C" int egpt_int8_gemm_workspace(int M, int N, int K, size_t* bytes) {
  if (!bytes || M < 0 || N < 0 || K < 0) return EGPT_ERR_INVALID;
  int splits, kchunk;
  gemm_split(M, N, K, splits, kchunk);
  *bytes = splits > 1 ? (size_t)splits * (size_t)M * (size_t)N * sizeof(float) : 0;
  return EGPT_OK;
}

extern "C" int egpt_int8_gemm_tile(int M, int N, int swiglu, int* rows, int* columns, int* ring) {
  if (M < 1 || N < 1 || !rows || !columns || !ring) return EGPT_ERR_INVALID;
  const GemmTile& t = best_tile(M, N, swiglu != 0);
  *rows = t.bm;
  *columns = t.bn;
  *ring = t.ring;
  return EGPT_OK;
}

extern "C" int egpt_int8_gemm_ws(const void* x, int64_t ldx, const int8_t* w, int64_t ldw, const float* scale,
                                 void* y, int64_t ldy, int M, int N, int K, void* workspace, size_t workspace_bytes,
                                 hipStream_t stream) {
  if (!x || !w || !scale || !y || M < 0 || N < 0 || K < 0) return EGPT_ERR_INVALID;
  if (ldx < K || ldw < K || ldy < N) return EGPT_ERR_INVALID;
  if (M == 0 || N == 0) return EGPT_OK;
  GemmArgs a{(const uint16_t*)x, ldx, w, ldw, scale, (uint16_t*)y, ldy, M, N, K, 0, 0, 1, K, nullptr, 0};
  // The LDS-direct tiles take K a multiple of 64, 16-byte aligned rows and operands their
  // 32-bit byte offsets reach; every other shape runs the ragged kernel.
  if (K == 0 || K % kBK || ldx % 8 || ldw % 16 || (uintptr_t)x % 16 || (uintptr_t)w % 16 ||
      (int64_t)M * ldx * 2 >= ((int64_t)1 << 31) || (int64_t)N * ldw >= ((int64_t)1 << 31) ||
      (int64_t)M * ldy * 2 >= ((int64_t)1 << 31) ||
      ((int64_t)M + 63) / 64 * (((int64_t)N + 63) / 64) > (int64_t)INT32_MAX / kMaxSplits)
    return launch_ragged(a, stream);
  if (workspace) {  // a workspace lets short-M shapes split K
    int splits, kchunk;
    gemm_split(M, N, K, splits, kchunk);
    if (splits > 1) {
      if (workspace_bytes < (size_t)splits * (size_t)M * (size_t)N * sizeof(float) || (uintptr_t)workspace % 16)
        return EGPT_ERR_WORKSPACE;
      a.splits = splits;
      a.kchunk = kchunk;
      a.part = (float*)workspace;
      return launch_split(a, stream);
    }
  }
  return launch_best_tile(a, false, stream);
}

extern "C" int egpt_int8_gemm_swiglu(const void* x, int64_t ldx, const int8_t* w, int64_t ldw, const float* scale,
                                     void* act, int64_t ld_act, int M, int inter, int K, hipStream_t stream) {
  if (!x || !w || !scale || !act || M < 0 || inter < 0 || K < 0) return EGPT_ERR_INVALID;
  if (ldx < K || ldw < K || ld_act < inter) return EGPT_ERR_INVALID;
  if (M == 0 || inter == 0) return EGPT_OK;
  const int64_t N = 2 * (int64_t)inter;
  if (K == 0 || K % kBK || ldx % 8 || ldw % 16 || (uintptr_t)x % 16 || (uintptr_t)w % 16 ||
      (int64_t)M * ldx * 2 >= ((int64_t)1 << 31) || N * ldw >= ((int64_t)1 << 31) ||
      (int64_t)M * ld_act * 2 >= ((int64_t)1 << 31) || N > INT32_MAX)
    return EGPT_ERR_UNSUPPORTED;
  GemmArgs a{(const uint16_t*)x, ldx, w, ldw, scale, (uint16_t*)act, ld_act, M, (int)N, K, 0, 0, 1, K, nullptr,
             inter};
  // Not where the plain product would split K, which this form cannot.
  int splits, kchunk;
  gemm_split(M, N, K, splits, kchunk);
  if (splits > 1 || N > INT32_MAX / 2) return EGPT_ERR_UNSUPPORTED;
  return launch_best_tile(a, true, stream);
}

extern "C" int egpt_int8_gemm_add_rmsnorm(const void* x, int64_t ldx, const int8_t* w, int64_t ldw,
                                          const float* scale, void* resid, int64_t ld_resid, const void* norm_w,
                                          void* y, int64_t ldy, int M, int N, int K, float eps, void* workspace,
                                          size_t workspace_bytes, hipStream_t stream) {
  if (!x || !w || !scale || !resid || !norm_w || !y || M < 0 || N < 0 || K < 0) return EGPT_ERR_INVALID;
  if (ldx < K || ldw < K || ld_resid < N || ldy < N) return EGPT_ERR_INVALID;
  if (M == 0 || N == 0) return EGPT_OK;
  if (K == 0 || K % kBK || ldx % 8 || ldw % 16 || (uintptr_t)x % 16 || (uintptr_t)w % 16)
    return EGPT_ERR_UNSUPPORTED;
  if ((int64_t)M * ldx * 2 >= ((int64_t)1 << 31) || (int64_t)N * ldw >= ((int64_t)1 << 31)) return EGPT_ERR_UNSUPPORTED;
  if ((size_t)N * sizeof(float) > 64 * 1024) return EGPT_ERR_UNSUPPORTED;  // the row kernel stages a row in LDS
  int splits, kchunk;
  gemm_split(M, N, K, splits, kchunk);
  if (splits < 2) return EGPT_ERR_UNSUPPORTED;  // nothing to fold: egpt_int8_gemm_ws, then egpt_add_rmsnorm
  if (!workspace || workspace_bytes < (size_t)splits * (size_t)M * (size_t)N * sizeof(float) ||
      (uintptr_t)workspace % 16)
    return EGPT_ERR_WORKSPACE;
  GemmArgs a{(const uint16_t*)x, ldx, w, ldw, scale, nullptr, N, M, N, K, 0, 0, splits, kchunk, (float*)workspace,
             0};
  const int st = launch_split_partials(a, stream);
  if (st != EGPT_OK) return st;
  return launch_reduce_add_rmsnorm((const float*)workspace, splits, scale, resid, ld_resid, norm_w, y, ldy, M, N,
                                   eps, stream);
}

extern "C" int egpt_int8_gemm_qk_norm_rope(const void* x, int64_t ldx, const int8_t* w, int64_t ldw,
                                           const float* scale, const int64_t* positions, const void* q_norm_w,
                                           const void* k_norm_w, const void* cos_t, const void* sin_t, void* q_out,
                                           int64_t ld_q, void* k_cache, void* v_cache, int64_t cache_head_stride,
                                           int64_t cache_slot_stride, int M, int Hq, int Hkv, int D, int K, int cap,
                                           float eps, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (!x || !w || !scale || M < 0 || K < 0 || Hq < 1 || Hkv < 1 || D < 1) return EGPT_ERR_INVALID;
  const int64_t N = (int64_t)(Hq + 2 * Hkv) * D;
  if (ldx < K || ldw < K || N > INT32_MAX) return EGPT_ERR_INVALID;
  if (M == 0) return EGPT_OK;
  if (K == 0 || K % kBK || ldx % 8 || ldw % 16 || (uintptr_t)x % 16 || (uintptr_t)w % 16)
    return EGPT_ERR_UNSUPPORTED;
  if ((int64_t)M * ldx * 2 >= ((int64_t)1 << 31) || N * ldw >= ((int64_t)1 << 31)) return EGPT_ERR_UNSUPPORTED;
  int splits, kchunk;
  gemm_split(M, N, K, splits, kchunk);
  if (splits < 2) return EGPT_ERR_UNSUPPORTED;  // nothing to fold: egpt_int8_gemm_ws, then egpt_qk_norm_rope
  const int c = check_reduce_qk_norm_rope(splits, positions, q_norm_w, k_norm_w, cos_t, sin_t, q_out, ld_q, k_cache,
                                          v_cache, cache_head_stride, cache_slot_stride, M, Hq, Hkv, D, cap);
  if (c != EGPT_OK) return c;
  if (!workspace || workspace_bytes < (size_t)splits * (size_t)M * (size_t)N * sizeof(float) ||
      (uintptr_t)workspace % 16)
    return EGPT_ERR_WORKSPACE;
  GemmArgs a{(const uint16_t*)x, ldx, w, ldw, scale, nullptr, N, M, (int)N, K, 0, 0, splits, kchunk,
             (float*)workspace, 0};
  const int st = launch_split_partials(a, stream);
  if (st != EGPT_OK) return st;
  return launch_reduce_qk_norm_rope((const float*)workspace, splits, scale, positions, q_norm_w, k_norm_w, cos_t,
                                    sin_t, q_out, ld_q, k_cache, v_cache, cache_head_stride, cache_slot_stride, M, Hq,
                                    Hkv, D, cap, eps, stream);
}

extern "C" int egpt_int8_gemm(const void* x, int64_t ldx, const int8_t* w, int64_t ldw, const float* scale, void* y,
                              int64_t ldy, int M, int N, int K, hipStream_t stream) {
  return egpt_int8_gemm_ws(x, ldx, w, ldw, scale, y, ldy, M, N, K, nullptr, 0, stream);
}
