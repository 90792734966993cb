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
//   * Large products run tiles of 128 x 128 to 256 x 256 on v_mfma_f32_16x16x32_bf16 (int8_gemm_dma_kernel): operands
//     straight into LDS, the weights as int8, eight wavefronts whose two halves take turns at the matrix cores.
//   * Small ones run 64 x 64 and 128 x 64 tiles of 4 wavefronts on v_mfma_f32_32x32x16_bf16 (int8_gemm_kernel). K
//     advances 64 (128 where the tiles are few) at a time through two LDS buffers and two register staging sets: the
//     global loads of step k + 2 are issued before the MFMAs of step k; one barrier per step. The padding of the LDS
//     rows puts the fragment reads of 16 consecutive rows on distinct banks.
//   * int8 -> bf16 is exact: every value in [-127, 127] is a bf16.
//   * Rows past M or N read a valid row and are never stored.
//   * Split-K (short M, long K: too few output tiles to give every CU a block):
//     block (split, tile) sums its K slice and stores the fp32 tile to a caller's
//     workspace [splits][M][N]; a second kernel adds the slices in split order and
//     applies the two roundings. The fp32 sum is the same product in another
//     order, as any GEMM blocking is.
// Operand layouts of v_mfma_f32_32x32x16_bf16 (checked on the MI355X): lane l holds A[l % 32][8 (l / 32) + e]
// and B[8 (l / 32) + e][l % 32], e = 0..7; accumulator register r of lane l is
// C[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace egpt {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kBK = 64;        // K per LDS stage of the one-pass kernel: K must be a multiple of it
constexpr int kBKSplit = 128;  // K per LDS stage of the split-K slices (half the dependent steps)

template <int BM, int BN, int BK, int WN, int NW>
struct GemmShape {
  static constexpr int NT = NW * kWave;      // threads of the block
  static constexpr int WM = NW / WN;          // wavefronts along M (the block's NW as WM x WN)
  static constexpr int TM = BM / (32 * WM);  // 32 x 32 tiles per wavefront along M
  static constexpr int TN = BN / (32 * WN);  // ... along N
  static constexpr int kLdsRow = BK + 8;    // bf16 elements per x or weight row in LDS (16 bytes of padding)
  static constexpr int kALoads = BM * BK * 2 / (NT * 16);  // 16-byte x loads per thread per step
  static constexpr int kBLoads = BN * BK / (NT * 16);      // 16-byte int8 loads per thread per step
  static_assert(WM * WN == NW && TM >= 1 && TN >= 1 && kALoads >= 1 && kBLoads >= 1, "tile too small for the block");
};

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

// SwiGLU form of the small tiles: block tile column j (of BN) -> weight row. Each wavefront's BN / WN columns hold its
// features' gate rows and then the same features' up rows. Features past `inter` read the last one.
template <int BN, int WN>
__device__ __forceinline__ int64_t swiglu_row(int64_t pid_n, int j, int inter) {
  constexpr int kPerWave = BN / WN, kHalf = kPerWave / 2;
  const int wn = j / kPerWave, o = j % kPerWave;
  const int64_t f = min(pid_n * (BN / 2) + wn * kHalf + (o % kHalf), (int64_t)inter - 1);
  return o < kHalf ? f : inter + f;
}

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

// The store of a block's accumulators (TM x TN 32 x 32 tiles per wavefront, wavefront tile origin wm0, wn0 in the
// block tile m0, n0): y = bf16(bf16(acc) * scale), the reference's two roundings, or with SWIGLU the activation
// of each feature from its gate and up columns.
template <int BM, int BN, int TM, int TN, int WN, bool SWIGLU>
__device__ __forceinline__ void gemm_store(const GemmArgs& a, const f32x16 (&acc)[TM][TN], int64_t m0, int64_t n0,
                                           int wm0, int wn0, int pid_n, int lane, int wave) {
  // y = bf16(bf16(acc) * scale): the reference's two roundings. Stores address y
  // by 32-bit byte offsets from the row of this lane's first accumulator (the
  // host checks that y spans < 2 GiB); row r of a tile is a constant multiple of
  // the row pitch away.
  char* yb = (char*)a.y;
  const int64_t mrow0 = m0 + wm0 + 4 * (lane / 32);
  const uint32_t pitch = (uint32_t)(a.ldy * 2);
  if constexpr (SWIGLU && TN == 1) {
    // One 32-column tile per wavefront: its columns 0-15 are the gate rows of 16 features and 16-31 their up
    // rows (swiglu_row), so lane l (column l % 32 < 16) takes u from lane l ^ 16, the same rows one tile half
    // over. The arithmetic per element is the form below.
    const int c = lane % 32;
    const int64_t f = (int64_t)pid_n * (BN / 2) + (wave % WN) * (BN / WN / 2) + (c % 16);
    const int64_t fc = min(f, (int64_t)a.inter - 1);
    const float sg_scale = a.scale[fc], su_scale = a.scale[a.inter + fc];
    const uint32_t base = (uint32_t)((mrow0 * a.ldy + f) * 2);
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float up = __shfl_xor(acc[tm][0][r], 16);
        const int dm = tm * 32 + 8 * (r / 4) + r % 4;
        if (c < 16 && mrow0 + dm < a.M && f < a.inter) {
          const float g = bf16_to_f32(f32_to_bf16(bf16_to_f32(f32_to_bf16(acc[tm][0][r])) * sg_scale));
          const float u = bf16_to_f32(f32_to_bf16(bf16_to_f32(f32_to_bf16(up)) * su_scale));
          const float sg = bf16_to_f32(f32_to_bf16(g / (1.0f + expf(-g))));
          *(uint16_t*)(yb + (base + (uint32_t)dm * pitch)) = f32_to_bf16(sg * u);
        }
      }
    }
    return;
  }
#pragma unroll
  for (int tn = 0; tn < TN; ++tn) {
    const int64_t n = n0 + wn0 + tn * 32 + lane % 32;
    const float sc = a.scale[min(n, (int64_t)a.N - 1)];
    const uint32_t base = (uint32_t)((mrow0 * a.ldy + n) * 2);
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int dm = tm * 32 + 8 * (r / 4) + r % 4;
        if (mrow0 + dm < a.M && n < a.N) {
          const float v = bf16_to_f32(f32_to_bf16(acc[tm][tn][r]));
          *(uint16_t*)(yb + (base + (uint32_t)dm * pitch)) = f32_to_bf16(v * sc);
        }
      }
    }
  }
}

// The small tiles (64 x 64 and 128 x 64): the weights are converted to bf16 once, by the thread that loaded them, as
// they are written to LDS, and the wavefronts read bf16 fragments.
template <int BM, int BN, int BK, bool SPLIT, int WN, int NW, bool SWIGLU = false>
__global__ __launch_bounds__(NW * kWave, 1) void int8_gemm_kernel(const GemmArgs a) {
  using S = GemmShape<BM, BN, BK, WN, NW>;
  constexpr int TM = S::TM, TN = S::TN;
  static_assert(!SWIGLU || (!SPLIT && TN == 1), "the SwiGLU form pairs the two halves of a wavefront's one column tile");
  constexpr int kLdsRow = S::kLdsRow;
  __shared__ __align__(16) uint16_t As[2][BM * kLdsRow];
  __shared__ __align__(16) uint16_t Bs[2][BN * kLdsRow];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  const int wm0 = (wave / WN) * (BM / S::WM);  // wavefront tile origin in the block tile
  const int wn0 = (wave % WN) * (BN / WN);
  const int tiles = a.tiles_m * a.tiles_n;
  const int split = SPLIT ? (int)blockIdx.x / tiles : 0;
  int pid_m, pid_n;
  gemm_tile((int)blockIdx.x - split * tiles, a.tiles_m, a.tiles_n, pid_m, pid_n);
  const int64_t m0 = (int64_t)pid_m * BM;
  const int64_t n0 = (int64_t)pid_n * BN;
  const int kbeg = SPLIT ? split * a.kchunk : 0;  // this block's K slice [kbeg, kbeg + nk * BK)

  // global -> register staging of one K step: 32-bit byte offsets from the
  // operands' base pointers (the host checks that both operands span < 2 GiB)
  const char* xb = (const char*)a.x;
  const char* wb = (const char*)a.w;
  uint32_t xoff[S::kALoads];
  int a_lds[S::kALoads];
#pragma unroll
  for (int j = 0; j < S::kALoads; ++j) {
    const int i = tid + j * S::NT;
    const int row = i / (BK / 8), chunk = i % (BK / 8);
    xoff[j] = (uint32_t)((min(m0 + row, (int64_t)a.M - 1) * a.ldx + kbeg + chunk * 8) * 2);
    a_lds[j] = row * kLdsRow + chunk * 8;
  }
  uint32_t woff[S::kBLoads];
  int b_lds[S::kBLoads];
#pragma unroll
  for (int j = 0; j < S::kBLoads; ++j) {
    const int i = tid + j * S::NT;
    const int row = i / (BK / 16), chunk = i % (BK / 16);
    const int64_t wrow = SWIGLU ? swiglu_row<BN, WN>(pid_n, row, a.inter) : min(n0 + row, (int64_t)a.N - 1);
    woff[j] = (uint32_t)(wrow * a.ldw + kbeg + chunk * 16);
    b_lds[j] = row * kLdsRow + chunk * 16;
  }
  // Two register staging sets: the loads of step k + 2 are issued while step k is
  // multiplied and land in LDS among the MFMAs of step k + 1, one to two steps of
  // MFMA work later. Loads past the last step re-read the last K slice (in bounds, never
  // stored), so every load is unconditional and each wait is for one set only.
  const int nk = (SPLIT ? min(a.kchunk, a.K - kbeg) : a.K) / BK;
  u32x4 xr[2][S::kALoads], wr[2][S::kBLoads];
  auto load_step = [&](int kt, int set) {
    const uint32_t k0 = (uint32_t)(min(kt, nk - 1) * BK);
#pragma unroll
    for (int j = 0; j < S::kALoads; ++j) xr[set][j] = ld16(xb + (xoff[j] + 2 * k0));
#pragma unroll
    for (int j = 0; j < S::kBLoads; ++j) wr[set][j] = ld16_stream(wb + (woff[j] + k0));
  };
  auto store_step = [&](int buf, int set) {
#pragma unroll
    for (int j = 0; j < S::kALoads; ++j) *(u32x4*)&As[buf][a_lds[j]] = xr[set][j];
#pragma unroll
    for (int j = 0; j < S::kBLoads; ++j) {
      *(bf16x8*)&Bs[buf][b_lds[j]] = int8x8_to_bf16(wr[set][j].x, wr[set][j].y);
      *(bf16x8*)&Bs[buf][b_lds[j] + 8] = int8x8_to_bf16(wr[set][j].z, wr[set][j].w);
    }
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int tm = 0; tm < TM; ++tm)
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) acc[tm][tn] = f32x16{};

  // fragment offsets (elements) inside one LDS buffer
  const int frag_k = 8 * (lane / 32);
  int a_frag[TM], b_frag[TN];
#pragma unroll
  for (int tm = 0; tm < TM; ++tm) a_frag[tm] = (wm0 + tm * 32 + lane % 32) * kLdsRow + frag_k;
#pragma unroll
  for (int tn = 0; tn < TN; ++tn) b_frag[tn] = (wn0 + tn * 32 + lane % 32) * kLdsRow + frag_k;

  // The MFMAs of one K step from LDS buffer `buf`, then, with sbuf >= 0, the next step's LDS stores (staging set `set`
  // into buffer sbuf). One wavefront per SIMD with a short MFMA chain per 16 columns leaves nothing to cover an LDS
  // read issued just before its MFMA, so every fragment of the step is read first.
  auto mma_step = [&](int buf, int sbuf = -1, int set = 0) {
    bf16x8 af[BK / 16][TM], bh[BK / 16][TN];
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) af[ks][tm] = *(const bf16x8*)&As[buf][a_frag[tm] + ks * 16];
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) bh[ks][tn] = *(const bf16x8*)&Bs[buf][b_frag[tn] + ks * 16];
    }
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks)
#pragma unroll
      for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
          acc[tm][tn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ks][tm], bh[ks][tn], acc[tm][tn], 0, 0, 0);
    if (sbuf >= 0) store_step(sbuf, set);
  };

  load_step(0, 0);
  load_step(1, 1);
  store_step(0, 0);
  __syncthreads();
  // Pairs of steps so the staging sets are fixed registers: step kt computes LDS
  // buffer kt & 1, refills set kt & 1 with step kt + 2 and stores set (kt + 1) & 1
  // into the other buffer among its MFMAs; an odd last step runs after the loop. Scheduling barriers keep each phase in
  // place (hoisting the second step's fragment reads above the first step's MFMAs
  // would double the live registers).
  int kt = 0;
  for (; kt + 1 < nk; kt += 2) {
    load_step(kt + 2, 0);
    __builtin_amdgcn_sched_barrier(0);
    mma_step(0, 1, 1);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    load_step(kt + 3, 1);
    __builtin_amdgcn_sched_barrier(0);
    mma_step(1, kt + 2 < nk ? 0 : -1, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (kt + 2 < nk) __syncthreads();
  }
  if (kt < nk) mma_step(0);

  if constexpr (SPLIT) {  // the fp32 tile of this K slice; the reduce kernel rounds
    float* part = a.part + (int64_t)split * a.M * a.N;
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      const int64_t n = n0 + wn0 + tn * 32 + lane % 32;
#pragma unroll
      for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int64_t m = m0 + wm0 + tm * 32 + 8 * (r / 4) + 4 * (lane / 32) + r % 4;
          if (m < a.M && n < a.N) part[m * a.N + n] = acc[tm][tn][r];
        }
    }
    return;
  }
  gemm_store<BM, BN, TM, TN, WN, SWIGLU>(a, acc, m0, n0, wm0, wn0, pid_n, lane, wave);
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

typedef uint32_t u32x4_h __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x2_h __attribute__((ext_vector_type(2), aligned(2)));

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
    if constexpr (C % 8)
      *(global_ptr<u32x2_h>)(p + C - 4) = u32x2{w[C / 2 - 2], w[C / 2 - 1]};
  } else {
#pragma unroll
    for (int i = 0; i < C; ++i)
      if (c0 + i < cols) gstore(p + i, f32_to_bf16(o[i]));
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

  if constexpr (SWIGLU) {
    const int64_t f0 = (int64_t)pid_n * (BN / 2) + (wave % WN) * (8 * TN) + 2 * TN * h;
    float gs[2 * TN], us[2 * TN];
#pragma unroll
    for (int e = 0; e < 2 * TN; ++e) {
      const int64_t f = min(f0 + e, (int64_t)a.inter - 1);
      gs[e] = a.scale[f];
      us[e] = a.scale[a.inter + f];
    }
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
      const int64_t m = m0 + wm0 + 16 * tm + r16;
      float o[2 * TN];
#pragma unroll
      for (int e = 0; e < 2 * TN; ++e) {
        const float g = bf16_to_f32(f32_to_bf16(bf16_to_f32(f32_to_bf16(acc[tm][e / 4][e % 4])) * gs[e]));
        const float u = bf16_to_f32(f32_to_bf16(bf16_to_f32(f32_to_bf16(acc[tm][TN / 2 + e / 4][e % 4])) * us[e]));
        o[e] = bf16_to_f32(f32_to_bf16(g / (1.0f + expf(-g)))) * u;
      }
      store_row<2 * TN>(a, m, f0, a.inter, o);
    }
  } else {
    const int64_t c0 = n0 + wn0 + 4 * TN * h;
    float sc[4 * TN];
#pragma unroll
    for (int e = 0; e < 4 * TN; ++e) sc[e] = a.scale[min(c0 + e, (int64_t)a.N - 1)];
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
      const int64_t m = m0 + wm0 + 16 * tm + r16;
      float o[4 * TN];
#pragma unroll
      for (int e = 0; e < 4 * TN; ++e) o[e] = bf16_to_f32(f32_to_bf16(acc[tm][e / 4][e % 4])) * sc[e];
      store_row<4 * TN>(a, m, c0, a.N, o);
    }
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

template <int BM, int BN>
unsigned gemm_blocks(const GemmArgs& a) {
  return (unsigned)(((int64_t)a.N + BN - 1) / BN) * (unsigned)(((int64_t)a.M + BM - 1) / BM);
}

constexpr int kMaxSplits = 16;

// 128 x 128 tiles of a product from which the LDS-direct tiles take it. With fewer, most CUs would run one block's
// chain of K steps alone (measured on the MI355X, us against the 64-row tiles: 144 tiles 300 x 4096 -> 6144 41.8 / 46.5,
// 192 tiles 700 x 2048 -> 4096 23.4 / 27.7 and 130 x 2048 -> 12288 23.1 / 27.5, 256 tiles 1000 x 12288 -> 4096 126.1 /
// 126.4; but 128 tiles 1000 x 2048 -> 2048 23.0 / 20.7 and 512 x 4096 -> 4096 41.7 / 34.4, 96 tiles 200 x 4096 -> 6144
// 41.7 / 32.5).
constexpr int kDmaMinTiles = 144;

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

// The split slices' fp32 tiles into a.part (64 x 64 tiles, a.splits > 1); no reduce.
int launch_split_partials(GemmArgs a, hipStream_t st) {
  a.tiles_m = (int)(((int64_t)a.M + 63) / 64);
  a.tiles_n = (int)(((int64_t)a.N + 63) / 64);
  const unsigned tiles = (unsigned)a.tiles_m * (unsigned)a.tiles_n;
  hipLaunchKernelGGL((int8_gemm_kernel<64, 64, kBKSplit, true, 2, 4>),
                     dim3(tiles * (unsigned)a.splits), dim3(4 * kWave), 0, st, a);
  return EGPT_LAUNCH_STATUS();
}

template <int BM, int BN, int WN = 2, int NW = 4>
int launch_gemm(GemmArgs a, hipStream_t st) {
  a.tiles_m = (int)(((int64_t)a.M + BM - 1) / BM);
  a.tiles_n = (int)(((int64_t)a.N + BN - 1) / BN);
  const unsigned tiles = (unsigned)a.tiles_m * (unsigned)a.tiles_n;
  if constexpr (BM == 64 && BN == 64 && WN == 2 && NW == 4) {  // split-K runs 64 x 64 tiles
    if (a.splits > 1) {
      if (launch_split_partials(a, st) != EGPT_OK) return EGPT_ERR_LAUNCH;
      const int64_t mn = (int64_t)a.M * a.N;
      const unsigned blocks = (unsigned)std::min<int64_t>((mn + kReduceThreads - 1) / kReduceThreads, 4096);
      if (!launch_reduce<kMaxSplits>(a, blocks, st)) return EGPT_ERR_INVALID;
      return EGPT_LAUNCH_STATUS();
    }
  }
  if constexpr (BM == 64 && BN == 64 && WN == 2 && NW == 4) {
    // Fewer tiles than CUs: each block's chain of dependent K steps is the time,
    // and a 128-wide step halves it (measured on the MI355X: 200 x 2048 -> 2048
    // 16.5 -> 12.5 us, 160 x 2048 -> 4096 16.8 -> 13.2; with 320 tiles, 300 x 2048
    // -> 4096, 1.7% slower).
    if (a.K % kBKSplit == 0 && tiles < 256) {
      hipLaunchKernelGGL((int8_gemm_kernel<64, 64, kBKSplit, false, 2, 4>), dim3(tiles),
                         dim3(4 * kWave), 0, st, a);
      return EGPT_LAUNCH_STATUS();
    }
  }
  hipLaunchKernelGGL((int8_gemm_kernel<BM, BN, kBK, false, WN, NW>), dim3(tiles),
                     dim3(NW * kWave), 0, st, a);
  return EGPT_LAUNCH_STATUS();
}

// The LDS-direct tiles (K a multiple of 64); with SWIGLU each block covers 32 TN features.
template <int TM, int TN, bool SWIGLU>
int launch_gemm_dma(GemmArgs a, hipStream_t st) {
  constexpr int BM = 32 * TM, BN = 64 * TN;
  a.tiles_m = (int)(((int64_t)a.M + BM - 1) / BM);
  a.tiles_n = SWIGLU ? (int)(((int64_t)a.inter + BN / 2 - 1) / (BN / 2)) : (int)(((int64_t)a.N + BN - 1) / BN);
  hipLaunchKernelGGL((int8_gemm_dma_kernel<TM, TN, SWIGLU>), dim3((unsigned)a.tiles_m * (unsigned)a.tiles_n),
                     dim3(kDmaWaves * kWave), 0, st, a);
  return EGPT_LAUNCH_STATUS();
}

// Which LDS-direct tile: the least time of the launch's rounds of 256 blocks (one per CU; the 128 x 128 tile fits two
// blocks on a CU, and a pair of them takes less than two rounds). The costs are the us of one full round over
// K = 4096, launch excluded, measured on the MI355X; their ratios hold for other K.
struct DmaTile {
  int tm, tn;
  float round;  // 256 blocks
  float pair;   // 512 blocks, where two fit on a CU
};
constexpr DmaTile kDmaTiles[] = {{8, 4, 95.0f, 0.f}, {6, 4, 79.5f, 0.f}, {8, 3, 79.5f, 0.f}, {6, 3, 65.3f, 0.f},
                                 {4, 4, 61.7f, 0.f}, {8, 2, 59.5f, 0.f}, {4, 3, 53.8f, 0.f}, {6, 2, 50.0f, 0.f},
                                 {4, 2, 39.7f, 64.0f}};

float dma_cost(const DmaTile& t, int64_t M, int64_t N) {
  const int64_t tiles = ((M + 32 * t.tm - 1) / (32 * t.tm)) * ((N + 64 * t.tn - 1) / (64 * t.tn));
  if (t.pair == 0.f) return t.round * (float)((tiles + 255) / 256);
  const int64_t rest = tiles % 512;
  return t.pair * (float)(tiles / 512) + (rest == 0 ? 0.f : rest <= 256 ? t.round : t.pair);
}

// N counts a SwiGLU product's gate and up columns; its tiles need an even TN.
template <bool SWIGLU>
int launch_gemm_dma_best(const GemmArgs& a, hipStream_t st) {
  const DmaTile* best = nullptr;
  for (const DmaTile& t : kDmaTiles)
    if (!(SWIGLU && t.tn % 2) && (!best || dma_cost(t, a.M, a.N) < dma_cost(*best, a.M, a.N))) best = &t;
  switch (best->tm * 8 + best->tn) {
    case 8 * 8 + 4: return launch_gemm_dma<8, 4, SWIGLU>(a, st);
    case 6 * 8 + 4: return launch_gemm_dma<6, 4, SWIGLU>(a, st);
    case 4 * 8 + 4: return launch_gemm_dma<4, 4, SWIGLU>(a, st);
    case 8 * 8 + 2: return launch_gemm_dma<8, 2, SWIGLU>(a, st);
    case 6 * 8 + 2: return launch_gemm_dma<6, 2, SWIGLU>(a, st);
    case 4 * 8 + 2: return launch_gemm_dma<4, 2, SWIGLU>(a, st);
    default: break;
  }
  if constexpr (!SWIGLU) {
    switch (best->tm * 8 + best->tn) {
      case 8 * 8 + 3: return launch_gemm_dma<8, 3, false>(a, st);
      case 6 * 8 + 3: return launch_gemm_dma<6, 3, false>(a, st);
      case 4 * 8 + 3: return launch_gemm_dma<4, 3, false>(a, st);
      default: break;
    }
  }
  return EGPT_ERR_INVALID;
}

// The same product for shapes the MFMA kernel does not take (K not a multiple of
// 64, rows not 16-byte aligned, operands past its 32-bit offsets): one wavefront
// per output feature n and group of kGenericRows rows, lanes striding K with
// element loads (any alignment, 64-bit indexing), fp32 sums reduced across the
// wavefront in a fixed order, then the two roundings of the prefill formula,
// y = bf16(bf16(sum) * scale[n]). No MFMA and no LDS: a correct form for the
// odd shapes, not a fast one.
constexpr int kGenericRows = 4;
constexpr int kGenericWaves = 4;

__global__ __launch_bounds__(kGenericWaves * kWave) void int8_gemm_generic_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, const int8_t* __restrict__ w, int64_t ldw,
    const float* __restrict__ scale, uint16_t* __restrict__ y, int64_t ldy, int M, int N, int K) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t mgroups = ((int64_t)M + kGenericRows - 1) / kGenericRows;
  const int64_t wv = (int64_t)blockIdx.x * kGenericWaves + threadIdx.x / kWave;
  if (wv >= mgroups * N) return;  // wave-uniform
  const int64_t n = wv / mgroups;  // neighbouring wavefronts share a weight row
  const int64_t m0 = (wv - n * mgroups) * kGenericRows;
  const int8_t* wr = w + n * ldw;
  float acc[kGenericRows] = {};
  for (int64_t k = lane; k < K; k += kWave) {
    const float wk = (float)gload(wr + k);
#pragma unroll
    for (int r = 0; r < kGenericRows; ++r)
      if (m0 + r < M) acc[r] = fmaf(bf16_to_f32(gload(x + (m0 + r) * ldx + k)), wk, acc[r]);
  }
#pragma unroll
  for (int r = 0; r < kGenericRows; ++r) {
    const float sum = wave_sum(acc[r]);
    if (lane == r && m0 + r < M) gstore(y + (m0 + r) * ldy + n, f32_to_bf16(bf16_to_f32(f32_to_bf16(sum)) * scale[n]));
  }
}

int launch_generic(const uint16_t* x, int64_t ldx, const int8_t* w, int64_t ldw, const float* scale, uint16_t* y,
                   int64_t ldy, int M, int N, int K, hipStream_t st) {
  const int64_t waves = ((int64_t)M + kGenericRows - 1) / kGenericRows * N;
  const int64_t blocks = (waves + kGenericWaves - 1) / kGenericWaves;
  if (blocks > (int64_t)UINT32_MAX) return EGPT_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(int8_gemm_generic_kernel, dim3((unsigned)blocks), dim3(kGenericWaves * kWave), 0, st, x, ldx, w,
                     ldw, scale, y, ldy, M, N, K);
  return EGPT_LAUNCH_STATUS();
}

// K slices for a short-M GEMM (at most 256 rows) whose 64 x 64 tiles leave CUs
// idle: the fewest (a power of two, at most 16) that give every CU a block, each
// slice a multiple of kBKSplit and at least 256 wide. 1 when the tiles already fill
// the chip, or K is short or not a multiple of kBKSplit.
constexpr int kMinSliceSteps = 4;
constexpr int kSplitTargetBlocks = 256;

void gemm_split(int64_t M, int64_t N, int64_t K, int& splits, int& kchunk) {
  const int64_t tiles = ((M + 63) / 64) * ((N + 63) / 64);
  splits = 1;
  kchunk = (int)K;
  if (M > 256 || K % kBKSplit) return;  // taller blocks take the larger tiles below
  // Past 128 rows only grids that fill at most half the CUs split (measured on the
  // MI355X: 200 x 2048 -> 2048, 128 tiles, 12.6 -> 10.1 us with 2 splits; 160 x 2048
  // -> 4096, 192 tiles, 13.4 -> 16.2 us with 2)
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

extern "C" int egpt_int8_gemm_ws(const void* x, int64_t ldx, const int8_t* w, int64_t ldw, const float* scale,
                                 void* y, int64_t ldy, int M, int N, int K, void* workspace, size_t workspace_bytes,
                                 hipStream_t stream) {
  if (!x || !w || !scale || !y || M < 0 || N < 0 || K < 0) return EGPT_ERR_INVALID;
  if (ldx < K || ldw < K || ldy < N) return EGPT_ERR_INVALID;
  if (M == 0 || N == 0) return EGPT_OK;
  // The MFMA kernel takes K a multiple of 64, 16-byte aligned rows and operands its
  // 32-bit byte offsets reach; every other shape runs the generic kernel.
  if (K == 0 || K % kBK || ldx % 8 || ldw % 16 || (uintptr_t)x % 16 || (uintptr_t)w % 16 ||
      (int64_t)M * ldx * 2 >= ((int64_t)1 << 31) || (int64_t)N * ldw >= ((int64_t)1 << 31) ||
      (int64_t)M * ldy * 2 >= ((int64_t)1 << 31) ||
      ((int64_t)M + 63) / 64 * (((int64_t)N + 63) / 64) > (int64_t)INT32_MAX / kMaxSplits)
    return launch_generic((const uint16_t*)x, ldx, w, ldw, scale, (uint16_t*)y, ldy, M, N, K, stream);
  GemmArgs a{(const uint16_t*)x, ldx, w, ldw, scale, (uint16_t*)y, ldy, M, N, K, 0, 0, 1, K, nullptr, 0};
  if (workspace) {  // a workspace lets short-M shapes split K
    int splits, kchunk;
    gemm_split(M, N, K, splits, kchunk);
    if (splits > 1) {
      if (workspace_bytes < (size_t)splits * (size_t)M * (size_t)N * sizeof(float) || (uintptr_t)workspace % 16)
        return EGPT_ERR_WORKSPACE;
      a.splits = splits;
      a.kchunk = kchunk;
      a.part = (float*)workspace;
      return launch_gemm<64, 64>(a, stream);
    }
  }
  // The LDS-direct tiles from kDmaMinTiles tiles of their smallest size; below, the 64-row tiles, whose more and
  // shorter blocks fill more of the chip.
  if (M > 64 && gemm_blocks<128, 128>(a) >= kDmaMinTiles) return launch_gemm_dma_best<false>(a, stream);
  if (M > 64 && gemm_blocks<128, 64>(a) >= 256) return launch_gemm<128, 64>(a, stream);
  return launch_gemm<64, 64>(a, stream);
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
  // The LDS-direct tiles where the plain product would take them.
  if (M > 64 && gemm_blocks<128, 128>(a) >= kDmaMinTiles) return launch_gemm_dma_best<true>(a, stream);
  // 64 x 64 tiles (32 features each, gate and up in the two halves of a wavefront's tile) where the plain
  // product would run them too: not where it would split K, which this form cannot.
  int splits, kchunk;
  gemm_split(M, N, K, splits, kchunk);
  if (splits > 1 || N > INT32_MAX / 2) return EGPT_ERR_UNSUPPORTED;
  a.tiles_m = (M + 63) / 64;
  a.tiles_n = (inter + 31) / 32;
  const unsigned tiles = (unsigned)a.tiles_m * (unsigned)a.tiles_n;
  if (K % kBKSplit == 0 && tiles < 256)
    hipLaunchKernelGGL((int8_gemm_kernel<64, 64, kBKSplit, false, 2, 4, true>), dim3(tiles),
                       dim3(4 * kWave), 0, stream, a);
  else
    hipLaunchKernelGGL((int8_gemm_kernel<64, 64, kBK, false, 2, 4, true>), dim3(tiles),
                       dim3(4 * kWave), 0, stream, a);
  return EGPT_LAUNCH_STATUS();
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
