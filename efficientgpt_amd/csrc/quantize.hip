// Per-output-channel symmetric int8 quantisation on the device: the int8 codes and
// fp32 steps of research/realmodel/int8_linear.py:106-117 (quantize_weight),
//   s[n]    = max(max_k |w[n, k]| / 127, 1e-12)              fp32, correctly rounded
//   q[n, k] = clamp(round_half_even(w[n, k] / s[n]), -127, 127)
// with the weight first converted exactly to fp32 (the reference's `.float()`).
//
// Max and abs are exact and both quotients are the correctly rounded ones
// (__fdiv_rn, or the multiplications of code_mul that give the same bits), so
// the codes and steps are the bits of the formula evaluated on the CPU, whatever
// the order of the max.
#include <algorithm>

#include "common.h"

namespace egpt {
namespace {

constexpr int kQuantWaves = 4;  // wavefronts per block

template <typename T>
__device__ __forceinline__ float load_as_f32(const T* p) {
  return Elem<T>::load1(p);
}

// NaN-propagating max of non-negative floats (torch.amax and numpy's max both propagate NaN): their bit patterns
// order as unsigned integers, with every NaN above infinity.
__device__ __forceinline__ uint32_t max_bits(uint32_t a, uint32_t b) { return a > b ? a : b; }
__device__ __forceinline__ uint32_t abs_bits(float v) { return __float_as_uint(v) & 0x7fffffffu; }

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_max_bits(uint32_t v) {
  return max_bits(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false));
}

__device__ __forceinline__ uint32_t wave_max_bits(uint32_t v) {
  v = dpp_max_bits<kDppXor1>(v);
  v = dpp_max_bits<kDppXor2>(v);
  v = dpp_max_bits<kDppHalfMirror>(v);
  v = dpp_max_bits<kDppMirror>(v);
  const uint32_t r0 = (uint32_t)__builtin_amdgcn_readlane((int)v, 0);
  const uint32_t r1 = (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
  const uint32_t r2 = (uint32_t)__builtin_amdgcn_readlane((int)v, 32);
  const uint32_t r3 = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
  return max_bits(max_bits(r0, r1), max_bits(r2, r3));
}

__device__ __forceinline__ float row_step(uint32_t amax_bits) {
  const float step = __fdiv_rn(__uint_as_float(amax_bits), 127.0f);
  return step < 1e-12f ? 1e-12f : step;  // clamp_min; NaN stays NaN
}

// The code of one value by the formula itself: one correctly rounded division, round half to even, clamp (a NaN
// quotient gives -127).
__device__ __forceinline__ uint32_t code_div(float w, float step) {
  const float r = rintf(__fdiv_rn(w, step));
  return (uint32_t)(int)fminf(fmaxf(r, -127.f), 127.f);
}

// The same code without a division, for a finite step. y is the correctly rounded 1 / step, and after one residual
// step q1 is within one ulp of w / step, so by Markstein's theorem the second one rounds w / step correctly (its
// conditions: y correctly rounded, the significand of step not all ones, nothing over- or underflows where it could
// matter: quotients too small for an exact residual are below 2^-50 and round to 0 either way). Adding
// 1.5 * 2^23 rounds the quotient to an integer half to even and leaves its two's complement in the low bits.
// |w| <= amax bounds the quotient by 127 (1 + 2^-23), which rounds to 127: no clamp is needed.
__device__ __forceinline__ uint32_t code_mul(float w, float step, float y) {
  const float q0 = w * y;
  const float q1 = fmaf(fmaf(-step, q0, w), y, q0);
  const float q2 = fmaf(fmaf(-step, q1, w), y, q1);
  return __float_as_uint(q2 + 12582912.0f);
}

// Rows where code_mul's conditions hold (wave-uniform).
__device__ __forceinline__ bool step_multiplies(float step) {
  return step < 1.2676506e30f && (__float_as_uint(step) & 0x7fffffu) != 0x7fffffu;
}

// 16 bytes of a weight row at any element alignment, and 4 or 8 codes at any byte alignment (the target takes
// unaligned vector accesses; aligned rows lose nothing by the wider type).
template <typename T>
__device__ __forceinline__ u32x4 ld16_el(const T* p) {
  return __builtin_nontemporal_load((global_ptr<const u32x4_h>)p);
}
typedef uint32_t u32_any __attribute__((aligned(1)));
typedef uint32_t u32x2_any __attribute__((ext_vector_type(2), aligned(1)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <typename T>
__device__ __forceinline__ uint32_t chunk_max(const u32x4& v, uint32_t m) {
  constexpr int VE = 16 / Elem<T>::kBytes;
  float f[VE];
  Elem<T>::unpack(v, f);
#pragma unroll
  for (int e = 0; e < VE; ++e) m = max_bits(m, abs_bits(f[e]));
  return m;
}

// The codes of one 16-byte chunk, stored as 4 (fp32) or 8 bytes.
template <typename T>
__device__ __forceinline__ void chunk_store(const u32x4& v, float step, float y, bool mul, int8_t* out) {
  constexpr int VE = 16 / Elem<T>::kBytes;
  float f[VE];
  Elem<T>::unpack(v, f);
  uint32_t c[VE];
  if (mul) {
#pragma unroll
    for (int e = 0; e < VE; ++e) c[e] = code_mul(f[e], step, y);
  } else {
#pragma unroll
    for (int e = 0; e < VE; ++e) c[e] = code_div(f[e], step);
  }
  uint32_t o[VE / 4];
#pragma unroll
  for (int i = 0; i < VE / 4; ++i) {  // the low bytes of four codes in one word
    const uint32_t lo = __builtin_amdgcn_perm(c[4 * i + 1], c[4 * i], 0x0c0c0400u);
    const uint32_t hi = __builtin_amdgcn_perm(c[4 * i + 3], c[4 * i + 2], 0x04000c0cu);
    o[i] = lo | hi;
  }
  if constexpr (VE == 8)
    *(global_ptr<u32x2_any>)out = u32x2{o[0], o[1]};
  else
    *(global_ptr<u32_any>)out = o[0];
}

// W wavefronts per row (kQuantWaves / W rows per block), each lane holding NC 16-byte chunks of the row in
// registers between the max and the codes, so the weight crosses memory once, 16 bytes a lane, and every load of a
// row is in flight before the first is used. NC = 0: rows too long for that, read twice.
// The chunks of a row that K ends in are moved back to end at K: their elements are also another lane's, which
// changes neither the max nor, as both lanes store the same codes, the result. K must be at least 16 bytes.
//
// Bound by memory, with the VALU (about 9 instructions a value) close behind. Measured on the MI355X (one element a
// lane, two passes over the row and a division per value before -> this): bf16 151936 x 2048 498 -> 154 us, 6.05 TB/s
// of weight read and codes written; 24576 x 4096 48 us (6.3 TB/s), fp32 151936 x 2048 269 us (5.8 TB/s).
template <typename T, int NC, int W>
__global__ __launch_bounds__(kQuantWaves * kWave) void quantize_rows_kernel(const T* __restrict__ w, int64_t ldw,
                                                                              int N, int K, int8_t* __restrict__ q,
                                                                              int64_t ldq, float* __restrict__ s) {
  constexpr int VE = 16 / Elem<T>::kBytes;
  constexpr int kRows = kQuantWaves / W;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int64_t row = (int64_t)blockIdx.x * kRows + wave / W;
  if (W == 1 && row >= N) return;  // W = kQuantWaves: the grid is the rows
  const T* wr = w + row * ldw;
  const int first = ((wave % W) * kWave + lane) * VE;  // the lane's chunk c starts at first + c * kStride
  constexpr int kStride = W * kWave * VE;
  uint32_t m = 0;
  u32x4 v[NC > 0 ? NC : 1];
  if constexpr (NC > 0) {
#pragma unroll
    for (int c = 0; c < NC; ++c) v[c] = ld16_el(wr + min(first + c * kStride, K - VE));
#pragma unroll
    for (int c = 0; c < NC; ++c) m = chunk_max<T>(v[c], m);
  } else {
    for (int64_t k = first; k < K; k += kStride) m = chunk_max<T>(ld16_el(wr + min(k, (int64_t)K - VE)), m);
  }
  m = wave_max_bits(m);
  if constexpr (W > 1) {
    __shared__ uint32_t wmax[kQuantWaves];
    if (lane == 0) wmax[wave] = m;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < W; ++i) m = max_bits(m, wmax[i]);
  }
  const float step = row_step(m);
  const float y = __fdiv_rn(1.0f, step);
  const bool mul = step_multiplies(step);
  if (first == 0) s[row] = step;
  int8_t* qr = q + row * ldq;
  if constexpr (NC > 0) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int k = first + c * kStride;
      if (k < K) chunk_store<T>(v[c], step, y, mul, qr + min(k, K - VE));
    }
  } else {
    for (int64_t k = first; k < K; k += kStride) {
      const int64_t kc = min(k, (int64_t)K - VE);
      chunk_store<T>(ld16_el(wr + kc), step, y, mul, qr + kc);
    }
  }
}

// Short rows (up to 64 E elements): one wavefront per row, element by element, E per lane. In 16-byte chunks most lanes
// would idle while each of the others works through 4 or 8 values (us, bf16 16384 x 64 8.9 -> 4.0, x 160 8.6 -> 6.5, x 200
// 8.9 -> 7.6, but 64 x 200 2.38 -> 2.41).
template <typename T, int E>
__global__ __launch_bounds__(kQuantWaves * kWave) void quantize_short_rows_kernel(const T* __restrict__ w, int64_t ldw,
                                                                                    int N, int K,
                                                                                    int8_t* __restrict__ q, int64_t ldq,
                                                                                    float* __restrict__ s) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t row = (int64_t)blockIdx.x * kQuantWaves + threadIdx.x / kWave;
  if (row >= N) return;
  float v[E];
  uint32_t m = 0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    v[e] = lane + e * kWave < K ? load_as_f32(w + row * ldw + lane + e * kWave) : 0.f;
    m = max_bits(m, abs_bits(v[e]));
  }
  const float step = row_step(wave_max_bits(m));
  if (lane == 0) s[row] = step;
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (lane + e * kWave < K) q[row * ldq + lane + e * kWave] = (int8_t)code_div(v[e], step);
}

template <typename T, int E>
void launch_short(const T* w, int64_t ldw, int N, int K, int8_t* q, int64_t ldq, float* s, hipStream_t st) {
  hipLaunchKernelGGL((quantize_short_rows_kernel<T, E>),
                     dim3((unsigned)(((int64_t)N + kQuantWaves - 1) / kQuantWaves)), dim3(kQuantWaves * kWave), 0, st, w,
                     ldw, N, K, q, ldq, s);
}

// A launch holds fewer than 2^32 threads: with a block per row, 2^23 rows take half of that.
constexpr int kLaunchRows = 1 << 23;
static_assert((uint64_t)kLaunchRows * kQuantWaves * kWave < (1ull << 32), "");

template <typename T, int NC, int W>
void launch_rows(const T* w, int64_t ldw, int N, int K, int8_t* q, int64_t ldq, float* s, hipStream_t st) {
  constexpr int kRows = kQuantWaves / W;
  for (int64_t n0 = 0; n0 < N; n0 += kLaunchRows) {
    const int rows = (int)std::min<int64_t>(N - n0, kLaunchRows);
    hipLaunchKernelGGL((quantize_rows_kernel<T, NC, W>), dim3((unsigned)((rows + kRows - 1) / kRows)),
                       dim3(kQuantWaves * kWave), 0, st, w + n0 * ldw, ldw, rows, K, q + n0 * ldq, ldq, s + n0);
  }
}

// Element by element up to 3 a lane, then one wavefront per row up to 8 chunks a lane (32 registers of row), then a block
// per row up to 16 a lane, then the form that reads the row twice.
template <typename T>
void launch_quantize(const T* w, int64_t ldw, int N, int K, int8_t* q, int64_t ldq, float* s, hipStream_t st) {
  constexpr int VE = 16 / Elem<T>::kBytes;
  constexpr int kChunk = kWave * VE;  // elements per wavefront load
  if (K <= kWave)
    launch_short<T, 1>(w, ldw, N, K, q, ldq, s, st);
  else if (K <= 2 * kWave)
    launch_short<T, 2>(w, ldw, N, K, q, ldq, s, st);
  else if (K <= 3 * kWave)
    launch_short<T, 3>(w, ldw, N, K, q, ldq, s, st);
  else if (K <= kChunk)
    launch_rows<T, 1, 1>(w, ldw, N, K, q, ldq, s, st);
  else if (K <= 2 * kChunk)
    launch_rows<T, 2, 1>(w, ldw, N, K, q, ldq, s, st);
  else if (K <= 4 * kChunk)
    launch_rows<T, 4, 1>(w, ldw, N, K, q, ldq, s, st);
  else if (K <= 8 * kChunk)
    launch_rows<T, 8, 1>(w, ldw, N, K, q, ldq, s, st);
  else if (K <= 4 * kQuantWaves * kChunk)
    launch_rows<T, 4, kQuantWaves>(w, ldw, N, K, q, ldq, s, st);
  else if (K <= 8 * kQuantWaves * kChunk)
    launch_rows<T, 8, kQuantWaves>(w, ldw, N, K, q, ldq, s, st);
  else if (K <= 16 * kQuantWaves * kChunk)
    launch_rows<T, 16, kQuantWaves>(w, ldw, N, K, q, ldq, s, st);
  else
    launch_rows<T, 0, kQuantWaves>(w, ldw, N, K, q, ldq, s, st);
}

}  // namespace
}  // namespace egpt

using namespace egpt;

extern "C" int egpt_quantize_rows(int dtype, const void* w, int64_t ldw, int N, int K, int8_t* q, int64_t ldq,
                                  float* s, hipStream_t stream) {
  if (!w || !q || !s || N < 0 || K < 1 || ldw < K || ldq < K) return EGPT_ERR_INVALID;
  if (N == 0) return EGPT_OK;
  switch (dtype) {
    case EGPT_F32:
      launch_quantize((const float*)w, ldw, N, K, q, ldq, s, stream);
      break;
    case EGPT_BF16:
      launch_quantize((const __bf16*)w, ldw, N, K, q, ldq, s, stream);
      break;
    case EGPT_F16:
      launch_quantize((const _Float16*)w, ldw, N, K, q, ldq, s, stream);
      break;
    default:
      return EGPT_ERR_UNSUPPORTED;
  }
  return EGPT_LAUNCH_STATUS();
}
