// The prompt pass of a Qwen3 decoder on gfx950: every launch of it from one call.
//
//   embed + RMSNorm -> per layer: QKV GEMM -> q/k norm + RoPE + cache write -> causal attention -> o GEMM + residual +
//   RMSNorm -> gate/up GEMM + SwiGLU -> down GEMM + residual + the next layer's RMSNorm -> lm_head of the last row ->
//   argmax.
//
// Rounding is that of the kernels it launches (transformers' bf16 Qwen3, models/qwen3/modeling_qwen3.py, with every
// linear on the reference's int8 formulas, research/realmodel/int8_linear.py:88-97): up to 16 rows the decode GEMV, more
// the prefill GEMM. Where a product splits K, its reduce takes the work that follows (norm, RoPE); elsewhere separate
// launches do the same arithmetic.
//
// A short prompt is bound by its launches: a pass of 128 tokens over four Qwen3-1.7B layers is 40 of them, 7.5 us each
// from Python (302 us of host work for 300 us of kernels). The pass needs one workspace and no allocation of its own.
#include "step_core.h"

namespace egpt {
namespace {

constexpr int kThreads = 256;

// Row r of the prompt: x = table[token], h = RMSNorm(x) * w, positions[r] = pos0 + r; block 0 sets *position to the last
// row's. The sums run in add_rmsnorm_kernel's order (V8: add_rmsnorm_v8_kernel's), so x and h have the bits of
// egpt_embed followed by egpt_rmsnorm. One launch for four, 16-byte accesses where the rows allow: 6001 rows of 4096
// took 48 us in the gather alone with 2-byte ones.
template <bool V8>
__global__ __launch_bounds__(kThreads) void prompt_start_kernel(const int64_t* __restrict__ tokens,
                                                                const uint16_t* __restrict__ table, int vocab, int n,
                                                                const uint16_t* __restrict__ w, float eps,
                                                                uint16_t* __restrict__ x, uint16_t* __restrict__ h,
                                                                int64_t* __restrict__ positions,
                                                                int64_t* __restrict__ position, int64_t pos0) {
  __shared__ float red[kThreads / kWave];
  extern __shared__ float rowbuf[];  // n floats
  const int64_t row = blockIdx.x;
  const int64_t tok = tokens[row];
  const int64_t id = tok < 0 ? 0 : (tok >= vocab ? vocab - 1 : tok);
  const uint16_t* t = table + id * n;
  uint16_t* xr = x + row * n;
  uint16_t* hr = h + row * n;
  if (threadIdx.x == 0) {
    positions[row] = pos0 + row;
    if (row == 0) *position = pos0 + (int64_t)gridDim.x - 1;
  }
  float ss = 0.f;
  if (V8) {
    for (int g = threadIdx.x; g * 8 < n; g += kThreads) {
      const u32x4 raw = *(global_ptr<const u32x4_h>)(t + g * 8);  // the table may start at any element
      *(u32x4*)(xr + g * 8) = raw;
      float v[8];
      Elem<__bf16>::unpack(raw, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        rowbuf[g * 8 + e] = v[e];
        ss = fmaf(v[e], v[e], ss);
      }
    }
  } else {
    for (int i = threadIdx.x; i < n; i += kThreads) {
      const float v = bf16_to_f32(t[i]);
      xr[i] = t[i];
      rowbuf[i] = v;
      ss = fmaf(v, v, ss);
    }
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = ss;
  __syncthreads();
  const float inv = rsqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)n + eps);
  if (V8) {
    for (int g = threadIdx.x; g * 8 < n; g += kThreads) {
      float wv[8];
      Elem<__bf16>::unpack(ld16(w + g * 8), wv);
      uint32_t u[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        u[i] = pack2_bf16(wv[2 * i] * bf16r(rowbuf[g * 8 + 2 * i] * inv),
                          wv[2 * i + 1] * bf16r(rowbuf[g * 8 + 2 * i + 1] * inv));
      *(u32x4*)(hr + g * 8) = u32x4{u[0], u[1], u[2], u[3]};
    }
  } else {
    for (int i = threadIdx.x; i < n; i += kThreads) hr[i] = f32_to_bf16(bf16_to_f32(w[i]) * bf16r(rowbuf[i] * inv));
  }
}

// Byte offsets into the workspace. qkv, qrot, attn and the decode attention's partials live from the QKV product to the
// o product, gu and act from the gate/up product to the down product: the two groups share their memory.
struct Layout {
  size_t positions, x, h, qkv, qrot, attn, o, gu, act, split, split_bytes, attn_ws, attn_ws_bytes, arg, arg_bytes, total;
  int attn_splits;
};

bool prompt_layout(const egpt_qwen3_step* s, int rows, Layout* out) {
  const int D = s->head_dim, nq = s->heads * D, nqkv = (s->heads + 2 * s->kv_heads) * D;
  Layout l{};
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t a = at;
    at += (bytes + 255) / 256 * 256;
    return a;
  };
  const size_t r = (size_t)rows;
  l.positions = take(r * sizeof(int64_t));
  l.x = take(r * s->hidden * 2);
  l.h = take(r * s->hidden * 2);
  l.o = take(r * s->hidden * 2);
  const int shape[4][2] = {{nqkv, s->hidden}, {s->hidden, nq}, {2 * s->inter, s->hidden}, {s->hidden, s->inter}};
  if (rows > EGPT_MAX_DECODE_ROWS)
    for (const auto& nk : shape) {
      size_t need = 0;
      if (egpt_int8_gemm_workspace(rows, nk[0], nk[1], &need) != EGPT_OK) return false;
      if (need > l.split_bytes) l.split_bytes = need;
    }
  l.split = take(l.split_bytes);
  l.attn_splits = rows == 1 ? s->nsplit : egpt_decode_attn_default_splits(rows, s->kv_heads, s->cap);
  if (egpt_decode_attn_workspace(rows, s->heads, s->kv_heads, s->cap, D, l.attn_splits, &l.attn_ws_bytes) != EGPT_OK ||
      egpt_argmax_workspace(s->vocab, &l.arg_bytes) != EGPT_OK)
    return false;
  l.arg = take(l.arg_bytes);
  const size_t shared = at;
  l.qkv = take(r * nqkv * 2);
  l.qrot = take(r * nq * 2);
  l.attn = take(r * nq * 2);
  l.attn_ws = take(l.attn_ws_bytes);
  l.total = at;
  at = shared;
  l.gu = take(r * 2 * (size_t)s->inter * 2);
  l.act = take(r * s->inter * 2);
  if (at > l.total) l.total = at;
  *out = l;
  return true;
}

bool prompt_args(const egpt_qwen3_step* s, int rows) {
  return s && s->layers >= 1 && s->hidden >= 1 && s->inter >= 1 && s->heads >= 1 && s->kv_heads >= 1 &&
         s->heads % s->kv_heads == 0 && s->head_dim >= 1 && s->vocab >= 1 && s->cap >= 1 && rows >= 1 && rows <= s->cap;
}

// The split-K workspace every GEMM of the pass shares (they run in stream order).
struct Split {
  void* ws;
  size_t bytes;
};

int linear(const void* x, int64_t ldx, const int8_t* w, const float* sc, void* y, int N, int K, int rows, bool gemm,
           const Split& sp, hipStream_t st) {
  if (!gemm) return egpt_int8_gemv(x, ldx, w, K, sc, y, N, rows, N, K, st);
  return egpt_int8_gemm_ws(x, ldx, w, K, sc, y, N, rows, N, K, sp.bytes ? sp.ws : nullptr, sp.bytes, st);
}

// x = bf16(x + linear(in)), h = RMSNorm(x) * norm: in the split product's reduce where there is one, else the linear
// into `tmp` and egpt_add_rmsnorm (the same bits).
int linear_add_norm(const void* in, int K, const int8_t* w, const float* sc, void* tmp, void* x, const void* norm,
                    void* h, int N, int rows, bool gemm, float eps, const Split& sp, hipStream_t st) {
  if (gemm && sp.bytes) {
    const int r = egpt_int8_gemm_add_rmsnorm(in, K, w, K, sc, x, N, norm, h, N, rows, N, K, eps, sp.ws, sp.bytes, st);
    if (r != EGPT_ERR_UNSUPPORTED) return r;
  }
  const int r = linear(in, K, w, sc, tmp, N, K, rows, gemm, sp, st);
  if (r != EGPT_OK) return r;
  return egpt_add_rmsnorm(x, N, tmp, N, norm, h, N, rows, N, eps, st);
}

}  // namespace
}  // namespace egpt

using namespace egpt;

extern "C" int egpt_qwen3_prefill_workspace(const egpt_qwen3_step* s, int rows, size_t* bytes) {
  Layout l;
  if (!bytes || !prompt_args(s, rows) || !prompt_layout(s, rows, &l)) return EGPT_ERR_INVALID;
  *bytes = l.total;
  return EGPT_OK;
}

extern "C" int egpt_qwen3_prefill(const egpt_qwen3_step* s, const int64_t* tokens, int rows, int pos0,
                                  int prompt_attn, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (!prompt_args(s, rows) || !tokens || pos0 < 0 || (int64_t)pos0 + rows > s->cap) return EGPT_ERR_INVALID;
  if (!s->layer || !s->embed || !s->final_norm || !s->head_w || !s->head_s || !s->rope_cos || !s->rope_sin || !s->token ||
      !s->position || !s->logits)
    return EGPT_ERR_INVALID;
  Layout l;
  if (!prompt_layout(s, rows, &l)) return EGPT_ERR_INVALID;
  if (!workspace || workspace_bytes < l.total || (uintptr_t)workspace % 256) return EGPT_ERR_WORKSPACE;
  const int n = s->hidden, D = s->head_dim, nq = s->heads * D, nqkv = (s->heads + 2 * s->kv_heads) * D;
  if ((size_t)n * sizeof(float) > 64 * 1024) return EGPT_ERR_UNSUPPORTED;  // the norms keep a row in LDS
  const bool gemm = rows > EGPT_MAX_DECODE_ROWS;
  const float scale = (float)(1.0 / sqrt((double)D));
  const int64_t c_sh = (int64_t)s->cap * D;
  char* ws = (char*)workspace;
  int64_t* positions = (int64_t*)(ws + l.positions);
  char *x = ws + l.x, *h = ws + l.h, *qrot = ws + l.qrot, *attn = ws + l.attn, *o = ws + l.o, *act = ws + l.act;
  const Split sp{ws + l.split, l.split_bytes};

  const uint16_t* norm0 = (const uint16_t*)s->layer[0].in_norm;
  const bool v8 = n % 8 == 0 && (uintptr_t)norm0 % 16 == 0;  // as egpt_rmsnorm chooses over the aligned x and h
  hipLaunchKernelGGL(v8 ? prompt_start_kernel<true> : prompt_start_kernel<false>, dim3(rows), dim3(kThreads),
                     n * sizeof(float), stream, tokens, (const uint16_t*)s->embed, s->vocab, n, norm0, s->eps,
                     (uint16_t*)x, (uint16_t*)h, positions, s->position, (int64_t)pos0);
  int st = EGPT_LAUNCH_STATUS();
  if (st != EGPT_OK) return st;

  for (int i = 0; i < s->layers; ++i) {
    const egpt_qwen3_layer& L = s->layer[i];
    st = gemm && l.split_bytes
             ? egpt_int8_gemm_qk_norm_rope(h, n, L.qkv_w, n, L.qkv_s, positions, L.q_norm, L.k_norm, s->rope_cos,
                                           s->rope_sin, qrot, nq, L.k_cache, L.v_cache, c_sh, D, rows, s->heads,
                                           s->kv_heads, D, n, s->cap, s->eps, sp.ws, sp.bytes, stream)
             : EGPT_ERR_UNSUPPORTED;
    if (st == EGPT_ERR_UNSUPPORTED) {
      char* qkv = ws + l.qkv;
      if ((st = linear(h, n, L.qkv_w, L.qkv_s, qkv, nqkv, n, rows, gemm, sp, stream)) != EGPT_OK) return st;
      st = egpt_qk_norm_rope(qkv, nqkv, positions, L.q_norm, L.k_norm, s->rope_cos, s->rope_sin, qrot, nq, L.k_cache,
                             L.v_cache, c_sh, D, rows, s->heads, s->kv_heads, D, s->cap, s->eps, stream);
    }
    if (st != EGPT_OK) return st;
    if (prompt_attn)
      st = egpt_prefill_attn(qrot, nq, L.k_cache, L.v_cache, c_sh, D, attn, nq, rows, s->heads, s->kv_heads, D, s->cap,
                             pos0, scale, stream);
    else
      st = egpt_decode_attn(EGPT_BF16, qrot, nq, D, L.k_cache, 0, c_sh, D, L.v_cache, 0, c_sh, D, positions, 1, attn, nq,
                            D, ws + l.attn_ws, l.attn_ws_bytes, rows, s->heads, s->kv_heads, s->cap, D, l.attn_splits,
                            scale, stream);
    if (st != EGPT_OK) return st;
    st = linear_add_norm(attn, nq, L.o_w, L.o_s, o, x, L.post_norm, h, n, rows, gemm, s->eps, sp, stream);
    if (st != EGPT_OK) return st;
    st = gemm ? egpt_int8_gemm_swiglu(h, n, L.gu_w, n, L.gu_s, act, s->inter, rows, s->inter, n, stream)
              : EGPT_ERR_UNSUPPORTED;
    if (st == EGPT_ERR_UNSUPPORTED) {
      char* gu = ws + l.gu;
      if ((st = linear(h, n, L.gu_w, L.gu_s, gu, 2 * s->inter, n, rows, gemm, sp, stream)) != EGPT_OK) return st;
      st = egpt_silu_mul(gu, 2 * (int64_t)s->inter, s->inter, act, s->inter, rows, stream);
    }
    if (st != EGPT_OK) return st;
    if (i + 1 < s->layers) {
      st = linear_add_norm(act, s->inter, L.down_w, L.down_s, o, x, s->layer[i + 1].in_norm, h, n, rows, gemm, s->eps, sp,
                           stream);
    } else {
      st = linear(act, s->inter, L.down_w, L.down_s, o, n, s->inter, rows, gemm, sp, stream);
    }
    if (st != EGPT_OK) return st;
  }
  const size_t last = (size_t)(rows - 1) * n * 2;
  st = egpt_add_rmsnorm(x + last, n, o + last, n, s->final_norm, h + last, n, 1, n, s->eps, stream);
  if (st != EGPT_OK) return st;
  st = egpt_int8_gemv(h + last, n, s->head_w, n, s->head_s, s->logits, s->vocab, 1, s->vocab, n, stream);
  if (st != EGPT_OK) return st;
  return egpt_argmax(s->logits, s->vocab, ws + l.arg, l.arg_bytes, s->token, s->position, stream);
}
