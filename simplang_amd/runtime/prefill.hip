// prefill.hip -- the tokens of a prompt through the decode engine's layers
// together.  The reference's host feeds the prompt to the single-token step one
// token at a time (examples/llama2/generate_stories110M.cpp:236-257); the K/V
// rows that these steps leave behind are all that generation needs of them, and
// the tokens of a prompt depend on each other only through the attention.  So a
// pass takes up to `rows` positions as the rows of matrices: per layer RMSNorm,
// one product over Wq|Wk|Wv, RoPE and the cache store, causal attention, Wo
// added to the residual, RMSNorm, one product over W1|W3, SwiGLU, W2 added to
// the residual.  The weights are read once per pass instead of once per token,
// and no logits are formed: the last prompt token goes through the step.
// The products run on the split-bf16 kernel (gemm_x3.hip), the attention on
// v_mfma_f32_16x16x4_f32; every sum is fp32, as in the step.
// Measured: 199 prompt tokens of the 110M fp32 model, steps 61 ms, one pass 1.4;
// 31 of the 3B W4 model 27 ms against 3.7.
#include <algorithm>

#include "rt_device.h"
#include "rt_internal.h"

namespace simp {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

// x[t] = emb[prompt[t]]
__global__ void __launch_bounds__(256)
    embed_rows_k(const float *__restrict__ emb, const int *__restrict__ prompt,
                 float *__restrict__ x, int dim) {
  const int64_t tok = prompt[blockIdx.y];
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < dim) x[(int64_t)blockIdx.y * dim + i] = emb[tok * dim + i];
}

// out[t] = x[t] / sqrt(mean(x[t]^2) + eps) * w, one block per row
__global__ void __launch_bounds__(256)
    rmsnorm_rows_k(const float *__restrict__ x, const float *__restrict__ w,
                   float *__restrict__ out, int dim, float eps) {
  __shared__ float scratch[16];
  const float *xr = x + (int64_t)blockIdx.x * dim;
  float ss = 0.f;
  for (int i = threadIdx.x; i < dim; i += 256) ss = fmaf(xr[i], xr[i], ss);
  ss = block_sum_lds<true>(ss, scratch);
  const float rms = sqrtf(ss / (float)dim + eps);
  for (int i = threadIdx.x; i < dim; i += 256)
    out[(int64_t)blockIdx.x * dim + i] = (xr[i] / rms) * w[i];
}

// Row t of qkv = (q[dim], k[kv], v[kv]): q rotated in place, k rotated and v
// copied into the cache rows of position p0 + t.  One thread per pair.
__global__ void __launch_bounds__(256)
    rope_store_rows_k(float *__restrict__ qkv, float *__restrict__ kc, float *__restrict__ vc,
                      const float2 *__restrict__ rope, int p0, int dim, int kv, int hs) {
  const int t = blockIdx.y, i = 2 * (blockIdx.x * 256 + threadIdx.x), ld = dim + 2 * kv;
  if (i >= ld) return;
  float2 *p = (float2 *)(qkv + (int64_t)t * ld + i);
  const float2 v = *p;
  const int64_t pos = p0 + t;
  if (i >= dim + kv) {
    *(float2 *)(vc + pos * kv + (i - dim - kv)) = v;
    return;
  }
  const int d = (i < dim ? i : i - dim) % hs;
  const float2 f = rope ? rope[pos * (hs >> 1) + (d >> 1)] : make_float2(1.f, 0.f);
  const float2 r = make_float2(v.x * f.x - v.y * f.y, v.x * f.y + v.y * f.x);
  if (i < dim) *p = r;
  else *(float2 *)(kc + pos * kv + (i - dim)) = r;
}

// h[t][i] = silu(h[t][i]) * h[t][hid + i]
__global__ void __launch_bounds__(256) swiglu_rows_k(float *__restrict__ h, int hid) {
  float *r = h + (int64_t)blockIdx.y * 2 * hid;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < hid) {
    const float g = r[i];
    r[i] = (g / (1.f + expf(-g))) * r[hid + i];
  }
}

// Causal attention of T queries at positions p0 .. p0 + T - 1 over the cache
// rows 0 .. position (the queries' own rows are in the cache).  A block takes
// 16 queries of one head; its four waves take the 16-key tiles in turn, each
// with its own running maximum, sum and output, combined through LDS at the end.
//   * v_mfma_f32_16x16x4_f32 on S^T = K Q^T: a lane ends with the scores of four
//     keys (4g .. 4g+3) for one query (lane % 16), which is the B operand that
//     O^T += V^T P^T wants with step r taking key 4g + r: no transposition.
//     Both operands of S^T take dimensions 16 j + 4 g + i at step (j, i), so a
//     lane's K or Q is one float4 per 16 dimensions.
//   * Latency bounds it (a handful of tiles per wave at these lengths): V of the
//     tile and K of the next are requested before the scores are formed.
// HB: 16-dimension blocks of a head (hs <= 16 HB, hs % 4 == 0).
template <int HB>
__global__ void __launch_bounds__(256)
    attn_rows_k(const float *__restrict__ qkv, const float *__restrict__ kc,
                const float *__restrict__ vc, float *__restrict__ out, int T, int p0, int dim,
                int kv, int n_heads, int n_kv_heads, int hs) {
  __shared__ float so[4][16 * HB][17];
  __shared__ float sm[4][16], sl[4][16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r16 = lane & 15, g = lane >> 4;
  const int h = blockIdx.y, kvh = h * n_kv_heads / n_heads;
  const int q0 = 16 * (int)(gridDim.x - 1 - blockIdx.x);  // the longest rows first
  const int qpos = p0 + min(q0 + r16, T - 1);             // this lane's query
  const int last = p0 + min(q0 + 15, T - 1);              // the block's last key
  const float *kb = kc + kvh * hs, *vb = vc + kvh * hs;
  const float scale = 1.f / sqrtf((float)hs);

  float4 q[HB], k[HB];
  {
    const float *qr = qkv + (int64_t)min(q0 + r16, T - 1) * (dim + 2 * kv) + h * hs;
#pragma unroll
    for (int j = 0; j < HB; j++) {
      const int d = 16 * j + 4 * g;
      q[j] = d < hs ? *(const float4 *)(qr + d) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  auto loadk = [&](int key0) {
    const float *kr = kb + (int64_t)min(key0 + r16, last) * kv;
#pragma unroll
    for (int j = 0; j < HB; j++) {
      const int d = 16 * j + 4 * g;
      k[j] = d < hs ? *(const float4 *)(kr + d) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  v4f o[HB];
#pragma unroll
  for (int j = 0; j < HB; j++) o[j] = v4f{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  loadk(16 * wave);
  for (int key0 = 16 * wave; key0 <= last; key0 += 64) {
    float v[HB][4];  // V[key0 + 4g + r][16 j + r16]
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const float *vr = vb + (int64_t)min(key0 + 4 * g + r, last) * kv;
#pragma unroll
      for (int j = 0; j < HB; j++) v[j][r] = vr[min(16 * j + r16, hs - 1)];
    }
    v4f s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < HB; j++) {
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(k[j].x, q[j].x, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(k[j].y, q[j].y, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(k[j].z, q[j].z, s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(k[j].w, q[j].w, s, 0, 0, 0);
    }
    loadk(key0 + 64);  // clamped to the last key past the end
    float mt = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      s[r] = key0 + 4 * g + r <= qpos ? s[r] * scale : -INFINITY;
      mt = fmaxf(mt, s[r]);
    }
    {  // over the four groups of lanes that share the query
      float a = mt, b = mt;
      permlane16_swap(a, b);
      mt = fmaxf(a, b);
      a = b = mt;
      permlane32_swap(a, b);
      mt = fmaxf(a, b);
    }
    const float mn = fmaxf(m, mt), mu = mn == -INFINITY ? 0.f : mn;  // every key masked so far
    const float alpha = expf(m - mu);
    float p[4], pl = 0.f;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      p[r] = expf(s[r] - mu);
      pl += p[r];
    }
    m = mn;
    l = l * alpha + pl;
#pragma unroll
    for (int j = 0; j < HB; j++) {
#pragma unroll
      for (int r = 0; r < 4; r++) o[j][r] *= alpha;
#pragma unroll
      for (int r = 0; r < 4; r++)
        o[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[j][r], p[r], o[j], 0, 0, 0);
    }
  }
  {
    float a = l, b = l;
    permlane16_swap(a, b);
    l = a + b;
    a = b = l;
    permlane32_swap(a, b);
    l = a + b;
  }
  if (g == 0) {
    sm[wave][r16] = m;
    sl[wave][r16] = l;
  }
#pragma unroll
  for (int j = 0; j < HB; j++)
#pragma unroll
    for (int r = 0; r < 4; r++) so[wave][16 * j + 4 * g + r][r16] = o[j][r];
  __syncthreads();
  for (int e = threadIdx.x; e < 16 * hs; e += 256) {
    const int qi = e / hs, d = e - qi * hs;
    if (q0 + qi >= T) break;  // queries in increasing order
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; w++) M = fmaxf(M, sm[w][qi]);
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      const float f = expf(sm[w][qi] - M);
      num = fmaf(f, so[w][d][qi], num);
      den = fmaf(f, sl[w][qi], den);
    }
    out[(int64_t)(q0 + qi) * dim + h * hs + d] = num / den;
  }
}

}  // namespace

bool prefill_supported(const simp_rt_llama_config &c, const simp_rt_llama_weights &w, int hs) {
  const int64_t kv = (int64_t)hs * c.n_kv_heads;
  // float4 rows of a head, in the attention kernel's registers
  if (hs % 4 != 0 || hs > 128 || c.dim % 4 != 0 || kv % 4 != 0 || c.hidden_dim > INT32_MAX / 2) return false;
  if (c.weight_format != SIMP_RT_W_W4S) return true;
  // 4-byte loads of W4 rows, which are whole 16 bytes apart
  for (const void *p : {w.q_wq, w.q_wk, w.q_wv, w.q_wo, w.q_w1, w.q_w2, w.q_w3})
    if (((uintptr_t)p & 3) != 0) return false;
  return c.dim % 32 == 0 && c.hidden_dim % 32 == 0 && c.group_size % 32 == 0;
}

size_t prefill_floats(const simp_rt_llama_config &c, int rows) {
  const int64_t kv = c.dim / c.n_heads * c.n_kv_heads;
  return (size_t)rows * (size_t)(2 * c.dim + (c.dim + 2 * kv) + 2 * c.hidden_dim);
}

int prefill(const PrefillArgs &a, int64_t n_tokens, hipStream_t st) {
  const auto &c = *a.cfg;
  const auto &w = *a.w;
  const int dim = (int)c.dim, hid = (int)c.hidden_dim, kv = a.kv_dim, hs = a.hs, gs = c.group_size;
  const bool w4 = c.weight_format == SIMP_RT_W_W4S;
  const int ldq = dim + 2 * kv;
  float *x = a.ws, *xb = x + (size_t)a.rows * dim, *qkv = xb + (size_t)a.rows * dim,
        *h13 = qkv + (size_t)a.rows * ldq;
  int rc;
  for (int64_t p0 = 0; p0 < n_tokens; p0 += a.rows) {
    const int T = (int)std::min<int64_t>(a.rows, n_tokens - p0);
    auto product = [&](const X3Mat *m, int nm, int K, const float *A, int64_t lda, float *C,
                       int64_t ldc, float beta) {
      return launch_x3(m, nm, w4 ? K / 2 : K, w4 ? X3Fmt::kW4 : X3Fmt::kT, w4 ? K / gs : 0, gs, A,
                       lda, C, ldc, T, K, beta, true, false, st);
    };
    auto mat = [&](const float *f, const uint8_t *q, const float *s, int64_t off, int n) {
      return w4 ? X3Mat{q + off / 2, s + off / gs, n} : X3Mat{f + off, nullptr, n};
    };
    hipLaunchKernelGGL(embed_rows_k, dim3((unsigned)cdiv(dim, 256), (unsigned)T), dim3(256), 0, st,
                       w.token_embedding, a.prompt + p0, x, dim);
    for (int64_t l = 0; l < c.n_layers; l++) {
      const int64_t lq = l * dim * dim, lk = l * kv * dim, lf = l * hid * dim;
      float *kc = a.kcache + l * c.seq_len * kv, *vc = a.vcache + l * c.seq_len * kv;
      hipLaunchKernelGGL(rmsnorm_rows_k, dim3((unsigned)T), dim3(256), 0, st, x, w.rms_att + l * dim,
                         xb, dim, c.eps);
      const X3Mat mq[3] = {mat(w.wq, w.q_wq, w.s_wq, lq, dim), mat(w.wk, w.q_wk, w.s_wk, lk, kv),
                           mat(w.wv, w.q_wv, w.s_wv, lk, kv)};
      if ((rc = product(mq, 3, dim, xb, dim, qkv, ldq, 0.f))) return rc;
      hipLaunchKernelGGL(rope_store_rows_k, dim3((unsigned)cdiv(ldq / 2, 256), (unsigned)T),
                         dim3(256), 0, st, qkv, kc, vc, a.rope, (int)p0, dim, kv, hs);
      if (l + 1 == c.n_layers) break;  // the last layer's K and V are all that is left to fill
      const dim3 ga((unsigned)cdiv(T, 16), (unsigned)c.n_heads);
#define ATTN(HB)                                                                              \
  hipLaunchKernelGGL(attn_rows_k<HB>, ga, dim3(256), 0, st, qkv, kc, vc, xb, T, (int)p0, dim, \
                     kv, (int)c.n_heads, (int)c.n_kv_heads, hs)
      if (hs <= 32) ATTN(2);
      else if (hs <= 64) ATTN(4);
      else if (hs <= 112) ATTN(7);
      else ATTN(8);
#undef ATTN
      const X3Mat mo = mat(w.wo, w.q_wo, w.s_wo, lq, dim);
      if ((rc = product(&mo, 1, dim, xb, dim, x, dim, 1.f))) return rc;
      hipLaunchKernelGGL(rmsnorm_rows_k, dim3((unsigned)T), dim3(256), 0, st, x, w.rms_ffn + l * dim,
                         xb, dim, c.eps);
      const X3Mat mf[2] = {mat(w.w1, w.q_w1, w.s_w1, lf, hid), mat(w.w3, w.q_w3, w.s_w3, lf, hid)};
      if ((rc = product(mf, 2, dim, xb, dim, h13, 2 * hid, 0.f))) return rc;
      hipLaunchKernelGGL(swiglu_rows_k, dim3((unsigned)cdiv(hid, 256), (unsigned)T), dim3(256), 0,
                         st, h13, hid);
      const X3Mat m2 = mat(w.w2, w.q_w2, w.s_w2, lf, dim);
      if ((rc = product(&m2, 1, hid, h13, 2 * hid, x, dim, 1.f))) return rc;
    }
    SIMP_HIP(hipGetLastError());
  }
  return SIMP_RT_OK;
}

}  // namespace simp
