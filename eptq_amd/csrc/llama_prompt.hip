// Attention of a prompt (many tokens per sequence) in the Llama harness.
//
// Counterpart of the reference driver's HuggingFace attention over a static
// cache (bench_decode.py:44-71), for T tokens at positions pos[0..T) of each
// of B sequences:
//   k_rope_cache   rotary on k, k and v into the caches;
//   k_prompt_attn  rotary on q, out = softmax(q·Kᵀ/√D)·V over the cache rows
//                  0..pos[t] of each token.
// head_dim 128, fp16 data.  Rotary in fp32 with one fp16 rounding, scores,
// softmax and sums in fp32, one fp16 rounding of the output: the roundings of
// the same steps as separate PyTorch operators.
//
// k_prompt_attn.  A workgroup takes 64 tokens of one head (16 per wave) and
// walks the cache in blocks of 64 rows staged in LDS (K as it is, V transposed).
// Both products run on v_mfma_f32_16x16x32_f16 in transposed form: Sᵀ = K·Qᵀ
// leaves lane (token n = l%16, lg = l/16) with the scores of its own token
// at rows 16j + 4lg + v, so the softmax needs two lane exchanges per block, and
// those values, two tiles of 16 rows at a time, are the B operand of Oᵀ = Vᵀ·Pᵀ
// as they lie (the rows' order inside an MFMA is free as long as Vᵀ follows it):
// the probabilities never leave their lane.  A probability goes into the MFMA
// as two fp16 terms (2048·p = hi + lo, 22 bits: its error stays below that of
// the fp32 sums), so nothing is lost against fp32 products.
//
// Bound by latency and the serial softmax chain, not by the matrix cores (4
// GFLOP for 2 x 500 tokens of 32 heads).  Two Llama-2-7B layers and the lm_head
// on 2 x 500 tokens: 2625 -> 1464 us with this kernel and the RMSNorm and SwiGLU
// kernels in place of PyTorch operators (fp32 matmuls over the whole cache,
// softmax, masks, rotary, conversions, copies); same error against 64 bits.

#include "common.h"
#include "eptq_llama.h"

namespace eptq {
namespace {

constexpr int kD = 128;
constexpr int kQ = 64;          // tokens per workgroup
constexpr int kKB = 64;         // cache rows per block
constexpr int kKLd = kD + 8;    // K row stride in halves: 16 rows at one chunk spread over the banks
constexpr int kVLd = kKB + 8;   // Vᵀ row stride in halves

typedef f16 h8 __attribute__((ext_vector_type(8)));

// Dims d .. d+7 of a rotated row: x·cos + rot(x)·sin with rot(x)[d] = -x[d+64]
// below 64 and x[d-64] from 64 (xp: the partner dims).
__device__ __forceinline__ h8 rope8(const h8 x, const h8 xp, const float* __restrict__ c, const float* __restrict__ s,
                                    bool upper) {
  h8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float r = upper ? (float)xp[e] : -(float)xp[e];
    o[e] = (f16)((float)x[e] * c[e] + r * s[e]);
  }
  return o;
}

// One thread per (token row, kv head, 8 dims).
__global__ __launch_bounds__(256) void k_rope_cache(const f16* __restrict__ qkv, const int64_t* __restrict__ posp,
                                                    const float* __restrict__ cosv, const float* __restrict__ sinv,
                                                    f16* __restrict__ kc, f16* __restrict__ vc, int B, int T, int H,
                                                    int Hk, int L) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  const int c = (int)(i & 15), d = 8 * c;
  const size_t rh = i >> 4;
  const int hk = (int)(rh % Hk);
  const size_t row = rh / Hk;   // b·T + t
  if (row >= (size_t)B * T) return;
  const int b = (int)(row / T), t = (int)(row - (size_t)b * T);
  const int64_t pos = posp[t];
  if (pos < 0 || pos >= L) return;
  const f16* src = qkv + row * (size_t)(H + 2 * Hk) * kD;
  const f16* k = src + (size_t)(H + hk) * kD;
  const size_t dst = (((size_t)b * Hk + hk) * L + (size_t)pos) * kD + d;
  *(h8*)(kc + dst) = rope8(*(const h8*)(k + d), *(const h8*)(k + (d ^ 64)), cosv + pos * kD + d, sinv + pos * kD + d, d >= 64);
  *(h8*)(vc + dst) = *(const h8*)(src + (size_t)(H + Hk + hk) * kD + d);
}

__device__ __forceinline__ float max4(float v) {   // over the four lanes of a token
  v = fmaxf(v, partner<16>(v));
  return fmaxf(v, partner<32>(v));
}
__device__ __forceinline__ float sum4(float v) {
  v += partner<16>(v);
  return v + partner<32>(v);
}

__global__ __launch_bounds__(256) void k_prompt_attn(const f16* __restrict__ qkv, const int64_t* __restrict__ posp,
                                                     const float* __restrict__ cosv, const float* __restrict__ sinv,
                                                     const f16* __restrict__ kc, const f16* __restrict__ vc,
                                                     f16* __restrict__ out, int T, int H, int Hk, int L, float scale) {
  __shared__ __attribute__((aligned(16))) f16 Ks[kKB][kKLd];
  __shared__ __attribute__((aligned(16))) f16 Vt[kD][kVLd];
  __shared__ int wlast[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = lane & 15, kg = lane >> 4;
  // The last tokens (the most cache rows) first.
  const int tb = (int)(gridDim.x - 1 - blockIdx.x), h = blockIdx.y, b = blockIdx.z;
  const int hk = h / (H / Hk);
  const int t = tb * kQ + 16 * wave + n;
  const bool live = t < T;
  const int64_t p64 = posp[live ? t : T - 1];
  const int pos = live && p64 >= 0 && p64 < L ? (int)p64 : -1;   // none of the cache for a row outside it

  // q: rotated, as the B operand (dims 32c + 8·kg ..; the partner dims are
  // fragment c ^ 2 of the same lane).
  h8 qf[4];
  {
    const size_t row = (size_t)b * T + (live ? t : T - 1);
    const f16* q = qkv + row * (size_t)(H + 2 * Hk) * kD + (size_t)h * kD + 8 * kg;
    h8 raw[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) raw[c] = *(const h8*)(q + 32 * c);
    const size_t cs = (size_t)(pos < 0 ? 0 : pos) * kD + 8 * kg;
#pragma unroll
    for (int c = 0; c < 4; ++c) qf[c] = rope8(raw[c], raw[c ^ 2], cosv + cs + 32 * c, sinv + cs + 32 * c, c >= 2);
  }
  int last = pos;
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) last = max(last, __shfl_xor(last, o));
  if (lane == 0) wlast[wave] = last;
  __syncthreads();
  last = max(max(wlast[0], wlast[1]), max(wlast[2], wlast[3]));

  const f16* kb = kc + ((size_t)b * Hk + hk) * L * kD;
  const f16* vb = vc + ((size_t)b * Hk + hk) * L * kD;
  // Block loads: K 64 rows x 16 chunks, four per thread; V row pairs x 16
  // chunks, two pairs per thread (rows past L read row L - 1, never used).
  h8 kr[4], vr[2][2];
  auto load = [&](int r0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = min(r0 + (tid >> 4) + 16 * u, L - 1);
      kr[u] = *(const h8*)(kb + (size_t)r * kD + 8 * (tid & 15));
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const int r = min(r0 + 2 * ((tid & 15) + 16 * u) + w, L - 1);
        vr[u][w] = *(const h8*)(vb + (size_t)r * kD + 8 * (tid >> 4));
      }
  };
  f32x4 o[8];
#pragma unroll
  for (int d = 0; d < 8; ++d) o[d] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m = -1e30f, l = 0.0f;
  if (last >= 0) load(0);
  for (int r0 = 0; r0 <= last; r0 += kKB) {
    __syncthreads();   // the previous block's reads are done
#pragma unroll
    for (int u = 0; u < 4; ++u) *(h8*)&Ks[(tid >> 4) + 16 * u][8 * (tid & 15)] = kr[u];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        *(f16x2*)&Vt[8 * (tid >> 4) + e][2 * ((tid & 15) + 16 * u)] = (f16x2){vr[u][0][e], vr[u][1][e]};
    __syncthreads();
    if (r0 + kKB <= last) load(r0 + kKB);

    // Scores of rows r0 + 16j + 4·kg + v for token n.
    f32x4 s[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      s[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 4; ++c)
        s[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(*(const h8*)&Ks[16 * j + n][32 * c + 8 * kg], qf[c], s[j], 0, 0, 0);
    }
    float mx = m;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        s[j][v] = r0 + 16 * j + 4 * kg + v <= pos ? s[j][v] * scale : -INFINITY;
        mx = fmaxf(mx, s[j][v]);
      }
    mx = max4(mx);
    const float down = __expf(m - mx);
    m = mx;
    l *= down;
#pragma unroll
    for (int d = 0; d < 8; ++d)
#pragma unroll
      for (int v = 0; v < 4; ++v) o[d][v] *= down;
#pragma unroll
    for (int j2 = 0; j2 < 2; ++j2) {
      h8 hi, lo;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float p = __expf(s[2 * j2 + (e >> 2)][e & 3] - m);
        l += p;
        const float p2 = p * 2048.0f;
        hi[e] = (f16)p2;
        lo[e] = (f16)(p2 - (float)hi[e]);
      }
#pragma unroll
      for (int d = 0; d < 8; ++d) {
        const f16x4 v0 = *(const f16x4*)&Vt[16 * d + n][32 * j2 + 4 * kg];
        const f16x4 v1 = *(const f16x4*)&Vt[16 * d + n][32 * j2 + 16 + 4 * kg];
        const h8 vf = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
        o[d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, hi, o[d], 0, 0, 0);
        o[d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, lo, o[d], 0, 0, 0);
      }
    }
  }
  l = sum4(l);
  if (!live) return;
  const float inv = 1.0f / (l * 2048.0f);
  f16* dst = out + ((size_t)b * T + t) * (size_t)H * kD + (size_t)h * kD + 4 * kg;
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    f16x4 r;
#pragma unroll
    for (int v = 0; v < 4; ++v) r[v] = (f16)(o[d][v] * inv);
    *(f16x4*)(dst + 16 * d) = r;
  }
}

}  // namespace
}  // namespace eptq

extern "C" int eptq_llama_prompt_attn(const void* qkv, const void* pos, const void* cos_tab, const void* sin_tab,
                                      void* k_cache, void* v_cache, void* out, int B, int T, int H, int Hk, int D,
                                      int L, void* stream) {
  if (!qkv || !pos || !cos_tab || !sin_tab || !k_cache || !v_cache || !out) return 1;
  if (B <= 0 || T <= 0 || H <= 0 || Hk <= 0 || H % Hk || L <= 0) return 1;
  if (D != eptq::kD || B > 65535 || H > 65535) return 2;
  if (((uintptr_t)qkv | (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)out) & 15) return 2;
  using eptq::f16;
  const hipStream_t s = (hipStream_t)stream;
  const size_t threads = (size_t)B * T * Hk * 16;
  if ((threads + 255) / 256 > 0x7fffffff) return 2;
  hipLaunchKernelGGL(eptq::k_rope_cache, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, (const f16*)qkv,
                     (const int64_t*)pos, (const float*)cos_tab, (const float*)sin_tab, (f16*)k_cache, (f16*)v_cache, B,
                     T, H, Hk, L);
  hipLaunchKernelGGL(eptq::k_prompt_attn, dim3((T + eptq::kQ - 1) / eptq::kQ, H, B), dim3(256), 0, s, (const f16*)qkv,
                     (const int64_t*)pos, (const float*)cos_tab, (const float*)sin_tab, (const f16*)k_cache,
                     (const f16*)v_cache, (f16*)out, T, H, Hk, L, 1.0f / sqrtf((float)D));
  return hipGetLastError() == hipSuccess ? 0 : 3;
}
