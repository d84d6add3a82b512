// gg_kernels.hip -- gfx950 (CDNA4) kernels of the Gemma-3 Q8_0 token loop.
//
// One forward pass over a token is five kernels per layer:
//   k_gemv_mg<EMBED_NORM|RESID_NORM, OUT>  fused QKV projection; its prologue
//        finishes the previous layer (post-FFN norm + residual) and applies
//        attn_norm (engine.ts:768-774, 794)
//   k_attn_dec      QK-norm + RoPE + KV store + one chunk of decode attention
//                   per block, chunk partials to memory (engine.ts:775-783)
//   k_gemv_mg<ATTN_MERGE, OUT>  merges the attention chunks in its prologue,
//                   then the attention output projection (engine.ts:784);
//                   spans above 4096 positions: k_attn_merge, then
//                   k_gemv_mg<NONE, OUT>
//   k_gemv_mg<RESID_NORM, GEGLU>  post-attn norm + residual + ffn_norm, gate
//                   and up rows side by side, GeGLU in the epilogue (engine.ts:785-792)
//   k_gemv_mg<NONE, OUT>       down projection (engine.ts:793)
// then k_final (post-FFN norm + residual + output_norm, engine.ts:794-801),
// and for a sampled step the LM head GEMV plus k_select1/k_select2
// (engine.ts:817-901).
//
// A batched prefill runs per layer the bf16-MFMA GEMMs (k_gemm: int8 weights
// exact in bf16, activations split into bf16 hi + lo), the row kernels
// (norms, residuals, QK-norm + RoPE + KV store) and the MFMA attention
// k_attn_pf (+ k_attn_pf_merge for long spans).
//
// On this multi-XCD part a device-scope fence is a whole-L2 write-back, so
// kernels never fence and never exchange data across blocks of one launch:
// every cross-block step is a kernel boundary.
//
// Decode arithmetic is fp32 except the int8 weight payload (dequantised
// exactly in registers) and the sampler's f64 steps, which mirror the JS
// host's. The batched prefill's bf16 products use hi + lo splits of their
// fp32 operands and accumulate in fp32.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "gg_device.h"
#include "gg_internal.h"
#include "gg_pf_schedule.h"

namespace gg {


// ---------------------------------------------------------------------------
// GEMV prologues: build the GEMV input x (K floats) in LDS.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float embed_elem(const GemvArgs& a, int token, int e) {
  return embed_value(a.embd, a.embd_KpS, a.embed_scale, token, e);
}

// Prologue inputs are read into registers before any reduction so that the
// prologue costs one memory latency, overlapped with the weight stream.
constexpr int kMaxEPT = kMaxK / 256;   // elements of x per thread

template <int PRO>
__device__ __forceinline__ void gemv_prologue(const GemvArgs& a, float* xs, int K, float* sh4) {
  const int tid = threadIdx.x;
  const int n = (K - tid + 255) / 256;   // elements this thread owns
  if (PRO == PRO_NONE) {
    float xv[kMaxEPT];
#pragma unroll
    for (int i = 0; i < kMaxEPT; ++i)
      if (i < n) xv[i] = a.x[tid + 256 * i];
#pragma unroll
    for (int i = 0; i < kMaxEPT; ++i)
      if (i < n) xs[xs_index(tid + 256 * i)] = xv[i];
    return;
  }
  float r[kMaxEPT / 4], wp[kMaxEPT / 4];  // K <= 2048 for the norm prologues
  float ss = 0.f;
  if (PRO == PRO_EMBED_NORM) {
    const int cur = a.st->cursor;
    const int token = cur < 0 ? a.st->token : a.tokens[cur];
#pragma unroll
    for (int i = 0; i < kMaxEPT / 4; ++i)
      if (i < n) {
        const int e = tid + 256 * i;
        r[i] = embed_elem(a, token, e);
        wp[i] = a.w_pre[e];
      }
#pragma unroll
    for (int i = 0; i < kMaxEPT / 4; ++i)
      if (i < n) {
        ss = fmaf(r[i], r[i], ss);
        if (blockIdx.x == 0) a.res_out[tid + 256 * i] = r[i];
      }
  } else {  // PRO_RESID_NORM: res = pre_res + norm(pre_vec) * w_post
    float v[kMaxEPT / 4], res[kMaxEPT / 4], wq[kMaxEPT / 4];
#pragma unroll
    for (int i = 0; i < kMaxEPT / 4; ++i)
      if (i < n) {
        const int e = tid + 256 * i;
        v[i] = a.pre_vec[e];
        res[i] = a.pre_res[e];
        wq[i] = a.w_post[e];
        wp[i] = a.w_pre[e];
      }
    float s1 = 0.f;
#pragma unroll
    for (int i = 0; i < kMaxEPT / 4; ++i)
      if (i < n) s1 = fmaf(v[i], v[i], s1);
    const float ri1 = rsq(block_sum256(s1, sh4) / (float)K + a.eps);
#pragma unroll
    for (int i = 0; i < kMaxEPT / 4; ++i)
      if (i < n) {
        const float t = (v[i] * wq[i]) * ri1;   // fusedNormAdd, shaders.ts:415
        r[i] = res[i] + t;
        ss = fmaf(r[i], r[i], ss);
        if (blockIdx.x == 0) {
          a.res_out[tid + 256 * i] = r[i];
          if (a.hist_out) a.hist_out[tid + 256 * i] = r[i];
        }
      }
  }
  const float ri = rsq(block_sum256(ss, sh4) / (float)K + a.eps);   // rmsNorm, shaders.ts:50-53
#pragma unroll
  for (int i = 0; i < kMaxEPT / 4; ++i)
    if (i < n) {
      const float x = (r[i] * wp[i]) * ri;
      xs[xs_index(tid + 256 * i)] = x;
      if (PRO == PRO_RESID_NORM && blockIdx.x == 0 && a.x_out) a.x_out[tid + 256 * i] = x;
    }
  // the LM head carrying k_final's work also carries its step of the state
  if (PRO == PRO_RESID_NORM && blockIdx.x == 0 && tid == 0 && a.st_advance) {
    a.st_advance->pos += 1;
    a.st_advance->cursor += 1;
  }
}

// ---------------------------------------------------------------------------
// Q8_0 dequant-GEMV, one row group per block (used with CI = 1: the tied LM
// head, 64 rows per block). Block = 256 threads = 4 wavefronts on one group
// of GR rows; lane l holds slot l of each item (row l % GR, pair-column phase
// l / GR). Wave w takes items w, w+4, ... of the group. Up to kStepsInFlight
// items per wave are issued at kernel entry, before the prologue (weights
// never depend on x); longer rows continue with a two-item prefetch.
// ---------------------------------------------------------------------------
template <int PRO, int EPI, int CI, int kStepsInFlight>
__global__ __launch_bounds__(256) void k_gemv(GemvArgs a) {
  constexpr int GR = 64 / CI;
  extern __shared__ float4 xs4[];
  float* xs = (float*)xs4;
  __shared__ float red[4][GR];
  __shared__ float sh4[4];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int g = blockIdx.x;
  const int cp = lane / GR;
  const int Kp = a.Kp, KpS = a.KpS;
  const uint8_t* base = a.W + (size_t)g * KpS * kColBytes;

  Pair st[kStepsInFlight];
#pragma unroll
  for (int i = 0; i < kStepsInFlight; ++i) {
    const int s = wv + 4 * i;
    if (s < KpS && s * CI + cp < Kp) load_planes(base + (size_t)s * kColBytes, lane, st[i]);
  }

  gemv_prologue<PRO>(a, xs, Kp * 64, sh4);
  __syncthreads();

  float acc = 0.f;
#pragma unroll
  for (int i = 0; i < kStepsInFlight; ++i) {
    const int s = wv + 4 * i;
    const int c = s * CI + cp;
    if (s < KpS && c < Kp) acc = dot_pair(st[i], xs + c * kXPad, acc);
  }
  int s = wv + 4 * kStepsInFlight;
  if (s < KpS) {
    Pair cur, nxt;
    if (s * CI + cp < Kp) load_planes(base + (size_t)s * kColBytes, lane, cur);
    if (s + 4 < KpS && (s + 4) * CI + cp < Kp) load_planes(base + (size_t)(s + 4) * kColBytes, lane, nxt);
    for (; s < KpS; s += 4) {
      Pair nn;
      const int s3 = s + 8;
      if (s3 < KpS && s3 * CI + cp < Kp) load_planes(base + (size_t)s3 * kColBytes, lane, nn);
      const int c = s * CI + cp;
      if (c < Kp) acc = dot_pair(cur, xs + c * kXPad, acc);
      cur = nxt;
      nxt = nn;
    }
  }
  // the CI column phases of a row sit in lanes r, r+GR, ...: butterfly sum
#pragma unroll
  for (int m = GR; m < 64; m <<= 1) acc += __shfl_xor(acc, m, 64);
  if (lane < GR) red[wv][lane] = acc;
  __syncthreads();
  if (wv != 0) return;
  const float r = lane < GR ? ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane] : 0.f;
  if (EPI == EPI_OUT) {
    if (lane < GR) a.out[g * GR + lane] = r;
  } else {
    // gate rows g*GR/2 + i sit in lanes 0..GR/2-1, the matching up rows in GR/2..GR-1
    const float up = __shfl(r, lane + GR / 2, 64);
    if (lane < GR / 2) a.act_out[g * (GR / 2) + lane] = gelu_mul(r, up);
  }
}

// ---------------------------------------------------------------------------
// Q8_0 dequant-GEMV over balanced ranges of row groups (used with CI = 8 or 2:
// QKV, O, gate/up, down). Block b owns groups [b G / nb, (b+1) G / nb); their
// items (memory-contiguous, KpS per group) are split evenly over the W
// waves. Every load is issued unconditionally (indices clamped into range)
// so the wait counters stay exact: the prologue's vector loads go first, then
// all NIF weight items of the wave, and the prologue only waits for its own
// loads. Dot products accumulate per lane while a wave stays in one group;
// one butterfly over the CI column phases per group lands the row sums in
// the wave's LDS slots, and a fixed-order sum over the waves gives the rows
// (deterministic). Prologue reductions run on the DPP network.
// ---------------------------------------------------------------------------
constexpr size_t kDecStatOff = (size_t)kDecMaxChunks * kAttnMaxQ * kHeadDim;   // (m, l) after the o block

constexpr int kMgRows = 256;   // rows one block may own
template <int PRO, int EPI, int CI, int W, int NIF, int EPT>
__global__ __launch_bounds__(64 * W) void k_gemv_mg(GemvArgs a) {
  // the prologue (x from the previous kernel's output: a latency chain of
  // loads and block reductions) runs at raised wave priority over the other
  // block's dot products on the CU (0.7797 -> 0.7780 ms per 1B token)
  __builtin_amdgcn_s_setprio(1);
  constexpr int GR = 64 / CI;
  constexpr int NT = 64 * W;
  extern __shared__ float4 xs4[];
  float* xs = (float*)xs4;
  __shared__ float red[W][kMgRows];
  __shared__ float shw[2][W];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int cp = lane / GR;
  const int Kp = a.Kp, KpS = a.KpS, K = Kp * 64;
  const int G = a.N / GR;
  const int b = blockIdx.x, nb = gridDim.x;
  const int g0 = (int)(((long long)b * G) / nb), g1 = (int)(((long long)(b + 1) * G) / nb);
  const int i0 = g0 * KpS, ni = (g1 - g0) * KpS;
  const int wi0 = i0 + (wv * ni) / W, wi1 = i0 + ((wv + 1) * ni) / W;
  const int K4 = K / 4;   // thread t owns the float4 chunks t + NT i (i < EPT) of x

  // Lanes of a padding column phase (c >= Kp, the tail item of a row group
  // when Kp % CI != 0) load the phase-0 lane of their row instead: the same
  // cache lines, so the padding bytes are not fetched (their products are
  // masked below).
  auto issue_weights = [&](Pair* w) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < NIF; ++k) {
      const int it = max(min(wi0 + k, wi1 - 1), i0);
      const int sp = it % KpS;
      const int ll = sp * CI + cp < Kp ? lane : (lane & (GR - 1));
      load_planes(a.W + (size_t)it * kColBytes, ll, w[k]);
    }
  };
  Pair st[NIF];
  // 1. prologue loads (16 bytes per lane, clamped indices: always issued)
  float4 v[EPT], res[EPT], wq[EPT], wp[EPT];
  // PRO_ATTN_MERGE: thread t merges x[4t .. 4t+3] (head t / 64) from the
  // first 16 chunk partials (more are merged in batches of 16 below)
  constexpr int kMB = 16;
  float am_m[kMB], am_l[kMB];
  float4 am_o[kMB];
  int nch = 0, ahd = 0;
  if (PRO == PRO_ATTN_MERGE) {
    issue_weights(st);
    nch = a.attn_chunks;   // every chunk of the launch, empty ones included: no wait for the position
    // head of this wave (uniform): its (max, sum) pairs come through scalar loads
    ahd = __builtin_amdgcn_readfirstlane(min(wv, K / kHeadDim - 1));
#pragma unroll
    for (int k = 0; k < kMB; ++k) {
      const int c = min(k, nch - 1);
      const float2 ml = *(const float2*)(a.attn_part + kDecStatOff + ((size_t)c * kAttnMaxQ + ahd) * 2);
      am_m[k] = ml.x;
      am_l[k] = ml.y;
      am_o[k] = *(const float4*)(a.attn_part + ((size_t)c * kAttnMaxQ + ahd) * kHeadDim + 4 * (tid & 63));
    }
  } else if (PRO == PRO_EMBED_NORM) {
    const int cur = a.st->cursor;
    const int token = cur < 0 ? a.st->token : a.tokens[cur];
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int c = min(tid + NT * i, K4 - 1);
      v[i] = make_float4(embed_elem(a, token, 4 * c), embed_elem(a, token, 4 * c + 1),
                         embed_elem(a, token, 4 * c + 2), embed_elem(a, token, 4 * c + 3));
      wp[i] = ((const float4*)a.w_pre)[c];
    }
  } else {
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int c = min(tid + NT * i, K4 - 1);
      if (PRO == PRO_NONE) {
        v[i] = ((const float4*)a.x)[c];
      } else {
        v[i] = ((const float4*)a.pre_vec)[c];
        res[i] = ((const float4*)a.pre_res)[c];
        wq[i] = ((const float4*)a.w_post)[c];
        wp[i] = ((const float4*)a.w_pre)[c];
      }
    }
  }
  // 2. this wave's weight items (clamped into the block's range); with
  // ATTN_MERGE they went out first, ahead of the position-dependent chunk loads
  if (PRO != PRO_ATTN_MERGE) issue_weights(st);
  for (int i = tid; i < W * kMgRows; i += NT) (&red[0][0])[i] = 0.f;

  // 3. prologue -> x in LDS
  auto has = [&](int i) { return tid + NT * i < K4; };
  auto sq4 = [](float4 q, float acc) {
    acc = fmaf(q.x, q.x, acc);
    acc = fmaf(q.y, q.y, acc);
    acc = fmaf(q.z, q.z, acc);
    return fmaf(q.w, q.w, acc);
  };
  if (PRO == PRO_NONE) {
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if (has(i)) *(float4*)&xs[xs_index(4 * (tid + NT * i))] = v[i];
  } else if (PRO == PRO_ATTN_MERGE) {
    // chunk weights 2^(m_c - M) (maxima in log2 units) with M the running
    // max, in chunk order
    float M = -INFINITY;
#pragma unroll
    for (int k = 0; k < kMB; ++k)
      if (k < nch) M = fmaxf(M, am_m[k]);
    float L = 0.f;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    auto add = [&](int k, float Mx) {
      const float f = __builtin_amdgcn_exp2f(am_m[k] - Mx);
      L = fmaf(f, am_l[k], L);
      acc.x = fmaf(f, am_o[k].x, acc.x);
      acc.y = fmaf(f, am_o[k].y, acc.y);
      acc.z = fmaf(f, am_o[k].z, acc.z);
      acc.w = fmaf(f, am_o[k].w, acc.w);
    };
#pragma unroll
    for (int k = 0; k < kMB; ++k)
      if (k < nch) add(k, M);
    for (int c0 = kMB; c0 < nch; c0 += kMB) {   // spans above 4096 positions
#pragma unroll
      for (int k = 0; k < kMB; ++k) {
        const int c = min(c0 + k, nch - 1);
        const float2 ml = *(const float2*)(a.attn_part + kDecStatOff + ((size_t)c * kAttnMaxQ + ahd) * 2);
        am_m[k] = ml.x;
        am_l[k] = ml.y;
        am_o[k] = *(const float4*)(a.attn_part + ((size_t)c * kAttnMaxQ + ahd) * kHeadDim + 4 * (tid & 63));
      }
      float Mb = M;
#pragma unroll
      for (int k = 0; k < kMB; ++k)
        if (c0 + k < nch) Mb = fmaxf(Mb, am_m[k]);
      const float sc = __builtin_amdgcn_exp2f(M - Mb);
      L *= sc;
      acc.x *= sc;
      acc.y *= sc;
      acc.z *= sc;
      acc.w *= sc;
      M = Mb;
#pragma unroll
      for (int k = 0; k < kMB; ++k)
        if (c0 + k < nch) add(k, M);
    }
    if (4 * tid < K) {
      const float iL = 1.f / L;
      const float4 xo = make_float4(acc.x * iL, acc.y * iL, acc.z * iL, acc.w * iL);
      *(float4*)&xs[xs_index(4 * tid)] = xo;
      if (b == 0) *(float4*)(a.x_out + 4 * tid) = xo;
    }
  } else {
    float4 r[EPT];
    if (PRO == PRO_EMBED_NORM) {
#pragma unroll
      for (int i = 0; i < EPT; ++i) r[i] = v[i];
    } else {   // res = pre_res + norm(pre_vec) * w_post (fusedNormAdd, shaders.ts:415)
      float s1 = 0.f;
#pragma unroll
      for (int i = 0; i < EPT; ++i)
        if (has(i)) s1 = sq4(v[i], s1);
      s1 = wave_sum_dpp(s1);
      if (lane == 0) shw[0][wv] = s1;
      __syncthreads();
      float t1 = 0.f;
#pragma unroll
      for (int w = 0; w < W; ++w) t1 += shw[0][w];
      const float ri1 = rsq(t1 / (float)K + a.eps);
#pragma unroll
      for (int i = 0; i < EPT; ++i)
        r[i] = make_float4(res[i].x + (v[i].x * wq[i].x) * ri1, res[i].y + (v[i].y * wq[i].y) * ri1,
                           res[i].z + (v[i].z * wq[i].z) * ri1, res[i].w + (v[i].w * wq[i].w) * ri1);
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if (has(i)) ss = sq4(r[i], ss);
    if (b == 0) {
#pragma unroll
      for (int i = 0; i < EPT; ++i)
        if (has(i)) {
          ((float4*)a.res_out)[tid + NT * i] = r[i];
          if (PRO == PRO_RESID_NORM && a.hist_out) ((float4*)a.hist_out)[tid + NT * i] = r[i];
        }
    }
    ss = wave_sum_dpp(ss);
    if (lane == 0) shw[1][wv] = ss;
    __syncthreads();
    float t2 = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) t2 += shw[1][w];
    const float ri = rsq(t2 / (float)K + a.eps);   // rmsNorm, shaders.ts:50-53
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if (has(i))
        *(float4*)&xs[xs_index(4 * (tid + NT * i))] =
            make_float4((r[i].x * wp[i].x) * ri, (r[i].y * wp[i].y) * ri, (r[i].z * wp[i].z) * ri,
                        (r[i].w * wp[i].w) * ri);
  }
  __syncthreads();

  // 4. dot products in item order
  __builtin_amdgcn_s_setprio(0);
  float acc = 0.f;
  int gcur = wi0 / KpS - g0;
  auto flush = [&](int gl) {
    float t = acc;
#pragma unroll
    for (int m = GR; m < 64; m <<= 1) t += __shfl_xor(t, m, 64);
    if (lane < GR) red[wv][gl * GR + lane] = t;
  };
#pragma unroll
  for (int k = 0; k < NIF; ++k) {
    const int it = wi0 + k;
    const int g = it / KpS, s = it - g * KpS;
    const int c = s * CI + cp;
    float d = dot_pair(st[k], xs + min(c, Kp - 1) * kXPad, 0.f);
    d = (c < Kp && it < wi1) ? d : 0.f;
    if (it < wi1 && g - g0 != gcur) {
      flush(gcur);
      gcur = g - g0;
      acc = 0.f;
    }
    acc += d;
  }
  if (wi1 > wi0) flush(gcur);
  __syncthreads();

  // 5. fixed-order sum over the waves; epilogue
  const int nrows = (g1 - g0) * GR;
  for (int t = tid; t < nrows; t += NT) {
    float r = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) r += red[w][t];
    if (EPI == EPI_OUT) {
      a.out[g0 * GR + t] = r;
    } else {
      // gate rows of a group in its first GR/2 slots, the matching up rows next
      const int rr = t % GR;
      if (rr < GR / 2) {
        float up = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) up += red[w][t + GR / 2];
        a.act_out[(g0 * GR + t - rr) / 2 + rr] = gelu_mul(r, up);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Decode attention (one KV head, head_dim 256, up to 4 query heads). Block
// (x, y) = (chunk of positions, query head); the chunk partials (max, sum, o)
// go to memory and the attention output projection merges them in its
// prologue (no cross-block step here). Chunks: 32 * ceil(span / (32 * mc))
// positions, mc = 16 while the span is <= 4096 (else kDecMaxChunks), so the
// merge reads at most 16 partials per head at Gemma-3 1B lengths. Blocks past
// the span write empty partials (m = -inf), so the merge always reads the
// launch's chunk count and does not wait for the position. One head
// per block keeps each wave's serial chain short (the pass is bound by
// instruction latency, not by the K/V bytes).
//
// Per block: QK-norm + NEOX RoPE of query head y and, in the chunk holding
// `pos`, of the key; that chunk's head-0 block also stores k/v to the cache
// (fusedPerHeadNormRope + kvCacheStore, shaders.ts:209-227, 420-467). Wave w
// then runs passes of 8 positions t0 + 32 p + 8 w + i: lane (i, o) =
// (lane / 8, lane % 8) holds key dims 4 (o + 8 j) .. +3 (j < 8), so each key
// load instruction reads 8 whole 128-byte segments, and the dot product
// finishes with a butterfly over the 8 lanes of a position; lane l holds
// value dims 4 l .. 4 l + 3 for the weighted sum (shaders.ts:229-325).
// Softmax statistics are kept online per pass; all reductions run on DPP,
// probabilities reach every lane through readlane.
// ---------------------------------------------------------------------------
template <int HPB>
__global__ __launch_bounds__(256) void k_attn_dec(AttnArgs a) {
  __shared__ float4 qs4[HPB][64];
  __shared__ float4 ks4[64], vs4[64];
  __shared__ float4 wo[4][HPB][64];
  __shared__ float wm[4][HPB], wl[4][HPB];

  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int nq = a.n_q;
  const int nqd = nq * kHeadDim;
  const int h0 = HPB == 1 ? (int)blockIdx.y : 0;   // first query head of the block
  // loads that do not depend on the position: q of the head this wave
  // normalises (HPB = 1: wave 0, head h0; else wave w, head w), this token's
  // k and v, the norm weights
  const int qh = HPB == 1 ? h0 : min(wv, nq - 1);
  float hx[4], kx[4], nwt[4], kwt[4], cs[2], sn[2];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    hx[i] = a.qkv[qh * kHeadDim + lane + 64 * i];
    nwt[i] = a.q_norm[lane + 64 * i];
    kx[i] = a.qkv[nqd + lane + 64 * i];
    kwt[i] = a.k_norm[lane + 64 * i];
  }
  const float4 vme = *(const float4*)(a.qkv + nqd + kHeadDim + 4 * lane);
  const int pos = a.st->pos;
  int t_lo, ch, nch;
  dec_span(pos, a.window, gridDim.x, &t_lo, &ch, &nch);
  const int b = blockIdx.x;
  if (b >= nch) {   // past the span: empty partials, so that the merge needs no position
#pragma unroll
    for (int hh = 0; hh < HPB; ++hh) {
      const int h = h0 + hh;
      if (h >= nq) break;
      if (tid < 64) *(float4*)(a.part + ((size_t)b * kAttnMaxQ + h) * kHeadDim + 4 * tid) = make_float4(0.f, 0.f, 0.f, 0.f);
      if (tid == 0) {
        a.part[kDecStatOff + ((size_t)b * kAttnMaxQ + h) * 2] = -INFINITY;
        a.part[kDecStatOff + ((size_t)b * kAttnMaxQ + h) * 2 + 1] = 0.f;
      }
    }
    return;
  }
  const int t0 = t_lo + b * ch;
  const int t1 = min(t0 + ch, pos + 1);
  const int npass = (t1 - t0 + 31) >> 5;
  const int kv_last = max(pos - 1, 0);     // cache rows [0, pos) hold earlier tokens
  const int pl = lane >> 3, oc = lane & 7;
  const bool holder = (b == nch - 1);      // this block's chunk contains pos

  // loads of pass p: key rows in the score layout, value rows in the PV
  // layout; rows are clamped into the cache (positions >= t1 are masked,
  // pos itself is substituted from LDS). Nontemporal: with HPB = 1 each row
  // is read by the four head blocks of its chunk (same XCD) within one launch.
  float4 kr[8], vr[8];
  auto load_k = [&](int p) {
    const int t = min(t0 + 32 * p + 8 * wv + pl, kv_last);
    const f32x4* kp = (const f32x4*)(a.k_cache + (size_t)t * kHeadDim);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const f32x4 v = __builtin_nontemporal_load(kp + oc + 8 * j);
      kr[j] = make_float4(v.x, v.y, v.z, v.w);
    }
  };
  auto load_v = [&](int p) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int t = min(t0 + 32 * p + 8 * wv + i, kv_last);
      const f32x4 v = __builtin_nontemporal_load((const f32x4*)(a.v_cache + (size_t)t * kHeadDim) + lane);
      vr[i] = make_float4(v.x, v.y, v.z, v.w);
    }
  };
  // this position's RoPE row, then the first pass of K / V rows (the norm
  // below waits only for the loads issued before these)
  const float* rt = a.rope + (size_t)pos * kHeadDim;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    cs[j] = rt[lane + 64 * j];
    sn[j] = rt[kHeadDim / 2 + lane + 64 * j];
  }
  load_k(0);
  load_v(0);

  // RMSNorm + NEOX RoPE of one head: lane owns dims lane + 64 i; pairs (i, i + 128)
  auto norm_rope = [&](float* x, const float* w, float* dst) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) ss = fmaf(x[i], x[i], ss);
    ss = wave_sum_dpp(ss);
    const float ri = rsq(ss / (float)kHeadDim + a.eps);
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = (x[i] * w[i]) * ri;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float x0 = x[j], x1 = x[j + 2];
      dst[lane + 64 * j] = x0 * cs[j] - x1 * sn[j];
      dst[lane + 64 * j + 128] = x0 * sn[j] + x1 * cs[j];
    }
  };
  if (HPB == 1) {
    if (wv == 0) norm_rope(hx, nwt, (float*)qs4[0]);
  } else if (wv < HPB) {
    if (wv < nq) norm_rope(hx, nwt, (float*)qs4[wv]);
    else qs4[wv][lane] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  if (holder && wv == 1) norm_rope(kx, kwt, (float*)ks4);
  if (holder && wv == 2) vs4[lane] = vme;
  __syncthreads();
  if (holder && h0 == 0) {
    a.k_cache[(size_t)pos * kHeadDim + tid] = ((const float*)ks4)[tid];
    a.v_cache[(size_t)pos * kHeadDim + tid] = ((const float*)vs4)[tid];
  }
  if (b == 0 && a.q_dbg && tid < 64)
#pragma unroll
    for (int hh = 0; hh < HPB; ++hh)
      if (h0 + hh < nq) *(float4*)(a.q_dbg + (h0 + hh) * kHeadDim + 4 * tid) = qs4[hh][tid];

  float4 qr[HPB][8];
#pragma unroll
  for (int hh = 0; hh < HPB; ++hh)
#pragma unroll
    for (int j = 0; j < 8; ++j) qr[hh][j] = qs4[hh][oc + 8 * j];

  // scores in log2 units: the online softmax and every merge of its
  // partials (chunk maxima in the same units) run in base 2 on v_exp_f32
  const float sl2 = a.scale * 1.4426950408889634f;
  float m[HPB], l[HPB];
  float4 o4[HPB];
#pragma unroll
  for (int hh = 0; hh < HPB; ++hh) {
    m[hh] = -INFINITY;
    l[hh] = 0.f;
    o4[hh] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  for (int p = 0; p < npass; ++p) {
    const int tb = t0 + 32 * p + 8 * wv;       // first position of this wave's pass
    const int t = tb + pl;
    if (t == pos) {
#pragma unroll
      for (int j = 0; j < 8; ++j) kr[j] = ks4[oc + 8 * j];
    }
    float sc[HPB];
#pragma unroll
    for (int hh = 0; hh < HPB; ++hh) {
      float d = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        d = fmaf(qr[hh][j].x, kr[j].x, d);
        d = fmaf(qr[hh][j].y, kr[j].y, d);
        d = fmaf(qr[hh][j].z, kr[j].z, d);
        d = fmaf(qr[hh][j].w, kr[j].w, d);
      }
      d = group8_sum(d);
      sc[hh] = (t < t1 && h0 + hh < nq) ? d * sl2 : -INFINITY;
    }
    if (p + 1 < npass) load_k(p + 1);          // next pass (wave-uniform)
    float pr[HPB], alpha[HPB];
#pragma unroll
    for (int hh = 0; hh < HPB; ++hh) {
      const float mx = across8_max(sc[hh]);
      const float mn = fmaxf(m[hh], mx);
      alpha[hh] = (m[hh] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m[hh] - mn);
      pr[hh] = (sc[hh] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(sc[hh] - mn);
      l[hh] = fmaf(l[hh], alpha[hh], across8_sum(pr[hh]));
      m[hh] = mn;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (tb + i == pos) vr[i] = vs4[lane];
#pragma unroll
    for (int hh = 0; hh < HPB; ++hh) {
      o4[hh].x *= alpha[hh];
      o4[hh].y *= alpha[hh];
      o4[hh].z *= alpha[hh];
      o4[hh].w *= alpha[hh];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float pv = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, pr[hh]), 8 * i));
        o4[hh].x = fmaf(pv, vr[i].x, o4[hh].x);
        o4[hh].y = fmaf(pv, vr[i].y, o4[hh].y);
        o4[hh].z = fmaf(pv, vr[i].z, o4[hh].z);
        o4[hh].w = fmaf(pv, vr[i].w, o4[hh].w);
      }
    }
    if (p + 1 < npass) load_v(p + 1);
  }

  // merge the four waves (fixed order) into the chunk's (max, sum, o) per
  // head: one barrier, then every lane of wave 0 forms the weights itself
#pragma unroll
  for (int hh = 0; hh < HPB; ++hh) {
    wo[wv][hh][lane] = o4[hh];
    if (lane == 0) {
      wm[wv][hh] = m[hh];
      wl[wv][hh] = l[hh];
    }
  }
  __syncthreads();
  if (tid < 64) {
#pragma unroll
    for (int hh = 0; hh < HPB; ++hh) {
      const int h = h0 + hh;
      if (h >= nq) break;
      const float M = fmaxf(fmaxf(wm[0][hh], wm[1][hh]), fmaxf(wm[2][hh], wm[3][hh]));
      float L = 0.f;
      float4 O = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float f = wm[w][hh] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(wm[w][hh] - M);
        L = fmaf(f, wl[w][hh], L);
        const float4 v = wo[w][hh][tid];
        O.x = fmaf(f, v.x, O.x);
        O.y = fmaf(f, v.y, O.y);
        O.z = fmaf(f, v.z, O.z);
        O.w = fmaf(f, v.w, O.w);
      }
      *(float4*)(a.part + ((size_t)b * kAttnMaxQ + h) * kHeadDim + 4 * tid) = O;
      if (tid == 0) {
        a.part[kDecStatOff + ((size_t)b * kAttnMaxQ + h) * 2] = M;
        a.part[kDecStatOff + ((size_t)b * kAttnMaxQ + h) * 2 + 1] = L;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Long-span decode attention merge: per query head, the softmax-weighted sum
// of the launch's nch chunk partials, o = sum_c f_c o_c / sum_c f_c l_c with
// f_c = 2^(m_c - max_c m_c) (maxima in log2 units; empty chunks have m_c =
// -inf, f_c = 0), written
// to attn_out, the O GEMV's input. Block (32-dim slice, head); thread (chunk
// group tid / 32 of 8, dim tid % 32) sums chunks g, g + 8, ..., then the
// groups add in a fixed order (deterministic).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_attn_merge(AttnArgs a, int nch) {
  constexpr int kPer = kDecMaxChunks / 8;   // chunks per thread
  __shared__ float gmax[8], gl[8], go[8][32];
  const int tid = threadIdx.x, cg = tid >> 5, d = tid & 31;
  const int h = blockIdx.y, dim = 32 * blockIdx.x + d;
  const float* ml = a.part + kDecStatOff;
  // every partial of this thread is loaded before any is used (the loads
  // are independent; one at a time each would wait a full memory latency)
  float2 st[kPer];
  float ov[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int c = min(cg + 8 * k, nch - 1);
    st[k] = *(const float2*)(ml + ((size_t)c * kAttnMaxQ + h) * 2);
    ov[k] = a.part[((size_t)c * kAttnMaxQ + h) * kHeadDim + dim];
  }
  float mx = -INFINITY;
#pragma unroll
  for (int k = 0; k < kPer; ++k)
    if (cg + 8 * k < nch) mx = fmaxf(mx, st[k].x);
  if (d == 0) gmax[cg] = mx;
  __syncthreads();
  float M = gmax[0];
#pragma unroll
  for (int i = 1; i < 8; ++i) M = fmaxf(M, gmax[i]);
  float L = 0.f, O = 0.f;
#pragma unroll
  for (int k = 0; k < kPer; ++k)
    if (cg + 8 * k < nch) {
      const float f = __builtin_amdgcn_exp2f(st[k].x - M);
      L = fmaf(f, st[k].y, L);
      O = fmaf(f, ov[k], O);
    }
  go[cg][d] = O;
  if (d == 0) gl[cg] = L;
  __syncthreads();
  if (cg == 0) {
    float So = 0.f, Sl = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      So += go[i][d];
      Sl += gl[i];
    }
    a.attn_out[h * kHeadDim + dim] = So / Sl;
  }
}

// ---------------------------------------------------------------------------
// End of a forward pass: hidden = residual + norm(down) * post_ffw_norm, then
// normed = rmsNorm(hidden, output_norm) (engine.ts:794-801); advance pos.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_final(FinalArgs a) {
  __shared__ float sh4[4];
  const int tid = threadIdx.x, H = a.H;
  const int n = (H - tid + 255) / 256;
  float v[8], res[8], wq[8], wo[8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (i < n) {
      const int e = tid + 256 * i;
      v[i] = a.pre_vec[e];
      for (int p = 1; p < a.pre_planes; ++p) v[i] += a.pre_vec[p * a.pre_stride + e];
      res[i] = a.pre_res[e];
      wq[i] = a.w_post[e];
      wo[i] = a.w_out[e];
    }
  float s1 = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (i < n) s1 = fmaf(v[i], v[i], s1);
  const float ri1 = rsq(block_sum256(s1, sh4) / (float)H + a.eps);
  float s2 = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (i < n) {
      const float r = res[i] + (v[i] * wq[i]) * ri1;
      v[i] = r;
      a.hidden[tid + 256 * i] = r;
      if (a.hist_out) a.hist_out[tid + 256 * i] = r;
      s2 = fmaf(r, r, s2);
    }
  const float ri2 = rsq(block_sum256(s2, sh4) / (float)H + a.eps);
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (i < n) a.normed[tid + 256 * i] = (v[i] * wo[i]) * ri2;
  if (tid == 0) {
    a.st->pos += 1;
    a.st->cursor += 1;
  }
}

// ---------------------------------------------------------------------------
// Token selection over the logits (engine.ts:823-901).
// k_select1: per stride class c = i mod 256, the first index of the class
// maximum over the block's stripes (strict >, init (-1e30, 0)), as in
// argmax/topk256 (shaders.ts:337-347, 371-381).
// k_select2: merge stripes in order -> topk256; then either the argmax
// halving tree (shaders.ts:351-357) or the host sampler (engine.ts:862-901):
// repetition penalty in f64, stable descending sort, f32-stored exp, f64
// sums, top-p cutoff, walk with the injected draw u.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_select1(SelectArgs a) {
  const int tid = threadIdx.x;
  const int nb = gridDim.x;
  const int stripes = (a.V + 255) / 256;
  const int per = (stripes + nb - 1) / nb;
  const int j0 = blockIdx.x * per, j1 = min(j0 + per, stripes);
  float m = -1e30f;
  uint32_t id = 0;
  for (int j = j0; j < j1; j += 32) {
    float v[32];
#pragma unroll
    for (int k = 0; k < 32; ++k) {
      const int i = (j + k) * 256 + tid;
      v[k] = (j + k < j1 && i < a.V) ? a.logits[i] : -INFINITY;
    }
#pragma unroll
    for (int k = 0; k < 32; ++k)
      if (v[k] > m) { m = v[k]; id = (uint32_t)((j + k) * 256 + tid); }
  }
  a.cand_val[blockIdx.x * 256 + tid] = m;
  a.cand_id[blockIdx.x * 256 + tid] = id;
}

__global__ __launch_bounds__(256) void k_select2(SelectArgs a, int nb) {
  __shared__ SelShared sh;
  const int tid = threadIdx.x;
  float m = -1e30f;
  uint32_t id = 0;
  for (int b0 = 0; b0 < nb; b0 += 32) {
    float v[32];
    uint32_t ix[32];
#pragma unroll
    for (int k = 0; k < 32; ++k) {
      v[k] = b0 + k < nb ? a.cand_val[(b0 + k) * 256 + tid] : -INFINITY;
      ix[k] = b0 + k < nb ? a.cand_id[(b0 + k) * 256 + tid] : 0u;
    }
#pragma unroll
    for (int k = 0; k < 32; ++k)
      if (v[k] > m) { m = v[k]; id = ix[k]; }
  }
  a.top[2 * tid] = __float_as_uint(m);
  a.top[2 * tid + 1] = id;
  const int token = select_token(sh, m, id, true, a.in_use ? a.in : sample_of(a.st), a.seen, a.V);
  if (tid == 0) {
    a.st->out_token = token;
    if (a.host_out) a.host_out[0] = token;
    if (a.auto_add && token >= 0 && token < a.V) {
      a.seen[token >> 5] |= 1u << (token & 31);
      a.st->seen_count += 1;
    }
  }
}

// ---------------------------------------------------------------------------
// Batched prefill attention (no reference counterpart: the reference attends
// one prompt token per decode pass, engine.ts:923-928, with the
// scores / softmax / weighted V of shaders.ts:229-325).
//
// k_rows_kv leaves q, k and v as bf16 hi / lo in MFMA operand order, so the
// splits are made once per value and staging is a plain copy. Block (x = key
// chunk, y = query tile) covers 16 RT prompt rows (32, or 16 where blocks are
// few: prefill_plan) with four waves, one per query head, each alone on its
// SIMD: a wave holds its 32 rows' q (128 registers) and output (128), so every
// K and V operand read from LDS feeds two row tiles; 16-row waves, two per
// SIMD, would read 170 bytes of LDS per MFMA cycle of a CU, above its 128.
// Long spans (global layers of 32760 ids, 1B shape): matrix cores busy 61% of
// the cycles at 1.85 GHz; 27% in 16-row tiles over a 512 window. All attention
// of that prefill with its merge takes 29.9 ms, 49.0 with the kernel that split
// K and V in every block.
//   S^T = K Q^T  on v_mfma_f32_16x16x32_bf16, q scaled by log2(e)/16 before
//                its split: per 32 dims the products hi.hi, lo.hi and hi.lo,
//                fp32 accumulate (the dropped lo.lo term is below 2^-16
//                |k| |q|). Operand row c of key tile j (j < 2) is key
//                8 (c / 4) + 4 j + c % 4, so lane l holds S^T[key 8 g + 4 j
//                + r][row l % 16] for r < 4, g = lane / 16.
//   O += P V     on v_mfma_f32_16x16x32_bf16, the same three products of
//                bf16 hi + lo splits: A = P from lane l's own S^T registers
//                (keys 8 g .. 8 g + 7 in order), B = V^T per dim; tile 2 k +
//                e column c is dim 32 k + 2 c + e, so lane l holds O[row
//                4 g + r] of adjacent dims and stores them as one word.
// Pipeline of 32-key tiles, one barrier each (pf_schedule_run, and one more
// behind the first tile's scores): while tile t's exponentials and
// splits run in the issue slots between the MFMAs of tile t + 1's scores and
// its P V follows, the next K and V tiles go to the other LDS stage by DMA
// (64 KB per tile, two stages, no registers).
// The softmax reference of a row (l % 16, per lane) moves only when a tile's
// maximum exceeds it by more than 2^8, so O is rescaled rarely; every
// probability is relative to the same reference until then, in fp32. A query
// tile whose span fits one chunk writes O / l; otherwise every chunk leaves
// (reference, l, O) in `part` for k_attn_pf_merge.
// ---------------------------------------------------------------------------

// x = hi + lo + e with hi = bf16(x), lo = bf16(x - hi), |e| <= 2^-17 |x|
// (the input format of the prefill GEMMs).
__device__ __forceinline__ void split_bf16(float x, uint16_t* hi, uint16_t* lo) {
  const __bf16 h = (__bf16)x;
  *hi = __builtin_bit_cast(uint16_t, h);
  *lo = __builtin_bit_cast(uint16_t, (__bf16)(x - (float)h));
}

typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ int a_slot(int e);   // below, with the GEMM's A rows
// The same split for two values at once, as packed bf16 pairs (element 0 in
// the low half): one packed conversion for hi, hi widened back by a shift and
// a mask, one packed conversion for lo.
__device__ __forceinline__ void split2_bf16(float x0, float x1, uint32_t& hi, uint32_t& lo) {
  hi = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2v){x0, x1}, bf16x2));
  const float h0 = __uint_as_float(hi << 16), h1 = __uint_as_float(hi & 0xffff0000u);
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2v){x0 - h0, x1 - h1}, bf16x2));
}
// bf16 hi / lo of four values as packed pairs
__device__ __forceinline__ void split4_bf16(float x0, float x1, float x2, float x3, bf16x4& hi, bf16x4& lo) {
  uint32_t h[2], l[2];
  split2_bf16(x0, x1, h[0], l[0]);
  split2_bf16(x2, x3, h[1], l[1]);
  hi = __builtin_bit_cast(bf16x4, h);
  lo = __builtin_bit_cast(bf16x4, l);
}

// max / sum with lane ^ 16 and lane ^ 32 on the gfx950 half-row and
// half-wave swaps (VALU) instead of ds_bpermute shuffles (an LDS round trip)
__device__ __forceinline__ float pf_xor16_max(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pf_xor32_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

__device__ __forceinline__ bf16x8 lds_bf16x8(const uint8_t* p) {
  return __builtin_bit_cast(bf16x8, *(const u32x4*)p);
}

constexpr int kPfKeys = 32;                    // keys per tile
constexpr int kPfTile = kPfKeys * 1024;        // bytes of a K (or V) tile: 256 dims, hi and lo
static_assert(kKvTileBytes == 2 * kPfTile, "a tile of the planes is its K part, then its V part");

__device__ __forceinline__ int pf_key_lo(const AttnArgs& a, int pos) {
  return a.window > 0 ? max(0, pos - a.window + 1) : 0;
}

// Key tiles [*t0, *t1] of query tile qt (16 pf_rt rows), in *nkc chunks of
// pf_chunk tiles.
__device__ __forceinline__ void pf_tile_span(const AttnArgs& a, int qt, int* t0, int* t1, int* nkc) {
  const int rows = 16 * a.pf_rt;
  const int p_first = a.pf_start + qt * rows;
  const int p_last = a.pf_start + min(qt * rows + rows - 1, a.pf_rows - 1);
  *t0 = pf_key_lo(a, p_first) / kPfKeys;
  *t1 = p_last / kPfKeys;
  *nkc = (*t1 - *t0 + a.pf_chunk) / a.pf_chunk;
}

template <int RT>
__global__ __launch_bounds__(256, 1) void k_attn_pf(AttnArgs a) {
  constexpr int kPfRows = 16 * RT;
  __shared__ __align__(16) uint8_t Ks[2][kPfTile];
  __shared__ __align__(16) uint8_t Vs[2][kPfTile];
  const int tid = threadIdx.x, lane = tid & 63, h = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c16 = lane & 15;
  const int M = a.pf_rows, nq = a.n_q, qt = blockIdx.y, kc = blockIdx.x;
  int t0, t1, nkc;
  pf_tile_span(a, qt, &t0, &t1, &nkc);
  if (kc >= nkc) return;
  const int tb = t0 + kc * a.pf_chunk, te = min(tb + a.pf_chunk, t1 + 1);   // key tiles [tb, te)
  // staging: a K or V tile goes to LDS as it is, by DMA: wave w copies KBs
  // 8 w .. 8 w + 7, each instruction one KB (lane l's 16 bytes to slot l of
  // M0 + offset; the offset counts on both sides). Inline asm, because the
  // compiler would wait for every DMA in flight before any LDS read; arrived()
  // waits for them explicitly before the barrier that precedes their readers.
  auto stage = [&](int t, int part, int st) __attribute__((always_inline)) {
    const uint8_t* src = a.kv_planes + (size_t)t * kKvTileBytes + part * kPfTile + h * 8192;
    uint8_t* lds = part ? Vs[st] : Ks[st];
    const uint32_t dst = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds + h * 8192;
#pragma unroll
    for (int half = 0; half < 2; ++half)
      asm volatile(
          "s_mov_b32 m0, %0\n\ts_nop 0\n\t"
          "global_load_lds_dwordx4 %1, %2\n\tglobal_load_lds_dwordx4 %1, %2 offset:1024\n\t"
          "global_load_lds_dwordx4 %1, %2 offset:2048\n\tglobal_load_lds_dwordx4 %1, %2 offset:3072"
          ::"s"(__builtin_amdgcn_readfirstlane(dst + half * 4096)), "v"(lane * 16), "s"(src + half * 4096)
          : "memory", "m0");
  };
  auto arrived = []() __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
  pf_schedule_fill(tb, te, stage);

  // q of row tiles RT qt + rt: [tile][head][t][plane][lane][8]; waves past the
  // last head repeat it and write nothing
  bf16x8 qh[RT][8], ql[RT][8];
  const u32x4* qp = (const u32x4*)(a.q_frag + (size_t)(RT * qt * nq + min(h, nq - 1)) * 16 * kHeadDim * 2) + lane;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      qh[rt][t] = __builtin_bit_cast(bf16x8, qp[(size_t)rt * nq * 1024 + t * 128]);
      ql[rt][t] = __builtin_bit_cast(bf16x8, qp[(size_t)rt * nq * 1024 + t * 128 + 64]);
    }

  int prow[RT], plo[RT];      // this lane's rows: position, first key
  bool row_ok[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int row = qt * kPfRows + 16 * rt + c16;
    row_ok[rt] = row < M;
    prow[rt] = a.pf_start + row;
    plo[rt] = pf_key_lo(a, prow[rt]);
  }
  // every key of the tile is valid for all rows: all rows exist, the last
  // key is at most the first row's position, the first key at least the last
  // row's window start
  const int r_first = a.pf_start + qt * kPfRows;
  const bool rows_full = qt * kPfRows + kPfRows <= M;
  const int lo_last = pf_key_lo(a, r_first + kPfRows - 1);
  auto tile_full = [&](int t) {
    return rows_full && t * kPfKeys + kPfKeys - 1 <= r_first && t * kPfKeys >= lo_last;
  };

  f32x4 o[RT][16];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[rt][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m[RT], mb[RT], l[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    m[rt] = -INFINITY;
    mb[rt] = l[rt] = 0.f;
  }
  f32x4 s[RT][2], nx[RT][2];  // [row tile][key tile j]: scores of this and of the next tile
  uint32_t ph[RT][4], pl[RT][4];

  // The wave runs alone on its SIMD, so its instruction order is the schedule:
  // it is written out and pinned slot by slot (fence), a few VALU instructions
  // behind each MFMA or pair, LDS operands read a whole group ahead.
  auto fence = []() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };

  // d[rt][j] = K Q^T of the K tile at kb: 8 dim blocks of 6 slots of RT MFMAs
  auto scores = [&](const uint8_t* kb, f32x4 (&d)[RT][2], auto slot) __attribute__((always_inline)) {
    bf16x8 k[2][4];
    auto read = [&](int t) __attribute__((always_inline)) {
#pragma unroll
      for (int x = 0; x < 4; ++x) k[t & 1][x] = lds_bf16x8(kb + (t * 4 + x) * 1024 + lane * 16);
    };
    read(0);
    fence();
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      if (t < 7) read(t + 1);
      fence();
#pragma unroll
      for (int q = 0; q < 6; ++q) {   // (product, key tile); both row tiles
        const int pr = q >> 1, j = q & 1;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
          d[rt][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[t & 1][2 * j + (pr == 1)], pr == 2 ? ql[rt][t] : qh[rt][t],
                                                             t == 0 && pr == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : d[rt][j], 0, 0, 0);
        slot(t * 6 + q);
        fence();
      }
    }
  };
  // slot q of the softmax of tile t: probabilities 2 (q / 6) and + 1 of the
  // lane's 16 are 2^(s - reference), added to the row's sum and split
  float p0 = 0.f, p1 = 0.f, h0 = 0.f, h1 = 0.f;
  auto probs = [&](int q) __attribute__((always_inline)) {
    if (q >= 24 * RT) return;
    const int pair = q / 6, rt = pair >> 2, j = (pair >> 1) & 1, r = 2 * (pair & 1);
    switch (q % 6) {
      case 0:
        p0 = s[rt][j][r] - mb[rt];
        p1 = s[rt][j][r + 1] - mb[rt];
        break;
      case 1:
        p0 = __builtin_amdgcn_exp2f(p0);
        p1 = __builtin_amdgcn_exp2f(p1);
        break;
      case 2:
        l[rt] += p0;
        l[rt] += p1;
        asm volatile("" : "+v"(l[rt]));
        break;
      case 3:
        ph[rt][pair & 3] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2v){p0, p1}, bf16x2));
        break;
      case 4:
        h0 = __uint_as_float(ph[rt][pair & 3] << 16);
        h1 = __uint_as_float(ph[rt][pair & 3] & 0xffff0000u);
        break;
      case 5:
        pl[rt][pair & 3] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2v){p0 - h0, p1 - h1}, bf16x2));
        asm volatile("" : "+v"(pl[rt][pair & 3]));
        break;
    }
    if (q % 6 < 2) asm volatile("" : "+v"(p0), "+v"(p1));   // or they sink past the MFMAs
  };
  // O += P V of the V tile at vb: 16 dim tiles of 3 slots of RT MFMAs
  auto weighted = [&](const uint8_t* vb, auto slot) __attribute__((always_inline)) {
    bf16x8 v[3][2];
    auto read = [&](int i) __attribute__((always_inline)) {
      v[i % 3][0] = lds_bf16x8(vb + (i * 2) * 1024 + lane * 16);
      v[i % 3][1] = lds_bf16x8(vb + (i * 2 + 1) * 1024 + lane * 16);
    };
    read(0);
    read(1);
    fence();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if (i < 14) read(i + 2);
      fence();
#pragma unroll
      for (int pr = 0; pr < 3; ++pr) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          const u32x4 pf = pr == 1 ? u32x4{pl[rt][0], pl[rt][1], pl[rt][2], pl[rt][3]}
                                   : u32x4{ph[rt][0], ph[rt][1], ph[rt][2], ph[rt][3]};
          o[rt][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, pf), v[i % 3][pr == 2], o[rt][i],
                                                             0, 0, 0);
        }
        slot(3 * i + pr);
        fence();
      }
    }
  };
  // causal / window mask of tile t's scores
  auto mask = [&](int t, f32x4 (&d)[RT][2]) __attribute__((always_inline)) {
    if (tile_full(t)) return;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = t * kPfKeys + 8 * g + 4 * j + r;
          const bool ok = row_ok[rt] && key >= plo[rt] && key <= prow[rt];
          d[rt][j][r] = ok ? d[rt][j][r] : -INFINITY;
        }
  };
  // row maxima of the scores d, one of the lane's 16 per slot, then across
  // the four lane groups
  float mx[RT];
  auto maxima = [&](const f32x4 (&d)[RT][2], int q) __attribute__((always_inline)) {
    const int rt = q >> 3;
    if (q < 8 * RT) mx[rt] = (q & 7) == 0 ? d[rt][0][0] : fmaxf(mx[rt], d[rt][(q >> 2) & 1][q & 3]);
    else if (q < 9 * RT) mx[q - 8 * RT] = pf_xor16_max(mx[q - 8 * RT]);
    else if (q < 10 * RT) mx[q - 9 * RT] = pf_xor32_max(mx[q - 9 * RT]);
  };
  // moves the softmax reference where a row needs it
  auto settle = [&]() __attribute__((always_inline)) {
    bool mv[RT], any = false;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) any |= mv[rt] = mx[rt] > m[rt] + 8.f;
    if (__ballot(any)) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const float mn = mv[rt] ? mx[rt] : m[rt];
        const float nb = mn == -INFINITY ? 0.f : mn;   // a row with no key yet keeps p = 0
        const float alpha = __builtin_amdgcn_exp2f(m[rt] - nb);
        m[rt] = mn;
        mb[rt] = nb;
        l[rt] *= alpha;
        // O rows 4 g + r take the factors of the lanes that hold those rows
        float ar[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) ar[r] = __shfl(alpha, 4 * g + r, 64);
#pragma unroll
        for (int i = 0; i < 16; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[rt][i][r] *= ar[r];
      }
    }
  };

  auto barrier = []() __attribute__((always_inline)) { __syncthreads(); };
  auto first = [&](int t, int ks) __attribute__((always_inline)) {
    scores(Ks[ks], s, [](int) {});
    mask(t, s);
#pragma unroll
    for (int q = 0; q < 10 * RT; ++q) maxima(s, q);
    settle();
  };
  auto step = [&](int t, int ks, int vs) __attribute__((always_inline)) {
    scores(Ks[ks], nx, probs);
    mask(t + 1, nx);
    weighted(Vs[vs], [&](int q) { maxima(nx, q); });
    settle();
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int j = 0; j < 2; ++j) s[rt][j] = nx[rt][j];
  };
  auto last = [&](int, int vs) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 24 * RT; ++q) probs(q);
    weighted(Vs[vs], [](int) {});
  };
  pf_schedule_run(tb, te, stage, arrived, barrier, first, step, last);
  if (h >= nq) return;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    float lt = l[rt];
    lt += __shfl_xor(lt, 16, 64);
    lt += __shfl_xor(lt, 32, 64);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float lr = __shfl(lt, 4 * g + r, 64), mr = __shfl(m[rt], 4 * g + r, 64);
      const int orow = qt * kPfRows + 16 * rt + 4 * g + r;
      if (orow >= M) continue;
      if (nkc == 1) {
        uint16_t* out = a.pf_out + ((size_t)orow * nq + h) * kHeadDim * 2;
        const float il = 1.f / lr;
#pragma unroll
        for (int i = 0; i < 16; i += 2) {   // dims 16 i + 2 c16 and + 1
          uint32_t hi, lo;
          split2_bf16(o[rt][i][r] * il, o[rt][i + 1][r] * il, hi, lo);
          uint16_t* e = out + a_slot(16 * i + 2 * c16);
          *(uint32_t*)e = hi;
          *(uint32_t*)(e + 32) = lo;
        }
      } else {
        float* pp = a.part + (((size_t)orow * kPrefillChunks + kc) * nq + h) * (2 + kHeadDim);
#pragma unroll
        for (int i = 0; i < 16; i += 2)
          *(float2*)(pp + 2 + 16 * i + 2 * c16) = make_float2(o[rt][i][r], o[rt][i + 1][r]);
        if (c16 == 0) {
          pp[0] = mr;
          pp[1] = lr;
        }
      }
    }
  }
}

// Rows of query tiles with more than one chunk: softmax-weighted sum of the
// chunks' (m, l, O) (maxima in log2 units, as k_attn_pf keeps them), one
// block per (row, query head), thread = head dim.
__global__ __launch_bounds__(256) void k_attn_pf_merge(AttnArgs a) {
  // one block per prompt row: wave h merges head h, lane l dims 4 l .. 4 l + 3
  // (16-byte loads of each chunk's o); the same per-element sums, in chunk
  // order, as one thread per dim
  const int row = blockIdx.x, tid = threadIdx.x, nq = a.n_q, h = tid >> 6, d4 = tid & 63;
  int t0, t1, nkc;
  pf_tile_span(a, row / (16 * a.pf_rt), &t0, &t1, &nkc);
  if (nkc == 1 || h >= nq) return;
  const float* pr = a.part + (size_t)row * kPrefillChunks * nq * (2 + kHeadDim);
  // chunks in groups of four, each group's loads issued together (clamped
  // indices; a group's chunks past nkc are skipped in the sums)
  constexpr int G = 4;
  float M = -INFINITY;
  for (int c0 = 0; c0 < nkc; c0 += G) {
    float m[G];
#pragma unroll
    for (int j = 0; j < G; ++j) m[j] = pr[(min(c0 + j, nkc - 1) * nq + h) * (2 + kHeadDim)];
#pragma unroll
    for (int j = 0; j < G; ++j)
      if (c0 + j < nkc) M = fmaxf(M, m[j]);
  }
  float L = 0.f;
  float4 O = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int c0 = 0; c0 < nkc; c0 += G) {
    float m[G], l[G];
    float4 o[G];
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const float* pc = pr + (min(c0 + j, nkc - 1) * nq + h) * (2 + kHeadDim);
      m[j] = pc[0];
      l[j] = pc[1];
      // a partial's o starts 2 floats into its 258-float record: 8-byte aligned
      const float2 lo2 = *(const float2*)(pc + 2 + 4 * d4), hi2 = *(const float2*)(pc + 4 + 4 * d4);
      o[j] = make_float4(lo2.x, lo2.y, hi2.x, hi2.y);
    }
#pragma unroll
    for (int j = 0; j < G; ++j) {
      if (c0 + j < nkc) {
        const float f = m[j] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m[j] - M);
        L = fmaf(f, l[j], L);
        O.x = fmaf(f, o[j].x, O.x);
        O.y = fmaf(f, o[j].y, O.y);
        O.z = fmaf(f, o[j].z, O.z);
        O.w = fmaf(f, o[j].w, O.w);
      }
    }
  }
  uint16_t* out = a.pf_out + ((size_t)row * nq + h) * kHeadDim * 2 + a_slot(4 * d4);
  bf16x4 hi, lo;
  split4_bf16(O.x / L, O.y / L, O.z / L, O.w / L, hi, lo);
  *(bf16x4*)out = hi;
  *(bf16x4*)(out + 32) = lo;
}

// ---------------------------------------------------------------------------
// Batched prefill GEMMs (no reference counterpart: the reference runs the
// decode pass once per prompt token, engine.ts:923-928).
//
// k_gemm: C[M x N] = A[M x K] * W[N x K]^T on bf16 MFMA
// (v_mfma_f32_16x16x32_bf16, K = 32 = one Q8_0 block). W holds the int8
// weights as bf16 (exact); A is split by its producer into hi = bf16(x) and
// lo = bf16(x - hi), so x - hi - lo is within 2^-17 |x| and every product
// q * hi, q * lo is exact in the fp32 accumulator. Per 32-block the two
// MFMAs give sum_j q_j x_j, which is scaled by the block's fp32 scale d and
// added to the output in fp32 -- the linearQ8 structure (shaders.ts:123-142)
// with the block sum on the matrix cores.
//
// A block is four waves side by side along the features: each owns 16 NJ
// weight rows and all 16 MI activation rows of the block. Weights are laid
// out as MFMA operands (one contiguous KB per 16 rows x 32 inputs), so they
// go from L2 straight to the registers of the one wave that uses them, PW
// steps ahead; only A, which the four waves share, passes through LDS (two
// stages of one 32-wide step, one barrier per step, PA steps of global loads
// in flight in registers). A 64 x 256 block so reads 16 bytes of LDS per
// MFMA cycle and SIMD where a 2 x 2 wave layout with W in LDS too read 24 and
// wrote 12, and its operand reads are prefetched one row tile ahead.
// What bounds it: at thousands of rows the cold weights of every layer and the
// power limit (in a prefill a 128 x 256 tile keeps the matrix cores busy 54% of
// the cycles at 1.83 GHz over 2048 rows, 57% at 1.92 over 4096; alone with warm
// weights 63% at 1.83 GHz, a 64 x 256 one 71% at 1.64, in the same time), at a
// hundred rows the latency of a step. The larger tiles use each weight for more
// rows and win where weights come from HBM, the small ones start more blocks.
// Gate/up of the 1B shape (N 13824, K 1152), weights cold: 4096 rows 283 -> 222
// to 229 us, 2048 rows 155 -> 124 to 129 us, 187 rows 33 -> 27 us against a
// 128 x 128 tile with both operands in LDS (ranges: two cards); gate/up of the
// 270M shape at 64 rows 20 -> 8.5 us.
//
// A rows are [K / 32][hi 32 | lo 32] bf16: one 128-byte line per 32-block.
// In LDS a 16-row tile's (plane, 8-wide chunk g) is 256 bytes of 16 rows, row
// r at slot r ^ (4 plane + g): the eight lanes that write one line and the
// eight that read one chunk each cover all banks. Rows past M are outside
// the buffer descriptors: their loads give zeros, their stores are dropped.
// ---------------------------------------------------------------------------
__device__ __forceinline__ u32x4 buf_load16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (uint32_t)bytes, 0x00020000);
}

// Position of input f of a 32-block in the planes that the GeGLU epilogue
// writes: a lane holds inputs c and 16 + c, stored as one dword, so the
// down weights carry their inputs in this order.
__device__ __forceinline__ int act_slot(int f) { return 2 * (f & 15) + (f >> 4); }

// KG > 1: KG groups of four waves split the block's K steps (its own A stages
// each) and add their tiles through LDS at the end, in a fixed order: the
// chain of steps, which bounds a hundred rows, is KG times shorter without
// more K slices for the consumer, and GeGLU tiles can be split too. The plan
// also takes it at up to a few thousand rows where N is small (64 x 128, N 640,
// 3264 rows).
template <int EPI, int MI, int NJ, int PW, int PA, int OCC, int KG>
__global__ __launch_bounds__(256 * KG, OCC) void k_gemm(GemmArgs a) {
  static_assert(EPI == EPI_OUT || NJ % 2 == 0, "GeGLU pairs adjacent column tiles");
  static_assert(KG == 1 || NJ <= 2, "half the groups' tiles fit the A stages");
  constexpr int BM = 16 * MI, BN = 64 * NJ;
  constexpr int AC = (BM * 8 + 255) / 256;   // 16-byte A chunks per thread and step
  constexpr int SL = PW + 1;                 // weight register stages
  static_assert(BM * 8 % 256 == 0, "whole chunks");
  __shared__ __align__(16) uint8_t stages[KG][2][BM * 128];
  const int kg = KG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  const int tid = threadIdx.x & 255, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  auto& As = stages[kg];
  const int M = a.M, N = a.N, KB = a.K / 32;
  // Tile order: workgroups go to the XCDs round-robin (from an XCD that
  // depends on earlier dispatches), so the blocks with one value of b % 8
  // (launch order) share an XCD; they take the contiguous range
  // [(b % 8) G / 8, (b % 8 + 1) G / 8) of an order with the K slice
  // slowest, then groups of 8 tile rows with the rows fastest, so that the
  // blocks sharing an XCD's L2 share A rows and W tiles (fewer L2 misses;
  // groups of 4, 8 or 16 are within 1%, of 2 4% slower).
  constexpr int GROUP = 8;
  const int NT = gridDim.x, MT = gridDim.y, G = NT * MT * gridDim.z;
  const int bid = blockIdx.x + NT * (blockIdx.y + MT * blockIdx.z);
  const int L = (G % 8 == 0) ? (bid % 8) * (G / 8) + bid / 8 : bid;
  const int kz = L / (NT * MT), Lp = L % (NT * MT);
  const int fm = (Lp / (GROUP * NT)) * GROUP, gm = min(MT - fm, GROUP);
  const int m0 = (fm + (Lp % (GROUP * NT)) % gm) * BM, n0 = ((Lp % (GROUP * NT)) / gm) * BN;
  // this block's K slice has KB / ks 32-blocks; a group's are [kb0, kb0 + ns)
  // of them, and every group goes through the same ng steps (and barriers)
  const int nb = KB / a.ks, ng = (nb + KG - 1) / KG;
  const int kb0 = kz * nb + min(kg * ng, nb - 1), ns = KG > 1 ? max(min(ng, nb - kg * ng), 0) : nb;
  const int rows = min(BM, M - m0);
  const uint32_t arow = (uint32_t)KB * 128;
  const int t0 = n0 / 16 + wv * NJ;          // this wave's first 16-row weight tile
  const auto ra = buf_rsrc((const uint8_t*)a.A + (size_t)m0 * arow, (size_t)rows * arow);
  const auto rw = buf_rsrc(a.W + (size_t)t0 * KB * 512, (size_t)NJ * KB * 1024);
  const auto rs = buf_rsrc(a.D + (size_t)t0 * KB * 16, (size_t)NJ * KB * 64);
  // staging: chunk tid + 256 i of a step is 16-byte unit q % 8 of row q / 8
  uint32_t ga[AC], la[AC];
#pragma unroll
  for (int i = 0; i < AC; ++i) {
    const int q = tid + 256 * i, row = q >> 3, c = q & 7;
    ga[i] = (uint32_t)row * arow + c * 16;
    la[i] = (row >> 4) * 2048 + c * 256 + (((row & 15) ^ c) * 16);
  }
  u32x4 ar[PA][AC], w[SL][NJ];
  float d[SL][NJ];
  // loads past the slice's end repeat its last step (never used)
  auto load_a = [&](int sl, int s) __attribute__((always_inline)) {
    const uint32_t so = (uint32_t)(kb0 + max(min(s, ns - 1), 0)) * 128u;
#pragma unroll
    for (int i = 0; i < AC; ++i) ar[sl][i] = buf_load16(ra, ga[i], so);
  };
  auto store_a = [&](int sl, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < AC; ++i) *(u32x4*)&As[st][la[i]] = ar[sl][i];
  };
  auto load_w = [&](int sl, int s) __attribute__((always_inline)) {
    const int k = kb0 + max(min(s, ns - 1), 0);
#pragma unroll
    for (int j = 0; j < NJ; ++j) w[sl][j] = buf_load16(rw, lane * 16, (uint32_t)(j * KB + k) * 1024u);
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      d[sl][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, r16 * 4, (uint32_t)(j * KB + k) * 64u, 0));
  };

  f32x4 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int rdh = g * 256 + ((r16 ^ g) * 16), rdl = 1024 + g * 256 + ((r16 ^ (4 + g)) * 16);
  load_a(0, 0);
#pragma unroll
  for (int p = 0; p < PW; ++p) load_w(p, p);
  store_a(0, 0);
#pragma unroll
  for (int q = 0; q < PA; ++q) load_a((1 + q) % PA, 1 + q);
  __syncthreads();
  // step s, u = s mod the unroll: stage s + 1 of A goes to LDS and the loads
  // of later steps go out, then this step's products
  auto step = [&](int s, int u) __attribute__((always_inline)) {
    const int sl = u % SL, st = u & 1;
    store_a((u + 1) % PA, st ^ 1);
    load_w((sl + PW) % SL, s + PW);
    load_a((u + 1) % PA, s + 1 + PA);
    if (KG > 1 && s >= ns) {   // a shorter group only keeps the barriers
      __syncthreads();
      return;
    }
    // the MFMA phase runs at raised wave priority: of the waves on a SIMD the
    // computing one issues ahead of the staging ones
    __builtin_amdgcn_s_setprio(1);
    f32x4 p[2][NJ];
    bf16x8 xh[2], xl[2];
    auto read = [&](int i) __attribute__((always_inline)) {
      xh[i & 1] = __builtin_bit_cast(bf16x8, *(const u32x4*)&As[st][i * 2048 + rdh]);
      xl[i & 1] = __builtin_bit_cast(bf16x8, *(const u32x4*)&As[st][i * 2048 + rdl]);
    };
    auto scale = [&](int i) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] = fmaf(d[sl][j], p[i & 1][j][r], acc[i][j][r]);
    };
    // the schedule: a row tile's operands are read while the previous row
    // tile multiplies, and its scale FMAs fill the issue slots between the
    // next tile's MFMAs, two behind each
    read(0);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      if (i + 1 < MI) read(i + 1);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        p[i & 1][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xh[i & 1], __builtin_bit_cast(bf16x8, w[sl][j]),
                                                              f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        p[i & 1][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xl[i & 1], __builtin_bit_cast(bf16x8, w[sl][j]),
                                                              p[i & 1][j], 0, 0, 0);
      if (i > 0) scale(i - 1);
      if (i == 0) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);       // LDS reads
      if (i + 1 < MI) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
      for (int q = 0; q < 2 * NJ; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);                   // MFMA
        if (i > 0) __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);        // VALU
      }
    }
    scale(MI - 1);
    __builtin_amdgcn_s_setprio(0);
    __syncthreads();
  };
  constexpr int U = SL % 2 == 0 ? SL : 2 * SL;
  static_assert(U % PA == 0, "the A registers rotate with the unroll");
  for (int s = 0; s < ng; s += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u > 0 && s + u >= ng) break;
      step(s + u, u);
    }
  }
  // groups h, 3 h, ... hand their tiles to groups 0, 2 h, ...
#pragma unroll
  for (int h = 1; h < KG; h *= 2) {
    f32x4* x = (f32x4*)&stages[0][0][0] + (size_t)(kg / (2 * h)) * 4 * MI * NJ * 64 + wv * MI * NJ * 64 + lane;
    if (kg % (2 * h) == h)
#pragma unroll
      for (int t = 0; t < MI * NJ; ++t) x[64 * t] = acc[t / NJ][t % NJ];
    __syncthreads();
    if (kg % (2 * h) == 0)
#pragma unroll
      for (int t = 0; t < MI * NJ; ++t) {
        const f32x4 y = x[64 * t];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[t / NJ][t % NJ][r] += y[r];
      }
    if (2 * h < KG) __syncthreads();
  }
  if (kg) return;

  // D of a 16x16 tile: lane l, register r -> row 4 (l / 16) + r, col l % 16
  if (EPI == EPI_OUT) {
    const auto rc = buf_rsrc(a.C + ((size_t)kz * M + m0) * N, (size_t)rows * N * 4);
    const uint32_t vo = ((uint32_t)(4 * g) * N + n0 + wv * 16 * NJ + r16) * 4u;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t v = vo + (uint32_t)(16 * i + r) * N * 4u;   // the checked part of the address
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[i][j][r]), rc, v + 64 * j, 0, 0);
      }
  } else {
    // 16 gate rows (tile j), then their 16 up rows (tile j + 1): 16 features
    // per pair, two pairs per 32-block of the output rows (2 N bytes each)
    const auto ro = buf_rsrc(a.act + (size_t)m0 * N, (size_t)rows * N * 2);
    const int f0 = (n0 + wv * 16 * NJ) / 2;   // this wave's first feature
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t vo = (uint32_t)(16 * i + 4 * g + r) * N * 2u + (f0 >> 5) * 128u + r16 * 4u;
        if (NJ % 4 == 0) {
#pragma unroll
          for (int j = 0; j < NJ; j += 4) {
            uint32_t hi, lo;
            split2_bf16(gelu_mul(acc[i][j][r], acc[i][(j + 1) % NJ][r]),
                        gelu_mul(acc[i][(j + 2) % NJ][r], acc[i][(j + 3) % NJ][r]), hi, lo);
            __builtin_amdgcn_raw_buffer_store_b32(hi, ro, vo + 32 * j, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b32(lo, ro, vo + 32 * j + 64, 0, 0);
          }
        } else {   // one pair: the low or high half of each dword
          uint16_t hi, lo;
          split_bf16(gelu_mul(acc[i][0][r], acc[i][1 % NJ][r]), &hi, &lo);
          const uint32_t vh = vo + (f0 & 16) / 8;
          __builtin_amdgcn_raw_buffer_store_b16(hi, ro, vh, 0, 0);
          __builtin_amdgcn_raw_buffer_store_b16(lo, ro, vh + 64, 0, 0);
        }
      }
  }
}

// Offset of element e of an A row: 32-blocks of hi then lo.
__device__ __forceinline__ int a_slot(int e) { return ((e >> 5) << 6) + (e & 31); }

// Row kernels (one block per prompt row, H <= 2048).
__device__ __forceinline__ void row_norm_out(const float* r, const float* w, int H, float eps, uint16_t* out,
                                             float* sh4, int n) {
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (i < n) ss = fmaf(r[i], r[i], ss);
  const float ri = rsq(block_sum256(ss, sh4) / (float)H + eps);
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (i < n) {
      const int e = threadIdx.x + 256 * i;
      split_bf16((r[i] * w[e]) * ri, &out[a_slot(e)], &out[a_slot(e) + 32]);
    }
}

__global__ __launch_bounds__(256) void k_rows_embed(RowArgs a) {
  __shared__ float sh4[4];
  const int row = blockIdx.x, tid = threadIdx.x, H = a.H;
  const int n = (H - tid + 255) / 256;
  const int token = a.tokens[row];
  float h[8];
  GemvArgs g{};
  g.embd = a.embd;
  g.embd_KpS = a.embd_KpS;
  g.embed_scale = a.embed_scale;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (i < n) {
      h[i] = embed_elem(g, token, tid + 256 * i);
      a.res_out[(size_t)row * H + tid + 256 * i] = h[i];
    }
  row_norm_out(h, a.w_pre, H, a.eps, a.x_out + (size_t)row * H * 2, sh4, n);
}

// One block per prompt row: thread t holds float4s t and t + 256, so every
// load of the row (all K slices of the GEMM output, the residual, both norm
// weights) is in flight before the sums. Memory-bound at thousands of rows
// (4096 rows, two slices, 94 MB: 19.1 -> 16.9 us), one memory latency and two
// barriers at few: 187 rows 8.6 -> 4.6 us, 64 rows of 640 6.1 -> 3.5 us,
// against one wave per row.
__global__ __launch_bounds__(256) void k_rows_resid(RowArgs a) {
  constexpr int KF = 2048 / 4 / 256;   // float4s per thread at the largest hidden size
  __shared__ float sh[2][4];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, H = a.H, row = blockIdx.x;
  const int F4 = H / 4;
  const size_t o4 = (size_t)row * F4;
  const float4* pre = (const float4*)a.pre;
  const float4* res = (const float4*)a.res;
  const size_t ps4 = a.pre_stride / 4;
  auto sum_row = [&](float x, int i) {
    x = wave_sum_dpp(x);
    if (lane == 0) sh[i][wv] = x;
    __syncthreads();
    return (sh[i][0] + sh[i][1]) + (sh[i][2] + sh[i][3]);
  };
  float4 v[KF], rs[KF], wq[KF], wp[KF];
#pragma unroll
  for (int k = 0; k < KF; ++k) {
    const int f = tid + 256 * k;
    if (f < F4) {
      v[k] = pre[o4 + f];
      float4 pv[kGemmMaxSlices - 1];
#pragma unroll
      for (int p = 1; p < kGemmMaxSlices; ++p)
        if (p < a.pre_planes) pv[p - 1] = pre[p * ps4 + o4 + f];
      rs[k] = res[o4 + f];
      wq[k] = ((const float4*)a.w_post)[f];
      wp[k] = ((const float4*)a.w_pre)[f];
      // K slices of the previous GEMM, added in slice order
#pragma unroll
      for (int p = 1; p < kGemmMaxSlices; ++p)
        if (p < a.pre_planes) {
          v[k].x += pv[p - 1].x;
          v[k].y += pv[p - 1].y;
          v[k].z += pv[p - 1].z;
          v[k].w += pv[p - 1].w;
        }
    }
  }
  float s1 = 0.f;
#pragma unroll
  for (int k = 0; k < KF; ++k)
    if (tid + 256 * k < F4) {
      s1 = fmaf(v[k].x, v[k].x, s1);
      s1 = fmaf(v[k].y, v[k].y, s1);
      s1 = fmaf(v[k].z, v[k].z, s1);
      s1 = fmaf(v[k].w, v[k].w, s1);
    }
  const float ri1 = rsq(sum_row(s1, 0) / (float)H + a.eps);
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < KF; ++k) {
    const int f = tid + 256 * k;
    if (f < F4) {
      float4 r;
      r.x = rs[k].x + (v[k].x * wq[k].x) * ri1;
      r.y = rs[k].y + (v[k].y * wq[k].y) * ri1;
      r.z = rs[k].z + (v[k].z * wq[k].z) * ri1;
      r.w = rs[k].w + (v[k].w * wq[k].w) * ri1;
      ((float4*)a.res_out)[o4 + f] = r;
      if (a.last_hidden && row == a.M - 1) ((float4*)a.last_hidden)[f] = r;
      v[k] = r;
      ss = fmaf(r.x, r.x, ss);
      ss = fmaf(r.y, r.y, ss);
      ss = fmaf(r.z, r.z, ss);
      ss = fmaf(r.w, r.w, ss);
    }
  }
  const float ri = rsq(sum_row(ss, 1) / (float)H + a.eps);
#pragma unroll
  for (int k = 0; k < KF; ++k) {
    const int f = tid + 256 * k;
    if (f < F4) {
      const float4 w = wp[k];
      bf16x4 hi, lo;
      split4_bf16((v[k].x * w.x) * ri, (v[k].y * w.y) * ri, (v[k].z * w.z) * ri, (v[k].w * w.w) * ri, hi, lo);
      uint16_t* xo = a.x_out + (size_t)row * H * 2 + a_slot(4 * f);
      *(bf16x4*)xo = hi;
      *(bf16x4*)(xo + 32) = lo;
    }
  }
}

// QK-norm + NEOX RoPE of every row's heads, k and v into the cache
// (fusedPerHeadNormRope, shaders.ts:420-467), and q, k, v as bf16 hi / lo in
// the attention kernel's MFMA operand order, each value split once. One block
// per 8 aligned positions from the first key that this slice's attention
// reads (kv_lo) to the end of its last 32-key tile: positions before the
// slice are converted from the cache, positions past its end are zeros (a
// masked key's probability 0 must meet a finite v). Waves w and w + n_q + 2 take
// positions 0-3 and 4-7 of query head w, of the keys (w = n_q) or the values
// (n_q + 1). Lane l holds dims l + 64 j, so the
// NEOX pairs (i, i + 128) are its own j and j + 2, and a head's sum of squares
// is one wave reduction; a wave's loads are all in flight at once. The operand order is reached through LDS in 16-byte units: a unit of
// v holds eight keys of one dim, which is why a block takes eight positions.
constexpr int kKvPos = 8, kKvWavePos = 4;
constexpr int kKvPitch = kHeadDim + 4;   // floats: eight rows' units fall into distinct banks
__global__ __launch_bounds__(128 * (kAttnMaxQ + 2)) void k_rows_kv(RowArgs a) {
  __shared__ __align__(16) float xs[kKvPos * (kAttnMaxQ + 2) * kKvPitch];
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, nq = a.n_q, nh = nq + 2;
  const int wv = wid >= nh ? wid - nh : wid, half = wid >= nh ? kKvWavePos : 0;
  const int p0 = (a.kv_lo / kPfKeys) * kPfKeys + kKvPos * blockIdx.x;
  const int row0 = p0 - a.pf_start;   // the block's positions as rows; wave position i is half + i
  const bool is_q = wv < nq, is_v = wv == nq + 1;
  const size_t stride = (size_t)nh * kHeadDim;
  auto fresh = [&](int i) { return row0 + half + i >= 0 && row0 + half + i < a.M; };
  float x[kKvWavePos][4];
  // every load is issued unconditionally (rows clamped into the slice, cache
  // rows into the context read so far) so that all of them are in flight together
  auto row_of = [&](int i) { return min(max(row0 + half + i, 0), a.M - 1); };
#pragma unroll
  for (int i = 0; i < kKvWavePos; ++i) {
    const float* src = a.qkv + (size_t)row_of(i) * stride + wv * kHeadDim;
    if (!is_q && row0 + half + i < 0) src = (is_v ? a.v_cache : a.k_cache) + (size_t)(p0 + half + i) * kHeadDim;
#pragma unroll
    for (int j = 0; j < 4; ++j) x[i][j] = src[lane + 64 * j];
  }
  // the QKV GEMM's K slices (pre_planes of them, pre_stride floats apart)
  // are added in slice order
  float y[kQkvMaxSlices - 1][kKvWavePos][4];
#pragma unroll
  for (int p = 1; p < kQkvMaxSlices; ++p)
    if (p < a.pre_planes)
#pragma unroll
      for (int i = 0; i < kKvWavePos; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          y[p - 1][i][j] = a.qkv[p * a.pre_stride + (size_t)row_of(i) * stride + wv * kHeadDim + lane + 64 * j];
#pragma unroll
  for (int p = 1; p < kQkvMaxSlices; ++p)
    if (p < a.pre_planes)
#pragma unroll
      for (int i = 0; i < kKvWavePos; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) x[i][j] += fresh(i) ? y[p - 1][i][j] : 0.f;
  if (!is_v && row0 + half + kKvWavePos > 0) {
    const float* w = is_q ? a.q_norm : a.k_norm;
    float nw[4], cs[kKvWavePos][2], sn[kKvWavePos][2];
#pragma unroll
    for (int j = 0; j < 4; ++j) nw[j] = w[lane + 64 * j];
#pragma unroll
    for (int i = 0; i < kKvWavePos; ++i) {
      const float* rt = a.rope + (size_t)(a.pf_start + row_of(i)) * kHeadDim;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        cs[i][j] = rt[lane + 64 * j];
        sn[i][j] = rt[kHeadDim / 2 + lane + 64 * j];
      }
    }
#pragma unroll
    for (int i = 0; i < kKvWavePos; ++i) {
      float ss = 0.f, y[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) ss = fmaf(x[i][j], x[i][j], ss);
      const float ri = rsq(wave_sum_dpp(ss) / (float)kHeadDim + a.eps);
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = (x[i][j] * nw[j]) * ri;
      if (fresh(i))
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          x[i][j] = y[j] * cs[i][j] - y[j + 2] * sn[i][j];
          x[i][j + 2] = y[j] * sn[i][j] + y[j + 2] * cs[i][j];
        }
    }
  }
  if (!is_q) {
    float* cache = is_v ? a.v_cache : a.k_cache;
#pragma unroll
    for (int i = 0; i < kKvWavePos; ++i)
      if (fresh(i))
#pragma unroll
        for (int j = 0; j < 4; ++j) cache[(size_t)(p0 + half + i) * kHeadDim + lane + 64 * j] = x[i][j];
  }
#pragma unroll
  for (int i = 0; i < kKvWavePos; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)   // positions past the slice: zeros
      xs[((half + i) * nh + wv) * kKvPitch + lane + 64 * j] = row0 + half + i < a.M ? x[i][j] : 0.f;
  __syncthreads();

  const int tid = threadIdx.x, nt = 128 * nh;
  auto split8 = [](const float* v, uint16_t* hi, uint16_t* lo) {
    uint32_t h4[4], l4[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) split2_bf16(v[2 * e], v[2 * e + 1], h4[e], l4[e]);
    *(u32x4*)hi = u32x4{h4[0], h4[1], h4[2], h4[3]};
    *(u32x4*)lo = u32x4{l4[0], l4[1], l4[2], l4[3]};
  };
  uint16_t* tile = (uint16_t*)(a.kv_planes + (size_t)(p0 / kPfKeys) * kKvTileBytes);
  // heads 0 .. n_q - 1 (q, scaled) and n_q (k): unit = (position, 8 dims)
  for (int u = tid; u < (nq + 1) * 256; u += nt) {
    const int i = u & 7, c = (u >> 3) & 31, hd = u >> 8, t = c >> 2, gd = c & 3;
    float v[8];
    const float4* src = (const float4*)&xs[(i * nh + hd) * kKvPitch + 8 * c];
    const float4 v0 = src[0], v1 = src[1];
    v[0] = v0.x; v[1] = v0.y; v[2] = v0.z; v[3] = v0.w;
    v[4] = v1.x; v[5] = v1.y; v[6] = v1.z; v[7] = v1.w;
    uint16_t* dst;
    if (hd < nq) {
      const int row = row0 + i;
      if (row < 0 || row >= a.M) continue;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] *= a.q_scale;
      dst = a.q_frag + ((size_t)((row >> 4) * nq + hd) * 16 + 2 * t) * 512 + (gd * 16 + (row & 15)) * 8;
    } else {
      const int kk = (p0 + i) % kPfKeys, j = (kk >> 2) & 1, r = (kk >> 3) * 4 + (kk & 3);
      dst = tile + ((t * 2 + j) * 2) * 512 + (gd * 16 + r) * 8;
    }
    split8(v, dst, dst + 512);
  }
  // v: unit = (dim, this block's eight keys)
  for (int d = tid; d < kHeadDim; d += nt) {
    float v[8];
#pragma unroll
    for (int i = 0; i < kKvPos; ++i) v[i] = xs[(i * nh + nq + 1) * kKvPitch + d];
    const int dt = 2 * (d >> 5) + (d & 1), c = (d & 31) >> 1;   // dim tile and column: adjacent dims in one lane
    uint16_t* dst = tile + kPfTile / 2 + (dt * 2) * 512 + (((p0 % kPfKeys) / kKvPos) * 16 + c) * 8;
    split8(v, dst, dst + 512);
  }
}

// ---------------------------------------------------------------------------
// Upload helpers.
// k_repack: GGUF row-major Q8_0 (rows of Kp 68-byte pairs) -> the
// item-planar layout L. interleave_half > 0 places source row r at fused
// row (r / half) * GR + (r % half) + dst_row_offset with half = GR / 2, i.e.
// gate rows in the first half of each row group and (dst_row_offset = half)
// the matching up rows in the second half.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_repack(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                long long rows, Q8Layout L, long long off, int half) {
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long total = rows * L.Kp;
  if (idx >= total) return;
  const long long r = idx / L.Kp;
  const int c = (int)(idx - r * L.Kp);
  const long long R = half > 0 ? (r / half) * L.GR + (r % half) + off : r + off;
  const long long g = R / L.GR;
  const int ln = (int)(R - g * L.GR);
  const uint32_t* s = (const uint32_t*)(src + (size_t)idx * kPairBytes);
  uint8_t* item = dst + ((size_t)g * L.KpS + c / L.CI) * kColBytes;
  const int slot = (c % L.CI) * L.GR + ln;
#pragma unroll
  for (int i = 0; i < 17; ++i) *(uint32_t*)(item + plane_offset(i, slot)) = s[i];
}

// Class-major copy of a CI = 1 item-planar matrix (the tied LM head): row
// c + 256 k (vocabulary stride class c, shaders.ts:337-347) goes to row
// c * (rows / 256) + k, so each 64-row group of the copy holds one class.
__global__ __launch_bounds__(256) void k_class_major(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                     long long rows, int Kp) {
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= rows * Kp) return;
  const long long r = idx / Kp;
  const int c = (int)(idx - r * Kp);
  const long long p = (r & 255) * (rows >> 8) + (r >> 8);
  const uint8_t* si = src + ((size_t)(r >> 6) * Kp + c) * kColBytes;
  uint8_t* di = dst + ((size_t)(p >> 6) * Kp + c) * kColBytes;
  const int ss = (int)(r & 63), ds = (int)(p & 63);
#pragma unroll
  for (int i = 0; i < 17; ++i) *(uint32_t*)(di + plane_offset(i, ds)) = *(const uint32_t*)(si + plane_offset(i, ss));
}

// Column-block layout of a Q8_0 matrix (the down projection of the
// persistent decode kernel): for each 32-wide input block m, the f16 scales
// of all rows [rows], then their 32 int8 values [rows][32]: 34 * rows bytes
// per block, so one block's column slice is contiguous.
__global__ __launch_bounds__(256) void k_repack_colblock(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                         long long rows, int nblk) {
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= rows * nblk) return;
  const long long r = idx / nblk;
  const int m = (int)(idx - r * nblk);
  const uint8_t* blk = src + (size_t)idx * 34;
  uint8_t* col = dst + (size_t)m * 34 * rows;
  col[2 * r] = blk[0];
  col[2 * r + 1] = blk[1];
  uint8_t* q = col + 2 * rows + 32 * r;
#pragma unroll
  for (int i = 0; i < 32; ++i) q[i] = blk[2 + i];
}

// Gate/up copy of the persistent decode kernel laid out as the B operands of
// v_mfma_i32_16x16x64_i8. Group g holds gate rows 32g .. 32g + 31 and up rows
// 32g .. 32g + 31 as four 16-row tiles t (0, 1: gate; 2, 3: up). For pair
// column c (k in [64c, 64c + 64)) tile t is 1 KB at c * 4096 + t * 1024, where
// lane l's 16 bytes are row 16 (t & 1) + l % 16 of its half at k = 64c +
// 16 (l / 16) .. +15. After the Kp * 4096 int8 bytes come the block scales,
// [t][m][lane < 32] dwords: the f16 scales of pair columns 2m (low half) and
// 2m + 1 (high half) for row 16 (t & 1) + lane % 16, Q8_0 block 2c + lane / 16.
// One thread per 16-byte chunk, then one per scale dword, of the gate (up = 0)
// or up (up = 1) half.
__global__ __launch_bounds__(256) void k_repack_gum(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                    long long rows, int K, int up) {
  const int Kp = K / 64, Kh = (Kp + 1) / 2;
  const size_t gbytes = gum_group_bytes(K), rowb = (size_t)K / 32 * 34;
  const long long groups = rows / 32;
  const long long nch = groups * Kp * 2 * 64, nsc = groups * 2 * Kh * 32;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i < nch) {
    const int lane = (int)(i % 64);
    long long q = i / 64;
    const int th = (int)(q % 2);
    q /= 2;
    const int c = (int)(q % Kp);
    const long long g = q / Kp;
    const long long row = 32 * g + 16 * th + lane % 16;
    const int k0 = 64 * c + 16 * (lane / 16);
    const uint8_t* sp = src + row * rowb + (size_t)(k0 / 32) * 34 + 2 + k0 % 32;
    uint8_t* dp = dst + g * gbytes + (size_t)c * 4096 + (size_t)(th + 2 * up) * 1024 + (size_t)lane * 16;
#pragma unroll
    for (int j = 0; j < 16; ++j) dp[j] = sp[j];
  } else if (i < nch + nsc) {
    long long q = i - nch;
    const int lane = (int)(q % 32);
    q /= 32;
    const int m = (int)(q % Kh);
    q /= Kh;
    const int th = (int)(q % 2);
    const long long g = q / 2;
    const long long row = 32 * g + 16 * th + lane % 16;
    uint32_t v = 0;
    for (int h = 0; h < 2; ++h) {
      const int c = 2 * m + h;
      if (c < Kp) {
        const uint8_t* bp = src + row * rowb + (size_t)(2 * c + lane / 16) * 34;
        v |= (uint32_t)(bp[0] | (bp[1] << 8)) << (16 * h);
      }
    }
    *(uint32_t*)(dst + g * gbytes + (size_t)Kp * 4096 + ((size_t)((th + 2 * up) * Kh + m) * 32 + lane) * 4) = v;
  }
}

// Embedding row of one token through embed_value (parity reads).
__global__ __launch_bounds__(256) void k_embed_row(const uint8_t* embd, int kps, float scale, int token, int H,
                                                   float* out) {
  for (int e = threadIdx.x; e < H; e += 256) out[e] = embed_value(embd, kps, scale, token, e);
}

// Bit-exact Q8_0 dequantisation of GGUF blocks (gguf.ts:107-124).
__global__ __launch_bounds__(256) void k_dequant(const uint8_t* __restrict__ src, float* __restrict__ out,
                                                 long long n) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint8_t* blk = src + (size_t)(i >> 5) * 34;
  const uint16_t sb = (uint16_t)(blk[0] | (blk[1] << 8));
  const float scale = (float)__builtin_bit_cast(_Float16, sb);
  out[i] = (float)(int8_t)blk[2 + (i & 31)] * scale;
}

// The same for 16-byte aligned src and out: a block takes 128 Q8_0 blocks
// (4352 bytes, a multiple of 16) through LDS in 16-byte loads and writes 4096
// floats in 16-byte stores; the byte loads and 4-byte stores above keep a
// quarter of the bytes in flight (8 M values, 40 MB: 12.4 -> 7.9 us).
// One block's chain (load, LDS, barrier, store) is longer than the byte
// kernel's, so dequant_wide takes it where the byte kernel has well more blocks
// than the chip holds at once (8 per CU: 524288 values), or for up to three
// blocks. Kernel times back to back, wide against byte: 128 values 1.50 / 1.32 us, 4096 1.71 / 1.97, 12288 1.98 / 1.98,
// 65536 2.60 / 2.00, 524288 2.81 / 2.45, 786432 2.94 / 2.93, 1 M 3.07 / 3.22,
// 2 M 3.84 / 4.68.
constexpr int kDeqBlocks = 128;
__global__ __launch_bounds__(256) void k_dequant16(const uint8_t* __restrict__ src, float* __restrict__ out,
                                                   long long nblk) {
  __shared__ __align__(16) uint8_t s[kDeqBlocks * 34];
  const int tid = threadIdx.x;
  const long long b0 = (long long)blockIdx.x * kDeqBlocks;
  const int nb = (int)(nblk - b0 < kDeqBlocks ? nblk - b0 : kDeqBlocks);
  const int bytes = nb * 34;
  const uint8_t* p = src + b0 * 34;
  for (int u = tid; u < kDeqBlocks * 34 / 16; u += 256) {
    if (16 * u + 16 <= bytes) *(u32x4*)&s[16 * u] = ((const u32x4*)p)[u];
    else
      for (int e = 16 * u; e < bytes; ++e) s[e] = p[e];   // the last block's tail
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = tid + 256 * j, q = i >> 3;   // float4 i: block q, values 4 (i % 8) .. + 3
    if (q < nb) {
      const uint16_t* h = (const uint16_t*)&s[q * 34];
      const float scale = (float)__builtin_bit_cast(_Float16, h[0]);
      const uint32_t w = h[1 + 2 * (i & 7)] | ((uint32_t)h[2 + 2 * (i & 7)] << 16);
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (float)(int8_t)(w >> (8 * e)) * scale;
      *((f32x4*)(out + b0 * 32) + i) = o;
    }
  }
}

// Class-major logits (row c + 256 k at c * V / 256 + k, as the persistent
// decode kernel leaves them) back in row order: 64 x 64 tiles through LDS.
__global__ __launch_bounds__(256) void k_logits_rows(const float* __restrict__ cm, float* __restrict__ out, int R) {
  __shared__ float t[64][65];
  const int x = threadIdx.x & 63, y0 = threadIdx.x >> 6;
  const int k0 = 64 * blockIdx.x, c0 = 64 * blockIdx.y;
  for (int y = y0; y < 64; y += 4)
    if (k0 + x < R) t[y][x] = cm[(size_t)(c0 + y) * R + k0 + x];
  __syncthreads();
  for (int y = y0; y < 64; y += 4)
    if (k0 + y < R) out[(size_t)(k0 + y) * 256 + c0 + x] = t[x][y];
}

// GGUF Q8_0 rows -> the prefill GEMM's weights: int8 values as bf16 (exact)
// and fp32 block scales, one thread per 32-block. Source row r goes to row
// r + off, or with half = 16 to (r / 16) * 32 + r % 16 + off (gate / up
// groups of 16 + 16 rows). The 16 rows of tile t and the 32 inputs of block b
// are the 1 KB at ((t nb) + b) * 1 KB: lane l of the MFMA operand holds row
// l % 16, inputs 8 (l / 16) .. + 7; their scales are 16 floats at t nb + b.
// act_order: inputs in the GeGLU epilogue's order (the down matrix).
__global__ __launch_bounds__(256) void k_q8_bf16(const uint8_t* __restrict__ src, uint16_t* __restrict__ wb,
                                                 float* __restrict__ wd, long long rows, int K, long long off,
                                                 int half, int act_order) {
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  const int nb = K / 32;
  if (idx >= rows * nb) return;
  const long long r = idx / nb;
  const int b = (int)(idx - r * nb);
  const long long R = half > 0 ? (r / half) * 2 * half + r % half + off : r + off;
  const uint8_t* blk = src + (size_t)idx * 34;
  const long long tb = (R >> 4) * nb + b;
  const int r16 = (int)(R & 15);
  wd[tb * 16 + r16] = (float)__builtin_bit_cast(_Float16, (uint16_t)(blk[0] | (blk[1] << 8)));
#pragma unroll
  for (int g = 0; g < 4; ++g) {   // operand slots 8 g .. + 7
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int p = 8 * g + 2 * e;   // slots p, p + 1 hold inputs p, p + 1 or (act_slot) p / 2, p / 2 + 16
      const float f0 = (float)(int8_t)blk[2 + (act_order ? p / 2 : p)];
      const float f1 = (float)(int8_t)blk[2 + (act_order ? p / 2 + 16 : p + 1)];
      o[e] = (__float_as_uint(f0) >> 16) | (__float_as_uint(f1) & 0xffff0000u);
    }
    *(u32x4*)(wb + tb * 512 + (g * 16 + r16) * 8) = u32x4{o[0], o[1], o[2], o[3]};
  }
}

// Add ids to the repetition-penalty bitmap (the turn's prompt tokens).
__global__ __launch_bounds__(256) void k_seen_add(uint32_t* seen, DevState* st, const int32_t* ids, int n,
                                                  int V) {
  for (int i = threadIdx.x; i < n; i += 256) {
    const int id = ids[i];
    if (id >= 0 && id < V) atomicOr(&seen[id >> 5], 1u << (id & 31));
  }
  if (threadIdx.x == 0) st->seen_count += n;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <int PRO, int EPI, int CI, int NIF>
static int launch_gemv_t(const GemvArgs& a, hipStream_t s) {
  const size_t lds = (size_t)a.Kp * kXPad * sizeof(float);
  hipLaunchKernelGGL((k_gemv<PRO, EPI, CI, NIF>), dim3(a.N / (64 / CI)), dim3(256), lds, s, a);
  return (int)hipGetLastError();
}

// Steps a wave issues before the prologue: all of them when a row group has
// at most 4, 8 or 20 column steps; longer rows continue with a prefetch loop.
template <int PRO, int EPI, int CI>
static int launch_gemv_nif(const GemvArgs& a, hipStream_t s) {
  if (a.KpS <= 4) return launch_gemv_t<PRO, EPI, CI, 1>(a, s);
  if (a.KpS <= 8) return launch_gemv_t<PRO, EPI, CI, 2>(a, s);
  return launch_gemv_t<PRO, EPI, CI, 5>(a, s);
}

template <int PRO, int EPI>
static int launch_gemv_ci(int ci, const GemvArgs& a, hipStream_t s) {
  switch (ci) {
    case 1: return launch_gemv_nif<PRO, EPI, 1>(a, s);
    case 2: return launch_gemv_nif<PRO, EPI, 2>(a, s);
    case 8: return launch_gemv_nif<PRO, EPI, 8>(a, s);
  }
  return (int)hipErrorInvalidValue;
}

// Launch plan of k_gemv_mg: W = 4 waves for K <= 2048, 16 above; about two
// blocks per CU (512 or 256 blocks, at most one per row group), more blocks
// when a wave would otherwise hold more than three items in registers.
// Returns false when no plan keeps every wave at <= 3 items.
struct MgPlan { int W, nb, nif, ept; };
static bool mg_plan(const GemvArgs& a, int pro, int ci, MgPlan& p) {
  const int K = a.Kp * 64, GR = 64 / ci, G = a.N / GR;
  p.W = K > 2048 ? 16 : 4;
  if ((pro != PRO_NONE || ci != 8) && p.W != 4) return false;
  p.ept = (K / 4 + 64 * p.W - 1) / (64 * p.W);   // float4 chunks of x per thread: 1 or 2
  if (p.ept > 2) return false;
  int nb = min(G, p.W == 4 ? 512 : 256);
  for (;;) {
    const int gpb = (G + nb - 1) / nb;
    const int nif = (gpb * a.KpS + p.W - 1) / p.W;
    if (nif <= 3 && gpb * GR <= kMgRows) {
      p.nb = nb;
      p.nif = nif;
      return true;
    }
    if (nb == G) return false;
    nb = min(G, nb * 2);
  }
}

template <int PRO, int EPI, int CI, int W, int NIF>
static int launch_mg_ept(const GemvArgs& a, const MgPlan& p, hipStream_t s) {
  const size_t lds = (size_t)a.Kp * kXPad * sizeof(float);
  switch (p.ept) {
#define GG_MG_EPT(E) \
    case E: hipLaunchKernelGGL((k_gemv_mg<PRO, EPI, CI, W, NIF, E>), dim3(p.nb), dim3(64 * W), lds, s, a); break;
    GG_MG_EPT(1) GG_MG_EPT(2)
#undef GG_MG_EPT
    default: return (int)hipErrorInvalidValue;
  }
  return (int)hipGetLastError();
}
template <int PRO, int EPI, int CI, int W>
static int launch_mg_nif(const GemvArgs& a, const MgPlan& p, hipStream_t s) {
  switch (p.nif) {
    case 1: return launch_mg_ept<PRO, EPI, CI, W, 1>(a, p, s);
    case 2: return launch_mg_ept<PRO, EPI, CI, W, 2>(a, p, s);
    case 3: return launch_mg_ept<PRO, EPI, CI, W, 3>(a, p, s);
  }
  return (int)hipErrorInvalidValue;
}
template <int CI>
static int launch_mg_ci(int pro, int epi, const GemvArgs& a, const MgPlan& p, hipStream_t s) {
  if (pro == PRO_ATTN_MERGE) return launch_mg_nif<PRO_ATTN_MERGE, EPI_OUT, CI, 4>(a, p, s);
  if (pro == PRO_NONE) {
    if (CI == 8 && p.W == 16) return launch_mg_nif<PRO_NONE, EPI_OUT, 8, 16>(a, p, s);
    return launch_mg_nif<PRO_NONE, EPI_OUT, CI, 4>(a, p, s);
  }
  if (epi == EPI_GEGLU) return launch_mg_nif<PRO_RESID_NORM, EPI_GEGLU, CI, 4>(a, p, s);
  if (pro == PRO_EMBED_NORM) return launch_mg_nif<PRO_EMBED_NORM, EPI_OUT, CI, 4>(a, p, s);
  return launch_mg_nif<PRO_RESID_NORM, EPI_OUT, CI, 4>(a, p, s);
}
static int launch_mg(int pro, int epi, int ci, const GemvArgs& a, const MgPlan& p, hipStream_t s) {
  return ci == 2 ? launch_mg_ci<2>(pro, epi, a, p, s) : launch_mg_ci<8>(pro, epi, a, p, s);
}

int launch_gemv(int pro, int epi, int ci, const GemvArgs& a, void* stream) {
  hipStream_t s = (hipStream_t)stream;
  if (a.Kp * 64 > kMaxK || a.Kp <= 0 || a.N <= 0 || (ci != 1 && ci != 2 && ci != 8) || a.N % (64 / ci) ||
      a.KpS != (a.Kp + ci - 1) / ci)
    return (int)hipErrorInvalidValue;
  if (pro != PRO_NONE && a.Kp * 64 > kMaxEPT / 4 * 256) return (int)hipErrorInvalidValue;
  if (epi == EPI_GEGLU && pro != PRO_RESID_NORM) return (int)hipErrorInvalidValue;
  MgPlan plan;
  if (pro == PRO_ATTN_MERGE) {   // only the multi-group kernel merges: K = n_q * 256 <= 1024 on 256 threads
    if (ci == 1 || a.Kp * 64 > kAttnMaxQ * kHeadDim || a.Kp % 4 || a.attn_chunks < 1 ||
        a.attn_chunks > kDecMaxChunks || !mg_plan(a, pro, ci, plan))
      return (int)hipErrorInvalidValue;
    return launch_mg(pro, epi, ci, a, plan, s);
  }
  if (ci != 1 && mg_plan(a, pro, ci, plan)) return launch_mg(pro, epi, ci, a, plan, s);
  if (epi == EPI_GEGLU) return launch_gemv_ci<PRO_RESID_NORM, EPI_GEGLU>(ci, a, s);
  if (pro == PRO_NONE) return launch_gemv_ci<PRO_NONE, EPI_OUT>(ci, a, s);
  if (pro == PRO_EMBED_NORM) return launch_gemv_ci<PRO_EMBED_NORM, EPI_OUT>(ci, a, s);
  if (pro == PRO_RESID_NORM) return launch_gemv_ci<PRO_RESID_NORM, EPI_OUT>(ci, a, s);
  return (int)hipErrorInvalidValue;
}

int launch_attention(const AttnArgs& a, int grid, void* stream) {
  if (a.n_q < 1 || a.n_q > kAttnMaxQ || grid < 1 || grid > kDecMaxChunks) return (int)hipErrorInvalidValue;
  if (grid <= kDecMergeInO) hipLaunchKernelGGL(k_attn_dec<1>, dim3(grid, a.n_q), dim3(256), 0, (hipStream_t)stream, a);
  else hipLaunchKernelGGL(k_attn_dec<kAttnMaxQ>, dim3(grid), dim3(256), 0, (hipStream_t)stream, a);
  return (int)hipGetLastError();
}

int launch_attention_merge(const AttnArgs& a, int chunks, void* stream) {
  if (a.n_q < 1 || a.n_q > kAttnMaxQ || chunks < 1 || chunks > kDecMaxChunks || !a.part || !a.attn_out)
    return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(k_attn_merge, dim3(kHeadDim / 32, a.n_q), dim3(256), 0, (hipStream_t)stream, a, chunks);
  return (int)hipGetLastError();
}

int launch_prefill_attention(const AttnArgs& a, int M, void* stream) {
  if (a.n_q < 1 || a.n_q > kAttnMaxQ || M < 1 || a.pf_rows != M || a.pf_start < 0 || a.window < 0 || a.pf_chunk < 1 ||
      (a.pf_rt != 1 && a.pf_rt != 2) || !a.q_frag || !a.kv_planes)
    return (int)hipErrorInvalidValue;
  const int nkc = (prefill_max_tiles(a.window, a.pf_start, M, 16 * a.pf_rt) + a.pf_chunk - 1) / a.pf_chunk;
  if (nkc > kPrefillChunks) return (int)hipErrorInvalidValue;   // `part` holds kPrefillChunks per row
  const dim3 grid(nkc, (M + 16 * a.pf_rt - 1) / (16 * a.pf_rt));
  if (a.pf_rt == 1) hipLaunchKernelGGL(k_attn_pf<1>, grid, dim3(256), 0, (hipStream_t)stream, a);
  else hipLaunchKernelGGL(k_attn_pf<2>, grid, dim3(256), 0, (hipStream_t)stream, a);
  if (nkc > 1) hipLaunchKernelGGL(k_attn_pf_merge, dim3(M), dim3(256), 0, (hipStream_t)stream, a);
  return (int)hipGetLastError();
}

int launch_final(const FinalArgs& a, void* stream) {
  if (a.H > 2048) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(k_final, dim3(1), dim3(256), 0, (hipStream_t)stream, a);
  return (int)hipGetLastError();
}

int launch_select(const SelectArgs& a, void* stream) {
  const int stripes = (a.V + 255) / 256;
  const int nb = stripes < kSelBlocks ? stripes : kSelBlocks;
  hipLaunchKernelGGL(k_select1, dim3(nb), dim3(256), 0, (hipStream_t)stream, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(k_select2, dim3(1), dim3(256), 0, (hipStream_t)stream, a, nb);
  return (int)hipGetLastError();
}

int launch_repack(const uint8_t* src, uint8_t* dst, const Q8Layout& L, long long rows, long long off, int half,
                  void* stream) {
  const long long total = rows * L.Kp;
  if (total <= 0) return 0;
  hipLaunchKernelGGL(k_repack, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream, src,
                     dst, rows, L, off, half);
  return (int)hipGetLastError();
}

int launch_embed_row(const uint8_t* embd, int kps, float scale, int token, int H, float* out, void* stream) {
  hipLaunchKernelGGL(k_embed_row, dim3(1), dim3(256), 0, (hipStream_t)stream, embd, kps, scale, token, H, out);
  return (int)hipGetLastError();
}

int launch_repack_gum(const uint8_t* src, uint8_t* dst, long long rows, int K, int up, void* stream) {
  if (rows <= 0 || rows % 32 || K <= 0 || K % 64) return (int)hipErrorInvalidValue;
  const int Kp = K / 64, Kh = (Kp + 1) / 2;
  const long long total = rows / 32 * (Kp * 2 * 64 + 2 * Kh * 32);
  hipLaunchKernelGGL(k_repack_gum, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream, src,
                     dst, rows, K, up);
  return (int)hipGetLastError();
}

int launch_repack_colblock(const uint8_t* src, uint8_t* dst, long long rows, int K, void* stream) {
  if (rows <= 0 || K <= 0 || K % 32) return (int)hipErrorInvalidValue;
  const long long total = rows * (K / 32);
  hipLaunchKernelGGL(k_repack_colblock, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     src, dst, rows, K / 32);
  return (int)hipGetLastError();
}

int launch_class_major(const uint8_t* src, uint8_t* dst, long long rows, int Kp, void* stream) {
  if (rows <= 0 || rows % 16384 || Kp <= 0) return (int)hipErrorInvalidValue;
  const long long total = rows * Kp;
  hipLaunchKernelGGL(k_class_major, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream, src,
                     dst, rows, Kp);
  return (int)hipGetLastError();
}

int launch_q8_bf16(const uint8_t* src, uint16_t* wb, float* wd, long long rows, int K, long long off, int half,
                   int act_order, void* stream) {
  if (K % 32 || off < 0 || (half != 0 && half != 16)) return (int)hipErrorInvalidValue;
  const long long total = rows * (K / 32);
  if (total <= 0) return 0;
  hipLaunchKernelGGL(k_q8_bf16, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream, src, wb,
                     wd, rows, K, off, half, act_order);
  return (int)hipGetLastError();
}

int launch_logits_rows(const float* cm, float* out, int V, void* stream) {
  if (V <= 0 || V % 256) return (int)hipErrorInvalidValue;
  const int R = V / 256;
  hipLaunchKernelGGL(k_logits_rows, dim3((R + 63) / 64, 4), dim3(256), 0, (hipStream_t)stream, cm, out, R);
  return (int)hipGetLastError();
}

// Sizes for k_dequant16 (measured beside it).
static bool dequant_wide(long long n) { return n >= 786432 || (n >= 512 && n <= 3 * 32 * kDeqBlocks); }

int launch_dequant(const uint8_t* src, float* out, long long n, void* stream) {
  if (n <= 0) return 0;
  if (n % 32 == 0 && ((uintptr_t)src | (uintptr_t)out) % 16 == 0 && dequant_wide(n)) {
    const long long nblk = n / 32;
    hipLaunchKernelGGL(k_dequant16, dim3((unsigned)((nblk + kDeqBlocks - 1) / kDeqBlocks)), dim3(256), 0,
                       (hipStream_t)stream, src, out, nblk);
    return (int)hipGetLastError();
  }
  hipLaunchKernelGGL(k_dequant, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, src, out,
                     n);
  return (int)hipGetLastError();
}

template <int EPI, int MI, int NJ, int PW, int PA, int OCC, int KG = 1>
static int launch_gemm_t(const GemmArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((k_gemm<EPI, MI, NJ, PW, PA, OCC, KG>),
                     dim3(a.N / (64 * NJ), (a.M + 16 * MI - 1) / (16 * MI), a.ks), dim3(256 * KG), 0, s, a);
  return (int)hipGetLastError();
}

int launch_gemm(int epi, const GemmArgs& a, void* stream) {
  if (a.tile < 0 || a.tile >= GT_COUNT) return (int)hipErrorInvalidValue;
  const GemmTile& t = kGemmTiles[a.tile];
  if (a.M < 1 || a.N < 64 || a.N % (64 * t.nj) || !((epi == EPI_OUT ? t.lat : t.glat) > 0.f) || a.K < 64 || a.ks < 1 ||
      a.ks > kGemmMaxSlices || a.K % (32 * a.ks) || !a.A || !a.W || !a.D ||
      (epi == EPI_OUT ? !a.C : (!a.act || a.ks != 1)))
    return (int)hipErrorInvalidValue;
  hipStream_t s = (hipStream_t)stream;
  if (epi == EPI_GEGLU) {
    switch (a.tile) {
      case GT_32x128: return launch_gemm_t<EPI_GEGLU, 2, 2, 3, 2, 4>(a, s);
      case GT_32x128_K2: return launch_gemm_t<EPI_GEGLU, 2, 2, 3, 2, 4, 2>(a, s);
      case GT_64x128: return launch_gemm_t<EPI_GEGLU, 4, 2, 3, 2, 3>(a, s);
      case GT_64x256: return launch_gemm_t<EPI_GEGLU, 4, 4, 1, 1, 3>(a, s);
      // two steps of weights in flight spill 9 of its 256 registers (40 bytes a
      // lane, reloaded once per six steps); one step needs 238 and none, and is
      // slower where weights come from HBM: 2048 ids 8.01 against 7.87 ms
      case GT_128x256: return launch_gemm_t<EPI_GEGLU, 8, 4, 2, 1, 2>(a, s);
    }
  } else {
    switch (a.tile) {
      case GT_32x64: return launch_gemm_t<EPI_OUT, 2, 1, 3, 2, 4>(a, s);
      case GT_32x64_K2: return launch_gemm_t<EPI_OUT, 2, 1, 3, 2, 4, 2>(a, s);
      case GT_32x128: return launch_gemm_t<EPI_OUT, 2, 2, 3, 2, 4>(a, s);
      case GT_32x128_K2: return launch_gemm_t<EPI_OUT, 2, 2, 3, 2, 4, 2>(a, s);
      case GT_64x128: return launch_gemm_t<EPI_OUT, 4, 2, 3, 2, 3>(a, s);
      case GT_64x128_K2: return launch_gemm_t<EPI_OUT, 4, 2, 3, 2, 3, 2>(a, s);
      case GT_64x192: return launch_gemm_t<EPI_OUT, 4, 3, 2, 1, 3>(a, s);
    }
  }
  return (int)hipErrorInvalidValue;
}

int launch_rows_embed(const RowArgs& a, void* stream) {
  if (a.H > 2048 || a.M < 1) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(k_rows_embed, dim3(a.M), dim3(256), 0, (hipStream_t)stream, a);
  return (int)hipGetLastError();
}

int launch_rows_resid(const RowArgs& a, void* stream) {
  if (a.H > 2048 || a.M < 1) return (int)hipErrorInvalidValue;
  if (a.H % 4 || a.pre_stride % 4) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(k_rows_resid, dim3(a.M), dim3(256), 0, (hipStream_t)stream, a);
  return (int)hipGetLastError();
}

int launch_rows_kv(const RowArgs& a, void* stream) {
  if (a.M < 1 || a.kv_lo < 0 || a.kv_lo > a.pf_start || !a.q_frag || !a.kv_planes) return (int)hipErrorInvalidValue;
  if (a.n_q < 1 || a.n_q > kAttnMaxQ || a.pre_planes > kQkvMaxSlices ||
      (a.pre_planes > 1 && a.pre_stride < (size_t)a.M * (a.n_q + 2) * kHeadDim))
    return (int)hipErrorInvalidValue;
  const int first = a.kv_lo / kPfKeys, last = (a.pf_start + a.M - 1) / kPfKeys;
  hipLaunchKernelGGL(k_rows_kv, dim3((last - first + 1) * (kPfKeys / kKvPos)), dim3(128 * (a.n_q + 2)), 0,
                     (hipStream_t)stream, a);
  return (int)hipGetLastError();
}

int launch_seen_add(uint32_t* seen, DevState* st, const int32_t* ids, int n, int V, void* stream) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(k_seen_add, dim3(1), dim3(256), 0, (hipStream_t)stream, seen, st, ids, n, V);
  return (int)hipGetLastError();
}

}  // namespace gg
