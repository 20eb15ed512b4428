// Importance scoring for the expert-level keep rule: the attention
// probabilities of the last query over every key, averaged over heads.
//
// Replaces HybridQwen3Attention._compute_and_cache_importance
// (models/qwen3_vl_moe/hybrid_attention.py:111-146: scores = (last_q K^T) in
// the model dtype, times `scaling` in the model dtype, softmax in fp32, mean
// over heads) and the DeepSeek variant _cache_last_token_attention
// (models/deepseek_vl2/deepseek_attention.py:206-249: fp32 scores, padded
// keys excluded, the last query_length keys kept).  Its output feeds
// tm_expert_keep_mask (the reference's build_prefill_keep_mask).
//
// Two launches.  scores_kernel: one workgroup per (key chunk, set of HG heads
// that share a KV head, batch row); 8 lanes per key (each lane a D / 8 slice,
// fp32 products summed in lane order, then an 8-lane DPP tree), every key read
// once for the set's heads; the chunk's scores to the workspace and each
// head's softmax statistics (max m_c, l_c = sum exp(s - m_c)).  mean_kernel: 64
// output keys per workgroup, a quarter of the heads per thread; per head, M =
// max_c m_c and L = sum_c l_c exp(m_c - M), p = exp(s - M) / L, then the p of
// each quarter summed in head order, the quarters in order, and divided by the
// head count.
//
// Both are chains of a few memory round trips, so what counts is how many
// workgroups share them: chunks of 64 keys (260 workgroups at 4099 keys of 4
// KV heads) instead of 512, and 64 keys x 4 head quarters instead of 256 keys
// x all heads (65 workgroups instead of 17).  Chunks of 512 keys stay for long
// prompts, whose statistics every workgroup of the mean reads, and for calls
// whose workspace holds no more.  32 heads on 4 KV heads, us before (one head per
// workgroup, 256 keys x all heads) and now: 4099 keys 14.8 + 16.3, 5.9 + 6.0; both
// together 16384 keys 39, 22; 16385 51, 24; 131072 141, 65; 524288 893, 355.
#include "tm_internal.h"
#include "tm_route_dev.h"

#include <type_traits>

namespace {

constexpr int kThreads = 256;  // 32 keys per pass (8 lanes each)
constexpr int kMaxHeads = 256;
constexpr int kMaxChunks = 1024;
constexpr int kShortKeys = 16384;  // up to here chunks of 64 keys, then of 512
constexpr int kMaxKeys = 512 * kMaxChunks;
constexpr int kMeanKeys = 64;      // output keys per workgroup of mean_kernel
constexpr int kBatch = 8;          // scores and statistics loaded per round trip

// Workspace of a call with chunks of `chunk` keys: scores, then statistics.
inline size_t score_bytes(int64_t batch, int n_heads, int64_t n_keys) {
  return ((size_t)batch * n_heads * n_keys * sizeof(float) + 255) / 256 * 256;
}
inline size_t ws_bytes(int64_t batch, int n_heads, int64_t n_keys, int chunk) {
  return score_bytes(batch, n_heads, n_keys) + (size_t)batch * n_heads * tm_cdiv(n_keys, chunk) * sizeof(float2);
}

// Maximum / sum over the wave in every lane (DPP: row shifts, row broadcasts).
__device__ __forceinline__ float wave_max_f(float v) {
  auto st = [&](auto c) {
    v = fmaxf(v, __uint_as_float(tm_dpp<decltype(c)::value>(__float_as_uint(v), __float_as_uint(v))));
  };
  st(std::integral_constant<int, 0x111>{});
  st(std::integral_constant<int, 0x112>{});
  st(std::integral_constant<int, 0x114>{});
  st(std::integral_constant<int, 0x118>{});
  v = fmaxf(v, __uint_as_float(tm_dpp<0x142, 0xA>(__float_as_uint(v), __float_as_uint(v))));
  v = fmaxf(v, __uint_as_float(tm_dpp<0x143, 0xC>(__float_as_uint(v), __float_as_uint(v))));
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), 63));
}
__device__ __forceinline__ float wave_sum_f(float v) {
  auto st = [&](auto c) { v += __uint_as_float(tm_dpp<decltype(c)::value>(0u, __float_as_uint(v))); };
  st(std::integral_constant<int, 0x111>{});
  st(std::integral_constant<int, 0x112>{});
  st(std::integral_constant<int, 0x114>{});
  st(std::integral_constant<int, 0x118>{});
  v += __uint_as_float(tm_dpp<0x142, 0xA>(0u, __float_as_uint(v)));
  v += __uint_as_float(tm_dpp<0x143, 0xC>(0u, __float_as_uint(v)));
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), 63));
}

template <int DT, int CH, int HG, int PASSES>
__global__ __launch_bounds__(kThreads) void scores_kernel(
    const typename Elem<DT>::T *__restrict__ q, int64_t qs_b, int64_t qs_h, const typename Elem<DT>::T *__restrict__ k,
    int64_t ks_b, int64_t ks_s, int64_t ks_h, int n_heads, int groups, int64_t n_keys, float scale, int score_mode,
    const uint8_t *__restrict__ key_mask, int64_t km_b, float *__restrict__ sc, float2 *__restrict__ stats) {
  using T = typename Elem<DT>::T;
  constexpr int kChunk = 32 * PASSES;
  constexpr int kAhead = PASSES < 4 ? PASSES : 4;  // passes whose keys are in flight together
  // head dim 64 * CH: lane `sub` of a key's 8 lanes holds chunks sub, sub + 8, ... (8 elements each)
  const int c = (int)blockIdx.x, h0 = (int)blockIdx.y * HG;
  const int64_t b = blockIdx.z;
  const int tid = threadIdx.x, sub = tid & 7, grp = tid >> 3;
  __shared__ float tile[HG][kChunk];
  const int64_t t0 = (int64_t)c * kChunk;
  const T *const kb = k + b * ks_b + (int64_t)(h0 / groups) * ks_h;
  float qv[HG][CH][8];
#pragma unroll
  for (int h = 0; h < HG; ++h)
#pragma unroll
    for (int j = 0; j < CH; ++j) tm_load8<DT>(q + b * qs_b + (int64_t)(h0 + h) * qs_h + (j * 8 + sub) * 8, qv[h][j]);
#pragma unroll 1
  for (int it0 = 0; it0 < PASSES; it0 += kAhead) {
    float kv[kAhead][CH][8];
#pragma unroll
    for (int a = 0; a < kAhead; ++a) {
      const int64_t t = t0 + (it0 + a) * 32 + grp;
      const T *kr = kb + (t < n_keys ? t : n_keys - 1) * ks_s;
#pragma unroll
      for (int j = 0; j < CH; ++j) tm_load8<DT>(kr + (j * 8 + sub) * 8, kv[a][j]);
    }
#pragma unroll
    for (int a = 0; a < kAhead; ++a)
#pragma unroll
      for (int h = 0; h < HG; ++h) {
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < CH; ++j)
#pragma unroll
          for (int i = 0; i < 8; ++i) acc = fmaf(qv[h][j][i], kv[a][j][i], acc);
        acc += tm_g8f<kG8Steps[0]>(acc);
        acc += tm_g8f<kG8Steps[1]>(acc);
        acc += tm_g8f<kG8Steps[2]>(acc);
        const float s = score_mode == TM_SCORE_MODEL ? tm_round<DT>(tm_round<DT>(acc) * scale) : acc * scale;
        if (sub == (h & 7)) tile[h][(it0 + a) * 32 + grp] = s;
      }
  }
  // which of this lane's keys count, for the statistics below
  const int lane = tid & 63, wave = tid >> 6;
  bool ok[kChunk / 64 > 0 ? kChunk / 64 : 1];
#pragma unroll
  for (int i = 0; i < kChunk / 64; ++i) {
    const int64_t t = t0 + i * 64 + lane;
    ok[i] = t < n_keys && (key_mask == nullptr || key_mask[b * km_b + (t < n_keys ? t : n_keys - 1)] != 0);
  }
  __syncthreads();
  // a wave per head: the scores out, the chunk's max, then the sum of
  // exp(s - max) over its valid keys
  for (int h = wave; h < HG; h += kThreads / 64) {
    float sv[kChunk / 64];
    float m = -__builtin_huge_valf();
#pragma unroll
    for (int i = 0; i < kChunk / 64; ++i) {
      sv[i] = tile[h][i * 64 + lane];
      m = ok[i] ? fmaxf(m, sv[i]) : m;
      const int64_t t = t0 + i * 64 + lane;
      if (t < n_keys) sc[(b * n_heads + h0 + h) * n_keys + t] = sv[i];
    }
    m = wave_max_f(m);
    float l = 0.f;
#pragma unroll
    for (int i = 0; i < kChunk / 64; ++i)  // (a chunk may hold scores of -inf alone: they add nothing)
      l += ok[i] && sv[i] != -__builtin_huge_valf() ? expf(sv[i] - m) : 0.f;
    l = wave_sum_f(l);
    if (lane == 0) stats[(b * n_heads + h0 + h) * gridDim.x + c] = make_float2(m, l);
  }
}

__global__ __launch_bounds__(kThreads) void mean_kernel(const float *__restrict__ sc, const float2 *__restrict__ stats,
                                                       int n_heads, int lanes_log2, int n_chunks, int64_t n_keys,
                                                       const uint8_t *__restrict__ key_mask, int64_t km_b,
                                                       int64_t out_len, float *__restrict__ out, int64_t ld_out) {
  __shared__ float hm[kMaxHeads], hl[kMaxHeads];
  __shared__ float part[kThreads / kMeanKeys][kMeanKeys];
  const int64_t b = blockIdx.y;
  const int tid = threadIdx.x;
  // thread: output key tid % 64, heads [ha, hb) (a quarter of them); its first
  // scores are requested before the statistics
  const int64_t j = (int64_t)blockIdx.x * kMeanKeys + (tid & (kMeanKeys - 1));
  const int64_t t = n_keys - out_len + (j < out_len ? j : out_len - 1);
  const int per = (n_heads + 3) / 4, ha = (tid / kMeanKeys) * per;
  const int hb = ha + per < n_heads ? ha + per : n_heads;
  const float *const col = sc + b * n_heads * n_keys + t;
  float s0[kBatch];
#pragma unroll
  for (int i = 0; i < kBatch; ++i) s0[i] = col[(int64_t)(ha + i < n_heads ? ha + i : n_heads - 1) * n_keys];
  const bool valid = key_mask == nullptr || key_mask[b * km_b + t] != 0;
  // the chunk statistics of head h, combined by 1 << lanes_log2 lanes
  const int lanes = 1 << lanes_log2, lane = tid & (lanes - 1);
  for (int hbase = 0; hbase < n_heads; hbase += kThreads >> lanes_log2) {
    const int h = hbase + (tid >> lanes_log2);
    const float2 *st = stats + (b * n_heads + (h < n_heads ? h : n_heads - 1)) * n_chunks;
    float M = -__builtin_huge_valf(), L = 0.f;
    for (int c0 = lane; c0 < n_chunks; c0 += lanes * kBatch) {
      float2 v[kBatch];
      float m = M;
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const int cc = c0 + i * lanes;
        v[i] = st[cc < n_chunks ? cc : n_chunks - 1];
        if (cc >= n_chunks) v[i] = make_float2(-__builtin_huge_valf(), 0.f);
        m = fmaxf(m, v[i].x);
      }
      // (where a maximum is -inf its sum is 0, or NaN from NaN scores, which stays)
      L *= M == -__builtin_huge_valf() ? 0.f : expf(M - m);
#pragma unroll
      for (int i = 0; i < kBatch; ++i) L += v[i].y == 0.f ? 0.f : v[i].y * expf(v[i].x - m);
      M = m;
    }
    for (int o = 1; o < lanes; o <<= 1) {
      const float om = __shfl_xor(M, o, 64), ol = __shfl_xor(L, o, 64);
      const float m = fmaxf(M, om);
      L = L * (M == -__builtin_huge_valf() ? 0.f : expf(M - m)) + ol * (om == -__builtin_huge_valf() ? 0.f : expf(om - m));
      M = m;
    }
    if (lane == 0 && h < n_heads) {
      hm[h] = M;
      hl[h] = L;
    }
  }
  __syncthreads();
  float acc = 0.f;
  for (int hh = ha; hh < hb; hh += kBatch) {
    float s1[kBatch];  // the next batch
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int hn = hh + kBatch + i;
      s1[i] = hh + kBatch < hb ? col[(int64_t)(hn < n_heads ? hn : n_heads - 1) * n_keys] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int h = hh + i < hb ? hh + i : hb - 1;
      const float p = expf(s0[i] - hm[h]) / hl[h];
      acc += (hh + i < hb && valid && hl[h] > 0.f) ? p : 0.f;
    }
#pragma unroll
    for (int i = 0; i < kBatch; ++i) s0[i] = s1[i];
  }
  part[tid / kMeanKeys][tid & (kMeanKeys - 1)] = acc;
  __syncthreads();
  if (tid < kMeanKeys && j < out_len)
    out[b * ld_out + j] = (((part[0][tid] + part[1][tid]) + part[2][tid]) + part[3][tid]) / (float)n_heads;
}

template <int DT, int CH>
void launch_scores(int chunk, const void *q, int64_t qs_b, int64_t qs_h, const void *k, int64_t ks_b, int64_t ks_s, int64_t ks_h,
                   int64_t batch, int n_heads, int groups, int64_t n_keys, float scale, int score_mode,
                   const uint8_t *key_mask, int64_t km_b, float *sc, float2 *stats, hipStream_t s) {
  using T = typename Elem<DT>::T;
  auto launch = [&](auto hg_c, auto passes_c) {
    constexpr int HG = decltype(hg_c)::value, PASSES = decltype(passes_c)::value;
    const dim3 grid((unsigned)tm_cdiv(n_keys, chunk), (unsigned)(n_heads / HG), (unsigned)batch);
    hipLaunchKernelGGL((scores_kernel<DT, CH, HG, PASSES>), grid, dim3(kThreads), 0, s, static_cast<const T *>(q),
                       qs_b, qs_h, static_cast<const T *>(k), ks_b, ks_s, ks_h, n_heads, groups, n_keys, scale,
                       score_mode, key_mask, km_b, sc, stats);
  };
  auto heads = [&](auto hg_c) {
    if (chunk == 64) launch(hg_c, std::integral_constant<int, 2>{});
    else launch(hg_c, std::integral_constant<int, 16>{});
  };
  // heads per workgroup: as many of a KV head's as the registers hold
  if (CH <= 2 && groups % 8 == 0) heads(std::integral_constant<int, CH <= 2 ? 8 : 4>{});
  else if (groups % 4 == 0) heads(std::integral_constant<int, 4>{});
  else if (groups % 2 == 0) heads(std::integral_constant<int, 2>{});
  else heads(std::integral_constant<int, 1>{});
}

}  // namespace

extern "C" size_t tm_importance_workspace_size(int64_t batch, int32_t n_heads, int64_t n_keys) {
  if (batch <= 0 || n_heads <= 0 || n_keys <= 0) return 0;
  // never less than that of a shorter prompt, so one buffer serves every prompt up to the one it was sized for
  const size_t chunks64 = ws_bytes(batch, n_heads, n_keys < kShortKeys ? n_keys : kShortKeys, 64);
  const size_t chunks512 = ws_bytes(batch, n_heads, n_keys, 512);
  return chunks64 > chunks512 ? chunks64 : chunks512;
}

extern "C" int tm_last_query_importance(int32_t dtype, const void *q, int64_t qs_b, int64_t qs_h, const void *k,
                                        int64_t ks_b, int64_t ks_s, int64_t ks_h, int64_t batch, int32_t n_heads,
                                        int32_t n_kv_heads, int32_t head_dim, int64_t n_keys, float scale,
                                        int32_t score_mode, const uint8_t *key_mask, int64_t km_b, int64_t out_len,
                                        float *out, int64_t ld_out, void *workspace, size_t workspace_bytes,
                                        tm_stream_t stream) {
  TM_REQUIRE(batch >= 0 && n_heads >= 1 && n_heads <= kMaxHeads && n_kv_heads >= 1 && n_heads % n_kv_heads == 0 &&
                 n_keys >= 0 && n_keys <= kMaxKeys && out_len >= 0 && out_len <= n_keys &&
                 ld_out >= out_len && batch < 65536,
             TM_EINVAL_SHAPE, "tm_last_query_importance: bad sizes (heads <= %d, keys <= %d)", kMaxHeads,
             kMaxKeys);
  TM_REQUIRE(head_dim == 64 || head_dim == 128 || head_dim == 192 || head_dim == 256, TM_EINVAL_SHAPE,
             "tm_last_query_importance: head_dim %d not in {64, 128, 192, 256}", head_dim);
  TM_REQUIRE(score_mode == TM_SCORE_MODEL || score_mode == TM_SCORE_F32, TM_EINVAL_ARG,
             "tm_last_query_importance: bad score mode");
  if (batch == 0 || n_keys == 0 || out_len == 0) return TM_OK;
  TM_REQUIRE(q && k && out, TM_EINVAL_ARG, "tm_last_query_importance: null pointer");
  const size_t need = ws_bytes(batch, n_heads, n_keys, 512);
  TM_REQUIRE(workspace != nullptr && workspace_bytes >= need && tm_aligned16(workspace), TM_EWORKSPACE,
             "tm_last_query_importance: workspace %zu bytes < %zu", workspace_bytes, need);
  hipStream_t s = tm_hip_stream(stream);
  // short prompts run in chunks of 64 keys where their statistics fit
  const int chunk = n_keys <= kShortKeys && workspace_bytes >= ws_bytes(batch, n_heads, n_keys, 64) ? 64 : 512;
  float *sc = static_cast<float *>(workspace);
  float2 *stats = reinterpret_cast<float2 *>(static_cast<char *>(workspace) + score_bytes(batch, n_heads, n_keys));
  const int groups = n_heads / n_kv_heads;
  return TM_DISPATCH_DTYPE(dtype, DT, [&] {
    const int E = Elem<DT>::kBytes;
    TM_REQUIRE(tm_aligned16(q) && tm_aligned16(k) && (qs_b * E) % 16 == 0 && (qs_h * E) % 16 == 0 &&
                   (ks_b * E) % 16 == 0 && (ks_s * E) % 16 == 0 && (ks_h * E) % 16 == 0,
               TM_EINVAL_SHAPE, "tm_last_query_importance: q/k rows must be 16-byte aligned");
    if constexpr (DT == TM_DT_F32) {
      TM_REQUIRE(score_mode == TM_SCORE_F32, TM_EINVAL_ARG, "tm_last_query_importance: fp32 inputs score in fp32");
    }
    switch (head_dim) {
      case 64: launch_scores<DT, 1>(chunk, q, qs_b, qs_h, k, ks_b, ks_s, ks_h, batch, n_heads, groups, n_keys, scale, score_mode, key_mask, km_b, sc, stats, s); break;
      case 128: launch_scores<DT, 2>(chunk, q, qs_b, qs_h, k, ks_b, ks_s, ks_h, batch, n_heads, groups, n_keys, scale, score_mode, key_mask, km_b, sc, stats, s); break;
      case 192: launch_scores<DT, 3>(chunk, q, qs_b, qs_h, k, ks_b, ks_s, ks_h, batch, n_heads, groups, n_keys, scale, score_mode, key_mask, km_b, sc, stats, s); break;
      default: launch_scores<DT, 4>(chunk, q, qs_b, qs_h, k, ks_b, ks_s, ks_h, batch, n_heads, groups, n_keys, scale, score_mode, key_mask, km_b, sc, stats, s); break;
    }
    TM_LAUNCH_CHECK("tm_last_query_importance(scores)");
    int lanes_log2 = 0;  // lanes per head that combine its chunk statistics
    while (lanes_log2 < 6 && (kThreads >> (lanes_log2 + 1)) >= n_heads) ++lanes_log2;
    hipLaunchKernelGGL(mean_kernel, dim3((unsigned)tm_cdiv(out_len, kMeanKeys), (unsigned)batch), dim3(kThreads), 0, s,
                       sc, stats, (int)n_heads, lanes_log2, (int)tm_cdiv(n_keys, chunk), n_keys, key_mask,
                       km_b, out_len, out, ld_out);
    TM_LAUNCH_CHECK("tm_last_query_importance(mean)");
    return TM_OK;
  });
}
