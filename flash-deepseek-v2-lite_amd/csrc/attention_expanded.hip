// q_len = 1 decode attention over an EXPANDED per-head K/V cache ([B, H, L, Dq] keys,
// [B, H, L, Dv] values, bf16): the reference's batched_attention_decode_q1_triton surface.
// The decode step itself never uses it (it reads the compressed 576-wide latent cache);
// it is here so a caller that keeps the reference's expanded cache layout can still call
// that function.
//
// Bound by the cache stream (every K and V row is read once, by one workgroup).  One 8-wave
// workgroup per (row, head, split of the tokens).  Eight lanes share a token: lane k of the
// group holds 16-byte chunks k, k + 8, ... of its K and V rows, so one load instruction
// covers 8 tokens x 128 contiguous bytes, and a group's 4 tokens (20 chunks per lane at
// Dq = 192, Dv = 128) are requested together.  Every 8-lane group keeps an online softmax
// (m, l, O) of its own -- nothing is exchanged and no barrier is met until the tokens are
// done, then the 8 groups of a wave meet by lane swaps and the 8 waves in LDS; fp32
// throughout, one bf16 round.  (Staging 64-token chunks through LDS with three barriers each kept
// one chunk's loads in flight at a time.)  MI355X, 12 rows x 16 heads x 1,381 tokens of 192 + 128
// dims (170 MB): 178 -> 28 us with five such caches read in turn (6.0 TB/s; the same one again 26,
// partly from the last-level cache).
#include "common.h"

namespace {
constexpr int kWaves = 8;
constexpr int kGroups = 8;              // 8-lane token groups per wave
constexpr int kTok = 4;                 // tokens of a group requested together
constexpr int kPass = kWaves * kGroups * kTok;  // tokens per workgroup pass
}  // namespace

struct ExpandedArgs {
  const bf16_t *q, *k, *v;
  int64_t qsb, qsh, ksb, ksh, kss, vsb, vsh, vss;
  bf16_t* out;
  int64_t osb, osh;
  int qd, vd, L, split_tokens, splits;
  const int64_t* cache_position;
  float scale_log2;
  int32_t* status;
  float* part;  // splits > 1: [B, H, splits, Dv + 2] fp32 (O, then m and l)
};

// the tokens a call attends: 0..cache_position, at most L; out-of-range positions are flagged
__device__ __forceinline__ int expanded_len(const ExpandedArgs& a, bool flag) {
  int64_t pos = a.cache_position[0];
  if (pos < 0 || pos >= a.L) {
    if (flag && a.status) atomicOr(a.status, DSV2_DEVERR_CACHE_FULL);
    pos = pos < 0 ? 0 : a.L - 1;
  }
  return static_cast<int>(pos) + 1;
}

// NK / NV: 16-byte chunks of a K / V row per lane (ceil(D / 64))
template <int NK, int NV>
__global__ __launch_bounds__(kWaves * 64, 2) void attention_expanded_kernel(const ExpandedArgs a) {
  __shared__ float s_o[kWaves][NV * 64];
  __shared__ float s_m[kWaves], s_l[kWaves];
  const int sp = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, grp = lane >> 3, k8 = lane & 7;
  const int len = expanded_len(a, tid == 0 && sp == 0 && h == 0 && b == 0);
  const int t_begin = sp * a.split_tokens, t_end = min(len, t_begin + a.split_tokens);
  const bf16_t* qr = a.q + b * a.qsb + h * a.qsh;
  const bf16_t* kr = a.k + b * a.ksb + h * a.ksh;
  const bf16_t* vr = a.v + b * a.vsb + h * a.vsh;
  // chunks past the row's dims read chunk 0 and count as zero (K) or are not stored (V)
  int kc[NK], vc[NV];
  float qf[NK][8];
#pragma unroll
  for (int j = 0; j < NK; ++j) {
    const bool on = (k8 + 8 * j) * 8 < a.qd;
    kc[j] = on ? (k8 + 8 * j) * 8 : 0;
    unpack8(keep_if(on, ldg16(qr + kc[j])), qf[j]);
  }
#pragma unroll
  for (int j = 0; j < NV; ++j) vc[j] = (k8 + 8 * j) * 8 < a.vd ? (k8 + 8 * j) * 8 : 0;
  float m = -INFINITY, l = 0.f, acc[NV][8];
#pragma unroll
  for (int j = 0; j < NV; ++j)
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[j][i] = 0.f;

  for (int c0 = t_begin + wv * kGroups * kTok; c0 < t_end; c0 += kPass) {
    // load u of the wave covers tokens c0 + 8u .. + 7 (one per group); past the end: the last
    uint4 kq[kTok][NK], vq[kTok][NV];
#pragma unroll
    for (int u = 0; u < kTok; ++u) {
      const int64_t t = min(c0 + 8 * u + grp, t_end - 1);
#pragma unroll
      for (int j = 0; j < NK; ++j) kq[u][j] = ldg16_nt(kr + t * a.kss + kc[j]);
    }
#pragma unroll
    for (int u = 0; u < kTok; ++u) {
      const int64_t t = min(c0 + 8 * u + grp, t_end - 1);
#pragma unroll
      for (int j = 0; j < NV; ++j) vq[u][j] = ldg16_nt(vr + t * a.vss + vc[j]);
    }
    float s[kTok];
#pragma unroll
    for (int u = 0; u < kTok; ++u) {
      s[u] = 0.f;
#pragma unroll
      for (int j = 0; j < NK; ++j) {
        const bool on = (k8 + 8 * j) * 8 < a.qd;
        const float d = dot8(kq[u][j], qf[j]);
        s[u] += on ? d : 0.f;
      }
    }
#pragma unroll
    for (int off = 4; off > 0; off >>= 1)
#pragma unroll
      for (int u = 0; u < kTok; ++u) s[u] = xor_sum(s[u], off);
    float mn = m;
#pragma unroll
    for (int u = 0; u < kTok; ++u) {
      s[u] = c0 + 8 * u + grp < t_end ? s[u] * a.scale_log2 : -INFINITY;
      mn = fmaxf(mn, s[u]);
    }
    const float ms = mn == -INFINITY ? 0.f : mn;  // nothing finite so far: every p is 0
    const float alpha = exp2f(m - ms);
    m = mn;
    l *= alpha;
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[j][i] *= alpha;
#pragma unroll
    for (int u = 0; u < kTok; ++u) {
      const bool on = c0 + 8 * u + grp < t_end;
      const float p = exp2f(s[u] - ms);
      l += p;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        float f[8];
        unpack8(keep_if(on, vq[u][j]), f);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[j][i] = __builtin_fmaf(p, f[i], acc[j][i]);
      }
    }
  }

  // the wave's 8 groups (lanes l ^ 8, 16, 32 hold the same chunks), then the workgroup's waves
  float M = m;
#pragma unroll
  for (int off = 32; off >= 8; off >>= 1) M = xor_max(M, off);
  const float f = m == -INFINITY ? 0.f : exp2f(m - M);
  l *= f;
#pragma unroll
  for (int off = 32; off >= 8; off >>= 1) l = xor_sum(l, off);
#pragma unroll
  for (int j = 0; j < NV; ++j)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float x = acc[j][i] * f;
#pragma unroll
      for (int off = 32; off >= 8; off >>= 1) x = xor_sum(x, off);
      acc[j][i] = x;
    }
  if (grp == 0) {
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i) s_o[wv][(k8 + 8 * j) * 8 + i] = acc[j][i];
    if (k8 == 0) {
      s_m[wv] = M;
      s_l[wv] = l;
    }
  }
  __syncthreads();
  if (tid >= a.vd) return;
  float Mw = s_m[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) Mw = fmaxf(Mw, s_m[w]);
  float o = 0.f, lt = 0.f;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const float g = s_m[w] == -INFINITY ? 0.f : exp2f(s_m[w] - Mw);
    lt = __builtin_fmaf(g, s_l[w], lt);
    o = __builtin_fmaf(g, s_o[w][tid], o);
  }
  if (a.splits == 1) {
    a.out[b * a.osb + h * a.osh + tid] = f2bf(o / lt);
    return;
  }
  float* p = a.part + (((int64_t)b * gridDim.y + h) * a.splits + sp) * (a.vd + 2);
  p[tid] = o;
  if (tid == 0) {
    p[a.vd] = Mw;
    p[a.vd + 1] = lt;
  }
}

// one workgroup per (row, head): the splits' (O, m, l) merged in order
__global__ __launch_bounds__(256) void attention_expanded_merge_kernel(const ExpandedArgs a) {
  const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x;
  if (tid >= a.vd) return;
  const int len = expanded_len(a, false);
  const int ns = min((len + a.split_tokens - 1) / a.split_tokens, a.splits);
  const float* p = a.part + ((int64_t)b * gridDim.x + h) * a.splits * (a.vd + 2);
  float M = -INFINITY;
  for (int s = 0; s < ns; ++s) M = fmaxf(M, p[s * (a.vd + 2) + a.vd]);
  float o = 0.f, lt = 0.f;
  for (int s = 0; s < ns; ++s) {
    const float* ps = p + s * (a.vd + 2);
    const float g = ps[a.vd] == -INFINITY ? 0.f : exp2f(ps[a.vd] - M);
    lt = __builtin_fmaf(g, ps[a.vd + 1], lt);
    o = __builtin_fmaf(g, ps[tid], o);
  }
  a.out[b * a.osb + h * a.osh + tid] = f2bf(o / lt);
}

extern "C" int dsv2_attention_decode_expanded(const void* q, int64_t q_stride_b, int64_t q_stride_h, const void* k,
                                              int64_t k_stride_b, int64_t k_stride_h, int64_t k_stride_s,
                                              const void* v, int64_t v_stride_b, int64_t v_stride_h,
                                              int64_t v_stride_s, void* out, int64_t out_stride_b,
                                              int64_t out_stride_h, int batch, int heads, int q_dim, int v_dim,
                                              int seq_len, const int64_t* cache_position, float softmax_scale,
                                              int32_t* status, void* stream) {
  return dsv2_attention_decode_expanded_split(q, q_stride_b, q_stride_h, k, k_stride_b, k_stride_h, k_stride_s, v,
                                              v_stride_b, v_stride_h, v_stride_s, out, out_stride_b, out_stride_h,
                                              batch, heads, q_dim, v_dim, seq_len, cache_position, softmax_scale, 1,
                                              nullptr, status, stream);
}

extern "C" int dsv2_attention_decode_expanded_split(
    const void* q, int64_t q_stride_b, int64_t q_stride_h, const void* k, int64_t k_stride_b, int64_t k_stride_h,
    int64_t k_stride_s, const void* v, int64_t v_stride_b, int64_t v_stride_h, int64_t v_stride_s, void* out,
    int64_t out_stride_b, int64_t out_stride_h, int batch, int heads, int q_dim, int v_dim, int seq_len,
    const int64_t* cache_position, float softmax_scale, int splits, float* workspace, int32_t* status, void* stream) {
  DSV2_REQUIRE(q && k && v && out && cache_position && (splits == 1 || workspace), DSV2_E_NULL,
               "attention_decode_expanded: null pointer");
  DSV2_REQUIRE(batch >= 0 && batch <= 65535 && heads > 0 && heads <= 65535 && q_dim > 0 && q_dim <= 256 &&
                   q_dim % 8 == 0 && v_dim > 0 && v_dim <= 256 && v_dim % 8 == 0 && seq_len > 0,
               DSV2_E_SHAPE, "attention_decode_expanded: bad shape (q_dim, v_dim <= 256 and %% 8, seq_len > 0)");
  DSV2_REQUIRE(splits >= 1 && splits <= 64, DSV2_E_SHAPE, "attention_decode_expanded: 1 to 64 splits");
  DSV2_REQUIRE(dsv2_aligned16(q) && dsv2_aligned16(k) && dsv2_aligned16(v) && q_stride_b % 8 == 0 &&
                   q_stride_h % 8 == 0 && k_stride_b % 8 == 0 && k_stride_h % 8 == 0 && k_stride_s % 8 == 0 &&
                   v_stride_b % 8 == 0 && v_stride_h % 8 == 0 && v_stride_s % 8 == 0,
               DSV2_E_ALIGN, "attention_decode_expanded: rows must be 16-byte aligned (strides %% 8 elements)");
  if (batch == 0) return DSV2_OK;
  ExpandedArgs a{};
  a.q = (const bf16_t*)q;
  a.k = (const bf16_t*)k;
  a.v = (const bf16_t*)v;
  a.qsb = q_stride_b, a.qsh = q_stride_h;
  a.ksb = k_stride_b, a.ksh = k_stride_h, a.kss = k_stride_s;
  a.vsb = v_stride_b, a.vsh = v_stride_h, a.vss = v_stride_s;
  a.out = (bf16_t*)out;
  a.osb = out_stride_b, a.osh = out_stride_h;
  a.qd = q_dim, a.vd = v_dim, a.L = seq_len;
  // splits are whole 32-token wave passes; rounding up may leave the last ones without tokens
  a.split_tokens = (int)((((int64_t)seq_len + splits - 1) / splits + 31) / 32 * 32);
  a.splits = splits;
  a.cache_position = cache_position;
  a.scale_log2 = softmax_scale * 1.4426950408889634f;
  a.status = status;
  a.part = workspace;
  const dim3 grid(splits, heads, batch);
  // 192 / 128 (the model's heads) and anything smaller take 3 + 2 chunks per lane
  if (q_dim <= 192 && v_dim <= 128)
    hipLaunchKernelGGL((attention_expanded_kernel<3, 2>), grid, dim3(kWaves * 64), 0, (hipStream_t)stream, a);
  else
    hipLaunchKernelGGL((attention_expanded_kernel<4, 4>), grid, dim3(kWaves * 64), 0, (hipStream_t)stream, a);
  if (splits > 1)
    hipLaunchKernelGGL(attention_expanded_merge_kernel, dim3(heads, batch), dim3(256), 0, (hipStream_t)stream, a);
  return dsv2_launch_status("attention_decode_expanded");
}
