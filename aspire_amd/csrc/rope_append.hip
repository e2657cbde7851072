// (f2) QK RMSNorm + rotary permute + interleaved RoPE + paged KV append, one launch.
//
// Per layer the reference runs q_norm, k_norm, two permutes, mylib::rope and
// mylib::update_kv_padded (aspire/models/sparse_draft_transformer.py:149-171):
// six launches and four round trips of q / k through HBM. Here a few waves
// take a token: 16 lanes own a head (lane j its rotated pairs 4j .. 4j + 3,
// dims 8j .. 8j + 7 after the permute), normalise and rotate it, write q in
// place and k / v into the page pool at the token's append position.
//
//   * RMSNorm (transformer.py:505-516): fp32 sum of squares (wave sum),
//     x * (1 / sqrt(mean + eps)) rounded to bf16, times the bf16 weight,
//     rounded again;
//   * permute (transformer.py:360-364): output pair i takes input dims i and
//     i + D/2 (the norm weight follows the input dim);
//   * RoPE, FlashInfer's interleaved convention (mixed_transformer.py:159-198):
//     angle = fp32(position) * fp32 frequency (the host computes the D/2
//     frequencies once, including the Llama 3.1 smoothing), accurate sincosf,
//     (a, b) -> (a cos - b sin, b cos + a sin) in fp32, rounded to bf16;
//   * append: the row / slot rule of the plain append (append_locate).
#include <cmath>
#include <type_traits>

#include "common.h"

namespace aspire {
namespace {

constexpr int kPairs = kHeadDim / 2;

struct RopeParams {
  uint16_t* q;
  int64_t q_st, q_sh;
  uint16_t* k;
  int64_t k_st, k_sh;
  const uint16_t* v;
  int64_t v_st, v_sh;
  int32_t hq, hkv;
  const uint16_t* q_w;
  const uint16_t* k_w;
  float eps;
  int32_t permute;
  float freq[kPairs];
  const int32_t* indptr;
  const int32_t* offsets;
  int32_t num_rows;
  uint16_t* cache;
  int64_t c_sp, c_skv, c_st, c_sh;
  int32_t page_size;
  const int32_t* page_indices;
  const int32_t* page_indptr;
  const int32_t* last_page_len;
  int32_t num_seq;
  int32_t write_k;
  const float* partials;  // fp32 slabs [splits][T][(hq + 2 hkv) * 128] of the fused projection, or null
  int32_t splits;
};

// Head slots of one wave pass: 4 groups of 16 lanes, one head each.
constexpr int kRopeHeads = 4;
constexpr int kRopeWaves = 4;   // waves per workgroup
constexpr int64_t kRopeMaxWaves = 2816;  // 11 a CU: waves past that cost more than the passes they spare

__device__ __forceinline__ float lo_bf(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi_bf(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// Sum over the 16 lanes of each DPP row.
__device__ __forceinline__ float row_sum_f(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xF, 0xF, false));
  return v;
}

// The 8 inputs of lane j of a head as 4 words: pairs 4j .. 4j + 3 are dims (4j + e, 64 + 4j + e)
// with the permute (words 0-1: the first halves, 2-3: the second), (8j + 2e, 8j + 2e + 1) without.
template <bool kWide>
__device__ __forceinline__ uint4 load_lane_dims(const uint16_t* row, int j, bool permute) {
  const int d0 = permute ? 4 * j : 8 * j, d1 = permute ? kPairs + 4 * j : 8 * j + 4;
  if (kWide) {
    const uint2 x = *reinterpret_cast<const uint2*>(row + d0), y = *reinterpret_cast<const uint2*>(row + d1);
    return make_uint4(x.x, x.y, y.x, y.y);
  }
  auto word = [&](int d) { return uint32_t(row[d]) | (uint32_t(row[d + 1]) << 16); };
  return make_uint4(word(d0), word(d0 + 2), word(d1), word(d1 + 2));
}
// The same words from a row of fp32 slabs: summed, and rounded once as the projection's output would be.
__device__ __forceinline__ uint4 sum_lane_dims(const float* row, int splits, int64_t slab, int j, bool permute) {
  const int d0 = permute ? 4 * j : 8 * j, d1 = permute ? kPairs + 4 * j : 8 * j + 4;
  float4 a = *reinterpret_cast<const float4*>(row + d0), b = *reinterpret_cast<const float4*>(row + d1);
  for (int k = 1; k < splits; ++k) {
    row += slab;
    const float4 c = *reinterpret_cast<const float4*>(row + d0), d = *reinterpret_cast<const float4*>(row + d1);
    a.x += c.x, a.y += c.y, a.z += c.z, a.w += c.w;
    b.x += d.x, b.y += d.y, b.z += d.z, b.w += d.w;
  }
  return make_uint4(pack_bf16x2_rne(a.x, a.y), pack_bf16x2_rne(a.z, a.w), pack_bf16x2_rne(b.x, b.y), pack_bf16x2_rne(b.z, b.w));
}
__device__ __forceinline__ void split_pairs(const uint4& w, bool permute, float* a, float* b) {
  if (permute) {
    a[0] = lo_bf(w.x), a[1] = hi_bf(w.x), a[2] = lo_bf(w.y), a[3] = hi_bf(w.y);
    b[0] = lo_bf(w.z), b[1] = hi_bf(w.z), b[2] = lo_bf(w.w), b[3] = hi_bf(w.w);
  } else {
    a[0] = lo_bf(w.x), a[1] = lo_bf(w.y), a[2] = lo_bf(w.z), a[3] = lo_bf(w.w);
    b[0] = hi_bf(w.x), b[1] = hi_bf(w.y), b[2] = hi_bf(w.z), b[3] = hi_bf(w.w);
  }
}
__device__ __forceinline__ void round_pair(float& x, float& y) {
  const uint32_t w = pack_bf16x2_rne(x, y);
  x = lo_bf(w);
  y = hi_bf(w);
}

// wpt consecutive waves share a token; wave `part` of them takes head quads part, part + wpt, ...
// of the token's q heads, k heads and (when appending) v heads, in that order. A head is read
// with 8-byte and written with 16-byte accesses (kWide: q, k and the weights allow them), and a
// wave computes the token's 64 angles once, one per lane, handing every lane its four through the
// wave's LDS slice. Bound by HBM at prompt-chunk sizes, by the chain of loads (row search, row
// metadata, page id) plus one sincosf at decode sizes. One wave per (token, head) with 2-byte
// loads, two searches and a sincosf for every head took 168 us for 8,192 tokens of 32 q / 8 kv
// heads (1.2 TB/s, bound by the sincosf and address arithmetic) where this takes 48 us (4.2 TB/s);
// 208 tokens 6.3 -> 4.8 us.
// kSum: the inputs are the slabs of a split projection; q is written to p.q, nothing is read from it.
// kNorm (not with kSum, which looks) / kAppend: with the norm weights / a cache. The rotation alone is 0.15 us
// shorter without their code.
template <bool kWide, bool kSum, bool kNorm, bool kAppend>
__global__ __launch_bounds__(64 * kRopeWaves) void qk_norm_rope_append_kernel(RopeParams p, int total_tokens, int wpt_log2) {
  __shared__ float2 rot[kRopeWaves][kPairs];
  const int lane = threadIdx.x & 63;
  const int wave = wave_uniform(threadIdx.x >> 6);
  const int unit = blockIdx.x * kRopeWaves + wave;
  const int tok = unit >> wpt_log2;
  const int part = unit & ((1 << wpt_log2) - 1);
  if (tok >= total_tokens) return;
  const int j = lane & 15, grp = lane >> 4;
  const bool norm = kSum ? p.q_w != nullptr : kNorm, permute = norm && p.permute != 0;
  const int n_qk = p.hq + p.hkv;
  const int n_all = kAppend && p.v != nullptr ? n_qk + p.hkv : n_qk;
  const int step = kRopeHeads << wpt_log2;

  // a head's words: q / k dims for the rotation, 16 bytes of v for the copy
  auto load = [&](int h) -> uint4 {
    uint4 w = make_uint4(0, 0, 0, 0);
    if (kSum) {
      const int64_t width = int64_t(p.hq + 2 * p.hkv) * kHeadDim;
      if (h < n_all)
        w = sum_lane_dims(p.partials + tok * width + h * kHeadDim, p.splits, total_tokens * width, j, permute && h < n_qk);
    } else if (h < p.hq) {
      w = load_lane_dims<kWide>(p.q + int64_t(tok) * p.q_st + int64_t(h) * p.q_sh, j, permute);
    } else if (h < n_qk) {
      w = load_lane_dims<kWide>(p.k + int64_t(tok) * p.k_st + int64_t(h - p.hq) * p.k_sh, j, permute);
    } else if (kAppend && h < n_all) {
      w = *reinterpret_cast<const uint4*>(p.v + int64_t(tok) * p.v_st + int64_t(h - n_qk) * p.v_sh + 8 * j);
    }
    return w;
  };
  // the first quad's loads and the weights are requested before the position look-up they do not need
  int h = part * kRopeHeads + grp;
  uint4 cur = load(h);
  uint4 qw = make_uint4(0, 0, 0, 0), kw = qw;
  if (norm) {
    qw = load_lane_dims<kWide>(p.q_w, j, permute);
    kw = load_lane_dims<kWide>(p.k_w, j, permute);
  }

  // one search serves both positions: the row b that owns the token (last b with indptr[b] <= tok),
  // and the append's rows are its first num_seq
  int pos = -1;
  uint16_t* page_k = nullptr;
  const int b = wave_last_le(p.indptr, p.num_rows, tok);
  if (b >= 0) {
    const int begin = p.indptr[b], end = p.indptr[b + 1];
    if (tok < end) {
      pos = wave_uniform(p.offsets[b] + tok - begin);
      if (kAppend && b < p.num_seq) {
        const int first = p.page_indptr[b];
        const int pages = p.page_indptr[b + 1] - first;
        const int seq_len = max(pages - 1, 0) * p.page_size + p.last_page_len[b];
        const int ps = tok + seq_len - end;
        if (pages != 0 && ps >= 0 && ps < (pages - 1) * p.page_size + p.last_page_len[b])
          page_k = p.cache + int64_t(p.page_indices[first + ps / p.page_size]) * p.c_sp +
                   int64_t(ps % p.page_size) * p.c_st;
      }
    }
  }

  {
    float c = 1.f, s = 0.f;
    if (pos >= 0) sincosf(static_cast<float>(pos) * p.freq[lane], &s, &c);
    rot[wave][lane] = make_float2(c, s);
  }
  float c[4], s[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float2 r = rot[wave][4 * j + e];
    c[e] = r.x;
    s[e] = r.y;
  }

  for (; wave_uniform(h - grp) < n_all; h += step) {
    const uint4 next = load(h + step);  // heads past the last one load nothing
    const uint4 w = cur;
    cur = next;
    if (h >= n_qk) {
      if (kAppend && h < n_all && page_k != nullptr)
        *reinterpret_cast<uint4*>(page_k + p.c_skv + int64_t(h - n_qk) * p.c_sh + 8 * j) = w;
      continue;
    }
    const bool is_q = h < p.hq;
    float x[4], y[4];
    split_pairs(w, permute, x, y);
    if (norm) {
      float ss = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) ss += x[e] * x[e] + y[e] * y[e];
      const float r = 1.f / sqrtf(row_sum_f(ss) / float(kHeadDim) + p.eps);
      float wx[4], wy[4];
      split_pairs(is_q ? qw : kw, permute, wx, wy);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] *= r;
        y[e] *= r;
        round_pair(x[e], y[e]);
        x[e] *= wx[e];
        y[e] *= wy[e];
        round_pair(x[e], y[e]);
      }
    }
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[e] = pos >= 0 ? pack_bf16x2_rne(x[e] * c[e] - y[e] * s[e], y[e] * c[e] + x[e] * s[e])
                      : pack_bf16x2_rne(x[e], y[e]);
    }
    // every lane of the wave has read its inputs before any lane stores
    if (is_q || p.write_k) {
      uint16_t* row = is_q ? p.q + int64_t(tok) * p.q_st + int64_t(h) * p.q_sh
                           : p.k + int64_t(tok) * p.k_st + int64_t(h - p.hq) * p.k_sh;
      if (kWide) {
        *reinterpret_cast<uint4*>(row + 8 * j) = make_uint4(o[0], o[1], o[2], o[3]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) *reinterpret_cast<uint32_t*>(row + 8 * j + 2 * e) = o[e];
      }
    }
    if (kAppend && !is_q && page_k != nullptr)
      *reinterpret_cast<uint4*>(page_k + int64_t(h - p.hq) * p.c_sh + 8 * j) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

inline bool aligned(const void* ptr, uintptr_t a) { return (reinterpret_cast<uintptr_t>(ptr) & (a - 1)) == 0; }

}  // namespace
}  // namespace aspire

extern "C" int aspire_rope_frequencies(int32_t head_dim, float rope_theta, float rope_scale, int32_t llama31,
                                       float low_freq_factor, float high_freq_factor, float old_context_len,
                                       float* out) {
  using namespace aspire;
  ASPIRE_CHECK_ARG(out && head_dim > 0 && head_dim % 2 == 0, "bad arguments");
  ASPIRE_CHECK_ARG(rope_theta > 0.f && rope_scale > 0.f, "rope_theta and rope_scale must be positive");
  const double two_pi = 6.283185307179586;
  for (int i = 0; i < head_dim / 2; ++i) {
    const double f = std::pow(double(rope_theta), -2.0 * i / head_dim);
    double g = f / rope_scale;
    if (llama31) {
      // Llama 3.1: unchanged above the high-frequency cut, divided by the scale
      // below the low-frequency cut, interpolated in between
      const double wavelen = two_pi / f;
      if (wavelen < double(old_context_len) / high_freq_factor) {
        g = f;
      } else if (wavelen <= double(old_context_len) / low_freq_factor) {
        const double sm = (old_context_len / wavelen - low_freq_factor) / (double(high_freq_factor) - low_freq_factor);
        g = (1.0 - sm) * f / rope_scale + sm * f;
      }
    }
    out[i] = static_cast<float>(g);
  }
  return ASPIRE_OK;
}

namespace {

int prepare_qkv(const aspire_rope_args* a, const float* partials, int32_t splits, void* stream) {
  using namespace aspire;
  ASPIRE_CHECK_ARG(a != nullptr, "null arguments");
  ASPIRE_CHECK_ARG(a->head_dim == kHeadDim, "head_dim must be 128");
  ASPIRE_CHECK_ARG(a->total_tokens >= 0 && a->num_qo_heads >= 0 && a->num_kv_heads >= 0, "bad sizes");
  if (a->total_tokens == 0 || a->num_qo_heads + a->num_kv_heads == 0) return ASPIRE_OK;
  ASPIRE_CHECK_ARG((a->num_qo_heads == 0 || a->q) && (a->num_kv_heads == 0 || a->k || partials), "null q / k");
  ASPIRE_CHECK_ARG(a->num_rows >= 0 && (a->num_rows == 0 || (a->indptr && a->offsets)), "null indptr / offsets");
  ASPIRE_CHECK_ARG((a->q_norm_weight == nullptr) == (a->k_norm_weight == nullptr),
                   "q and k norm weights go together");
  ASPIRE_CHECK_ARG(aligned(a->q, 4) && aligned(a->k, 4) && a->q_stride_h % 2 == 0 && a->k_stride_h % 2 == 0 &&
                       a->q_stride_t % 2 == 0 && a->k_stride_t % 2 == 0,
                   "q / k rows must be 4-byte aligned");
  RopeParams p;
  p.q = static_cast<uint16_t*>(a->q);
  p.q_st = a->q_stride_t;
  p.q_sh = a->q_stride_h;
  p.k = static_cast<uint16_t*>(a->k);
  p.k_st = a->k_stride_t;
  p.k_sh = a->k_stride_h;
  p.v = static_cast<const uint16_t*>(a->v);
  p.v_st = a->v_stride_t;
  p.v_sh = a->v_stride_h;
  p.hq = a->num_qo_heads;
  p.hkv = a->num_kv_heads;
  p.q_w = static_cast<const uint16_t*>(a->q_norm_weight);
  p.k_w = static_cast<const uint16_t*>(a->k_norm_weight);
  p.eps = a->norm_eps;
  p.permute = a->permute && a->q_norm_weight != nullptr;
  p.partials = partials;
  p.splits = splits;
  const int rc = aspire_rope_frequencies(kHeadDim, a->rope_theta, a->rope_scale, a->llama31, a->low_freq_factor,
                                         a->high_freq_factor, a->old_context_len, p.freq);
  if (rc != ASPIRE_OK) return rc;
  p.indptr = a->indptr;
  p.offsets = a->offsets;
  p.num_rows = a->num_rows;
  p.cache = static_cast<uint16_t*>(a->kv_cache);
  p.c_sp = a->cache_stride_p;
  p.c_skv = a->cache_stride_kv;
  p.c_st = a->cache_stride_t;
  p.c_sh = a->cache_stride_h;
  p.page_size = a->page_size;
  p.page_indices = a->kv_page_indices;
  p.page_indptr = a->kv_page_indptr;
  p.last_page_len = a->kv_last_page_len;
  p.num_seq = a->num_seq;
  p.write_k = a->write_k;
  if (p.cache != nullptr) {
    ASPIRE_CHECK_ARG(a->num_seq > 0 && a->num_seq <= a->num_rows, "append rows must be a prefix of the rope rows");
    ASPIRE_CHECK_ARG(a->kv_page_indices && a->kv_page_indptr && a->kv_last_page_len, "null page table");
    ASPIRE_CHECK_ARG(a->page_size > 0, "page_size must be positive");
    ASPIRE_CHECK_ARG(aligned(a->kv_cache, 16) && a->cache_stride_p % 8 == 0 && a->cache_stride_kv % 8 == 0 &&
                         a->cache_stride_t % 8 == 0 && a->cache_stride_h % 8 == 0,
                     "cache must be 16-byte aligned with strides in multiples of 8 elements");
    if (partials != nullptr) p.v = reinterpret_cast<const uint16_t*>(partials);  // the v heads follow in the slabs
    ASPIRE_CHECK_ARG(partials != nullptr || a->v == nullptr || (aligned(a->v, 16) && a->v_stride_t % 8 == 0 && a->v_stride_h % 8 == 0),
                     "v rows must be 16-byte aligned");
  }
  const bool wide = aligned(a->q, 16) && aligned(a->k, 16) && aligned(p.q_w, 8) && aligned(p.k_w, 8) &&
                    a->q_stride_t % 8 == 0 && a->q_stride_h % 8 == 0 && a->k_stride_t % 8 == 0 &&
                    a->k_stride_h % 8 == 0;
  // Waves per token: one for each quad of heads, so that a token is done in one pass of its waves, as
  // long as that keeps the launch within kRopeMaxWaves; past it as many as fit, then 4, which share one sincosf
  // (8,192 tokens: 81 / 62 / 48 us at 16 / 8 / 4). us at 4 / 8 / 16 / 32 waves, 32 q / 8 kv heads (12 quads):
  // 33 tokens 5.7 / 5.0 / 4.4 / 4.6, 160: 5.9 / 5.5 / 5.5 / 6.5, 208: 6.0 / 5.7 / 5.9 / 7.6, 400: 6.9 / 7.0 / 7.6;
  // 64 / 8 (20): 33: 7.1 / 5.7 / 5.0 / 4.6, 104: 7.3 / 5.9 / 5.6 / 5.8, 300: 8.8 / 7.7 / 8.0; 16 / 8 (8): 33: 5.0 / 4.4 /
  // 4.4, 300: 5.7 / 5.4 / 6.4. (One wave a head, as it was once, takes 4.4, 6.0, 7.0 and 10.0 in the first row's places.)
  const int quads = (a->num_qo_heads + a->num_kv_heads * (p.cache && p.v ? 2 : 1) + kRopeHeads - 1) / kRopeHeads;
  int wpt_log2 = 2;
  while ((1 << wpt_log2) < quads && (int64_t(a->total_tokens) << (wpt_log2 + 1)) <= kRopeMaxWaves) ++wpt_log2;
  ASPIRE_CHECK_ARG(partials == nullptr || (p.cache != nullptr && wide && aligned(partials, 16) && splits >= 1 && !a->write_k),
                   "partials need a cache, 16-byte aligned slabs and q rows, and write_k 0");
  const int64_t units = int64_t(a->total_tokens) << wpt_log2;
  const dim3 grid(unsigned((units + kRopeWaves - 1) / kRopeWaves));
  const auto pick = [&](auto kWide, auto kNorm) {
    return p.cache ? qk_norm_rope_append_kernel<kWide(), false, kNorm(), true>
                   : qk_norm_rope_append_kernel<kWide(), false, kNorm(), false>;
  };
  const std::true_type yes;
  const std::false_type no;
  const bool norm = p.q_w != nullptr;
  const auto kernel = p.partials ? qk_norm_rope_append_kernel<true, true, true, true>
                      : wide     ? (norm ? pick(yes, yes) : pick(yes, no))
                                 : (norm ? pick(no, yes) : pick(no, no));
  hipLaunchKernelGGL(kernel, grid, dim3(64 * kRopeWaves), 0, static_cast<hipStream_t>(stream), p, a->total_tokens,
                     wpt_log2);
  ASPIRE_CHECK_LAUNCH();
  return ASPIRE_OK;
}

}  // namespace

extern "C" int aspire_qk_norm_rope_append(const aspire_rope_args* a, void* stream) {
  return prepare_qkv(a, nullptr, 0, stream);
}

extern "C" int aspire_qk_norm_rope_append_partials(const aspire_rope_args* a, const float* partials, int32_t splits,
                                                   void* stream) {
  if (partials == nullptr) return aspire::fail(ASPIRE_ERR_INVALID, "aspire_qk_norm_rope_append_partials: null partials");
  return prepare_qkv(a, partials, splits, stream);
}
