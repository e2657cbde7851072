// Linear layers of a decode step: y[m, n] = sum_k x[m, k] * w[n, k] for up to 224 token rows against
// a weight matrix that is read once; bf16 operands, fp32 accumulation, no compiler-visible copies.
//
// Bound by the weight stream from HBM, and past some 64 rows by what one CU can take in: a CU's loads
// return in order, so x (from L2) queues behind w (from HBM) and w + x together ran at 55-60 GB/s a CU
// whatever the LDS reads and products beside them (a copy without either took the same time; x alone
// from L2 runs at 145 GB/s). So a workgroup takes all rows of x against a tile of 64 to 128 weight
// rows, k is split over workgroups where the tiles do not fill the chip, and the fp32 partial sums go
// to a kernel that reads the layer's output anyway (aspire_add_rms_norm_partials, the q/k preparation).
//   * Both operands travel HBM -> LDS directly (buffer_load ... lds, full 128- or 256-byte row pieces)
//     into rings of 3 to 7 steps of 64 or 128 k: 40-100 KB a CU in flight. Past 64 rows half of the
//     waves load w and half x, so that the w ring can be deeper than the larger x ring.
//   * One barrier a step; a wave multiplies one set of fragments (16x16x32 MFMAs, w as the A operand:
//     a lane's 4 results are 4 neighbouring output columns) while it reads the next.
//   * Workgroups start their walk over k at different places (tile * 7 steps): started together, they
//     all read the same few memory channels (24,576 x 4,096, 12 rows: 43 -> 36 us; 151,936 x 4,096:
//     224 -> 196 us).
// us here / with hipBLASLt's kernels (torch.nn.functional.linear) on MI355X, weights cold:
//   rows   6,144 x 4,096  4,096 x 4,096  24,576 x 4,096 + swiglu  4,096 x 12,288  151,936 x 2,048
//     12    11.6 / 14.3     8.4 / 15.4     36 / 43 + 4             18.5 / 21.5      98 / 203
//     48    14.3 / 17.6     9.9 / 15.0     41 / 46 + 4             21.4 / 36        128 / 152
//    208    21   / 26      16.6 / 21.8     59 / 62 + 5             37   / 50        (203 / 181)
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"

namespace aspire {
namespace {

struct LinearParams {
  const uint16_t* x;
  int64_t x_st;
  const uint16_t* w;
  int64_t w_st;
  uint16_t* out;
  int64_t o_st;
  float* partials;      // [splits][rows][n] fp32, in place of out
  int32_t rows, n, k, splits;   // swiglu: n gate rows of w, then n up rows
};

constexpr uint32_t kBufferConfig = 0x00020000u;  // gfx9 raw buffer dword 3

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

// A raw buffer over [base, base + span): loads past span return zeros.
__device__ __forceinline__ u32x4 buffer_desc(const char* base, int span) {
  const uint64_t v = reinterpret_cast<uint64_t>(base);
  return u32x4{uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(v))),
               uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(v >> 32))) & 0xffffu, uint32_t(span), kBufferConfig};
}

// 64 lanes x 16 bytes from the buffer straight into 1 KiB of LDS at `dst`. Issued from inline asm: for
// the builtin the compiler waits for every such load in flight before the next LDS read, which would
// empty the ring at each step; here the explicit waits before the step barriers order them. The load
// has no register output, so nothing it writes can be reused early.
template <bool kNonTemporal>
__device__ __forceinline__ void load_lds(u32x4 desc, int voff, const uint4* dst) {
  const uint32_t at = wave_uniform(int(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void*)dst)));
  if (kNonTemporal)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen nt lds"
                 :: "s"(at), "v"(voff), "s"(desc) : "memory");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :: "s"(at), "v"(voff), "s"(desc) : "memory");
}

__device__ __forceinline__ float bf_round(float f) { return __uint_as_float(pack_bf16x2_rne(0.f, f) & 0xffff0000u); }

// silu(g) rounded to bf16, times u; the store rounds again (FeedForward, transformer.py:490-502).
__device__ __forceinline__ float swiglu(float g, float u) {
  const float gb = bf_round(g);
  return bf_round(gb / (1.f + expf(-gb))) * bf_round(u);
}

// Chunk c of row q of a stage is placed at c ^ swizzle(q): the 16 rows of a fragment read then cover
// every 16-byte slot of LDS's 64 banks once (128-byte rows: two rows share the banks' 256 bytes).
template <int kCh>
__device__ __forceinline__ int swizzle(int row) {
  return kCh == 8 ? (row >> 1) & 7 : row & 15;
}

enum class Out { kBf16, kPartial, kSwiglu };

// WM x WN waves; wave (wm, wn) computes the 16-row tiles wm, wm + WM, ... (TM of them) of x against TN
// tiles of 16 weight rows. BK: k elements of a step. DW / DA: LDS ring stages of w / x.
template <int WM, int WN, int TM, int TN, int BK, int DW, int DA, bool kRoles, Out kOut>
__global__ __launch_bounds__(64 * WM * WN) void linear_kernel(LinearParams p) {
  constexpr int kWaves = WM * WN;
  constexpr int kBN = 16 * WN * TN, kBM = 16 * WM * TM;
  constexpr int kCh = BK / 8;            // 16-byte chunks of a row's step
  constexpr int kRpi = 64 / kCh;         // rows of one 1 KiB load
  constexpr int kLoadersW = kRoles ? kWaves / 2 : kWaves, kLoadersA = kLoadersW;
  constexpr int kNlw = kBN / kRpi / kLoadersW, kNla = kBM / kRpi / kLoadersA;
  static_assert(kBN % (kRpi * kLoadersW) == 0 && kBM % (kRpi * kLoadersA) == 0, "whole loads a wave");
  static_assert(kRoles || DW == DA, "one ring depth where a wave loads both");
  constexpr int kStW = kBN * kCh, kStA = kBM * kCh;  // stage sizes in chunks
  __shared__ uint4 ring_w[DW * kStW];
  __shared__ uint4 ring_a[DA * kStA];
  const int lane = threadIdx.x & 63;
  const int wave = wave_uniform(threadIdx.x >> 6);
  const int r = lane & 15, grp = lane >> 4;
  const int wm = wave % WM, wn = wave / WM;

  const int z = wave_uniform(int(blockIdx.x) % p.splits), tile = wave_uniform(int(blockIdx.x) / p.splits);
  const int ksteps = p.k / BK;
  const int s0 = wave_uniform(int(int64_t(ksteps) * z / p.splits)), s1 = wave_uniform(int(int64_t(ksteps) * (z + 1) / p.splits));
  const int steps = s1 - s0;
  const int turn = wave_uniform(steps > 0 ? int(int64_t(tile) * 7 % steps) : 0);
  auto at_step = [&](int s) { return s + turn < steps ? s + turn : s + turn - steps; };
  const int n0 = tile * (kOut == Out::kSwiglu ? kBN / 2 : kBN);

  // ---- loads: slot L of a stage holds rows kRpi L .. of it, chunk c of row q at c ^ swizzle(q)
  const int lrow = lane / kCh, lpos = lane % kCh;
  const bool loads_w = !kRoles || wave < kLoadersW;
  const int lw = wave, la = kRoles ? wave - kLoadersW : wave;
  const int w_row_bytes = int(p.w_st) * 2, x_row_bytes = int(p.x_st) * 2;
  int woff[kNlw], aoff[kNla];
#pragma unroll
  for (int i = 0; i < kNlw; ++i) {
    const int row = (lw * kNlw + i) * kRpi + lrow;
    woff[i] = row * w_row_bytes + (lpos ^ swizzle<kCh>(row)) * 16;
  }
#pragma unroll
  for (int i = 0; i < kNla; ++i) {
    const int row = (la * kNla + i) * kRpi + lrow;
    aoff[i] = row * x_row_bytes + (lpos ^ swizzle<kCh>(row)) * 16;
  }
  // weight rows of this wave's slots: for a swiglu block the first half of the tile's rows are gate
  // rows n0 .., the second half the up rows n + n0 ..; a wave's slots lie in one half
  const int half = kOut == Out::kSwiglu && lw * kNlw * kRpi >= kBN / 2 ? 1 : 0;
  const int first = half * (kBN / 2);
  const int w_rows = min(kOut == Out::kSwiglu ? kBN / 2 : kBN, p.n - n0);
  const char* w_base = reinterpret_cast<const char*>(p.w + (int64_t(n0) + (half ? p.n : 0)) * p.w_st) -
                       int64_t(first) * w_row_bytes + int64_t(s0) * BK * 2;
  const int w_span = (first + w_rows - 1) * w_row_bytes + BK * 2;
  const char* a_base = reinterpret_cast<const char*>(p.x) + int64_t(s0) * BK * 2;
  const int a_span = (p.rows - 1) * x_row_bytes + BK * 2;

  auto desc_w = [&](int s) { return buffer_desc(w_base + int64_t(at_step(s)) * (BK * 2), s < steps ? w_span : 0); };
  auto desc_a = [&](int s) { return buffer_desc(a_base + int64_t(at_step(s)) * (BK * 2), s < steps ? a_span : 0); };
  auto issue_w = [&](u32x4 desc, int slot, int i) {
    load_lds<true>(desc, woff[i], ring_w + slot * kStW + (lw * kNlw + i) * 64);
  };
  auto issue_a = [&](u32x4 desc, int slot, int i) {
    load_lds<false>(desc, aoff[i], ring_a + slot * kStA + (la * kNla + i) * 64);
  };

  f32x4 acc[TM][TN];
#pragma unroll
  for (int t = 0; t < TM; ++t)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int kSub = BK / 32;  // even: the fragment buffers alternate
  static_assert(kSub % 2 == 0, "whole pairs of 32-k steps");
  int foff[kSub];  // this lane's chunk of a 16-row tile, per 32 k
#pragma unroll
  for (int c = 0; c < kSub; ++c) foff[c] = r * kCh + ((4 * c + grp) ^ swizzle<kCh>(r));

  // one 32-k step's fragments: TN of w, TM of x
  struct Frags {
    bf16x8 w[TN], a[TM];
  };
  auto read_w = [&](Frags& f, int slot, int c, int j) {
    f.w[j] = __builtin_bit_cast(bf16x8, ring_w[slot * kStW + (wn * TN + j) * 16 * kCh + foff[c]]);
  };
  auto read_a = [&](Frags& f, int slot, int c, int t) {
    f.a[t] = __builtin_bit_cast(bf16x8, ring_a[slot * kStA + (wm + t * WM) * 16 * kCh + foff[c]]);
  };
  auto multiply = [&](const Frags& f, int t) {
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[t][j] = mfma_16x16x32_bf16(f.w[j], f.a[t], acc[t][j]);
  };

  auto run = [&](auto role) {
    constexpr int kRole = decltype(role)::value;  // 0: loads both, 1: weights, 2: x
    constexpr int kDepth = kRole == 2 ? DA : DW;
    constexpr int kLoads = kRole == 0 ? kNlw + kNla : kRole == 1 ? kNlw : kNla;
    constexpr int kWaitN = (kDepth - 1) * kLoads, kWaitStep = (kDepth - 2) * kLoads;
    static_assert(kWaitN < 64, "vmcnt has 6 bits");
    // this wave's loads of the wanted stage have landed, later ones may be in flight (vmcnt(n)
    // lgkmcnt(0); gfx9 encoding: vmcnt in bits 3:0 and 15:14, expcnt 6:4 at 7)
    constexpr int kWait0 = (kWaitN & 15) | ((kWaitN >> 4) << 14) | 0x70;
    constexpr int kWait = (kWaitStep & 15) | ((kWaitStep >> 4) << 14) | 0x70;
    constexpr int kLw = kRole == 2 ? 0 : kNlw, kLa = kRole == 1 ? 0 : kNla;
    for (int s = 0; s < kDepth; ++s) {
      const u32x4 dw = desc_w(s), da = desc_a(s);
#pragma unroll
      for (int i = 0; i < kLw; ++i) issue_w(dw, s, i);
#pragma unroll
      for (int i = 0; i < kLa; ++i) issue_a(da, s, i);
    }
    Frags f[2];
    __builtin_amdgcn_s_waitcnt(kWait0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < TN; ++j) read_w(f[0], 0, 0, j);
#pragma unroll
    for (int t = 0; t < TM; ++t) read_a(f[0], 0, 0, t);
    int cw = 0, ca = 0;  // ring slots of step s
    for (int s = 0; s < steps; ++s) {
      // A 32-k step multiplies one set of fragments while the next set is read, a tile's read beside a
      // tile's products (the fences keep that order: left alone, the compiler moves the reads behind
      // the products, and LDS and matrix cores take turns).
#pragma unroll
      for (int c = 0; c < kSub - 1; ++c) {
#pragma unroll
        for (int t = 0; t < TM; ++t) {
#pragma unroll
          for (int j = t; j < TN; j += TM) read_w(f[(c + 1) & 1], cw, c + 1, j);
          read_a(f[(c + 1) & 1], ca, c + 1, t);
          multiply(f[c & 1], t);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      // every fragment of step s is in registers once the wait is over, so its slots take step s + depth
      const int nw = cw + 1 == DW ? 0 : cw + 1, na = ca + 1 == DA ? 0 : ca + 1;
      const u32x4 dw = desc_w(s + kDepth), da = desc_a(s + kDepth);
      __builtin_amdgcn_s_waitcnt(kWait);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
#pragma unroll
      for (int t = 0; t < TM; ++t) {
#pragma unroll
        for (int j = t; j < TN; j += TM) read_w(f[0], nw, 0, j);
        read_a(f[0], na, 0, t);
        multiply(f[1], t);
#pragma unroll
        for (int i = t * kLw / TM; i < (t + 1) * kLw / TM; ++i) issue_w(dw, cw, i);
#pragma unroll
        for (int i = t * kLa / TM; i < (t + 1) * kLa / TM; ++i) issue_a(da, ca, i);
        __builtin_amdgcn_sched_barrier(0);
      }
      cw = nw;
      ca = na;
    }
    __builtin_amdgcn_s_waitcnt(0x70);  // vmcnt(0) lgkmcnt(0): no load may land after the ring is given up
    asm volatile("" ::: "memory");
    // the sums move to vector registers here; without this the compiler keeps some there all along
    // and copies them to the accumulation registers and back at every step
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        f32x4& sum = acc[t][j];
        asm volatile("" : "+v"(sum));
      }
  };
  if constexpr (kRoles) {
    if (loads_w)
      run(std::integral_constant<int, 1>{});
    else
      run(std::integral_constant<int, 2>{});
  } else {
    run(std::integral_constant<int, 0>{});
  }

  if constexpr (kOut == Out::kSwiglu) {
    // gate and up tiles of a column lie in different waves: exchange through LDS (bf16-rounded values)
    __syncthreads();
    float* ex = reinterpret_cast<float*>(ring_a);  // up values [kBM rows][kBN / 2] fp32
    constexpr int kHalfTiles = WN * TN / 2;
    static_assert(sizeof(ring_a) >= sizeof(float) * WM * 16 * (kBN / 2 + 4), "the exchange fits the x ring");
#pragma unroll
    for (int t = 0; t < TM; ++t) {
      // one pass per TM tile: WM * 16 rows x kBN / 2 columns of fp32
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int nt = wn * TN + j;
        if (nt >= kHalfTiles)
          *reinterpret_cast<float4*>(ex + (wm * 16 + r) * (kBN / 2 + 4) + (nt - kHalfTiles) * 16 + 4 * grp) =
              make_float4(acc[t][j][0], acc[t][j][1], acc[t][j][2], acc[t][j][3]);
      }
      __syncthreads();
      const int row = (wm + WM * t) * 16 + r;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int nt = wn * TN + j;
        if (nt < kHalfTiles) {
          const float4 u = *reinterpret_cast<const float4*>(ex + (wm * 16 + r) * (kBN / 2 + 4) + nt * 16 + 4 * grp);
          const int col = n0 + nt * 16 + 4 * grp;
          if (row < p.rows && col < p.n)
            *reinterpret_cast<uint2*>(p.out + int64_t(row) * p.o_st + col) =
                make_uint2(pack_bf16x2_rne(swiglu(acc[t][j][0], u.x), swiglu(acc[t][j][1], u.y)),
                           pack_bf16x2_rne(swiglu(acc[t][j][2], u.z), swiglu(acc[t][j][3], u.w)));
        }
      }
      __syncthreads();
    }
  } else {
#pragma unroll
    for (int t = 0; t < TM; ++t) {
      const int row = (wm + WM * t) * 16 + r;
      if (row >= p.rows) continue;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int col = n0 + (wn * TN + j) * 16 + 4 * grp;
        if (col >= p.n) continue;
        const f32x4 v = acc[t][j];
        if (kOut == Out::kPartial)
          *reinterpret_cast<float4*>(p.partials + (int64_t(z) * p.rows + row) * p.n + col) = make_float4(v[0], v[1], v[2], v[3]);
        else
          *reinterpret_cast<uint2*>(p.out + int64_t(row) * p.o_st + col) =
              make_uint2(pack_bf16x2_rne(v[0], v[1]), pack_bf16x2_rne(v[2], v[3]));
      }
    }
  }
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

template <int WM, int WN, int TM, int TN, int BK, int DW, int DA, bool kRoles>
void launch(const LinearParams& p, Out out, hipStream_t s) {
  const int cols = 16 * WN * TN / (out == Out::kSwiglu ? 2 : 1);
  const dim3 grid((p.n + cols - 1) / cols * p.splits), block(64 * WM * WN);
  if (out == Out::kSwiglu)
    hipLaunchKernelGGL((linear_kernel<WM, WN, TM, TN, BK, DW, DA, kRoles, Out::kSwiglu>), grid, block, 0, s, p);
  else if (out == Out::kPartial)
    hipLaunchKernelGGL((linear_kernel<WM, WN, TM, TN, BK, DW, DA, kRoles, Out::kPartial>), grid, block, 0, s, p);
  else
    hipLaunchKernelGGL((linear_kernel<WM, WN, TM, TN, BK, DW, DA, kRoles, Out::kBf16>), grid, block, 0, s, p);
}

constexpr int kMaxRows = 224;
constexpr int kMaxSplits = 8;
constexpr int kCus = 256;

struct Shape {
  int cols;    // weight rows of a tile: 64, 96 or 128
  int splits;
};

// Tile and split: the least bytes through the busiest CU. A block of `cols` weight rows moves
// (rows + cols) k bytes twice over, divided by the splits, writes its fp32 partials, and every slab
// is read once more by the consumer; 256 blocks run at a time, in whole rounds where a CU holds one
// block (two of the 64-row tiles fit up to 64 rows, and even the rounds out). Up to 16 rows only
// 64-row tiles; 96-row tiles past 64 rows, 128-row ones up to 128.
// Measured either side (us): 24,576 x 4,096 + swiglu at 48 rows 41 with 128 / 43 with 64, 12,288 x
// 2,048 + swiglu 20 / 13; 6,144 x 4,096 at 208 rows 21 with 96 rows x 4 splits / 30 with 64 x 4.
Shape choose(int rows, int n, int k, Out out) {
  const double m = (rows + 15) / 16 * 16;
  Shape best{64, 1};
  double least = 1e30;
  for (int cols = 64; cols <= 128; cols += 32) {
    if (cols == 96 ? rows <= 64 : cols == 128 && (rows <= 16 || rows > 128)) continue;
    const int out_cols = out == Out::kSwiglu ? cols / 2 : cols;
    const double tiles = (n + out_cols - 1) / out_cols;
    const int most = out == Out::kPartial ? std::max(1, std::min(kMaxSplits, k / 256)) : 1;
    for (int s = 1; s <= most; ++s) {
      const double slabs = out == Out::kPartial ? 4.0 * rows : 0.0;
      const double rounds = rows <= 64 && cols == 64 ? std::max(1.0, tiles * s / kCus) : std::ceil(tiles * s / kCus);
      const double cost = rounds * ((m + cols) * 2.0 * k / s + slabs * cols) + s * slabs * n / kCus;
      if (cost <= least) {
        least = cost;
        best = Shape{cols, s};
      }
    }
  }
  return best;
}

const char* refused(const void* x, int64_t x_st, const void* w, int64_t w_st, int rows, int n, int k) {
  if (!x || !w) return "null pointer";
  if (k % 128 != 0 || n % 16 != 0) return "k must be a multiple of 128 and n of 16";
  if (rows > kMaxRows) return "at most 224 rows";
  if (x_st % 8 != 0 || w_st % 8 != 0 || !aligned16(x) || !aligned16(w)) return "x and w rows must be 16-byte aligned";
  if (x_st < k || w_st < k) return "row strides smaller than k";
  // a tile's byte offsets (128 rows of w, 224 of x) stay below 2^31
  if (x_st >= (1 << 22) || w_st >= (1 << 22)) return "row strides of 2^22 elements or more";
  return nullptr;
}

void run(const LinearParams& p, int cols, Out out, hipStream_t s) {
  if (p.rows <= 16) {
    launch<1, 4, 1, 1, 128, 4, 4, false>(p, out, s);
  } else if (p.rows <= 32) {
    if (cols == 64) launch<1, 4, 2, 1, 64, 6, 6, false>(p, out, s);
    else launch<1, 4, 2, 2, 64, 6, 6, false>(p, out, s);
  } else if (p.rows <= 64) {
    if (cols == 64) launch<1, 4, 4, 1, 64, 5, 5, false>(p, out, s);
    else launch<1, 4, 4, 2, 64, 6, 6, false>(p, out, s);
  } else if (p.rows <= 128) {
    if (cols == 64) launch<2, 2, 4, 2, 64, 7, 4, true>(p, out, s);
    else if (cols == 96) launch<2, 2, 4, 3, 64, 7, 4, true>(p, out, s);
    else launch<2, 2, 4, 4, 64, 6, 3, true>(p, out, s);
  } else {
    if (cols == 64) launch<2, 2, 7, 2, 64, 7, 3, true>(p, out, s);
    else launch<2, 2, 7, 3, 64, 6, 3, true>(p, out, s);
  }
}

}  // namespace
}  // namespace aspire

extern "C" int aspire_linear(const void* x, int64_t x_stride, const void* w, int64_t w_stride, void* out,
                             int64_t out_stride, int32_t rows, int32_t n, int32_t k, int32_t swiglu, void* stream) {
  using namespace aspire;
  ASPIRE_CHECK_ARG(rows >= 0 && n >= 0 && k > 0, "bad sizes");
  if (rows == 0 || n == 0) return ASPIRE_OK;
  if (const char* why = refused(x, x_stride, w, w_stride, rows, n, k)) ASPIRE_CHECK_ARG(false, why);
  ASPIRE_CHECK_ARG(out && out_stride >= n && out_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 7u) == 0,
                   "out rows must be 8-byte aligned and hold n values");
  const Out kind = swiglu ? Out::kSwiglu : Out::kBf16;
  const LinearParams p{static_cast<const uint16_t*>(x), x_stride, static_cast<const uint16_t*>(w), w_stride,
                       static_cast<uint16_t*>(out), out_stride, nullptr, rows, n, k, 1};
  run(p, choose(rows, n, k, kind).cols, kind, static_cast<hipStream_t>(stream));
  ASPIRE_CHECK_LAUNCH();
  return ASPIRE_OK;
}

extern "C" int32_t aspire_linear_splits(int32_t rows, int32_t n, int32_t k) {
  using namespace aspire;
  if (rows <= 0 || rows > kMaxRows || n <= 0 || n % 16 != 0 || k <= 0 || k % 128 != 0) return 0;
  return choose(rows, n, k, Out::kPartial).splits;
}

extern "C" int aspire_linear_partials(const void* x, int64_t x_stride, const void* w, int64_t w_stride, float* partials,
                                      int64_t partials_size, int32_t rows, int32_t n, int32_t k, void* stream) {
  using namespace aspire;
  ASPIRE_CHECK_ARG(rows >= 0 && n >= 0 && k > 0, "bad sizes");
  if (rows == 0 || n == 0) return ASPIRE_OK;
  if (const char* why = refused(x, x_stride, w, w_stride, rows, n, k)) ASPIRE_CHECK_ARG(false, why);
  const Shape shape = choose(rows, n, k, Out::kPartial);
  ASPIRE_CHECK_ARG(partials && aligned16(partials) && partials_size >= int64_t(shape.splits) * rows * n,
                   "partials must be 16-byte aligned and hold splits * rows * n floats");
  const LinearParams p{static_cast<const uint16_t*>(x), x_stride, static_cast<const uint16_t*>(w), w_stride,
                       nullptr, 0, partials, rows, n, k, shape.splits};
  run(p, shape.cols, Out::kPartial, static_cast<hipStream_t>(stream));
  ASPIRE_CHECK_LAUNCH();
  return ASPIRE_OK;
}
