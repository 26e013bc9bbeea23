// Route scoring and per-KV-group top-k chunk selection.
//
// Semantics follow ref_softmax_topk_max_pooling (ops/topk_head_softmax.py:15-156):
//   s[q,g,c]     = (q[q,g] . lmk[c,g]) * sm_scale        (causal-masked -> -inf)
//   x[q,g,c]     = s + bias[c,g]
//   post_softmax: y = x - logaddexp(lse_local[q,g], logsumexp_c x[q,g,:])
//   pre_softmax:  y = x
//   score[q,c]   = max_g y ; dropped chunks -> -inf
//   top-k over c; -inf picks become -1; indices sorted ascending with -1 last;
//   returned scores are s (no bias) at the picked chunks for every g.
// The logsumexp runs over every chunk, dropped ones included.  Ties in the
// selection score go to the lower chunk index (the rule of the reference's
// fused selection kernel, topk_head_softmax.py:614-626).
//
// One-pass path (route_heads_kernel, route_tile_kernel): head_dim 128, chunks
// <= 256, bf16 scores, up to 8 heads per KV group, no workspace.  Either a
// workgroup holds 16 or 32 queries of one KV head with one or two waves per
// head, whose logits stay in registers while the maxima over heads are
// selected from, or each of its waves takes 16 queries through every head in
// two passes.
//
// Scan path (route_lse_kernel, route_scan_kernel and route_pick_kernel, with a
// caller workspace): many rows against up to 4096 chunks; the selection scores
// pass through the workspace and the picks' raw scores are formed again.
//
// Short-block path (route_logits_kernel + route_select_kernel, with a caller
// workspace): logits of few query rows against up to 4096 chunks on the
// matrix cores, then one workgroup per (row, KV head) for LSE, scores and
// selection with the keys in registers.
//
// General path (route_topk_generic_kernel): one workgroup per (token, KV head)
// with scalar dot products; any head_dim / chunk count that fits LDS.
#include <mutex>
#include <type_traits>
#include <utility>

#include "block_select.h"
#include "mrsa_device.h"

using namespace mrsa;

namespace {

struct RouteArgs {
  const uint16_t* q;
  const uint16_t* lmk;
  const float* lse;
  const float* bias;
  const int32_t* drop;
  const uint8_t* key_valid;
  int64_t derive_window;
  int64_t B, L, C;
  int Hkv, G, D, K;
  int64_t block_size;
  int per_head_lmk;
  int is_causal;
  int64_t window_size;
  int64_t q_offset;
  int pre_softmax;
  float sm_scale;
  int32_t* indices;
  void* scores;
  int scores_fp32;
  int vec32_out;  // K % 32 == 0, indices and scores 16-byte aligned: 16-byte stores of both
  int vec_out;  // K % 8 == 0 and the scores 16-byte aligned: stores of 8 or 16 bytes
};

__device__ __forceinline__ int64_t floor_div(int64_t a, int64_t b) {
  int64_t q = a / b;
  if ((a % b != 0) && ((a < 0) != (b < 0))) --q;
  return q;
}

// First chunk index hidden by the causal mask for query row r (global offset applied).
__device__ __forceinline__ int64_t causal_limit(const RouteArgs& a, int64_t r) {
  const int64_t tq = r + a.q_offset;
  if (a.window_size > 0) return floor_div(tq - a.window_size + 1, a.block_size);
  return floor_div(tq, a.block_size);
}

// Whether a chunk has a valid real key: one of its first block_size - 1
// valid bytes (the last slot is the landmark) is set.  Four 16-byte loads
// for 64-key chunks at a 16-byte aligned address.
__device__ __forceinline__ bool chunk_has_valid_key(const uint8_t* kv, int64_t block_size) {
  if (block_size == 64 && ((uintptr_t)kv & 15) == 0) {
    u32x4_t acc = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const u32x4_t x = *reinterpret_cast<const u32x4_t*>(kv + 16 * v);
      acc[0] |= x[0];
      acc[1] |= x[1];
      acc[2] |= x[2];
      acc[3] |= v == 3 ? (x[3] & 0x00ffffffu) : x[3];
    }
    return (acc[0] | acc[1] | acc[2] | acc[3]) != 0u;
  }
  bool any = false;
  for (int64_t t = 0; t < block_size - 1; ++t) any |= kv[t] != 0;
  return any;
}

__device__ __forceinline__ const uint16_t* lmk_row(const RouteArgs& a, int64_t b, int64_t c, int h,
                                                   int g) {
  if (a.per_head_lmk) return a.lmk + ((b * a.C + c) * (int64_t)(a.Hkv * a.G) + h * a.G + g) * a.D;
  return a.lmk + ((b * a.C + c) * (int64_t)a.Hkv + h) * a.D;
}

// ---------------------------------------------------------------------------
// One-pass path (C <= 256): a wave per head.
//
// A workgroup of 8 waves holds 16 QT queries of one KV head; wave g computes
// head g's logits S^T = lmk . q^T, NT 16-chunk tiles (16 chunks x 16 queries
// per matrix product: lane (j, grp) holds query j's chunks 16 t + 4 grp + i),
// and keeps them in registers, so each logit is formed once:
//   scores  the head's LSE over all chunks (the four lanes sharing j), then
//           x - logaddexp(local LSE, LSE) into the workgroup's [chunk][query]
//           maxima with LDS float-max atomics;
//   picks   each wave selects 2 QT queries' K largest, lanes over chunks, and
//           lists them in LDS;
//   output  the scoring waves write their bf16 raw logits to LDS (over the
//           maxima, dead by then) and gather them at the picks.
// A wave's landmark rows stream through its own ring of 16-chunk LDS slots,
// filled by DMA and read with no workgroup barrier.
//
// Bound: a chain of short phases (loads, products, three passes over the
// logits, selection, output) rather than any one unit, so what counts is how
// many waves share a phase and how many workgroups share a CU.  Each workgroup
// reads all G C landmark rows from L2 (458 KB at G = 7, C = 256): 32 queries
// (QT = 2) halve that, 16 (QT = 1) give a short sequence twice the workgroups.
// ---------------------------------------------------------------------------
constexpr int kHeadThreads = 512;
constexpr int kHeadWaves = kHeadThreads / 64;
constexpr int kHeadRing = 2;   // landmark tiles in flight per wave
constexpr int kFastMaxTopk = 64;
constexpr int kFastMaxChunks = 256;

typedef __attribute__((address_space(3))) void lds_void_t;

// logaddexp(local LSE, LSE of the logits) from the latter in base 2.  A -inf
// total (no visible logit at all) is clamped to -FLT_MAX: finite x - tot then
// ties at the top like x - (-inf) = +inf would, and -inf stays.
__device__ __forceinline__ float route_total(float lse, float lse2) {
  const float lv2 = lse * kLog2e;
  const float hi = fmaxf(lv2, lse2), lo = fminf(lv2, lse2);
  return hi == neg_inf() ? -__FLT_MAX__ : (hi + log2_hw(1.f + exp2_hw(lo - hi))) * kLn2;
}

// The same from the LSE itself: totals scaled to base 2 and back round three
// times at the size of the total, this form once.
__device__ __forceinline__ float route_total_ln(float lse, float lse_h) {
  const float hi = fmaxf(lse, lse_h), lo = fminf(lse, lse_h);
  return hi == neg_inf()
             ? -__FLT_MAX__
             : __builtin_fmaf(log2_hw(1.f + exp2_hw((lo - hi) * kLog2e)), kLn2, hi);
}

__device__ __forceinline__ void lds_max(float* p, float v) {
  __hip_atomic_fetch_max(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Buffer resource of one batch's landmark keys (under 2 GB on the paths that
// use it), read by 24-bit lane offsets with the head slot in the scalar offset.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t lmk_rsrc(const RouteArgs& a, int64_t b,
                                                           uint32_t rowlen) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.lmk + b * a.C * (int64_t)rowlen),
                                           (short)0, (int)((uint32_t)a.C * rowlen * 2u),
                                           0x00020000);
}

template <int NT, int QT>
struct HeadsLayout {
  static constexpr int kQ = 16 * QT;           // queries
  static constexpr int kC = 16 * NT;           // chunks, padded
  static constexpr int kPitch = kQ + 4;        // floats per chunk of the maxima (4 mod 16: the
                                               // four lane groups meet distinct banks)
  static constexpr int kStage = kHeadRing * 4096;  // ring bytes per wave
  static constexpr int kRaw = kQ * kC * 2;         // raw-logit bytes per head
  static constexpr int kMax = kC * kPitch * 4;
  // One region holds the rings, then the maxima, then the raw logits; after
  // it the bias rows [G][kC], the pick lists [kQ][K] int16 and the chunk flags
  // [kC].
  static int bias(int G) {
    int n = G * kStage;
    if (n < G * kRaw) n = G * kRaw;
    return n < kMax ? kMax : n;
  }
  static int picks(int G) { return bias(G) + G * kC * 4; }
  static size_t total(int G, int K) { return (size_t)picks(G) + kQ * K * 2 + kC; }
};

template <int NT, int QT>
__global__ void __launch_bounds__(kHeadThreads, 4)
    route_heads_kernel(RouteArgs a, int bias_at, int picks_at) {
  using Lay = HeadsLayout<NT, QT>;
  constexpr int kQ = Lay::kQ, kC = Lay::kC, kPitch = Lay::kPitch;
  constexpr int kPer = NT / 4;        // chunks per selecting lane
  constexpr int kRows = kQ / kHeadWaves;  // queries a wave selects for
  static_assert(kPer * 64 == kC && kRows >= 1, "whole lanes and rows");
  extern __shared__ __align__(16) unsigned char smem[];
  const int G = a.G, K = a.K;
  float* mx_s = reinterpret_cast<float*>(smem);
  int16_t* picks = reinterpret_cast<int16_t*>(smem + picks_at);
  unsigned char* cbad = smem + picks_at + kQ * K * 2;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, grp = lane >> 4;
  const int64_t b = blockIdx.z;
  const int h = blockIdx.y;
  const int64_t L = a.L;
  const int C = (int)a.C;
  const int64_t q0 = (int64_t)blockIdx.x * kQ;
  const int g = wave;          // head of this wave's scores
  const bool scoring = g < G;  // wave-uniform

  // Every load of the prologue in flight together: the queries, their local
  // LSE and the head's bias; the flags of the chunk this thread looks at (the
  // last slot of a chunk is its landmark); an explicit drop mask's entries for
  // the rows and chunks this lane selects from.
  u32x4_t Q[QT][4];
  float lse[QT], bv[kPer];
  const int gl = min(g, G - 1);
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    // rows past L re-read row L - 1
    const int64_t qrow = ((b * L + min(q0 + 16 * u + j, L - 1)) * a.Hkv + h) * G + gl;
    const uint16_t* src = a.q + qrow * 128 + 8 * grp;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) Q[u][ks] = *reinterpret_cast<const u32x4_t*>(src + 32 * ks);
    lse[u] = a.pre_softmax ? 0.f : a.lse[qrow];
  }
#pragma unroll
  for (int i = 0; i < kPer; ++i)
    bv[i] = a.bias ? a.bias[((b * C + min(lane + 64 * i, C - 1)) * a.Hkv + h) * G + gl] : 0.f;
  uint32_t dropbits = 0u;
  if (a.derive_window >= 0) {
    if (tid < kC) {
      bool any = tid < C && a.block_size > 1;
      if (any && a.key_valid)
        any = chunk_has_valid_key(a.key_valid + b * L + (int64_t)tid * a.block_size, a.block_size);
      cbad[tid] = !any;
    }
  } else if (a.drop) {
    int32_t d[kRows][kPer];
#pragma unroll
    for (int it = 0; it < kRows; ++it) {
      const int32_t* drow = a.drop + (b * L + min(q0 + wave * kRows + it, L - 1)) * C;
#pragma unroll
      for (int i = 0; i < kPer; ++i) d[it][i] = drow[min(lane + 64 * i, C - 1)];
    }
#pragma unroll
    for (int it = 0; it < kRows; ++it)
#pragma unroll
      for (int i = 0; i < kPer; ++i) dropbits |= (uint32_t)(d[it][i] != 0) << (kPer * it + i);
  }

  // ---- scores ---------------------------------------------------------------
  f32x4_t S[NT][QT];
  float* bias_s = reinterpret_cast<float*>(smem + bias_at) + g * kC;
  float tot[QT];
  // x = s * scale + bias (-inf past C), formed anew in each of the three
  // passes over the held logits.
  auto x_of = [&](int t, int u, const f32x4_t& bt, int i) {
    return __builtin_fmaf(S[t][u][i], a.sm_scale, bt[i]);
  };
  auto bias_of = [&](int t) {
    return *reinterpret_cast<const f32x4_t*>(bias_s + 16 * t + 4 * grp);
  };
  if (scoring) {
    unsigned char* ring = smem + wave * Lay::kStage;
#pragma unroll
    for (int i = 0; i < kPer; ++i) bias_s[lane + 64 * i] = lane + 64 * i < C ? bv[i] : neg_inf();
    // The loads above complete before the first DMA is in flight: a later wait
    // for one of them would wait for the ring too.
#pragma unroll
    for (int u = 0; u < QT; ++u) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) asm volatile("" : "+v"(Q[u][ks]));
      asm volatile("" : "+v"(lse[u]));
    }
    // Tile t into its slot: 4 instructions of 4 rows x 256 bytes.  Part p of
    // row r sits at unit p ^ r of the row.  Rows >= C re-read row C - 1 (their
    // bias is -inf).
    const uint32_t rowlen = (uint32_t)(a.per_head_lmk ? a.Hkv * G : a.Hkv) * 128u;
    const uint32_t head = 256u * (uint32_t)(a.per_head_lmk ? h * G + g : h);
    const __amdgpu_buffer_rsrc_t lrs = lmk_rsrc(a, b, rowlen);
    auto stage = [&](int t) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int r = 4 * k + grp;
        const uint32_t c = (uint32_t)min(16 * t + r, C - 1);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            lrs, (lds_void_t*)(ring + (t % kHeadRing) * 4096 + 1024 * k), 16,
            2u * (__umul24(c, rowlen) + 8u * (uint32_t)(j ^ r)), head, 0, 0);
      }
    };
#pragma unroll
    for (int t = 0; t < kHeadRing; ++t) stage(t);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      static_assert(kHeadRing == 2, "one tile (4 loads) is in flight behind the awaited one");
      if (t + 1 < NT) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      const unsigned char* arow = ring + (t % kHeadRing) * 4096 + j * 256;
      u32x4_t A[4];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        A[ks] = *reinterpret_cast<const u32x4_t*>(arow + (((4 * ks + grp) ^ j) * 16));
#pragma unroll
      for (int u = 0; u < QT; ++u) {
        S[t][u] = zero4();
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) S[t][u] = mfma_bf16_16x16x32(A[ks], Q[u][ks], S[t][u]);
      }
      if (t + kHeadRing < NT) {
        // the slot's reads are done before its next tile is requested
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        stage(t + kHeadRing);
      }
    }
    // LSE over all chunks with the hardware exp2 / log2.  With every x -inf the
    // stabiliser is 0 and the sum 0.  The terms are 2^(x log2e - m2) with m2 =
    // m log2e rounded.  With up to 6 heads the rounding goes back in as
    // fma(-m, log2e, m2), so that the LSE is as close as the short-block path's
    // m + logf(sum of expf(x - m)) (scores' rms error over 3..256 chunks 0.9..1.02
    // times that form's; 1..1.5 with the LSE held in base 2).  With 7 or 8 it
    // stays in base 2 as route_tile_kernel holds it: which of the two kernels
    // takes a call depends on its length, and near ties fall the same way.
#pragma unroll
    for (int u = 0; u < QT; ++u) tot[u] = 0.f;
    if (!a.pre_softmax) {  // uniform
      float m[QT], m2[QT], part[QT], p[QT][4];
#pragma unroll
      for (int u = 0; u < QT; ++u) {
        m[u] = neg_inf();
#pragma unroll
        for (int i = 0; i < 4; ++i) p[u][i] = 0.f;
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const f32x4_t bt = bias_of(t);
#pragma unroll
        for (int u = 0; u < QT; ++u)
          m[u] = max3_raw(m[u], max_raw(x_of(t, u, bt, 0), x_of(t, u, bt, 1)),
                          max_raw(x_of(t, u, bt, 2), x_of(t, u, bt, 3)));
      }
#pragma unroll
      for (int u = 0; u < QT; ++u) {
        m[u] = across4_max(m[u]);
        m2[u] = m[u] * kLog2e;
        if (m2[u] == neg_inf()) m[u] = m2[u] = 0.f;
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const f32x4_t bt = bias_of(t);
#pragma unroll
        for (int u = 0; u < QT; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            p[u][i] += exp2_hw(__builtin_fmaf(x_of(t, u, bt, i), kLog2e, -m2[u]));
      }
#pragma unroll
      for (int u = 0; u < QT; ++u)
        part[u] = across4_sum((p[u][0] + p[u][1]) + (p[u][2] + p[u][3]));
#pragma unroll
      for (int u = 0; u < QT; ++u)
        if (G >= 7) {  // uniform
          tot[u] = route_total(lse[u], m2[u] + log2_hw(part[u]));
        } else {
          const float back = __builtin_fmaf(-m[u], kLog2e, m2[u]);
          tot[u] = route_total_ln(lse[u], __builtin_fmaf(log2_hw(part[u]) + back, kLn2, m[u]));
        }
    }
  }
  __syncthreads();  // the rings are done
  for (int i = tid; i < Lay::kMax / 16; i += kHeadThreads) {
    const float n = neg_inf();
    reinterpret_cast<f32x4_t*>(mx_s)[i] = f32x4_t{n, n, n, n};
  }
  __syncthreads();
  if (scoring) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const f32x4_t bt = bias_of(t);
#pragma unroll
      for (int u = 0; u < QT; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          lds_max(mx_s + (16 * t + 4 * grp + i) * kPitch + 16 * u + j,
                  x_of(t, u, bt, i) - tot[u]);
    }
  }
  __syncthreads();

  // ---- picks ----------------------------------------------------------------
  const uint32_t kNeg = float_order_key(neg_inf());
  const int win = (int)min(max(a.derive_window, (int64_t)0), L);
  const uint32_t bsz = (uint32_t)min(a.block_size, (int64_t)0x7fffffff);
#pragma unroll
  for (int it = 0; it < kRows; ++it) {
    const int ql = wave * kRows + it;
    const int64_t r = q0 + ql;
    if (r >= L) break;  // uniform
    // (32-bit: row and window are below 2^31)
    const uint32_t lc = (uint32_t)max((int)r - win, 0) / bsz;
    const uint32_t rc = (uint32_t)min((int)r + win, (int)L - 1) / bsz;
    uint32_t key[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int c = lane + 64 * i;
      const float m = mx_s[min(c, kC - 1) * kPitch + ql];
      bool dropped = false;
      if (a.derive_window >= 0)
        dropped = ((uint32_t)c >= lc && (uint32_t)c <= rc) || cbad[min(c, kC - 1)] != 0;
      else
        dropped = (dropbits >> (kPer * it + i)) & 1u;
      // 0 is below every real key: never picked
      key[i] = c < C ? (dropped ? kNeg : float_order_key(m)) : 0u;
    }
    int16_t* plist = picks + ql * K;
    if (lane < K) plist[lane] = -1;
    const uint64_t sel = WaveSelect<kPer>::run(key, kPer, K);
    int base = 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const bool p = (sel >> i) & 1ull;
      const uint64_t pb = __builtin_amdgcn_ballot_w64(p);
      if (p) plist[base + __builtin_popcountll(pb & ((1ull << lane) - 1ull))] =
          (int16_t)(lane + 64 * i);
      base += __builtin_popcountll(pb);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's list
    if (lane < K) a.indices[((b * L + r) * a.Hkv + h) * K + lane] = plist[lane];
  }
  __syncthreads();
  if (!scoring) return;

  // ---- output ---------------------------------------------------------------
  // Query j's chunk c at unit (c >> 2) ^ (j & 15) of its row (8-byte units: a
  // tile's writes touch distinct banks).
  uint16_t* raw = reinterpret_cast<uint16_t*>(smem + g * Lay::kRaw);
  static_assert(kC % 64 == 0, "units come in blocks of 16");
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int u = 0; u < QT; ++u) {
      u32x2_t w;
      w[0] = pack_bf16x2(S[t][u][0] * a.sm_scale, S[t][u][1] * a.sm_scale);
      w[1] = pack_bf16x2(S[t][u][2] * a.sm_scale, S[t][u][3] * a.sm_scale);
      *reinterpret_cast<u32x2_t*>(raw + (16 * u + j) * kC + 4 * ((4 * t + grp) ^ j)) = w;
    }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's tile
  auto raw_at = [&](int ql, int c) {
    return c < 0 ? 0xff80u  // -inf past the picks
                 : (uint32_t)raw[ql * kC + 4 * ((c >> 2) ^ (ql & 15)) + (c & 3)];
  };
  uint16_t* out = reinterpret_cast<uint16_t*>(a.scores);
  const int nq = (int)min((int64_t)kQ, L - q0);
  if (a.vec_out) {
    const int k8 = K >> 3;
    for (int e = lane; e < nq * k8; e += 64) {
      const int ql = e / k8, s0 = 8 * (e - ql * k8);
      const u32x4_t pk = *reinterpret_cast<const u32x4_t*>(picks + ql * K + s0);
      u32x4_t o;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        o[i] = raw_at(ql, (int)(int16_t)(pk[i] & 0xffffu)) |
               (raw_at(ql, (int)(int16_t)(pk[i] >> 16)) << 16);
      *reinterpret_cast<u32x4_t*>(out + (((b * L + q0 + ql) * a.Hkv + h) * G + g) * K + s0) = o;
    }
  } else {
    for (int e = lane; e < nq * K; e += 64) {
      const int ql = e / K, s = e - ql * K;
      out[(((b * L + q0 + ql) * a.Hkv + h) * G + g) * K + s] =
          (uint16_t)raw_at(ql, picks[ql * K + s]);
    }
  }
}

// ---------------------------------------------------------------------------
// One-pass path, 129 to 256 chunks and enough queries to fill the chip with
// 128 of them per workgroup: every head in each wave.
//
// A workgroup takes 128 queries of one KV head, 16 per wave; a wave keeps
// its queries' running max over heads M for all 256 chunks in registers.
// Logits are computed transposed, S^T = lmk . q^T (16 chunks x 16 queries
// per matrix product): lane (j, grp) holds query j's chunks 16 t + 4 grp + i
// (t = 0..15, i = 0..3), so every per-query reduction runs over the four
// lanes sharing j.
//   pass 1, heads 0..G-1: x = s * scale + bias, the head's LSE over all
//           chunks, M = max(M, x - logaddexp(local LSE, LSE));
//   selection: the K-th largest M per query by bisection on order keys
//           (ties at the threshold to the lower chunk), the ascending pick
//           list of each query in LDS;
//   pass 2, heads G-1..0: the raw logits again, rounded to bf16 into the
//           wave's [16][256] LDS tile, gathered at the picks.
// One head's landmark keys sit in LDS while the next head's stream in.
// ---------------------------------------------------------------------------
constexpr int kTileThreads = 512;  // 8 waves x 16 queries
constexpr int kTileQ = 128;        // queries per workgroup

// LDS carve-up.  Two landmark buffers ([256][128] bf16, 16-byte parts
// XOR-swizzled: part p of row c at unit 16 c + (p ^ (c & 15))); in pass 2
// the one pass 1 ends off holds the waves' raw-logit tiles.  Two bias rows
// (-inf past C), the chunk flags and the pick lists [128][K] int16.
struct TileLayout {
  static constexpr size_t lmk = 0;                    // [2][256][128] bf16
  static constexpr size_t bias = 2 * 256 * 128 * 2;   // [2][256] f32
  static constexpr size_t cbad = bias + 2 * 256 * 4;  // [256] u8
  static constexpr size_t picks = cbad + 256;         // [128][K] i16
  static size_t total(int K) { return picks + (size_t)kTileQ * K * 2; }
};

__device__ __forceinline__ int across4_sum_i(int v) {
  const auto r = __builtin_amdgcn_permlane32_swap((uint32_t)v, (uint32_t)v, false, false);
  const int s = (int)r[0] + (int)r[1];
  const auto q = __builtin_amdgcn_permlane16_swap((uint32_t)s, (uint32_t)s, false, false);
  return (int)q[0] + (int)q[1];
}
__device__ __forceinline__ uint32_t across4_min_u(uint32_t v) {
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  const uint32_t s = min((uint32_t)r[0], (uint32_t)r[1]);
  const auto q = __builtin_amdgcn_permlane16_swap(s, s, false, false);
  return min((uint32_t)q[0], (uint32_t)q[1]);
}
__device__ __forceinline__ uint32_t across4_max_u(uint32_t v) {
  const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  const uint32_t s = max((uint32_t)r[0], (uint32_t)r[1]);
  const auto q = __builtin_amdgcn_permlane16_swap(s, s, false, false);
  return max((uint32_t)q[0], (uint32_t)q[1]);
}

// Position of chunk 16 t + 4 grp + i among the set bits of a query's four
// per-lane masks (bit 4 t + i of lane group grp'): the bits of all groups in
// tiles before t, of lower groups in tile t, and of lower i in this group.
__device__ __forceinline__ int chunk_rank(const uint64_t (&m)[4], int grp, int t, int i) {
  const uint64_t below = (1ull << (4 * t)) - 1ull;
  int r = 0;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    r += __popcll(m[g] & below);
    const int nib = (int)((m[g] >> (4 * t)) & 15u);
    r += g < grp ? __popc(nib) : (g == grp ? __popc(nib & ((1 << i) - 1)) : 0);
  }
  return r;
}

template <int G>
__global__ void __launch_bounds__(kTileThreads, 1) route_tile_kernel(RouteArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int K = a.K;
  float* bias_s = reinterpret_cast<float*>(smem + TileLayout::bias);
  unsigned char* cbad = smem + TileLayout::cbad;
  int16_t* picks = reinterpret_cast<int16_t*>(smem + TileLayout::picks);
  auto lmk_buf = [&](int i) {
    return reinterpret_cast<uint16_t*>(smem + TileLayout::lmk) + i * 256 * 128;
  };

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int j = lane & 15, grp = lane >> 4;
  const int64_t b = blockIdx.z;
  const int h = blockIdx.y;
  const int64_t L = a.L, C = a.C;
  const int64_t q0 = (int64_t)blockIdx.x * kTileQ;
  const int ql = 16 * wave + j;            // this lane's query within the workgroup
  const int64_t r = q0 + ql;
  const bool rvalid = r < L;
  const int64_t rr = rvalid ? r : L - 1;   // rows past L re-read row L - 1
  const int64_t qrow = ((b * L + rr) * a.Hkv + h) * G;  // (row, head 0) of q, lse

  // Chunks with no valid real key (the last slot of a chunk is its landmark).
  if (a.derive_window >= 0) {
    for (int c = tid; c < 256; c += kTileThreads) {
      bool any = false;
      if (c < C) {
        if (a.key_valid) {
          any = chunk_has_valid_key(a.key_valid + b * L + (int64_t)c * a.block_size, a.block_size);
        } else {
          any = a.block_size > 1;
        }
      }
      cbad[c] = !any;
    }
  }

  // Head g's landmark keys into buffer i, instruction k (0..7) of this wave:
  // LDS units (8 wave + k) * 64 + lane = row 4 (8 wave + k) + lane / 16,
  // stored part lane & 15 (global part (lane & 15) ^ (row & 15)).  Rows >= C
  // re-read row C - 1; their logits are masked by the bias row.  The keys
  // of batch b are one buffer (chunk c's head slot s at element c rowlen +
  // 128 s, under 2 GB on this path): the lane's offset is a 24-bit multiply
  // and the head slot rides in the scalar offset.
  const uint32_t rowlen = (uint32_t)(a.per_head_lmk ? a.Hkv * G : a.Hkv) * 128u;
  const __amdgpu_buffer_rsrc_t lrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(a.lmk + b * C * (int64_t)rowlen), (short)0,
      (int)((uint32_t)C * rowlen * 2u), 0x00020000);
  auto stage_part = [&](int g, int i, int k) {
    const int row = 4 * (8 * wave + k) + (lane >> 4);
    const uint32_t part = (uint32_t)((lane & 15) ^ (row & 15));
    const uint32_t c = (uint32_t)min(row, (int)C - 1);
    const uint32_t slot = a.per_head_lmk ? (uint32_t)(h * G + g) : (uint32_t)h;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(lrs, (lds_void_t*)(lmk_buf(i) + (8 * wave + k) * 512),
                                             16, 2u * (__umul24(c, rowlen) + 8u * part),
                                             256u * slot, 0, 0);
  };
  // Bias of chunk tid for head g (-inf past C), loaded ahead of its LDS write.
  auto bias_of = [&](int g) {
    float v = neg_inf();
    if (tid < C) v = a.bias ? a.bias[((b * C + tid) * a.Hkv + h) * G + g] : 0.f;
    return v;
  };
  // This lane's Q^T operand (query j, dims 32 ks + 8 grp ..) of head g.
  auto load_q = [&](int g, u32x4_t (&Q)[4]) {
    const uint16_t* src = a.q + (qrow + g) * 128 + 8 * grp;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) Q[ks] = *reinterpret_cast<const u32x4_t*>(src + 32 * ks);
  };

  // An explicit drop mask, read before pass 1 while few registers are live,
  // so that its loads are in flight together: bit 4 t + e of this lane's
  // word is chunk 16 t + 4 grp + e (chunks >= C dropped).
  uint64_t dropbits = 0ull;
  if (a.derive_window < 0 && a.drop) {
    const int32_t* drow = a.drop + (b * L + rr) * C;
    if (C == 256 && ((uintptr_t)a.drop & 15) == 0) {
      u32x4_t d[16];
#pragma unroll
      for (int t = 0; t < 16; ++t) d[t] = *reinterpret_cast<const u32x4_t*>(drow + 16 * t + 4 * grp);
#pragma unroll
      for (int t = 0; t < 16; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) dropbits |= (uint64_t)(d[t][e] != 0u) << (4 * t + e);
    } else {
      int32_t d[16][4];
#pragma unroll
      for (int t = 0; t < 16; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) d[t][e] = drow[min(16 * t + 4 * grp + e, (int)C - 1)];
#pragma unroll
      for (int t = 0; t < 16; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          dropbits |= (uint64_t)((16 * t + 4 * grp + e >= C) | (d[t][e] != 0)) << (4 * t + e);
    }
  }

  // ---- pass 1 -------------------------------------------------------------
  float M[16][4];
#pragma unroll
  for (int t = 0; t < 16; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) M[t][e] = neg_inf();
  u32x4_t Qc[4], Qn[4];
  float lse_c = 0.f, lse_n = 0.f;
  load_q(0, Qc);
  if (!a.pre_softmax) lse_c = a.lse[qrow];
#pragma unroll
  for (int k = 0; k < 8; ++k) stage_part(0, 0, k);
  if (tid < 256) bias_s[tid] = bias_of(0);
  for (int g = 0; g < G; ++g) {
    // Head g landed (this wave's DMA; the barrier covers the others') and
    // every wave is done with the other buffer.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    const bool more = g + 1 < G;
    float bnext = 0.f;
    if (more) {
      load_q(g + 1, Qn);
      if (!a.pre_softmax) lse_n = a.lse[qrow + g + 1];
      if (tid < 256) bnext = bias_of(g + 1);
    }
    // x = s * scale + bias (bias -inf past C), tile by tile after its
    // products, with the running max for the LSE.
    f32x4_t S[16];
    float mx = neg_inf();
    {
      const uint16_t* lmk_s = lmk_buf(g & 1);
      const float* brow = bias_s + 256 * (g & 1) + 4 * grp;
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        f32x4_t acc = zero4();
        const uint16_t* arow = lmk_s + (16 * t + j) * 128;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          const u32x4_t A =
              *reinterpret_cast<const u32x4_t*>(arow + (((4 * ks + grp) ^ j) * 8));
          acc = mfma_bf16_16x16x32(A, Qc[ks], acc);
        }
        if (more && (t & 1)) stage_part(g + 1, (g + 1) & 1, t >> 1);
        const f32x4_t bv = *reinterpret_cast<const f32x4_t*>(brow + 16 * t);
#pragma unroll
        for (int e = 0; e < 4; ++e) S[t][e] = __builtin_fmaf(acc[e], a.sm_scale, bv[e]);
        mx = max3_raw(mx, max_raw(S[t][0], S[t][1]), max_raw(S[t][2], S[t][3]));
      }
    }
    // LSE over all chunks in base 2 with the hardware exp2 / log2.
    const float m2 = across4_max(mx) * kLog2e;
    float sm = 0.f;
    if (m2 != neg_inf()) {
      float p[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < 16; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) p[e] += exp2_hw(__builtin_fmaf(S[t][e], kLog2e, -m2));
      sm = (p[0] + p[1]) + (p[2] + p[3]);
    }
    const float s2 = across4_sum(sm);
    const float lse2 = m2 == neg_inf() ? neg_inf() : m2 + log2_hw(s2);
    const float tot = a.pre_softmax ? 0.f : route_total(lse_c, lse2);
#pragma unroll
    for (int t = 0; t < 16; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) M[t][e] = max_raw(M[t][e], S[t][e] - tot);
    if (more) {
      if (tid < 256) bias_s[256 * ((g + 1) & 1) + tid] = bnext;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) Qc[ks] = Qn[ks];
      lse_c = lse_n;
    }
  }

  // ---- selection ----------------------------------------------------------
  // Order keys of M (dropped chunks and chunks >= C: -inf).
  const uint32_t kNeg = float_order_key(neg_inf());
  // One uniform branch per drop source; straight-line code per element.
  uint32_t key[16][4];
  if (a.derive_window >= 0) {
    const int lc = (int)(max(rr - a.derive_window, (int64_t)0) / a.block_size);
    const int rc = (int)(min(rr + a.derive_window, L - 1) / a.block_size);
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      const int c0 = 16 * t + 4 * grp;
      const uint32_t bad4 = *reinterpret_cast<const uint32_t*>(cbad + c0);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int c = c0 + e;
        const bool dropped =
            (c >= C) | ((c >= lc) & (c <= rc)) | (((bad4 >> (8 * e)) & 0xffu) != 0u);
        key[t][e] = dropped ? kNeg : float_order_key(M[t][e]);
      }
    }
  } else if (a.drop) {
#pragma unroll
    for (int t = 0; t < 16; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        key[t][e] = ((dropbits >> (4 * t + e)) & 1ull) ? kNeg : float_order_key(M[t][e]);
  } else {
#pragma unroll
    for (int t = 0; t < 16; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        key[t][e] = 16 * t + 4 * grp + e >= C ? kNeg : float_order_key(M[t][e]);
  }
  int nfin = 0;
  uint32_t kmin = 0xffffffffu, kmax = 0u;
#pragma unroll
  for (int t = 0; t < 16; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool fin = key[t][e] > kNeg;
      nfin += fin ? 1 : 0;
      kmin = min(kmin, fin ? key[t][e] : 0xffffffffu);
      kmax = max(kmax, key[t][e]);  // -inf keys are below every finite key
    }
  nfin = across4_sum_i(nfin);
  kmin = across4_min_u(kmin);
  kmax = across4_max_u(kmax);
  // Threshold: keys >= thr_hi are picked, plus the first `need` keys equal
  // to thr_tie in chunk order.  The search keeps count(key >= lo) = clo > K
  // and count(key >= hi) = chi < K and stops when a probe counts exactly K
  // (or hi = lo + 1: ties at lo).  Probes interpolate the count linearly in
  // key space; a probe that leaves more than half the interval is followed
  // by a bisection step, so the search never takes more than twice the
  // steps of plain bisection.
  uint32_t thr_hi, thr_tie = 0u, lo = kmin, hi = kmax + 1u;
  int clo = nfin, chi = 0;
  int need = 0;
  bool done = nfin <= K;
  thr_hi = done ? kNeg + 1u : 0u;
  bool bisect = false;
  for (int it = 0; it < 80; ++it) {
    if (!done && hi - lo <= 1u) done = true;
    if (!__any(!done)) break;
    uint32_t mid = lo + ((hi - lo) >> 1);
    if (!done && !bisect) {
      const float f = (float)(clo - K) / (float)(clo - chi);
      const uint32_t step = (uint32_t)((float)(hi - lo) * f);
      mid = min(max(lo + step, lo + 1u), hi - 1u);
    }
    int cnt = 0;
#pragma unroll
    for (int t = 0; t < 16; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) cnt += key[t][e] >= mid ? 1 : 0;
    cnt = across4_sum_i(cnt);
    if (!done) {
      const uint32_t width = hi - lo;
      if (cnt == K) {
        thr_hi = mid;
        done = true;
      } else if (cnt > K) {
        lo = mid;
        clo = cnt;
      } else {
        hi = mid;
        chi = cnt;
      }
      bisect = !bisect && (hi - lo) > (width >> 1);
    }
  }
  if (thr_hi == 0u) {  // hi = lo + 1: keys >= hi, then ties at lo
    thr_hi = hi;
    thr_tie = lo;
    need = K - chi;
  }
  // This lane's picks / ties as bit masks (bit 4 t + e), built per 32-bit half.
  uint32_t ph[2] = {0u, 0u}, th[2] = {0u, 0u};
  const uint32_t tie_key = need > 0 ? thr_tie : 0u;  // key 0 is never finite
#pragma unroll
  for (int t = 0; t < 16; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int bit = (4 * t + e) & 31;
      ph[t >> 3] |= (uint32_t)(key[t][e] >= thr_hi) << bit;
      th[t >> 3] |= (uint32_t)(key[t][e] == tie_key) << bit;
    }
  uint64_t pm = ((uint64_t)ph[1] << 32) | ph[0];
  const uint64_t tm = ((uint64_t)th[1] << 32) | th[0];
  // The four lanes' masks of this query, in lane-group order.
  auto gather4 = [&](uint64_t v, uint64_t (&m)[4]) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int src = j + 16 * g;
      const uint32_t lo32 = (uint32_t)__shfl((int)(uint32_t)v, src, 64);
      const uint32_t hi32 = (uint32_t)__shfl((int)(uint32_t)(v >> 32), src, 64);
      m[g] = ((uint64_t)hi32 << 32) | lo32;
    }
  };
  if (__any(need > 0)) {
    // Ties at the threshold: the first `need` in chunk order.
    uint64_t tall[4];
    gather4(tm, tall);
    uint64_t x = tm;
    while (x) {
      const int p = __builtin_ctzll(x);
      x &= x - 1ull;
      if (chunk_rank(tall, grp, p >> 2, p & 3) < need) pm |= 1ull << p;
    }
  }
  uint64_t pall[4];
  gather4(pm, pall);
  const int total = __popcll(pall[0]) + __popcll(pall[1]) + __popcll(pall[2]) + __popcll(pall[3]);
  int16_t* plist = picks + ql * K;  // this query's ascending pick list
  {
    uint64_t x = pm;
    while (x) {
      const int p = __builtin_ctzll(x);
      x &= x - 1ull;
      plist[chunk_rank(pall, grp, p >> 2, p & 3)] = (int16_t)(16 * (p >> 2) + 4 * grp + (p & 3));
    }
  }
  // The wave's own pick lists are read back below (LDS keeps one wave's
  // operations in order).
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  int32_t* irow = a.indices + ((b * L + r) * a.Hkv + h) * K;
  // Output slots: with vec32_out a lane writes the K / 4 consecutive slots
  // s0 .. s0 + K / 4 - 1 of its query (one 16-byte store per 8 scores, per
  // 4 indices), its picks held as int16 pairs in pk; else slots grp + 4 i.
  const bool vec = a.vec32_out != 0;
  const int per = K >> 2, nv = K >> 5, s0 = per * grp;
  uint32_t pk[8];
#pragma unroll
  for (int v = 0; v < 2; ++v) {
    u32x4_t x = {0u, 0u, 0u, 0u};
    if (vec && v < nv) x = *reinterpret_cast<const u32x4_t*>(plist + s0 + 8 * v);
#pragma unroll
    for (int e = 0; e < 4; ++e) pk[4 * v + e] = x[e];
  }
  // chunk of this lane's slot s0 + 8 v + e (0 past the picks)
  auto pick_at = [&](int v, int e) {
    const int c = (int)((pk[4 * v + (e >> 1)] >> (16 * (e & 1))) & 0xffffu);
    return s0 + 8 * v + e < total ? c : 0;
  };
  if (rvalid) {
    if (vec) {
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        if (v >= nv) break;
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          u32x4_t o;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o[e] = s0 + 8 * v + 4 * hh + e < total ? (uint32_t)pick_at(v, 4 * hh + e) : 0xffffffffu;
          *reinterpret_cast<u32x4_t*>(irow + s0 + 8 * v + 4 * hh) = o;
        }
      }
    } else {
      for (int s = grp; s < K; s += 4) irow[s] = s < total ? (int32_t)plist[s] : -1;
    }
  }

  // ---- pass 2 -------------------------------------------------------------
  // Raw logits bf16(s * scale) of the picks, heads G-1..0.  Pass 1 left head
  // G-1 in buffer pb; the other buffer holds the waves' tiles: query j's
  // chunk c at j * 256 + 4 ((c >> 2) ^ j) + (c & 3) (8-byte units swizzled
  // by query so a tile write touches distinct banks).
  const int pb = (G - 1) & 1;
  uint16_t* tile = lmk_buf(1 - pb) + wave * 16 * 256;
  uint16_t* sc16 = reinterpret_cast<uint16_t*>(a.scores);
  load_q(G - 1, Qc);
  for (int g = G - 1; g >= 0; --g) {
    if (g < G - 1) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();  // head g landed in buffer pb
    }
    if (g > 0) load_q(g - 1, Qn);
    // S^T tile by tile (S[e] = q_j . lmk[16 t + 4 grp + e]) into the LDS tile.
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      f32x4_t acc = zero4();
      const uint16_t* arow = lmk_buf(pb) + (16 * t + j) * 128;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const u32x4_t A = *reinterpret_cast<const u32x4_t*>(arow + (((4 * ks + grp) ^ j) * 8));
        acc = mfma_bf16_16x16x32(A, Qc[ks], acc);
      }
      u32x2_t w;
      w[0] = pack_bf16x2(acc[0] * a.sm_scale, acc[1] * a.sm_scale);
      w[1] = pack_bf16x2(acc[2] * a.sm_scale, acc[3] * a.sm_scale);
      *reinterpret_cast<u32x2_t*>(tile + j * 256 + 4 * ((4 * t + grp) ^ j)) = w;
    }
    if (g > 0) {
      __syncthreads();  // every wave is done with head g's keys
#pragma unroll
      for (int k = 0; k < 8; ++k) stage_part(g - 1, pb, k);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (rvalid) {
      uint16_t* orow = sc16 + (((b * L + r) * a.Hkv + h) * G + g) * K;
      if (vec) {
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          if (v >= nv) break;
          uint32_t w[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int c = pick_at(v, e);
            const uint32_t x = tile[j * 256 + 4 * ((c >> 2) ^ j) + (c & 3)];
            w[e] = s0 + 8 * v + e < total ? x : 0xff80u;  // -inf past the picks
          }
          u32x4_t o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = w[2 * e] | (w[2 * e + 1] << 16);
          *reinterpret_cast<u32x4_t*>(orow + s0 + 8 * v) = o;
        }
      } else {
        for (int s = grp; s < K; s += 4) {
          uint16_t v = 0xff80u;  // -inf past the picks
          if (s < total) {
            const int c = plist[s];
            v = tile[j * 256 + 4 * ((c >> 2) ^ j) + (c & 3)];
          }
          orow[s] = v;
        }
      }
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) Qc[ks] = Qn[ks];
  }
}

// ---------------------------------------------------------------------------
// Scan path, for many rows against more chunks than the one-pass path holds:
// the selection scores [B, L, Hkv, Cp] (fp32, Cp = C rounded up to 16) pass
// through the workspace, a seventh of the raw logits.  Three kernels:
//
// route_lse_kernel: a workgroup of 8 waves holds one head of 128 queries, 16
// per wave, and forms their logaddexp(local LSE, LSE over all chunks).
// route_scan_kernel: a workgroup of 8 waves holds 128 queries of one KV head,
// 16 per wave with every head's Q operand in registers, and forms the maximum
// over heads of x - that total, dropped chunks -inf.
// route_pick_kernel: a wave per row picks its K largest and forms the picks'
// raw logits again.
//
// Landmark rows stream through an LDS ring in both scans, filled by DMA.  The
// products are S = q . lmk^T: lane (j, grp) holds chunk 16 t + j for queries
// 4 grp + i.  A row's LSE is summed as the workgroup selection's wave form
// sums it -- chunks c mod 64 in running (max, sum) pairs, then a butterfly over
// the 64 -- here 4 pairs per lane and query, so that near ties between heads
// fall the same way as they always did.
//
// Measured at 65536 queries x 4 KV heads x 7 heads against 1024 chunks: 1490-1640
// (LSE) + 1140-1170 (scan) + 1350-1440 (pick) us; 7590 + 6260 us with the fp32
// logits of every head through memory (7.5 GB written and read).  The LSE kernel
// is bound by the ~30 VALU instructions of each term (the VALU never idles); the
// scan (VALU 43%, matrix cores 18%, waves waiting 35%) by its products and their
// 7-head epilogue at two waves per SIMD; the pick (waiting 50%) by the gather.
// ---------------------------------------------------------------------------
constexpr int kScanThreads = 512;
constexpr int kScanQ = 128;
constexpr int kScanRing = 4;
constexpr int kLseRing = 3;  // 64-chunk stages of one head
constexpr int kPickRing = 2;
constexpr int kScanMaxChunks = 4096;

inline int64_t scan_chunks(int64_t chunks) { return (chunks + 15) / 16 * 16; }

// The scaled logit plus the bias, each rounded (no fused multiply-add).
__device__ __forceinline__ float scaled_plus(float acc, float scale, float bias) {
#pragma clang fp contract(off)
  const float s = acc * scale;
  return s + bias;
}

// The causal limit of row r as a chunk count in [0, C].
__device__ __forceinline__ int chunk_limit(const RouteArgs& a, int64_t r) {
  return (int)(a.is_causal ? max((int64_t)0, min(a.C, causal_limit(a, r))) : a.C);
}

__global__ void __launch_bounds__(kScanThreads, 4)
    route_lse_kernel(RouteArgs a, float* __restrict__ total) {
  __shared__ __align__(16) unsigned char ring[kLseRing][64 * 256];
  __shared__ float bias_s[kLseRing][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, grp = lane >> 4;
  const int G = a.G;
  const int64_t b = blockIdx.z;
  const int h = blockIdx.y / G, g = blockIdx.y - h * G;
  const int64_t L = a.L;
  const int C = (int)a.C;
  const int ns = (C + 63) >> 6;  // stages
  const int64_t r0 = (int64_t)blockIdx.x * kScanQ + 16 * wave;
  u32x4_t Q[4];
  {
    const int64_t row = ((b * L + min(r0 + j, L - 1)) * a.Hkv + h) * G + g;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      Q[ks] = *reinterpret_cast<const u32x4_t*>(a.q + row * 128 + 8 * grp + 32 * ks);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) asm volatile("" : "+v"(Q[ks]));  // before any DMA
  }
  // Stage s: 64 chunks' rows, 2 of the 16 DMA instructions per wave (4 rows of
  // 256 bytes each; part p of row r at unit p ^ (r & 15)), and with a bias its
  // 64 values (every wave issues it: the same bytes, the same count of loads).
  const uint32_t rowlen = (uint32_t)(a.per_head_lmk ? a.Hkv * G : a.Hkv) * 128u;
  const uint32_t head = 256u * (uint32_t)(a.per_head_lmk ? h * G + g : h);
  const __amdgpu_buffer_rsrc_t lrs = lmk_rsrc(a, b, rowlen);
  const uint32_t blen = (uint32_t)(a.Hkv * G);
  const __amdgpu_buffer_rsrc_t brs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(a.bias ? a.bias + b * C * (int64_t)blen : a.lse), (short)0,
      a.bias ? (int)((uint32_t)C * blen * 4u) : 0, 0x00020000);
  if (!a.bias && tid < 64)
    for (int s = 0; s < kLseRing; ++s) bias_s[s][tid] = 0.f;
  auto stage = [&](int s) {
    const int slot = s % kLseRing;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int n = 2 * wave + i, row = 4 * n + grp;
      const uint32_t c = (uint32_t)min(64 * s + row, C - 1);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          lrs, (lds_void_t*)(ring[slot] + n * 1024), 16,
          2u * (__umul24(c, rowlen) + 8u * (uint32_t)(j ^ (row & 15))), head, 0, 0);
    }
    if (a.bias) {  // uniform
      const uint32_t c = (uint32_t)min(64 * s + lane, C - 1);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(brs, (lds_void_t*)bias_s[slot], 4,
                                               4u * __umul24(c, blen), 4u * (uint32_t)(h * G + g),
                                               0, 0);
    }
  };
  for (int s = 0; s < kLseRing - 1 && s < ns; ++s) stage(s);
  int climit[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) climit[i] = chunk_limit(a, min(r0 + 4 * grp + i, L - 1));
  // The pair of (query 4 grp + i, chunks with c mod 64 = 16 k + j).
  float m[4][4], sum[4][4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      m[k][i] = neg_inf();
      sum[k][i] = 0.f;
    }
  auto step = [&](int s, bool hide) {
    // one stage may be in flight behind the awaited one
    if (s + 1 < ns) {
      if (a.bias) asm volatile("s_waitcnt vmcnt(3)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (s + kLseRing - 1 < ns) stage(s + kLseRing - 1);
    const int slot = s % kLseRing;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const unsigned char* brow = ring[slot] + (16 * k + j) * 256;
      f32x4_t x = zero4();
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        x = mfma_bf16_16x16x32(
            Q[ks], *reinterpret_cast<const u32x4_t*>(brow + (((4 * ks + grp) ^ j) * 16)), x);
      const float bv = bias_s[slot][16 * k + j];
      const int c = 64 * s + 16 * k + j;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v = scaled_plus(x[i], a.sm_scale, bv);
        if (hide && c >= climit[i]) v = neg_inf();
        // a new max scales the sum so far: sum e + 1, else sum + e, with
        // e = exp(-|v - max|), one rounding each
        const bool up = v > m[k][i];
        float e = expf(-fabsf(v - m[k][i]));
        e = v == neg_inf() ? 0.f : e;
        sum[k][i] = __builtin_fmaf(up ? sum[k][i] : 1.f, e, up ? 1.f : sum[k][i]);
        m[k][i] = fmaxf(m[k][i], v);
      }
    }
  };
  const int whole = a.is_causal ? 0 : C >> 6;
  for (int s = 0; s < whole; ++s) step(s, false);
  for (int s = whole; s < ns; ++s) step(s, true);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    // over the 64 pairs: j by lane moves (1, 2, 4, 8), then k (16, 32)
    float mm = fmaxf(fmaxf(m[0][i], m[1][i]), fmaxf(m[2][i], m[3][i]));
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) mm = fmaxf(mm, __shfl_xor(mm, o, 64));
    float ss[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      ss[k] = m[k][i] == neg_inf() ? 0.f : sum[k][i] * expf(m[k][i] - mm);
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) ss[k] += __shfl_xor(ss[k], o, 64);
    }
    const float st = (ss[0] + ss[1]) + (ss[2] + ss[3]);
    const float lse_h = mm == neg_inf() ? mm : mm + logf(st);
    const int64_t r = r0 + 4 * grp + i;
    if (j == 0 && r < L) {
      const int64_t at = ((b * L + r) * a.Hkv + h) * G + g;
      total[at] = logaddexp_f(a.lse[at], lse_h);
    }
  }
}

template <int G>
struct ScanLayout {
  static constexpr int kTile = 16 * G * 256;             // a tile's landmark rows
  static constexpr int kBias = kScanRing * kTile;        // [ring][8][16] f32
  static constexpr int kBad = kBias + kScanRing * 512;   // [Cp / 64] u64
  static constexpr int kTotal = kBad + kScanMaxChunks / 8;
};

// total: [B, L, Hkv, G], or null (pre-softmax selection).
template <int G>
__global__ void __launch_bounds__(kScanThreads, 2)
    route_scan_kernel(RouteArgs a, const float* __restrict__ total, float* __restrict__ best,
                      int Cp) {
  using Lay = ScanLayout<G>;
  extern __shared__ __align__(16) unsigned char smem[];
  float* bias_s = reinterpret_cast<float*>(smem + Lay::kBias);
  uint64_t* bad_s = reinterpret_cast<uint64_t*>(smem + Lay::kBad);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, grp = lane >> 4;
  const int64_t b = blockIdx.z;
  const int h = blockIdx.y;
  const int64_t L = a.L;
  const int C = (int)a.C;
  const int nt = Cp >> 4;
  const int64_t r0 = (int64_t)blockIdx.x * kScanQ + 16 * wave;

  // Chunks with no valid real key, as bits.
  if (a.derive_window >= 0)
    for (int c0 = 64 * wave; c0 < Cp; c0 += kScanThreads) {
      const int c = c0 + lane;
      bool any = c < C && a.block_size > 1;
      if (any && a.key_valid)
        any = chunk_has_valid_key(a.key_valid + b * L + (int64_t)c * a.block_size, a.block_size);
      const uint64_t m = __builtin_amdgcn_ballot_w64(!any);
      if (lane == 0) bad_s[c0 >> 6] = m;
    }
  // Q rows r0 + j of every head; the totals of queries r0 + 4 grp + i (rows
  // past L re-read row L - 1).
  u32x4_t Q[G][4];
  float tot[G][4];
  {
    const int64_t row = ((b * L + min(r0 + j, L - 1)) * a.Hkv + h) * G;
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        Q[g][ks] =
            *reinterpret_cast<const u32x4_t*>(a.q + (row + g) * 128 + 8 * grp + 32 * ks);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t at = ((b * L + min(r0 + 4 * grp + i, L - 1)) * a.Hkv + h) * G;
#pragma unroll
      for (int g = 0; g < G; ++g) tot[g][i] = total ? total[at + g] : 0.f;
    }
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        asm volatile("" : "+v"(Q[g][i]));  // before any DMA
        asm volatile("" : "+v"(tot[g][i]));
      }
  }
  // Tile t into slot t % kScanRing: 4 DMA instructions of 4 rows x 256 bytes
  // per head (part p of row r at unit p ^ r; rows >= C re-read row C - 1) and,
  // with a bias, 2 of 64 floats for its [G][16] values, dealt to the waves in
  // turn.  Waves past the last one repeat it (the same bytes), so that every
  // wave counts the same number of loads in flight.
  const uint32_t rowlen = (uint32_t)(a.per_head_lmk ? a.Hkv * G : a.Hkv) * 128u;
  const __amdgpu_buffer_rsrc_t lrs = lmk_rsrc(a, b, rowlen);
  const uint32_t blen = (uint32_t)(a.Hkv * G);
  const __amdgpu_buffer_rsrc_t brs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(a.bias ? a.bias + b * C * (int64_t)blen : a.lse), (short)0,
      a.bias ? (int)((uint32_t)C * blen * 4u) : 0, 0x00020000);
  constexpr int kRows = 4 * G;
  constexpr int kMine = (kRows + 2 + 7) / 8;  // instructions per wave and tile
  const int ninstr = kRows + (a.bias ? 2 : 0);
  auto stage = [&](int t) {
    const int slot = t % kScanRing;
#pragma unroll
    for (int i = 0; i < kMine; ++i) {
      const int n = min(wave + 8 * i, ninstr - 1);
      if (n < kRows) {  // uniform
        const int row = 4 * (n & 3) + grp;
        const uint32_t c = (uint32_t)min(16 * t + row, C - 1);
        const uint32_t head = 256u * (uint32_t)(a.per_head_lmk ? h * G + (n >> 2) : h);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            lrs, (lds_void_t*)(smem + slot * Lay::kTile + n * 1024), 16,
            2u * (__umul24(c, rowlen) + 8u * (uint32_t)(j ^ row)), head, 0, 0);
      } else {
        const int e = 64 * (n - kRows) + lane;
        const uint32_t c = (uint32_t)min(16 * t + (e & 15), C - 1);
        const uint32_t g = (uint32_t)min(e >> 4, G - 1);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            brs, (lds_void_t*)(smem + Lay::kBias + slot * 512 + 256 * (n - kRows)), 4,
            4u * (__umul24(c, blen) + g), 4u * (uint32_t)(h * G), 0, 0);
      }
    }
  };
  if (!a.bias) {
    for (int i = tid; i < kScanRing * 128; i += kScanThreads) bias_s[i] = 0.f;
  }
#pragma unroll
  for (int t = 0; t < kScanRing - 1; ++t)
    if (t < nt) stage(t);
  int climit[4], lc[4], rc[4];
  const int win = (int)min(max(a.derive_window, (int64_t)0), L);
  const uint32_t bsz = (uint32_t)min(a.block_size, (int64_t)0x7fffffff);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t r = min(r0 + 4 * grp + i, L - 1);
    climit[i] = chunk_limit(a, r);
    lc[i] = (int)((uint32_t)max((int)r - win, 0) / bsz);
    rc[i] = (int)((uint32_t)min((int)r + win, (int)L - 1) / bsz);
  }
  auto step = [&](int t, bool hide) {
    // Tile t is in LDS for every wave once each has waited for its own share;
    // the barrier also frees slot t - 1 for tile t + ring - 1.
    const int later = min(kScanRing - 2, nt - 1 - t);
    if (later >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kMine) : "memory");
    else if (later == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kMine) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (t + kScanRing - 1 < nt) stage(t + kScanRing - 1);
    const int slot = t % kScanRing;
    const unsigned char* tile = smem + slot * Lay::kTile + j * 256;
    // the products of all heads first, so that their chains overlap
    f32x4_t x[G];
#pragma unroll
    for (int g = 0; g < G; ++g) x[g] = zero4();
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int g = 0; g < G; ++g)
        x[g] = mfma_bf16_16x16x32(Q[g][ks],
                                  *reinterpret_cast<const u32x4_t*>(
                                      tile + g * 4096 + (((4 * ks + grp) ^ j) * 16)),
                                  x[g]);
    float y[4] = {neg_inf(), neg_inf(), neg_inf(), neg_inf()};
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float bv = bias_s[slot * 128 + 16 * g + j];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // (an x of -inf stays -inf beside an infinite total)
        const float v = scaled_plus(x[g][i], a.sm_scale, bv);
        y[i] = fmaxf(y[i], v == neg_inf() ? v : v - tot[g][i]);
      }
    }
    const int c = 16 * t + j;
    const bool bad = a.derive_window >= 0 && ((bad_s[t >> 2] >> (16 * (t & 3) + j)) & 1ull);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t r = r0 + 4 * grp + i;
      if (hide && c >= climit[i]) y[i] = neg_inf();
      if (a.derive_window >= 0) {  // uniform
        if (bad | ((c >= lc[i]) & (c <= rc[i]))) y[i] = neg_inf();
      } else if (a.drop) {
        if (a.drop[(b * L + min(r, L - 1)) * C + min(c, C - 1)] != 0) y[i] = neg_inf();
      }
      if (r < L) best[((b * L + r) * a.Hkv + h) * Cp + c] = y[i];
    }
  };
  const int whole = a.is_causal ? 0 : C >> 4;
  for (int t = 0; t < whole; ++t) step(t, false);
  for (int t = whole; t < nt; ++t) step(t, true);
}

template <int G, int PER>
__global__ void __launch_bounds__(256)
    route_pick_kernel(RouteArgs a, const float* __restrict__ best, int Cp) {
  __shared__ int32_t list_s[4][64];
  __shared__ __align__(16) unsigned char ring_s[4][kPickRing * 4096];
  __shared__ __align__(16) unsigned char q_s[4][2048];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, grp = lane >> 4;
  const int64_t r = (int64_t)blockIdx.x * 4 + wv;
  if (r >= a.L) return;  // wave-uniform
  const int h = blockIdx.y;
  const int64_t b = blockIdx.z;
  const int C = (int)a.C, K = a.K;
  const int n = (C + 63) >> 6;  // <= PER
  const int64_t row = (b * a.L + r) * a.Hkv + h;
  // The row's G query heads to LDS (past them: zeros).
  {
    const __amdgpu_buffer_rsrc_t qrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(a.q + row * G * 128), (short)0, G * 256, 0x00020000);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(qrs, (lds_void_t*)(q_s[wv] + 1024 * i), 16,
                                               16u * lane, 1024u * i, 0, 0);
  }
  // The loads are unconditional (slots past the row read its last score), all
  // in flight together.
  uint32_t key[PER];
  {
    float v[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) v[i] = best[row * Cp + min(lane + 64 * i, C - 1)];
#pragma unroll
    for (int i = 0; i < PER; ++i)
      key[i] = lane + 64 * i < C ? float_order_key(v[i]) : 0u;  // 0: never picked
  }
  const uint64_t sel = WaveSelect<PER>::run(key, n, K);
  int32_t* list = list_s[wv];
  int total = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    if (i >= n) continue;  // uniform
    const bool p = (sel >> i) & 1ull;
    const uint64_t pb = __builtin_amdgcn_ballot_w64(p);
    if (p) list[total + __builtin_popcountll(pb & ((1ull << lane) - 1ull))] = lane + 64 * i;
    total += __builtin_popcountll(pb);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's list only
  if (lane < K) a.indices[row * K + lane] = lane < total ? list[lane] : -1;
  // Raw logits of the picks for every head: item (T, g) is a product whose
  // rows are picks 16 T .. 16 T + 15's landmark rows of head g and whose
  // every column is the query.  The rows pass through the wave's LDS ring, by
  // DMA in whole 256-byte rows (part p of row r at unit p ^ r; operand-shaped
  // loads would touch 16 rows per 16 bytes of each: 2.29 ms at 262144 rows of
  // 1024 chunks).  Lanes with j = g keep head g's picks 16 T + 4 grp + i.
  const uint32_t rowlen = (uint32_t)(a.per_head_lmk ? a.Hkv * G : a.Hkv) * 128u;
  const __amdgpu_buffer_rsrc_t lrs = lmk_rsrc(a, b, rowlen);
  unsigned char* ring = ring_s[wv];
  const int items = (K + 15) / 16 * G;
  auto stage = [&](int it) {
    const int T = it / G, g = it - T * G;
    const uint32_t head = 256u * (uint32_t)(a.per_head_lmk ? h * G + g : h);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int rr = 4 * k + grp, p = 16 * T + rr;
      const uint32_t c = p < total ? (uint32_t)list[p] : 0u;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          lrs, (lds_void_t*)(ring + (it % kPickRing) * 4096 + 1024 * k), 16,
          2u * (__umul24(c, rowlen) + 8u * (uint32_t)(j ^ rr)), head, 0, 0);
    }
  };
  for (int it = 0; it < kPickRing && it < items; ++it) stage(it);
  for (int T = 0; 16 * T < K; ++T) {
    f32x4_t keep = zero4();
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int it = T * G + g;
      if (it + 1 < items) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      const unsigned char* arow = ring + (it % kPickRing) * 4096 + j * 256;
      f32x4_t acc = zero4();
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        acc = mfma_bf16_16x16x32(
            *reinterpret_cast<const u32x4_t*>(arow + (((4 * ks + grp) ^ j) * 16)),
            *reinterpret_cast<const u32x4_t*>(q_s[wv] + 256 * g + 64 * ks + 16 * grp), acc);
#pragma unroll
      for (int i = 0; i < 4; ++i) keep[i] = j == g ? acc[i] : keep[i];
      if (it + kPickRing < items) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot has been read
        stage(it + kPickRing);
      }
    }
    const int s0 = 16 * T + 4 * grp;
    if (j < G) {
#pragma unroll
      for (int i = 0; i < 4; ++i) keep[i] = s0 + i < total ? keep[i] * a.sm_scale : neg_inf();
      const int64_t at = (row * G + j) * K + s0;
      if (a.scores_fp32) {
        for (int i = 0; i < 4; ++i)
          if (s0 + i < K) reinterpret_cast<float*>(a.scores)[at + i] = keep[i];
      } else if (a.vec_out) {  // K % 8 == 0: whole 8-byte groups
        if (s0 < K)
          *reinterpret_cast<u32x2_t*>(reinterpret_cast<uint16_t*>(a.scores) + at) =
              u32x2_t{pack_bf16x2(keep[0], keep[1]), pack_bf16x2(keep[2], keep[3])};
      } else {
        for (int i = 0; i < 4; ++i)
          if (s0 + i < K)
            reinterpret_cast<uint16_t*>(a.scores)[at + i] = (uint16_t)f32_to_bf16(keep[i]);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// General path.
// ---------------------------------------------------------------------------
constexpr int kGenThreads = 256;

__device__ __forceinline__ float block_reduce_max(float v, float* red) {
  v = wave_max(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float r = red[0];
  for (int w = 1; w < kGenThreads / 64; ++w) r = fmaxf(r, red[w]);
  return r;
}
__device__ __forceinline__ float block_reduce_sum(float v, float* red) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float r = 0.f;
  for (int w = 0; w < kGenThreads / 64; ++w) r += red[w];
  return r;
}
__device__ __forceinline__ int block_reduce_sum_i(int v, int* red) {
  v = wave_sum_i(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  int r = 0;
  for (int w = 0; w < kGenThreads / 64; ++w) r += red[w];
  return r;
}
// Exclusive prefix sum over the block (thread order), plus the total.
__device__ __forceinline__ int block_exclusive_scan(int v, int* scratch, int* total) {
  const int tid = threadIdx.x;
  __syncthreads();
  scratch[tid] = v;
  __syncthreads();
  for (int o = 1; o < kGenThreads; o <<= 1) {
    const int add = tid >= o ? scratch[tid - o] : 0;
    __syncthreads();
    scratch[tid] += add;
    __syncthreads();
  }
  const int incl = scratch[tid];
  *total = scratch[kGenThreads - 1];
  __syncthreads();
  return incl - v;
}

__global__ void __launch_bounds__(kGenThreads) route_topk_generic_kernel(RouteArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int64_t C = a.C, L = a.L;
  const int G = a.G, D = a.D, K = a.K;
  float* raw = reinterpret_cast<float*>(smem);  // [G][C]
  float* Ms = raw + (int64_t)G * C;             // [C]
  float* qs = Ms + C;                           // [G][D]
  float* tot = qs + G * D;                      // [G]
  float* redf = tot + G;                        // [8]
  int* redi = reinterpret_cast<int*>(redf + 8);  // [8]
  int* scan = redi + 8;                          // [256]

  const int tid = threadIdx.x;
  const int64_t r = blockIdx.x;
  const int h = blockIdx.y;
  const int64_t b = blockIdx.z;
  for (int e = tid; e < G * D; e += kGenThreads) {
    const int g = e / D, d = e - g * D;
    qs[e] = bf16_to_f32(a.q[(((b * L + r) * a.Hkv + h) * G + g) * D + d]);
  }
  __syncthreads();
  const int64_t climit = a.is_causal ? causal_limit(a, r) : C;
  for (int64_t p = tid; p < (int64_t)G * C; p += kGenThreads) {
    const int g = (int)(p / C);
    const int64_t c = p - (int64_t)g * C;
    const uint16_t* kr = lmk_row(a, b, c, h, g);
    const float* qr = qs + g * D;
    float acc = 0.f;
    for (int d = 0; d < D; ++d) acc = fmaf(qr[d], bf16_to_f32(kr[d]), acc);
    float x = acc * a.sm_scale;
    if (c >= climit) x = neg_inf();
    raw[p] = x;
  }
  __syncthreads();
  for (int g = 0; g < G; ++g) {
    float m = neg_inf();
    for (int64_t c = tid; c < C; c += kGenThreads) {
      const float bv = a.bias ? a.bias[((b * C + c) * a.Hkv + h) * G + g] : 0.f;
      m = fmaxf(m, raw[(int64_t)g * C + c] + bv);
    }
    m = block_reduce_max(m, redf);
    float s = 0.f;
    if (m != neg_inf())
      for (int64_t c = tid; c < C; c += kGenThreads) {
        const float bv = a.bias ? a.bias[((b * C + c) * a.Hkv + h) * G + g] : 0.f;
        s += expf(raw[(int64_t)g * C + c] + bv - m);
      }
    s = block_reduce_sum(s, redf);
    if (tid == 0) {
      const float lse_h = (m == neg_inf()) ? m : m + logf(s);
      const float lv = a.pre_softmax ? 0.f : a.lse[((b * L + r) * a.Hkv + h) * G + g];
      tot[g] = a.pre_softmax ? 0.f : logaddexp_f(lv, lse_h);
    }
  }
  __syncthreads();
  int64_t lc = 0, rc = -1;
  if (a.derive_window >= 0) {
    lc = max(r - a.derive_window, (int64_t)0) / a.block_size;
    rc = min(r + a.derive_window, L - 1) / a.block_size;
  }
  for (int64_t c = tid; c < C; c += kGenThreads) {
    float best = neg_inf();
    for (int g = 0; g < G; ++g) {
      const float bv = a.bias ? a.bias[((b * C + c) * a.Hkv + h) * G + g] : 0.f;
      const float xb = raw[(int64_t)g * C + c] + bv;
      best = fmaxf(best, xb == neg_inf() ? xb : xb - tot[g]);
    }
    bool dropped = false;
    if (a.derive_window >= 0) {
      bool any = false;
      if (a.key_valid) {
        const uint8_t* kv = a.key_valid + b * L + c * a.block_size;
        for (int64_t s = 0; s < a.block_size - 1; ++s) any |= kv[s] != 0;
      } else {
        any = a.block_size > 1;
      }
      dropped = (c >= lc && c <= rc) || !any;
    } else if (a.drop) {
      dropped = a.drop[(b * L + r) * C + c] != 0;
    }
    Ms[c] = dropped ? neg_inf() : best;
  }
  __syncthreads();

  // Threshold search on order keys (block-wide counts).
  const uint32_t kNeg = float_order_key(neg_inf());
  int nfin = 0;
  uint32_t kmin = 0xffffffffu, kmax = 0u;
  for (int64_t c = tid; c < C; c += kGenThreads) {
    const uint32_t key = float_order_key(Ms[c]);
    if (key > kNeg) {
      ++nfin;
      kmin = min(kmin, key);
      kmax = max(kmax, key);
    }
  }
  nfin = block_reduce_sum_i(nfin, redi);
  // min / max through float reductions on the key bits is not order-safe;
  // reduce the keys as ints instead.
  {
    int vmin = (int)(kmin ^ 0x80000000u), vmax = (int)(kmax ^ 0x80000000u);
    for (int o = 1; o < 64; o <<= 1) {
      vmin = min(vmin, __shfl_xor(vmin, o, 64));
      vmax = max(vmax, __shfl_xor(vmax, o, 64));
    }
    __syncthreads();
    if ((tid & 63) == 0) {
      redi[tid >> 6] = vmin;
      redi[4 + (tid >> 6)] = vmax;
    }
    __syncthreads();
    for (int w = 1; w < 4; ++w) {
      vmin = min(vmin, redi[w]);
      vmax = max(vmax, redi[4 + w]);
    }
    vmin = min(vmin, redi[0]);
    vmax = max(vmax, redi[4]);
    kmin = (uint32_t)vmin ^ 0x80000000u;
    kmax = (uint32_t)vmax ^ 0x80000000u;
  }
  uint32_t thr_hi, thr_tie = 0u;
  int need = 0;
  if (nfin <= K) {
    thr_hi = kNeg + 1u;
  } else {
    uint32_t lo = kmin, hi = kmax + 1u;
    bool exact = false;
    thr_hi = 0u;
    while (hi - lo > 1u) {
      const uint32_t mid = lo + ((hi - lo) >> 1);
      int cnt = 0;
      for (int64_t c = tid; c < C; c += kGenThreads) cnt += float_order_key(Ms[c]) >= mid ? 1 : 0;
      cnt = block_reduce_sum_i(cnt, redi);
      if (cnt == K) {
        thr_hi = mid;
        exact = true;
        break;
      }
      if (cnt > K) lo = mid; else hi = mid;
    }
    if (!exact) {
      int cnt_hi = 0;
      for (int64_t c = tid; c < C; c += kGenThreads) cnt_hi += float_order_key(Ms[c]) >= hi ? 1 : 0;
      cnt_hi = block_reduce_sum_i(cnt_hi, redi);
      thr_hi = hi;
      thr_tie = lo;
      need = K - cnt_hi;
    }
  }

  // Each thread owns a contiguous chunk range; scan counts for slots / tie ranks.
  const int64_t per = (C + kGenThreads - 1) / kGenThreads;
  const int64_t c0 = tid * per, c1 = min(C, c0 + per);
  int my_ties = 0;
  for (int64_t c = c0; c < c1; ++c) my_ties += (need > 0 && float_order_key(Ms[c]) == thr_tie) ? 1 : 0;
  int total_ties;
  int tie_base = block_exclusive_scan(my_ties, scan, &total_ties);
  int my_picks = 0;
  {
    int tr = tie_base;
    for (int64_t c = c0; c < c1; ++c) {
      const uint32_t key = float_order_key(Ms[c]);
      const bool tie = need > 0 && key == thr_tie;
      const bool pick = key >= thr_hi || (tie && tr < need);
      if (tie) ++tr;
      my_picks += pick ? 1 : 0;
    }
  }
  int total_picks;
  int slot = block_exclusive_scan(my_picks, scan, &total_picks);
  const int64_t row = (b * L + r) * a.Hkv + h;
  {
    int tr = tie_base;
    for (int64_t c = c0; c < c1; ++c) {
      const uint32_t key = float_order_key(Ms[c]);
      const bool tie = need > 0 && key == thr_tie;
      const bool pick = key >= thr_hi || (tie && tr < need);
      if (tie) ++tr;
      if (pick) {
        a.indices[row * K + slot] = (int32_t)c;
        for (int g = 0; g < G; ++g) {
          const float v = raw[(int64_t)g * C + c];
          if (a.scores_fp32)
            reinterpret_cast<float*>(a.scores)[(row * G + g) * K + slot] = v;
          else
            reinterpret_cast<uint16_t*>(a.scores)[(row * G + g) * K + slot] = (uint16_t)f32_to_bf16(v);
        }
        ++slot;
      }
    }
  }
  for (int s = total_picks + tid; s < K; s += kGenThreads) {
    a.indices[row * K + s] = -1;
    for (int g = 0; g < G; ++g) {
      if (a.scores_fp32)
        reinterpret_cast<float*>(a.scores)[(row * G + g) * K + s] = neg_inf();
      else
        reinterpret_cast<uint16_t*>(a.scores)[(row * G + g) * K + s] = 0xff80u;
    }
  }
}

// ---------------------------------------------------------------------------
// Short-block path: few query rows against many chunks (the cached block
// step: 32 rows, thousands of chunks).  Two kernels over a caller-provided
// fp32 workspace raw [B][L][Hkv][G][C] of scaled logits s = (q . lmk) * scale.
// ---------------------------------------------------------------------------
constexpr int kBlkQ = 32;        // query rows per logits workgroup
constexpr int kSelThreads = 512;
constexpr int kSelWaves = kSelThreads / 64;
constexpr int kSelMaxPer = 8;    // chunks per selection thread -> C <= 4096

// Logits: one workgroup per (16-chunk tile, 32-row tile, KV head, batch),
// one wave per query head g of the group.  S^T tiles on the matrix cores:
// A = 16 landmark rows, B = 16 query rows, both read straight from global
// memory (each landmark row is used by one wave only), all in one round trip.
__global__ void __launch_bounds__(512) route_logits_kernel(RouteArgs a, float* __restrict__ raw) {
  const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
  const int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t C = a.C, L = a.L;
  const int G = a.G;
  const int64_t c0 = (int64_t)blockIdx.x * 16;
  const int64_t q0 = (int64_t)blockIdx.y * kBlkQ;
  const int h = (int)(blockIdx.z % a.Hkv);
  const int64_t b = blockIdx.z / a.Hkv;
  const int64_t cl = min(c0 + col, C - 1);  // clamped: loads stay in bounds
  const int64_t qa = q0 + col, qb = q0 + 16 + col;
  const bool va = qa < L, vb = qb < L;
  const uint16_t* kr = lmk_row(a, b, cl, h, g) + 8 * grp;
  const uint16_t* qra = a.q + (((b * L + min(qa, L - 1)) * a.Hkv + h) * G + g) * 128 + 8 * grp;
  const uint16_t* qrb = a.q + (((b * L + min(qb, L - 1)) * a.Hkv + h) * G + g) * 128 + 8 * grp;
  u32x4_t A[4], Ba[4], Bb[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    A[j] = *reinterpret_cast<const u32x4_t*>(kr + 32 * j);
    Ba[j] = *reinterpret_cast<const u32x4_t*>(qra + 32 * j);
    Bb[j] = *reinterpret_cast<const u32x4_t*>(qrb + 32 * j);
  }
  f32x4_t Sa = zero4(), Sb = zero4();
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    Sa = mfma_bf16_16x16x32(A[j], Ba[j], Sa);
    Sb = mfma_bf16_16x16x32(A[j], Bb[j], Sb);
  }
  // Sa[i]: chunk c0 + 4 grp + i, row qa (Sb: row qb).
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t c = c0 + 4 * grp + i;
    if (c < C) {
      if (va) raw[(((b * L + qa) * a.Hkv + h) * G + g) * C + c] = Sa[i] * a.sm_scale;
      if (vb) raw[(((b * L + qb) * a.Hkv + h) * G + g) * C + c] = Sb[i] * a.sm_scale;
    }
  }
}

// Block-wide reduction of one value per head (G <= 8) with a single barrier
// (`red` holds kSelWaves x 8 floats and must not be read by a previous
// reduction any more).
template <bool MAX>
__device__ __forceinline__ void block_reduce8(float (&v)[8], int G, float* red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int g = 0; g < 8; ++g)
    if (g < G) v[g] = MAX ? wave_max(v[g]) : wave_sum(v[g]);
  if (lane == 0)
#pragma unroll
    for (int g = 0; g < 8; ++g)
      if (g < G) red[wave * 8 + g] = v[g];
  __syncthreads();
#pragma unroll
  for (int g = 0; g < 8; ++g) {
    if (g >= G) continue;
    float r = red[g];
#pragma unroll
    for (int w = 1; w < kSelWaves; ++w) r = MAX ? fmaxf(r, red[w * 8 + g]) : r + red[w * 8 + g];
    v[g] = r;
  }
}

// The K largest keys of a selection workgroup's row (K <= kTwoLevelMaxK,
// C <= 4096; key[i] of thread tid is chunk tid + 512 i) in two levels with
// one barrier.  Each wave first picks the K largest of its own chunks
// (chunks 512 i + 64 wave + lane: the wave order index 64 i + lane follows
// the chunk order, so its ties go to the lower chunk) and lists them in LDS;
// wave 0 then selects the K largest of the <= 8 K candidates, the ties at
// the threshold going to the lowest chunks, and writes the picks in
// ascending chunk order.  Each chunk of the row's K largest is among its
// wave's K largest, so the result is the one-level selection's.
constexpr int kTwoLevelMaxK = 64;

template <int G>
__device__ void select_two_level(const RouteArgs& a, const uint32_t (&key)[kSelMaxPer], int n,
                                 int64_t row, const float* xr) {
  constexpr int kCand = kSelWaves * kTwoLevelMaxK / 64;  // candidate slots per lane
  __shared__ uint32_t ck_s[kSelWaves * kTwoLevelMaxK];
  __shared__ uint16_t cc_s[kSelWaves * kTwoLevelMaxK];
  __shared__ int cn_s[kSelWaves];
  __shared__ uint32_t cmask[128];  // chunk bit sets (C <= 4096)
  __shared__ uint32_t cpre[128];   // set bits below each word
  const int K = a.K;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint64_t below = (1ull << lane) - 1ull;
  {
    const uint64_t wp = WaveSelect<kSelMaxPer>::run(key, n, K);
    int base = 0;
#pragma unroll
    for (int i = 0; i < kSelMaxPer; ++i) {
      if (i >= n) continue;
      const bool p = (wp >> i) & 1ull;
      const uint64_t bl = __builtin_amdgcn_ballot_w64(p);
      if (p) {
        const int pos = wave * K + base + __builtin_popcountll(bl & below);
        ck_s[pos] = key[i];
        cc_s[pos] = (uint16_t)(tid + kSelThreads * i);
      }
      base += __builtin_popcountll(bl);
    }
    if (lane == 0) cn_s[wave] = base;
  }
  __syncthreads();
  if (wave != 0) return;
  // candidate e = 64 j + lane: entry e - w K of wave w = e / K
  const int n2 = (kSelWaves * K + 63) / 64;
  uint32_t ckey[kCand];
  int cch[kCand];
#pragma unroll
  for (int j = 0; j < kCand; ++j) {
    const int e = 64 * j + lane;
    const int w = e / K;
    const bool ok = j < n2 && w < kSelWaves && e - w * K < cn_s[w < kSelWaves ? w : 0];
    ckey[j] = ok ? ck_s[e] : 0u;
    cch[j] = ok ? (int)cc_s[e] : 0;
  }
  uint32_t thr_hi, thr_tie;
  int need;
  WaveSelect<kCand>::threshold(ckey, n2, K, thr_hi, thr_tie, need);
  // rank[j] = the members of the set below chunk cch[j] (for members), from
  // a chunk bit set in LDS and its per-word prefix counts (this wave only:
  // the LDS runs one wave's operations in order).
  auto ranks = [&](const bool (&in)[kCand], int (&rank)[kCand]) {
    asm volatile("" ::: "memory");
    cmask[lane] = 0u;
    cmask[lane + 64] = 0u;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < kCand; ++j)
      if (in[j]) atomicOr(&cmask[cch[j] >> 5], 1u << (cch[j] & 31));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const uint32_t w0 = cmask[2 * lane], w1 = cmask[2 * lane + 1];
    const int cnt = __popc(w0) + __popc(w1);
    int incl = cnt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(incl, o, 64);
      if (lane >= o) incl += t;
    }
    cpre[2 * lane] = (uint32_t)(incl - cnt);
    cpre[2 * lane + 1] = (uint32_t)(incl - cnt + __popc(w0));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int j = 0; j < kCand; ++j) {
      rank[j] = 0;
      if (in[j]) {
        const int c = cch[j];
        rank[j] = (int)cpre[c >> 5] + __popc(cmask[c >> 5] & ((1u << (c & 31)) - 1u));
      }
    }
  };
  bool pick[kCand];
#pragma unroll
  for (int j = 0; j < kCand; ++j) pick[j] = j < n2 && ckey[j] >= thr_hi;
  if (need > 0) {  // wave-uniform: ties at the threshold to the lowest chunks
    bool tie[kCand];
    int tr[kCand];
#pragma unroll
    for (int j = 0; j < kCand; ++j) tie[j] = j < n2 && ckey[j] == thr_tie;
    ranks(tie, tr);
#pragma unroll
    for (int j = 0; j < kCand; ++j)
      if (tie[j] && tr[j] < need) pick[j] = true;
  }
  int slot[kCand];
  ranks(pick, slot);
  // The picks' chunks to lane slot order through the candidate area (free
  // now), then lane t writes output slot t with all its loads in flight.
  int total = 0;
#pragma unroll
  for (int j = 0; j < kCand; ++j) total += __builtin_popcountll(__builtin_amdgcn_ballot_w64(pick[j]));
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int j = 0; j < kCand; ++j)
    if (pick[j]) cc_s[slot[j]] = (uint16_t)cch[j];
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  if (lane < K) {
    const int t = lane;
    const bool live = t < total;
    const int64_t c = live ? (int64_t)cc_s[t] : 0;
    float v[G];
#pragma unroll
    for (int g = 0; g < G; ++g) v[g] = xr[(int64_t)g * a.C + c];
    a.indices[row * K + t] = live ? (int32_t)c : -1;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (a.scores_fp32)
        reinterpret_cast<float*>(a.scores)[(row * G + g) * K + t] = live ? v[g] : neg_inf();
      else
        reinterpret_cast<uint16_t*>(a.scores)[(row * G + g) * K + t] =
            live ? (uint16_t)f32_to_bf16(v[g]) : (uint16_t)0xff80u;
    }
  }
}

// Selection: one workgroup per (row, KV head, batch); chunk c = tid + 512 i.
// The row's logits and bias are read once into registers.  Same score, LSE,
// drop and tie rules as the general kernel.
template <int G>
__global__ void __launch_bounds__(kSelThreads) route_select_kernel(RouteArgs a,
                                                                   const float* __restrict__ raw) {
  using Select = BlockSelect<kSelThreads, kSelMaxPer>;
  __shared__ float redf[2][kSelWaves * 8];
  __shared__ typename Select::Lds sel;
  const int64_t C = a.C, L = a.L;
  const int K = a.K;
  const int tid = threadIdx.x;
  const int64_t r = blockIdx.x;
  const int h = blockIdx.y;
  const int64_t b = blockIdx.z;
  const int n = (int)((C + kSelThreads - 1) / kSelThreads);  // <= kSelMaxPer
  const int64_t row = (b * L + r) * a.Hkv + h;
  const float* xr = raw + row * (int64_t)G * C;
  const int64_t climit = a.is_causal ? causal_limit(a, r) : C;

  // 1. x = s + bias (-inf past the causal limit or the last chunk).  The
  //    loads are unconditional (slots past the row read chunk 0), with no
  //    branch between them, so that they are all in flight at once: loads
  //    inside per-element branches were each waited for at the branch's end.
  float x[kSelMaxPer][G];
#pragma unroll
  for (int i = 0; i < kSelMaxPer; ++i) {
    const int64_t c = tid + (int64_t)kSelThreads * i;
    const int64_t cc = i < n && c < C ? c : 0;
#pragma unroll
    for (int g = 0; g < G; ++g) x[i][g] = xr[(int64_t)g * C + cc];
  }
  if (a.bias) {
    const float* brow = a.bias + (b * C * a.Hkv + h) * G;  // chunk c at c Hkv G
    const int64_t bstride = (int64_t)a.Hkv * G;
#pragma unroll
    for (int i = 0; i < kSelMaxPer; ++i) {
      const int64_t c = tid + (int64_t)kSelThreads * i;
      const int64_t cc = i < n && c < C ? c : 0;
#pragma unroll
      for (int g = 0; g < G; ++g) x[i][g] += brow[cc * bstride + g];
    }
  }
#pragma unroll
  for (int i = 0; i < kSelMaxPer; ++i) {
    const int64_t c = tid + (int64_t)kSelThreads * i;
    const bool ok = i < n && c < C && c < climit;
#pragma unroll
    for (int g = 0; g < G; ++g) x[i][g] = ok ? x[i][g] : neg_inf();
  }

  // 2. Per-head LSE over every chunk (dropped ones included).
  float m[8], sum[8];
#pragma unroll
  for (int g = 0; g < 8; ++g) {
    m[g] = neg_inf();
    sum[g] = 0.f;
  }
#pragma unroll
  for (int i = 0; i < kSelMaxPer; ++i)
#pragma unroll
    for (int g = 0; g < G; ++g) m[g] = fmaxf(m[g], x[i][g]);
  block_reduce8<true>(m, G, redf[0]);
#pragma unroll
  for (int i = 0; i < kSelMaxPer; ++i)
#pragma unroll
    for (int g = 0; g < G; ++g)
      if (m[g] != neg_inf()) sum[g] += expf(x[i][g] - m[g]);
  block_reduce8<false>(sum, G, redf[1]);
  float tot[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const float lse_h = m[g] == neg_inf() ? m[g] : m[g] + logf(sum[g]);
    const float lv = a.pre_softmax ? 0.f : a.lse[row * G + g];
    tot[g] = a.pre_softmax ? 0.f : logaddexp_f(lv, lse_h);
  }

  // 3. Selection keys: max over heads of x - tot, dropped chunks -inf.
  int64_t lc = 0, rc = -1;
  if (a.derive_window >= 0) {
    lc = max(r - a.derive_window, (int64_t)0) / a.block_size;
    rc = min(r + a.derive_window, L - 1) / a.block_size;
  }
  // Drop flags first, one uniform branch per drop source (loads batched as
  // in step 1).
  bool dropped[kSelMaxPer];
  if (a.derive_window >= 0) {
#pragma unroll
    for (int i = 0; i < kSelMaxPer; ++i) {
      const int64_t c = tid + (int64_t)kSelThreads * i;
      const int64_t cc = i < n && c < C ? c : 0;
      bool any = a.block_size > 1;
      if (a.key_valid) any = chunk_has_valid_key(a.key_valid + b * L + cc * a.block_size,
                                                 a.block_size);
      dropped[i] = (c >= lc && c <= rc) || !any;
    }
  } else if (a.drop) {
#pragma unroll
    for (int i = 0; i < kSelMaxPer; ++i) {
      const int64_t c = tid + (int64_t)kSelThreads * i;
      const int64_t cc = i < n && c < C ? c : 0;
      dropped[i] = a.drop[(b * L + r) * C + cc] != 0;
    }
  } else {
#pragma unroll
    for (int i = 0; i < kSelMaxPer; ++i) dropped[i] = false;
  }
  uint32_t key[kSelMaxPer];
#pragma unroll
  for (int i = 0; i < kSelMaxPer; ++i) {
    const int64_t c = tid + (int64_t)kSelThreads * i;
    float best = neg_inf();
#pragma unroll
    for (int g = 0; g < G; ++g) best = fmaxf(best, x[i][g] == neg_inf() ? x[i][g] : x[i][g] - tot[g]);
    // 0 is below every real key: never picked
    key[i] = i < n && c < C ? float_order_key(dropped[i] ? neg_inf() : best) : 0u;
  }

  // 4. The K largest (ties to the lower chunk), in ascending chunk order.
  if (K <= kTwoLevelMaxK) {
    select_two_level<G>(a, key, n, row, xr);
    return;
  }
  bool pick[kSelMaxPer];
  int slot[kSelMaxPer];
  const int slot_base = Select::run(key, n, K, sel, pick, slot);
  // The picks' raw scores, all loaded before any store.
  float sv[kSelMaxPer][G];
#pragma unroll
  for (int i = 0; i < kSelMaxPer; ++i) {
    const int64_t c = tid + (int64_t)kSelThreads * i;
    const int64_t cc = i < n && c < C ? c : 0;
#pragma unroll
    for (int g = 0; g < G; ++g) sv[i][g] = xr[(int64_t)g * C + cc];
  }
#pragma unroll
  for (int i = 0; i < kSelMaxPer; ++i) {
    if (i >= n || !pick[i]) continue;
    const int64_t c = tid + (int64_t)kSelThreads * i;
    a.indices[row * K + slot[i]] = (int32_t)c;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float v = sv[i][g];
      if (a.scores_fp32)
        reinterpret_cast<float*>(a.scores)[(row * G + g) * K + slot[i]] = v;
      else
        reinterpret_cast<uint16_t*>(a.scores)[(row * G + g) * K + slot[i]] = (uint16_t)f32_to_bf16(v);
    }
  }
  for (int t = slot_base + tid; t < K; t += kSelThreads) {
    a.indices[row * K + t] = -1;
    for (int g = 0; g < G; ++g) {
      if (a.scores_fp32)
        reinterpret_cast<float*>(a.scores)[(row * G + g) * K + t] = neg_inf();
      else
        reinterpret_cast<uint16_t*>(a.scores)[(row * G + g) * K + t] = 0xff80u;
    }
  }
}

template <int G>
int launch_select(const RouteArgs& a, const float* raw, hipStream_t s) {
  dim3 g2((unsigned)a.L, (unsigned)a.Hkv, (unsigned)a.B);
  hipLaunchKernelGGL(route_select_kernel<G>, g2, dim3(kSelThreads), 0, s, a, raw);
  return mrsa_launch_status();
}

int launch_block(const RouteArgs& a, float* raw, hipStream_t s) {
  dim3 g1((unsigned)((a.C + 15) / 16), (unsigned)((a.L + kBlkQ - 1) / kBlkQ),
          (unsigned)(a.Hkv * a.B));
  hipLaunchKernelGGL(route_logits_kernel, g1, dim3(64 * a.G), 0, s, a, raw);
  int st = mrsa_launch_status();
  if (st != MRSA_OK) return st;
  switch (a.G) {
    case 1: return launch_select<1>(a, raw, s);
    case 2: return launch_select<2>(a, raw, s);
    case 3: return launch_select<3>(a, raw, s);
    case 4: return launch_select<4>(a, raw, s);
    case 5: return launch_select<5>(a, raw, s);
    case 6: return launch_select<6>(a, raw, s);
    case 7: return launch_select<7>(a, raw, s);
    default: return launch_select<8>(a, raw, s);
  }
}

template <int NT, int QT>
int launch_heads(const RouteArgs& a, hipStream_t s) {
  using Lay = HeadsLayout<NT, QT>;
  const size_t smem = Lay::total(a.G, a.K);
  auto kern = route_heads_kernel<NT, QT>;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
    return MRSA_ERR_LAUNCH;
  dim3 grid((unsigned)((a.L + Lay::kQ - 1) / Lay::kQ), (unsigned)a.Hkv, (unsigned)a.B);
  hipLaunchKernelGGL(kern, grid, dim3(kHeadThreads), smem, s, a, Lay::bias(a.G),
                     Lay::picks(a.G));
  return mrsa_launch_status();
}

template <int G>
int launch_tile(const RouteArgs& a, hipStream_t s) {
  const size_t smem = TileLayout::total(a.K);
  auto kern = route_tile_kernel<G>;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
    return MRSA_ERR_LAUNCH;
  dim3 grid((unsigned)((a.L + kTileQ - 1) / kTileQ), (unsigned)a.Hkv, (unsigned)a.B);
  hipLaunchKernelGGL(kern, grid, dim3(kTileThreads), smem, s, a);
  return mrsa_launch_status();
}

// The one-pass kernels.  At 7 heads x 4 KV heads, K = 32 (us, route_tile /
// route_heads): 1024 queries x 16 chunks 55 / 9, 8064 x 63 77 / 39, 8192 x 128
// 77 / 53, 32 x 128 66 / 13; 8192 x 256 79 / 98, 16384 x 256 157 / 198.  A
// wave of route_tile keeps all 256 chunks of its 16 queries for every head, so
// it pays for 256 chunks whatever C is and needs 256 workgroups of 128 queries
// to fill the chip; route_heads pays per chunk and forms each logit once, but
// reads the landmarks once per 16 or 32 queries.
constexpr int64_t kTileMinGroups = 256;
// 32 queries per workgroup of route_heads where that fills the chip twice.
constexpr int64_t kHeadsWide = 512;

int launch_fast(const RouteArgs& a, hipStream_t s) {
  const bool wide = (a.L + 31) / 32 * a.Hkv * a.B >= kHeadsWide;
  if (a.C <= 64) return wide ? launch_heads<4, 2>(a, s) : launch_heads<4, 1>(a, s);
  if (a.C <= 128) return wide ? launch_heads<8, 2>(a, s) : launch_heads<8, 1>(a, s);
  if (a.G >= 7 && (a.L + kTileQ - 1) / kTileQ * a.Hkv * a.B >= kTileMinGroups)
    return a.G == 7 ? launch_tile<7>(a, s) : launch_tile<8>(a, s);
  return launch_heads<16, 1>(a, s);
}

// Rows (token, KV head, batch) from which the scan path (128 queries per
// workgroup) replaces the logits + workgroup selection, which spreads few rows
// over more of the chip.
constexpr int64_t kScanRows = 4096;

template <int G>
int launch_scan(const RouteArgs& a, float* ws, hipStream_t s) {
  const int Cp = (int)scan_chunks(a.C);
  const unsigned blocks = (unsigned)((a.L + kScanQ - 1) / kScanQ);
  float* best = ws;                                  // [B, L, Hkv, Cp]
  float* total = ws + a.B * a.L * a.Hkv * (int64_t)Cp;  // [B, L, Hkv, G]
  int st;
  if (!a.pre_softmax) {
    hipLaunchKernelGGL(route_lse_kernel, dim3(blocks, (unsigned)(a.Hkv * G), (unsigned)a.B),
                       dim3(kScanThreads), 0, s, a, total);
    st = mrsa_launch_status();
    if (st != MRSA_OK) return st;
  }
  const size_t smem = ScanLayout<G>::kTotal;
  auto scan = route_scan_kernel<G>;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(scan),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
    return MRSA_ERR_LAUNCH;
  hipLaunchKernelGGL(scan, dim3(blocks, (unsigned)a.Hkv, (unsigned)a.B), dim3(kScanThreads), smem,
                     s, a, a.pre_softmax ? nullptr : total, best, Cp);
  st = mrsa_launch_status();
  if (st != MRSA_OK) return st;
  dim3 g2((unsigned)((a.L + 3) / 4), (unsigned)a.Hkv, (unsigned)a.B);
  auto pick = a.C <= 256    ? route_pick_kernel<G, 4>
              : a.C <= 1024 ? route_pick_kernel<G, 16>
              : a.C <= 2048 ? route_pick_kernel<G, 32>
                            : route_pick_kernel<G, 64>;
  hipLaunchKernelGGL(pick, g2, dim3(256), 0, s, a, best, Cp);
  return mrsa_launch_status();
}

int launch_scan(const RouteArgs& a, float* best, hipStream_t s) {
  switch (a.G) {
    case 1: return launch_scan<1>(a, best, s);
    case 2: return launch_scan<2>(a, best, s);
    case 3: return launch_scan<3>(a, best, s);
    case 4: return launch_scan<4>(a, best, s);
    case 5: return launch_scan<5>(a, best, s);
    case 6: return launch_scan<6>(a, best, s);
    case 7: return launch_scan<7>(a, best, s);
    default: return launch_scan<8>(a, best, s);
  }
}

}  // namespace

namespace {

// The one-pass matrix-core kernel (no workspace) serves the call.  Shared by
// the dispatcher and the no-allocation entry point, which must agree on
// which problems need the workspace.
bool fast_path(const void* q, const void* lmk, int64_t chunks, int64_t kv_heads, int64_t groups,
               int64_t head_dim, int64_t topk, int is_causal, int scores_fp32) {
  const bool aligned = ((uintptr_t)q % 16 == 0) && ((uintptr_t)lmk % 16 == 0);
  // (a batch's landmark keys, read through one buffer resource, stay under 2 GB)
  return !scores_fp32 && !is_causal && head_dim == 128 && chunks <= kFastMaxChunks &&
         topk <= kFastMaxTopk && aligned && groups <= 8 &&
         chunks * kv_heads * groups * head_dim * 2 < ((int64_t)1 << 31);
}

// Shapes the scan path serves (it needs a workspace of scan_bytes).
bool scan_path(int64_t batch, int64_t seq_len, int64_t chunks, int64_t kv_heads, int64_t groups,
               int64_t head_dim, int64_t topk) {
  return head_dim == 128 && groups <= 8 && topk <= kFastMaxTopk && chunks <= kScanMaxChunks &&
         batch * seq_len * kv_heads >= kScanRows && kv_heads * groups <= 65535 &&
         chunks * kv_heads * groups * head_dim * 2 < ((int64_t)1 << 31);
}
int64_t scan_bytes(int64_t batch, int64_t seq_len, int64_t chunks, int64_t kv_heads,
                   int64_t groups) {
  return batch * seq_len * kv_heads * (scan_chunks(chunks) + groups) * 4;
}

int route_topk_dispatch(const void* q, const void* lmk, const float* lse_local, const float* bias,
                        const int32_t* drop_mask, const uint8_t* key_valid,
                        int64_t derive_window, int64_t batch, int64_t seq_len, int64_t chunks,
                        int64_t kv_heads, int64_t groups, int64_t head_dim, int64_t topk,
                        int64_t block_size, int per_head_lmk, int is_causal,
                        int64_t window_size, int64_t q_offset, int selection_mode,
                        float sm_scale, int32_t* indices, void* scores, int scores_fp32,
                        void* workspace, int64_t workspace_bytes, void* stream) {
  if (batch < 0 || seq_len < 0 || chunks <= 0 || kv_heads <= 0 || groups <= 0 ||
      head_dim <= 0 || topk <= 0 || block_size <= 0 || (selection_mode != 0 && selection_mode != 1))
    return MRSA_ERR_INVALID_ARGUMENT;
  if (batch == 0 || seq_len == 0) return MRSA_OK;
  if (!q || !lmk || !indices || !scores) return MRSA_ERR_INVALID_ARGUMENT;
  if (selection_mode == 0 && !lse_local) return MRSA_ERR_INVALID_ARGUMENT;
  if (derive_window >= 0 && chunks * block_size != seq_len) return MRSA_ERR_INVALID_ARGUMENT;
  if (kv_heads > 65535 || batch > 65535) return MRSA_ERR_UNSUPPORTED;

  RouteArgs a;
  a.q = (const uint16_t*)q;
  a.lmk = (const uint16_t*)lmk;
  a.lse = lse_local;
  a.bias = bias;
  a.drop = drop_mask;
  a.key_valid = key_valid;
  a.derive_window = derive_window;
  a.B = batch;
  a.L = seq_len;
  a.C = chunks;
  a.Hkv = (int)kv_heads;
  a.G = (int)groups;
  a.D = (int)head_dim;
  a.K = (int)topk;
  a.block_size = block_size;
  a.per_head_lmk = per_head_lmk;
  a.is_causal = is_causal;
  a.window_size = window_size;
  a.q_offset = q_offset;
  a.pre_softmax = selection_mode;
  a.sm_scale = sm_scale;
  a.indices = indices;
  a.scores = scores;
  a.scores_fp32 = scores_fp32;
  a.vec32_out =
      topk % 32 == 0 && (uintptr_t)indices % 16 == 0 && (uintptr_t)scores % 16 == 0;
  a.vec_out = topk % 8 == 0 && (uintptr_t)scores % 16 == 0;
  hipStream_t s = (hipStream_t)stream;

  const bool aligned = ((uintptr_t)q % 16 == 0) && ((uintptr_t)lmk % 16 == 0);
  if (fast_path(q, lmk, chunks, kv_heads, groups, head_dim, topk, is_causal, scores_fp32)) 
    return launch_fast(a, s);
  if (workspace && (uintptr_t)workspace % 16 == 0 && aligned && seq_len <= 0x7fffffff &&
      scan_path(batch, seq_len, chunks, kv_heads, groups, head_dim, topk) &&
      workspace_bytes >= scan_bytes(batch, seq_len, chunks, kv_heads, groups))
    return launch_scan(a, (float*)workspace, s);
  const bool block = workspace && head_dim == 128 && groups <= 8 && aligned &&
                     chunks <= (int64_t)kSelThreads * kSelMaxPer && seq_len <= 0x7fffffff &&
                     (uintptr_t)workspace % 16 == 0 &&
                     workspace_bytes >= batch * seq_len * kv_heads * groups * chunks * 4;
  if (block) return launch_block(a, (float*)workspace, s);
  const size_t smem = ((size_t)groups * chunks + chunks + groups * head_dim + groups + 16) * 4 +
                      kGenThreads * 4;
  if (smem > 150 * 1024) return MRSA_ERR_UNSUPPORTED;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(&route_topk_generic_kernel),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
    return MRSA_ERR_LAUNCH;
  if (seq_len > 0x7fffffff) return MRSA_ERR_UNSUPPORTED;
  dim3 grid((unsigned)seq_len, (unsigned)kv_heads, (unsigned)batch);
  hipLaunchKernelGGL(route_topk_generic_kernel, grid, dim3(kGenThreads), smem, s, a);
  return mrsa_launch_status();
}

}  // namespace

extern "C" int mrsa_route_topk_fwd(const void* q, const void* lmk, const float* lse_local,
                                   const float* bias, const int32_t* drop_mask,
                                   const uint8_t* key_valid, int64_t derive_window, int64_t batch,
                                   int64_t seq_len, int64_t chunks, int64_t kv_heads,
                                   int64_t groups, int64_t head_dim, int64_t topk,
                                   int64_t block_size, int per_head_lmk, int is_causal,
                                   int64_t window_size, int64_t q_offset, int selection_mode,
                                   float sm_scale, int32_t* indices, void* scores,
                                   int scores_fp32, void* stream) {
  return route_topk_dispatch(q, lmk, lse_local, bias, drop_mask, key_valid, derive_window, batch,
                             seq_len, chunks, kv_heads, groups, head_dim, topk, block_size,
                             per_head_lmk, is_causal, window_size, q_offset, selection_mode,
                             sm_scale, indices, scores, scores_fp32, nullptr, 0, stream);
}

extern "C" int64_t mrsa_route_topk_workspace_bytes(int64_t batch, int64_t seq_len, int64_t chunks,
                                                   int64_t kv_heads, int64_t groups) {
  if (batch < 0 || seq_len < 0 || chunks < 0 || kv_heads < 0 || groups < 0) return -1;
  return batch * seq_len * kv_heads * groups * chunks * 4;
}

extern "C" int64_t mrsa_route_topk_needed_bytes(int64_t batch, int64_t seq_len, int64_t chunks,
                                                int64_t kv_heads, int64_t groups,
                                                int64_t head_dim, int64_t topk, int is_causal,
                                                int scores_fp32) {
  if (batch < 0 || seq_len < 0 || chunks < 0 || kv_heads < 0 || groups < 0) return -1;
  if (!scores_fp32 && !is_causal && head_dim == 128 && chunks <= kFastMaxChunks &&
      topk <= kFastMaxTopk && groups <= 8)
    return 0;
  if (scan_path(batch, seq_len, chunks, kv_heads, groups, head_dim, topk))
    return scan_bytes(batch, seq_len, chunks, kv_heads, groups);
  if (head_dim != 128 || groups > 8 || chunks > (int64_t)kSelThreads * kSelMaxPer) return 0;
  return batch * seq_len * kv_heads * groups * chunks * 4;
}

// ---------------------------------------------------------------------------
// No-allocation variant: the workspace is a file-scope device array.
//
// `scratch` is one fixed buffer per GPU (each device holds its own copy for
// the life of the process).  Host code never passes the array's name to a
// kernel: its device address is looked up once per device with
// hipGetSymbolAddress (with that device current) and kept in scratch_ptr.
// Every call on one GPU shares the buffer, so calls that overlap on one GPU
// (two streams, two threads) race; the kernels write every byte they later
// read, so nothing needs clearing between calls.
// ---------------------------------------------------------------------------
static __device__ __align__(256) uint8_t scratch[MRSA_ROUTE_TOPK_SCRATCH_BYTES];

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxScratchDevices] = {};

// The current device's address of `scratch` (looked up on first use).
int scratch_address(void** out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return MRSA_ERR_LAUNCH;
  if (dev < 0 || dev >= kMaxScratchDevices) return MRSA_ERR_UNSUPPORTED;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr)
      return MRSA_ERR_LAUNCH;
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return MRSA_OK;
}
}  // namespace

extern "C" int mrsa_route_topk_noalloc_fwd(
    const void* q, const void* lmk, const float* lse_local, const float* bias,
    const int32_t* drop_mask, const uint8_t* key_valid, int64_t derive_window, int64_t batch,
    int64_t seq_len, int64_t chunks, int64_t kv_heads, int64_t groups, int64_t head_dim,
    int64_t topk, int64_t block_size, int per_head_lmk, int is_causal, int64_t window_size,
    int64_t q_offset, int selection_mode, float sm_scale, int32_t* indices, void* scores,
    int scores_fp32, void* stream) {
  if (batch < 0 || seq_len < 0 || chunks <= 0 || kv_heads <= 0 || groups <= 0)
    return MRSA_ERR_INVALID_ARGUMENT;
  // What the caller may rely on is the size of the fp32 logits [batch, seq_len,
  // kv_heads, groups, chunks], except for the one-pass kernel with 7 or 8
  // groups: larger problems are refused also where the call would take less
  // (the one-pass kernel with fewer groups, the scan path).
  const bool one_pass = groups >= 7 && fast_path(q, lmk, chunks, kv_heads, groups, head_dim, topk,
                                                 is_causal, scores_fp32);
  const int64_t need = one_pass ? 0 : batch * seq_len * kv_heads * groups * chunks * 4;
  if (need > (int64_t)MRSA_ROUTE_TOPK_SCRATCH_BYTES) return MRSA_ERR_SCRATCH;
  void* ws = nullptr;
  if (need > 0) {
    const int st = scratch_address(&ws);
    if (st != MRSA_OK) return st;
  }
  return route_topk_dispatch(q, lmk, lse_local, bias, drop_mask, key_valid, derive_window, batch,
                             seq_len, chunks, kv_heads, groups, head_dim, topk, block_size,
                             per_head_lmk, is_causal, window_size, q_offset, selection_mode,
                             sm_scale, indices, scores, scores_fp32, ws, need, stream);
}

extern "C" int mrsa_route_topk_ws_fwd(const void* q, const void* lmk, const float* lse_local,
                                      const float* bias, const int32_t* drop_mask,
                                      const uint8_t* key_valid, int64_t derive_window,
                                      int64_t batch, int64_t seq_len, int64_t chunks,
                                      int64_t kv_heads, int64_t groups, int64_t head_dim,
                                      int64_t topk, int64_t block_size, int per_head_lmk,
                                      int is_causal, int64_t window_size, int64_t q_offset,
                                      int selection_mode, float sm_scale, int32_t* indices,
                                      void* scores, int scores_fp32, void* workspace,
                                      int64_t workspace_bytes, void* stream) {
  if (workspace_bytes < 0 || (workspace_bytes > 0 && !workspace)) return MRSA_ERR_INVALID_ARGUMENT;
  return route_topk_dispatch(q, lmk, lse_local, bias, drop_mask, key_valid, derive_window, batch,
                             seq_len, chunks, kv_heads, groups, head_dim, topk, block_size,
                             per_head_lmk, is_causal, window_size, q_offset, selection_mode,
                             sm_scale, indices, scores, scores_fp32, workspace, workspace_bytes,
                             stream);
}
