// Backward of the routed (selected-chunk) attention.
//
// Forward: out[q, g] = sum_k w[q, g, k] * softmax_{s in chunk idx[q, k], s visible}(q_g . k_s * scale) . V
// (the forward kernel's semantics: a list ends at its first negative entry,
// entries >= kv_len / 64 are skipped, the landmark slot and invalid / dropped
// keys are not visible).  The backward follows the reference kernel
// ops/hils_fwd_bwd_head.py:573-910, which also rounds P and w dO to bf16:
//   P      = softmax over the visible keys (recomputed here, fp32);
//   dP     = dO . V^T (fp32);  di = sum_s P dP  ->  dW[q, g, k] = di (bf16);
//   dS     = bf16(scale * w * P * (dP - di));
//   dQ    += dS . K            (fp32, summed over the query's chunks);
//   dK    += dS^T . Q,  dV += bf16(w * P)^T . dO  (fp32, summed over the
//            (query, slot) pairs that route to the chunk).
// A chunk listed twice is processed once per slot (its gradient terms add,
// as the weights do in the forward).
//
// Work split (chunk-major).  A list of the (query, slot) pairs of every
// chunk is built first (count, scan, fill); a workgroup then owns one chunk
// (or a segment of its pairs) and recomputes each pair's
// chunk softmax:
//   dK / dV  stay in the workgroup's registers and are written once per
//            chunk (added with atomics when the chunk's pairs span several
//            segments) -- the reference instead adds each query block's
//            dK / dV into global memory with atomics;
//   dS       each pair's bf16 dS tile is stored as a record (128 bytes per
//            (query, head, slot));
//   dW       written directly (one pair = one slot).
// dQ is then the forward kernel's walk over each query tile's chunks
// (routed_attention.hip, mrsa::routed_dq_walk): the tiles take the records
// as their P^T operand and K^T where the forward reads V, and the rows are
// summed in LDS and added into dQ once -- no atomics.
// Operands come from two fragment layouts of the same K / V:
//   fwd = mrsa_kv_fragments(k, v): K images (keys x dims) for S^T = K . Q^T;
//   bwd = mrsa_kv_fragments(v, k): V images (keys x dims) for dP^T = V . dO^T
//         and K^T images (dims x keys, tiled order) for the walk's dS . K.
#include "chunk_tile.h"
#include "mrsa_device.h"

#include <algorithm>
#include <type_traits>

using namespace mrsa;

namespace {

constexpr int kMaxTopk = 64;

struct BwdArgs {
  const uint16_t* q;
  const uint16_t* dout;
  const uint16_t* fwd;       // [B, Hkv, Ck, 16384]: K images | V^T images
  const uint16_t* bwd;       // [B, Hkv, Ck, 16384]: V images | K^T images
  const uint16_t* w;
  const int32_t* idx;
  const uint8_t* key_valid;
  const int8_t* keep;        // [B, Lq, Hkv, K, 64] or null
  int64_t B, Lq, Lk, Ck;
  int Hq, Hkv, G, K;
  int mask_last;
  float scale, scale_log2;
  float* dq;                 // [B, Lq, Hq, 128] fp32
  float* dk;                 // [B, Lk, Hkv, 128] fp32, accumulated
  float* dv;                 // [B, Lk, Hkv, 128] fp32, accumulated
  uint16_t* dw;              // [B, Lq, Hq, K] bf16
  // chunk-major pass: pair lists (entry = query | slot << 24), per chunk
  // (b, h, c) the list start and the first work unit
  const int32_t* list;
  const int32_t* start;      // [B * Hkv * Ck + 1]
  const int32_t* ustart;     // [B * Hkv * Ck + 1]
  const float* slope;        // [Hq] ALiBi slopes or null
  // dS records [B, Lq, Hq, K] x 64 bf16 (key 32 t + 16 m + j at 32 t + 2 j + m),
  // one per listed slot, for the dQ walk.
  uint16_t* ds_rec;
  uint16_t* sink;            // 256 elements nothing reads
  int seg;                   // pairs per work unit
};


__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes,
                                           (int)0x00020000);
}
// Bits of the nonzero bytes (bit j = byte j) of one 64-byte keep / key-valid
// row: one byte per lane and a wave ballot (every lane must be active).
__device__ __forceinline__ uint64_t nonzero_bits(const int8_t* row) {
  return __builtin_amdgcn_ballot_w64(row[threadIdx.x & 63] != 0);
}

// ---- chunk-major dK / dV ---------------------------------------------------
constexpr int kListBlock = 256;       // queries per list workgroup (one per thread)
constexpr int kMaxListChunks = 8192;  // LDS counters of the list kernels (32 KB)

// (query, slot) pairs per dK / dV work unit: about 4096 units (16 per CU), at
// least 256 pairs (a unit's K, V and dK / dV traffic) and at most 1024.  At
// 16384 queries the backward takes 3.51 ms with 512, 3.61 with 1024, 0.5 more with
// 2048.
int64_t segment_entries(int64_t pairs) {
  const int64_t n = (pairs / 4096 + 63) / 64 * 64;
  return n < 256 ? 256 : n > 1024 ? 1024 : n;
}

// The valid slots of one index row: up to the first negative entry, chunks
// below Ck.
template <class F>
__device__ __forceinline__ void for_each_slot(const int32_t* row, int K, int64_t Ck, F&& f) {
  for (int k = 0; k < K; ++k) {
    const int32_t c = row[k];
    if (c < 0) break;
    if (c < Ck) f(k, c);
  }
}

// 1. Pairs per (chunk, query block) in LDS; each block's run of a chunk's
//    list is reserved with one global add (blkbase = its offset).
__global__ void __launch_bounds__(kListBlock) list_count_kernel(BwdArgs a, int32_t* count,
                                                                int32_t* blkbase, int nqb) {
  __shared__ int32_t hist[kMaxListChunks];
  const int tid = threadIdx.x;
  const int qb = blockIdx.x;
  const int64_t bh = blockIdx.y;
  const int64_t b = bh / a.Hkv;
  const int h = (int)(bh % a.Hkv);
  for (int64_t c = tid; c < a.Ck; c += kListBlock) hist[c] = 0;
  __syncthreads();
  const int64_t q = (int64_t)qb * kListBlock + tid;
  if (q < a.Lq)
    for_each_slot(a.idx + ((b * a.Lq + q) * a.Hkv + h) * a.K, a.K, a.Ck,
                  [&](int, int32_t c) { atomicAdd(&hist[c], 1); });
  __syncthreads();
  for (int64_t c = tid; c < a.Ck; c += kListBlock) {
    const int n = hist[c];
    blkbase[(bh * nqb + qb) * a.Ck + c] = n ? atomicAdd(&count[bh * a.Ck + c], n) : 0;
  }
}

// 2. Exclusive scans over the chunks (b, h, c): list starts and work-unit
//    starts (ceil(count / seg) units per chunk).  One workgroup.
__global__ void __launch_bounds__(1024) list_scan_kernel(const int32_t* count, int64_t N,
                                                         int seg, int32_t* start,
                                                         int32_t* ustart) {
  __shared__ int32_t s1[1024], s2[1024];
  const int tid = threadIdx.x;
  const int64_t per = (N + 1023) / 1024;
  const int64_t lo = min(N, tid * per), hi = min(N, lo + per);
  int32_t t1 = 0, t2 = 0;
  for (int64_t i = lo; i < hi; ++i) {
    t1 += count[i];
    t2 += (count[i] + seg - 1) / seg;
  }
  s1[tid] = t1;
  s2[tid] = t2;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    const int32_t u1 = tid >= o ? s1[tid - o] : 0, u2 = tid >= o ? s2[tid - o] : 0;
    __syncthreads();
    s1[tid] += u1;
    s2[tid] += u2;
    __syncthreads();
  }
  int32_t r1 = s1[tid] - t1, r2 = s2[tid] - t2;
  for (int64_t i = lo; i < hi; ++i) {
    start[i] = r1;
    ustart[i] = r2;
    r1 += count[i];
    r2 += (count[i] + seg - 1) / seg;
  }
  if (tid == 1023) {
    start[N] = s1[1023];
    ustart[N] = s2[1023];
  }
}

// 3. Pairs written into their chunk's list: query | slot << 24.
__global__ void __launch_bounds__(kListBlock) list_fill_kernel(BwdArgs a, const int32_t* blkbase,
                                                               int nqb, int32_t* list) {
  __shared__ int32_t cur[kMaxListChunks];
  const int tid = threadIdx.x;
  const int qb = blockIdx.x;
  const int64_t bh = blockIdx.y;
  const int64_t b = bh / a.Hkv;
  const int h = (int)(bh % a.Hkv);
  for (int64_t c = tid; c < a.Ck; c += kListBlock) cur[c] = 0;
  __syncthreads();
  const int64_t q = (int64_t)qb * kListBlock + tid;
  if (q < a.Lq)
    for_each_slot(a.idx + ((b * a.Lq + q) * a.Hkv + h) * a.K, a.K, a.Ck, [&](int k, int32_t c) {
      const int p = atomicAdd(&cur[c], 1);
      const int64_t bhc = bh * a.Ck + c;
      list[(int64_t)a.start[bhc] + blkbase[(bh * nqb + qb) * a.Ck + c] + p] =
          (int32_t)(q | ((int64_t)k << 24));
    });
}

// One workgroup per work unit: chunk (b, h, c) and a segment of its pairs.  8
// waves: wave 2 w + s takes keys 32 s .. 32 s + 31 of the pairs of group w, 4 a
// round, as 32 matrix rows (row 8 p + g: pair p, head g):
//   S = Q . K^T and dP = dO . V^T: lane (grp, j) gets rows 16 ct + 4 grp + r of
//     keys 16 mt + j of its half; the rows' sums of p = 2^x and p dP over the
//     16 lanes, and over the two halves through LDS;
//   dK += dS^T . Q and dV += bf16(w P)^T . dO: a lane's rows are consecutive
//     elements of the products' reduction, so dS and w P are operands as they
//     leave the softmax, and Q and dO rows are read from LDS transposed.
// Q and dO rows arrive by DMA in whole 256-byte rows, a round ahead (row r's
// 16-byte part p at unit p ^ (r & 15)); half of a wave's K stays in registers,
// the rest and V in LDS, its dK and dV (32 keys x 128 dims, fp32) in 128 accumulators, summed
// over the four groups through LDS once per unit.  Halving the keys and not
// the pairs is what lets two waves share a SIMD; with 64 keys per wave the 256
// accumulators left no registers and the kernel ran 5090 us.  No unit is at its
// limit at 16384 queries x 28 heads x 32 slots: the matrix cores work 21% of the
// cycles, the VALU 43% (products included), LDS 31%; 8.4 GB read (the Q and dO
// rows, once per routed slot) and 2.7 GB written make 4.9 TB/s.  The waves wait
// 39% of their time, at a round's two barriers and for the rows, and two of them
// per SIMD do not cover it.  Measured there: 2270 us; with eight pairs per
// workgroup and round, element-wise transposes through LDS and no prefetch
// 3410 us.
constexpr int kGroups = 4;                 // pair groups of a workgroup
constexpr int kDkvThreads = 128 * kGroups;
constexpr int kPairs = 4;                  // per group and round
constexpr uint32_t kRowsBytes = 32 * 256;  // one round's Q or dO rows of a group
constexpr uint32_t kDkvK = 16384;          // K images of key tiles 1 and 3 (8 KB)
constexpr uint32_t kDkvExch = 24576;       // [2][2 kGroups][3][32] f32 row sums
constexpr uint32_t kDkvRows = kDkvExch + 2 * 2 * kGroups * 384;  // [group][2][Q, dO] rows
constexpr uint32_t kDkvLds = kDkvRows + kGroups * 4 * kRowsBytes;
static_assert(kDkvRows % 256 == 0 && kGroups * 32768 <= kDkvLds, "row alignment; the final sums");

template <bool ALIBI, bool KEEP>
__global__ void __launch_bounds__(kDkvThreads, 2) routed_attn_dkv_kernel(BwdArgs a) {
  extern __shared__ __align__(256) unsigned char sm[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wave >> 1, half = wave & 1;
  const int j = lane & 15, grp = lane >> 4;
  const int64_t N = a.B * a.Hkv * a.Ck;
  const int64_t u = blockIdx.x;
  if (u >= (int64_t)a.ustart[N]) return;  // workgroup-uniform
  // the chunk whose units hold u: ustart[lo] <= u < ustart[lo + 1]
  int64_t lo = 0, hi = N;
  while (hi - lo > 1) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)a.ustart[mid] <= u) lo = mid;
    else hi = mid;
  }
  const int64_t bhc = lo;
  const int cs = a.start[bhc], ce = a.start[bhc + 1];
  const int e0 = cs + (int)(u - a.ustart[bhc]) * a.seg;
  const int e1 = min(ce, e0 + a.seg);
  const bool whole = ce - cs <= a.seg;
  const int64_t c = bhc % a.Ck;
  const int64_t bh = bhc / a.Ck;
  const int h = (int)(bh % a.Hkv);
  const int64_t b = bh / a.Hkv;
  const int G = a.G, K = a.K;

  uint64_t excl = a.mask_last ? (1ull << 63) : 0ull;
  if (a.key_valid)
    excl |= ~nonzero_bits(reinterpret_cast<const int8_t*>(a.key_valid + b * a.Lk + c * 64));
  const uint32_t l16 = 16u * lane;
  const unsigned char* kimg = reinterpret_cast<const unsigned char*>(
      a.fwd + ((b * a.Hkv + h) * a.Ck + c) * 16384);
  u32x4_t kb[4];  // K images of the half's first key tile
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    kb[ks] = *reinterpret_cast<const u32x4_t*>(kimg + 1024 * (8 * half + ks) + l16);
  {
    // the other one's: image (half, ks) at 1024 (4 half + ks)
    const int o = 16 * tid;
    *reinterpret_cast<u32x4_t*>(sm + kDkvK + o) = *reinterpret_cast<const u32x4_t*>(
        kimg + 4096 + (o & 4095) + 2 * (o & 4096));
  }
  {
    // the V images: the first half of the chunk's bwd fragment (16 KB)
    const unsigned char* vsrc = reinterpret_cast<const unsigned char*>(
        a.bwd + ((b * a.Hkv + h) * a.Ck + c) * 16384);
#pragma unroll
    for (int i = 0; i < 16384 / 16 / kDkvThreads; ++i) {
      const int o = 16 * (tid + kDkvThreads * i);
      *reinterpret_cast<u32x4_t*>(sm + o) = *reinterpret_cast<const u32x4_t*>(vsrc + o);
    }
  }
  const float c2 = a.scale_log2;
  const int g4 = 4 * (grp & 1);  // this lane's rows: heads g4 + r of pair 2 ct + phalf
  const int phalf = grp >> 1;
  const float ninf = neg_inf();
  // 0, or -inf where key 16 mt + j of half t is excluded
  auto mask_of = [&](int t, int mt) {
    return ((excl >> (32 * t + 16 * mt + j)) & 1ull) ? ninf : 0.f;
  };
  const float madd[2] = {mask_of(half, 0), mask_of(half, 1)};
  float sl[4];                   // ALiBi: -slope c2 of this lane's heads
#pragma unroll
  for (int r = 0; r < 4; ++r)
    sl[r] = ALIBI ? -a.slope[(int64_t)h * G + min(g4 + r, G - 1)] * c2 : 0.f;
  auto alibi = [&](int t, int mt, int r, float x) {
    return ALIBI ? __builtin_fmaf(sl[r], fmaxf(0.f, (float)(62 - 32 * t - 16 * mt - j)), x) : x;
  };
  // DMA lane offsets: instruction k (0..7) fills rows 4 k + grp of the round
  // (pair k >> 1, head 4 (k & 1) + grp; heads past G - 1 repeat it).
  uint32_t voff[4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    voff[k] = 256u * (uint32_t)min(4 * (k & 1) + grp, G - 1) +
              16u * (uint32_t)(j ^ ((4 * k + grp) & 15));
  unsigned char* rows = sm + kDkvRows + group * 4 * kRowsBytes;  // [2][Q, dO]
  const int64_t row0 = b * a.Lq * a.Hq + (int64_t)h * G;         // row of query 0, head 0
  // the first pair of this group's round i; absent pairs repeat the last one
  auto base_of = [&](int i) { return e0 + kGroups * kPairs * i + kPairs * group; };
  auto entry = [&](int i) { return a.list[min(base_of(i) + (lane & 3), e1 - 1)]; };
  // half 0 brings the group's Q rows, half 1 its dO rows
  const uint16_t* src = half ? a.dout : a.q;
  auto stage = [&](const int32_t (&ent)[kPairs], int buf) {
#pragma unroll
    for (int p = 0; p < kPairs; ++p) {
      const __amdgpu_buffer_rsrc_t rs = make_rsrc(
          src + (row0 + (int64_t)(ent[p] & 0xffffff) * a.Hq) * 128, (uint32_t)G * 256u);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const int k = 2 * p + kk;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rs, (lds_void_t*)(rows + (2 * buf + half) * kRowsBytes + 1024 * k), 16, voff[k & 3], 0,
            0, 0);
      }
    }
  };
  auto split = [&](int32_t v, int32_t (&ent)[kPairs]) {
#pragma unroll
    for (int p = 0; p < kPairs; ++p) ent[p] = __builtin_amdgcn_readlane(v, p);
  };
  // The routing weights of this lane's rows (raw; padding heads repeat the last)
  auto load_w = [&](const int32_t (&ent)[kPairs], uint32_t (&w)[2][4]) {
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
      const int32_t v = phalf ? ent[2 * ct + 1] : ent[2 * ct];
      const uint16_t* wp =
          a.w + (row0 + (int64_t)(v & 0xffffff) * a.Hq + g4) * K + ((v >> 24) & 63);
#pragma unroll
      for (int r = 0; r < 4; ++r) w[ct][r] = wp[min(r, G - 1 - g4) * K];
    }
  };
  const unsigned char* vown = sm + 8192 * half + l16;  // V images of this wave's keys
  const unsigned char* kown = sm + kDkvK + 4096 * half + l16;
  f32x4_t dk[2][8], dv[2][8];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) {
      dk[mt][nt] = zero4();
      dv[mt][nt] = zero4();
    }
  int32_t ent[kPairs], ent2[kPairs], entn[kPairs];
  const int rounds = (e1 - e0 + kGroups * kPairs - 1) / (kGroups * kPairs);
  // One pass over the unit's pairs; true when some row's sum left fp32's range
  // (never with STAB: p is then stabilised by each half's maximum).
  auto pass = [&](auto stab) {
    constexpr bool STAB = decltype(stab)::value;
    bool fine = true;
    split(entry(0), ent);
    stage(ent, 0);
    asm volatile("" ::: "memory");
    int32_t evn = entry(1);
    for (int i = 0; i < rounds; ++i) {
      const int base = base_of(i);
      const int buf = i & 1;
      // This wave's rows of the round have landed; the barrier covers the other
      // waves' (and, first, the V and K images), and their reads of the buffers
      // written next.  Wait and barrier are one block: a wait that comes from
      // the use of a value loaded after the rows may be moved past the barrier.
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      split(evn, entn);
      uint32_t wraw[2][4];
      load_w(ent, wraw);
      asm volatile("" ::: "memory");
      stage(entn, buf ^ 1);
      asm volatile("" ::: "memory");
      evn = entry(i + 2);
      asm volatile("" ::: "memory");

      // Addresses of this lane's operand rows (row j + 16 ct, part 4 ks + grp:
      // ks flips bits 6 and 7), and below of the transposed reads.  Formed anew
      // each round from a redefined lane number: held across rounds they spill,
      // and a reload waits for every load and store in flight.
      uint32_t lj = lane;
      asm volatile("" : "+v"(lj));
      const uint32_t arow = lds_addr(rows) + (uint32_t)buf * 2u * kRowsBytes + 256u * (lj & 15u) +
                            16u * (((lj >> 4) ^ (lj & 3u)) | (lj & 12u));
      // S = Q . K^T and dP = dO . V^T of 16 rows
      auto products = [&](int ct, f32x4_t (&S)[2], f32x4_t (&dP)[2]) {
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) S[mt] = dP[mt] = zero4();
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          const uint32_t at = (arow ^ (64u * ks)) + 4096u * ct;
          const u32x4_t A = lds_read16(at), D = lds_read16(at + kRowsBytes);
#pragma unroll
          for (int mt = 0; mt < 2; ++mt) {
            S[mt] = mfma_bf16_16x16x32(
                A, mt ? *reinterpret_cast<const u32x4_t*>(kown + 1024 * ks) : kb[ks], S[mt]);
            dP[mt] = mfma_bf16_16x16x32(
                D, *reinterpret_cast<const u32x4_t*>(vown + 1024 * (4 * mt + ks)), dP[mt]);
          }
        }
      };
      f32x4_t dP[2][2];
      float e[2][2][4];        // p = 2^x (STAB: 2^(x - the half's maximum))
      float* ex = reinterpret_cast<float*>(sm + kDkvExch) + (buf * 2 * kGroups + wave) * 96;
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) {
        f32x4_t S[2];
        products(ct, S, dP[ct]);
        float ma[2] = {madd[0], madd[1]};
        if constexpr (KEEP) {
          const int32_t v = phalf ? ent[2 * ct + 1] : ent[2 * ct];
          const int64_t qrow = (row0 + (int64_t)(v & 0xffffff) * a.Hq) / G;  // (b Lq + q) Hkv + h
          const int8_t* kr = a.keep + (qrow * K + ((v >> 24) & 63)) * 64 + 32 * half + j;
#pragma unroll
          for (int mt = 0; mt < 2; ++mt)
            if (kr[16 * mt] == 0) ma[mt] = ninf;
        }
        f32x4_t psum, pd, pmax;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float x[2];
#pragma unroll
          for (int mt = 0; mt < 2; ++mt)
            x[mt] = alibi(half, mt, r, __builtin_fmaf(S[mt][r], c2, ma[mt]));
          if constexpr (STAB) {
            // (an excluded key's NaN or infinite logit is not made -inf by the
            // sum above; without STAB it fails the range test)
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) x[mt] = ma[mt] == ninf ? ninf : x[mt];
            const float m = group16_max(fmaxf(x[0], x[1]));
            pmax[r] = m;
            const float mb = m == ninf ? 0.f : m;
            x[0] -= mb;
            x[1] -= mb;
          }
#pragma unroll
          for (int mt = 0; mt < 2; ++mt) e[ct][mt][r] = exp2_hw(x[mt]);
          psum[r] = group16_sum(e[ct][0][r] + e[ct][1][r]);
          pd[r] = group16_sum(
              __builtin_fmaf(e[ct][0][r], dP[ct][0][r], e[ct][1][r] * dP[ct][1][r]));
        }
        // (the 16 lanes of a group write the same values)
        float* exc = ex + 16 * ct + 4 * grp;
        *reinterpret_cast<f32x4_t*>(exc) = psum;
        *reinterpret_cast<f32x4_t*>(exc + 32) = pd;
        if constexpr (STAB) *reinterpret_cast<f32x4_t*>(exc + 64) = pmax;
        __builtin_amdgcn_sched_barrier(0);  // one tile's operands at a time
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const float* exo = reinterpret_cast<const float*>(sm + kDkvExch) +
                         (buf * 2 * kGroups + (wave ^ 1)) * 96 + 4 * grp;
      u32x4_t dsb[2], wpb[2];  // dS^T and (w P)^T operands: element 4 ct + r
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) {
        const int32_t v = phalf ? ent[2 * ct + 1] : ent[2 * ct];
        const bool have = base + 2 * ct + phalf < e1;
        const int64_t prow = row0 + (int64_t)(v & 0xffffff) * a.Hq;
        const int slot = (v >> 24) & 63;
        // the rows' sums over both halves (the own ones are read back too: they
        // take no registers across the barrier)
        const float* exc = ex + 16 * ct + 4 * grp;
        f32x4_t psum = *reinterpret_cast<const f32x4_t*>(exc);
        f32x4_t pd = *reinterpret_cast<const f32x4_t*>(exc + 32);
        const f32x4_t so = *reinterpret_cast<const f32x4_t*>(exo + 16 * ct);
        const f32x4_t po = *reinterpret_cast<const f32x4_t*>(exo + 32 + 16 * ct);
        if constexpr (STAB) {
          const f32x4_t pm = *reinterpret_cast<const f32x4_t*>(exc + 64);
          const f32x4_t mo = *reinterpret_cast<const f32x4_t*>(exo + 64 + 16 * ct);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float m = fmaxf(pm[r], mo[r]), mb = m == ninf ? 0.f : m;
            const float f = exp2_hw(pm[r] - mb), fo = exp2_hw(mo[r] - mb);
            psum[r] = psum[r] * f + so[r] * fo;
            pd[r] = pd[r] * f + po[r] * fo;
            e[ct][0][r] *= f;
            e[ct][1][r] *= f;
          }
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            psum[r] += so[r];
            pd[r] += po[r];
            fine = fine && psum[r] >= 0x1p-64f && psum[r] <= 0x1p64f;
          }
        }
        float di[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float inv = psum[r] > 0.f ? rcp_hw(psum[r]) : 0.f;
          const float wi = have && g4 + r < G ? bf16_to_f32(wraw[ct][r]) * inv : 0.f;
          di[r] = pd[r] * inv;
          const float dis = -di[r] * a.scale;
#pragma unroll
          for (int mt = 0; mt < 2; ++mt) {
            const float wp = e[ct][mt][r] * wi;  // w P
            dP[ct][mt][r] = wp * __builtin_fmaf(dP[ct][mt][r], a.scale, dis);  // dS
            e[ct][mt][r] = wp;
          }
        }
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
          dsb[mt][2 * ct] = pack_bf16x2(dP[ct][mt][0], dP[ct][mt][1]);
          dsb[mt][2 * ct + 1] = pack_bf16x2(dP[ct][mt][2], dP[ct][mt][3]);
          wpb[mt][2 * ct] = pack_bf16x2(e[ct][mt][0], e[ct][mt][1]);
          wpb[mt][2 * ct + 1] = pack_bf16x2(e[ct][mt][2], e[ct][mt][3]);
        }
        // The dS records (key 32 t + 16 mt + j at 32 t + 2 j + mt) and dW = di;
        // absent rows write to the sink, so that no branch surrounds the stores.
        uint16_t* rec = a.ds_rec + ((prow + g4) * K + slot) * 64 + 32 * half + 2 * j;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          uint16_t* dst = have && g4 + r < G ? rec + (int64_t)r * K * 64 : a.sink + 2 * lane;
          *reinterpret_cast<uint32_t*>(dst) = pack_bf16x2(dP[ct][0][r], dP[ct][1][r]);
        }
        const float dj = (j & 2) ? ((j & 1) ? di[3] : di[2]) : ((j & 1) ? di[1] : di[0]);
        uint16_t* dwp = half == 0 && have && j < 4 && g4 + j < G
                            ? a.dw + (prow + g4 + j) * K + slot
                            : a.sink + 2 * lane;
        *dwp = (uint16_t)f32_to_bf16(dj);
        __builtin_amdgcn_sched_barrier(0);
      }
      // row 4 grp + (j >> 2) (+ 16 ct), dims 16 nt + 4 (j & 3): the dim tile
      // flips bits 5..7
      const uint32_t rr = lj >> 2;
      const uint32_t tb = lds_addr(rows) + (uint32_t)buf * 2u * kRowsBytes + 256u * rr +
                          16u * (rr & 14u) + 16u * (((lj >> 1) ^ rr) & 1u) + 8u * (lj & 1u);
#pragma unroll
      for (int nt = 0; nt < 8; ++nt) {
        const uint32_t ta = tb ^ (32u * nt);
        const u32x2_t q0 = read_transposed(ta), q1 = read_transposed(ta + 4096u);
        const u32x2_t o0 = read_transposed(ta + kRowsBytes);
        const u32x2_t o1 = read_transposed(ta + kRowsBytes + 4096u);
        const u32x4_t bq = {q0[0], q0[1], q1[0], q1[1]}, bo = {o0[0], o0[1], o1[0], o1[1]};
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
          dk[mt][nt] = mfma_bf16_16x16x32(dsb[mt], bq, dk[mt][nt]);
          dv[mt][nt] = mfma_bf16_16x16x32(wpb[mt], bo, dv[mt][nt]);
        }
        if (nt & 1) __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int p = 0; p < kPairs; ++p) ent[p] = entn[p];
    }
    return !fine;
  };
  // Unstabilised sums lie well inside fp32's range for any |x| well below 64;
  // a unit with a row outside it (extreme logits) runs again, stabilised.
  // Keep rows often drop a whole chunk and go there at once, as does a chunk
  // with no visible key.
  bool again = KEEP || ~excl == 0ull;
  if (!again) again = __syncthreads_or(pass(std::integral_constant<bool, false>{}) ? 1 : 0) != 0;
  if (again) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int nt = 0; nt < 8; ++nt) dk[mt][nt] = dv[mt][nt] = zero4();
    pass(std::integral_constant<bool, true>{});
  }
  // The groups' sums through LDS (a tensor at a time, [group][64][128]): lane
  // (grp, j) of tile (mt, nt) holds keys 16 mt + 4 grp + r of its half, dim
  // 16 nt + j.
  float* part = reinterpret_cast<float*>(sm);
  const int64_t krow = (int64_t)a.Hkv * 128;
  auto reduce = [&](const f32x4_t (&x)[2][8], float* out) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no DMA is in flight into the region
    __syncthreads();
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int nt = 0; nt < 8; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          part[group * 8192 + (32 * half + 16 * mt + 4 * grp + r) * 128 + 16 * nt + j] =
              x[mt][nt][r];
    __syncthreads();
#pragma unroll 4
    for (int i = 0; i < 8192 / kDkvThreads; ++i) {
      const int o = tid + kDkvThreads * i;  // element of [64][128]
      const float t = (part[o] + part[8192 + o]) + (part[2 * 8192 + o] + part[3 * 8192 + o]);
      float* dst = out + (int64_t)(o >> 7) * krow + (o & 127);
      if (whole) *dst = t;
      else atomicAdd(dst, t);
    }
  };
  reduce(dk, a.dk + ((b * a.Lk + c * 64) * a.Hkv + h) * 128);
  reduce(dv, a.dv + ((b * a.Lk + c * 64) * a.Hkv + h) * 128);
}

__global__ void __launch_bounds__(256) fill_zero_i32(int32_t* p, int64_t n) {
  for (int64_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] = 0;
}

struct ListPlan {
  int nqb;
  int64_t n;  // chunks B * Hkv * Ck
  int64_t count, blkbase, start, ustart, list, records, sink, total;  // byte offsets / size
  int64_t max_units, seg;
};

ListPlan list_plan(int64_t B, int64_t Lq, int64_t Hkv, int64_t K, int64_t Ck, int64_t Hq) {
  ListPlan p;
  p.nqb = (int)((Lq + kListBlock - 1) / kListBlock);
  p.n = B * Hkv * Ck;
  const int64_t pairs = B * Lq * Hkv * K;
  int64_t o = 0;
  auto take = [&](int64_t bytes) {
    const int64_t at = o;
    o += (bytes + 255) / 256 * 256;
    return at;
  };
  p.count = take(p.n * 4);
  p.blkbase = take(B * Hkv * p.nqb * Ck * 4);
  p.start = take((p.n + 1) * 4);
  p.ustart = take((p.n + 1) * 4);
  p.list = take(pairs * 4);
  p.records = take(B * Lq * Hq * K * 64 * 2);  // dS records of the dQ walk
  p.sink = take(512);
  p.total = o;
  p.seg = segment_entries(pairs);
  p.max_units = (pairs + p.seg - 1) / p.seg + p.n;
  return p;
}

}  // namespace

namespace {

int selected_backward(
    const void* q, const void* grad_out, const void* kv_frags, const void* kv_frags_bwd,
    const void* weights, const int32_t* indices, const uint8_t* key_valid,
    const int8_t* token_keep, int64_t batch, int64_t q_len, int64_t kv_len, int64_t q_heads,
    int64_t kv_heads, int64_t head_dim, int64_t topk, int64_t chunk_size, int mask_last_token,
    float sm_scale, float* grad_q, float* grad_k, float* grad_v, void* grad_weights,
    void* workspace, int64_t workspace_bytes, void* stream, const float* slope) {
  if (batch < 0 || q_len < 0 || kv_len < 0 || q_heads <= 0 || kv_heads <= 0 ||
      q_heads % kv_heads != 0 || head_dim <= 0 || topk <= 0 || chunk_size <= 0 ||
      !(sm_scale > 0.f) || sm_scale == __builtin_inff())
    return MRSA_ERR_INVALID_ARGUMENT;
  if (kv_len % chunk_size != 0) return MRSA_ERR_INVALID_ARGUMENT;
  if (chunk_size != 64 || head_dim != 128 || q_heads / kv_heads > 8 || topk > kMaxTopk)
    return MRSA_ERR_UNSUPPORTED;
  if (kv_len / 64 > kMaxListChunks || q_len >= (1 << 24)) return MRSA_ERR_UNSUPPORTED;
  if (batch * q_len * kv_heads * topk >= 0x7fffffff) return MRSA_ERR_UNSUPPORTED;
  if (batch == 0 || q_len == 0) return MRSA_OK;
  if (!q || !grad_out || !kv_frags || !kv_frags_bwd || !weights || !indices || !grad_q ||
      !grad_k || !grad_v || !grad_weights || !workspace)
    return MRSA_ERR_INVALID_ARGUMENT;
  const ListPlan lp = list_plan(batch, q_len, kv_heads, topk, kv_len / 64, q_heads);
  if (workspace_bytes < lp.total || (uintptr_t)workspace % 256 != 0)
    return MRSA_ERR_INVALID_ARGUMENT;
  if (((uintptr_t)q | (uintptr_t)grad_out | (uintptr_t)kv_frags | (uintptr_t)kv_frags_bwd |
       (uintptr_t)grad_q) % 16 != 0)
    return MRSA_ERR_INVALID_ARGUMENT;
  BwdArgs a;
  a.q = (const uint16_t*)q;
  a.dout = (const uint16_t*)grad_out;
  a.fwd = (const uint16_t*)kv_frags;
  a.bwd = (const uint16_t*)kv_frags_bwd;
  a.w = (const uint16_t*)weights;
  a.idx = indices;
  a.key_valid = key_valid;
  a.keep = token_keep;
  a.B = batch;
  a.Lq = q_len;
  a.Lk = kv_len;
  a.Ck = kv_len / 64;
  a.Hq = (int)q_heads;
  a.Hkv = (int)kv_heads;
  a.G = (int)(q_heads / kv_heads);
  a.K = (int)topk;
  a.mask_last = mask_last_token;
  a.scale = sm_scale;
  a.scale_log2 = sm_scale * kLog2e;
  a.dq = grad_q;
  a.dk = grad_k;
  a.dv = grad_v;
  a.dw = (uint16_t*)grad_weights;
  a.slope = slope;
  if (lp.max_units > 0x7fffffff || lp.nqb > 0x7fffffff || batch * kv_heads > 65535)
    return MRSA_ERR_UNSUPPORTED;
  hipStream_t st = (hipStream_t)stream;
  // pair lists, then the chunk-major pass
  char* ws = (char*)workspace;
  int32_t* count = (int32_t*)(ws + lp.count);
  int32_t* blkbase = (int32_t*)(ws + lp.blkbase);
  int32_t* start = (int32_t*)(ws + lp.start);
  int32_t* ustart = (int32_t*)(ws + lp.ustart);
  int32_t* list = (int32_t*)(ws + lp.list);
  hipLaunchKernelGGL(fill_zero_i32, dim3((unsigned)std::min<int64_t>((lp.n + 255) / 256, 4096)),
                     dim3(256), 0, st, count, lp.n);
  const dim3 lgrid((unsigned)lp.nqb, (unsigned)(batch * kv_heads));
  hipLaunchKernelGGL(list_count_kernel, lgrid, dim3(kListBlock), 0, st, a, count, blkbase, lp.nqb);
  hipLaunchKernelGGL(list_scan_kernel, dim3(1), dim3(1024), 0, st, (const int32_t*)count, lp.n,
                     (int)lp.seg, start, ustart);
  a.start = start;
  a.ustart = ustart;
  hipLaunchKernelGGL(list_fill_kernel, lgrid, dim3(kListBlock), 0, st, a,
                     (const int32_t*)blkbase, lp.nqb, list);
  a.list = list;
  a.ds_rec = (uint16_t*)(ws + lp.records);
  a.sink = (uint16_t*)(ws + lp.sink);
  a.seg = (int)lp.seg;
  auto dkv = slope ? (token_keep ? routed_attn_dkv_kernel<true, true>
                                 : routed_attn_dkv_kernel<true, false>)
                   : (token_keep ? routed_attn_dkv_kernel<false, true>
                                 : routed_attn_dkv_kernel<false, false>);
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(dkv),
                          hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)kDkvLds) != hipSuccess)
    return MRSA_ERR_LAUNCH;
  hipLaunchKernelGGL(dkv, dim3((unsigned)lp.max_units), dim3(kDkvThreads), kDkvLds, st, a);
  const int s2 = mrsa_launch_status();
  if (s2 != MRSA_OK) return s2;
  // dQ: the forward's walk over each query tile's chunks, adding dS . K
  // into rows it owns (no atomics) from the records just written
  return mrsa::routed_dq_walk(kv_frags_bwd, a.ds_rec, indices, key_valid, batch, q_len, kv_len,
                              q_heads, kv_heads, topk, grad_q, stream);
}

}  // namespace

extern "C" int mrsa_selected_attention_bwd(
    const void* q, const void* grad_out, const void* kv_frags, const void* kv_frags_bwd,
    const void* weights, const int32_t* indices, const uint8_t* key_valid,
    const int8_t* token_keep, int64_t batch, int64_t q_len, int64_t kv_len, int64_t q_heads,
    int64_t kv_heads, int64_t head_dim, int64_t topk, int64_t chunk_size, int mask_last_token,
    float sm_scale, float* grad_q, float* grad_k, float* grad_v, void* grad_weights,
    void* workspace, int64_t workspace_bytes, void* stream) {
  return selected_backward(q, grad_out, kv_frags, kv_frags_bwd, weights, indices, key_valid,
                           token_keep, batch, q_len, kv_len, q_heads, kv_heads, head_dim, topk,
                           chunk_size, mask_last_token, sm_scale, grad_q, grad_k, grad_v,
                           grad_weights, workspace, workspace_bytes, stream, nullptr);
}

extern "C" int mrsa_selected_attention_alibi_bwd(
    const void* q, const void* grad_out, const void* kv_frags, const void* kv_frags_bwd,
    const void* weights, const int32_t* indices, const uint8_t* key_valid,
    const int8_t* token_keep, const float* slope, int64_t batch, int64_t q_len, int64_t kv_len,
    int64_t q_heads, int64_t kv_heads, int64_t head_dim, int64_t topk, int64_t chunk_size,
    int mask_last_token, float sm_scale, float* grad_q, float* grad_k, float* grad_v,
    void* grad_weights, void* workspace, int64_t workspace_bytes, void* stream) {
  if (batch > 0 && q_len > 0 && !slope) return MRSA_ERR_INVALID_ARGUMENT;
  return selected_backward(q, grad_out, kv_frags, kv_frags_bwd, weights, indices, key_valid,
                           token_keep, batch, q_len, kv_len, q_heads, kv_heads, head_dim, topk,
                           chunk_size, mask_last_token, sm_scale, grad_q, grad_k, grad_v,
                           grad_weights, workspace, workspace_bytes, stream, slope);
}

extern "C" int64_t mrsa_selected_attention_bwd_workspace_bytes(int64_t batch, int64_t q_len,
                                                               int64_t kv_len, int64_t q_heads,
                                                               int64_t kv_heads, int64_t topk) {
  if (batch < 0 || q_len < 0 || kv_len < 0 || q_heads <= 0 || kv_heads <= 0 || topk <= 0 ||
      kv_len % 64 || q_heads % kv_heads)
    return -1;
  return list_plan(batch, q_len, kv_heads, topk, kv_len / 64, q_heads).total;
}
