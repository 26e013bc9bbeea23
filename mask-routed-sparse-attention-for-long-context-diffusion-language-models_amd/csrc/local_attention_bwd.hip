// Backward of the bidirectional window attention (the gradient flash-attn's
// flash_attn_func gives dream_dllm_hils/local_attention.py:67-107; the
// forward is local_attention.hip).
//
// With k' = k m, v' = v m (m = 0 for inert keys: failed key_valid, landmark
// slots), s = q . k' * scale over the window |i - j| <= W, P = exp(s - lse)
// (lse saved by the forward) and D_i = sum_d dO_i O_i:
//   dV'_j = sum_i P_ij dO_i,  dP_ij = dO_i . v'_j,  dS_ij = P_ij (dP_ij - D_i),
//   dQ_i = scale sum_j dS_ij k'_j,  dK'_j = scale sum_i dS_ij q_i,
// and dk = dK' m, dv = dV' m.  The LSE output carries no gradient (flash-attn's
// autograd drops it).  Rounding points as flash-attn's: P and dS are rounded
// to bf16 as matrix operands, every sum is fp32.
//
// Both passes are one kernel template: 16 matrix columns per wave in
// registers, 64-row tiles of two tensors streamed through a 2-slot LDS ring by
// buffer->LDS DMA, one barrier per tile.  The rows come as they lie in the
// tensors, whole 256-byte rows, and serve twice: read along the row (rows x
// dims) and by gfx950's transposing LDS reads (dims x rows).
//   per tile:  S^T  = A . X1^T,  dP^T = B . X2^T            (32 products)
//              acc4 += A^T . dS^T  (and acc3 += B^T . P^T)  (16 or 32 products)
//  dQ pass   (columns: (query, head); rows: keys):
//     A = K, B = V, X1 = Q, X2 = dO  ->  acc4 = dQ / scale
//  dK/dV pass (columns: keys; rows: (query, head) pairs, row = query G + head):
//     A = Q, B = dO, X1 = K, X2 = V  ->  acc3 = dV, acc4 = dK / scale
// The dQ pass also writes each (query, head) row's lse (log2 units) and D in
// row order for the dK/dV pass.
//
// No unit is at its limit (dQ / dK/dV pass, 28 heads over 4, 5003 queries, window
// 1280): LDS is busy 67 / 47% of the cycles, 40 / 33% of that bank conflicts, the
// matrix cores work 40 / 31%, and the waves wait 34 / 35% of their time, at the
// tile's barrier and for its rows and operands.  Operands read 4 (dQ) or 8
// ahead by explicit order; the dQ pass fits 128 registers and 68 KB of LDS, so
// that two workgroups share a CU.  16384 queries, window 319: dQ 330-365 us,
// dK/dV 407-443; with pre-transposed images in HBM (four layout launches, 214
// us) and 64 KB slots, one workgroup per CU, 473 and 527.
#include "chunk_tile.h"
#include "mrsa_device.h"

#include <algorithm>

using namespace mrsa;

namespace {

constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int kRing = 2;
constexpr int kTileBytes = 16384;     // 64 rows x 256 bytes
constexpr int kSlotBytes = 2 * kTileBytes;
constexpr int kMaskTiles = 512;       // inert-key words of the dQ pass kept in LDS
constexpr int kMaxParts = 8;          // row parts of the dK/dV pass

// Buffer resource of `bytes` bytes at a wave-uniform address, in scalar registers.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_rsrc(const uint16_t* at, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)uniform_u64((uint64_t)at), (short)0,
                                           __builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

// Row r's 16-byte part u lies at unit u ^ swizzle(r): 16 rows' reads of one
// part, and a transposing read's 8 rows x 2 parts, meet 16 different units of
// the 64 banks.
__device__ __forceinline__ uint32_t swizzle(uint32_t r) {
  return 2u * (r & 7u) + ((r >> 3) & 1u);
}

struct BwdArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const uint16_t* out;
  const uint16_t* dout;
  const float* lse;           // [B, L, Hq] natural log
  const uint8_t* key_valid;
  int64_t B, L;
  int Hq, Hkv, G;
  int64_t W;
  int64_t inert_chunk;
  float scale, scale_log2;
  int64_t row_pitch;          // L G rounded up to 64
  float* lse_rows;            // [B, Hkv, row_pitch] log2 units (written by the dQ pass)
  float* d_rows;              // [B, Hkv, row_pitch]
  int parts;                  // row parts of the dK/dV pass
  float* partial;             // parts > 1: [parts, 2 (dk, dv), B, L, Hkv, 128] fp32
  float* dq;                  // [B, L, Hq, 128] fp32
  float* dk;                  // [B, L, Hkv, 128] fp32
  float* dv;
};

// Inert-key bits of key tile kt (bit s = key 64 kt + s): failed key_valid and
// the landmark slots ((j + 1) % inert_chunk == 0).
__device__ __forceinline__ uint64_t inert_bits(const BwdArgs& a, int64_t b, int64_t kt) {
  const int lane = threadIdx.x & 63;
  const int64_t j0 = kt * 64;
  const int64_t j = j0 + lane;
  const bool bad = j < a.L && a.key_valid && a.key_valid[b * a.L + j] == 0;
  uint64_t m = __builtin_amdgcn_ballot_w64(bad);
  if (a.inert_chunk > 0) {
    const int64_t r = (j0 + 1) % a.inert_chunk;
    for (int64_t s = r == 0 ? 0 : a.inert_chunk - r; s < 64 && j0 + s < a.L; s += a.inert_chunk)
      m |= 1ull << s;
  }
  return m;
}

__device__ __forceinline__ bool key_inert(const BwdArgs& a, int64_t b, int64_t j) {
  if (a.key_valid && a.key_valid[b * a.L + j] == 0) return true;
  return a.inert_chunk > 0 && (j + 1) % a.inert_chunk == 0;
}

template <bool DKV>
__global__ void __launch_bounds__(kThreads, DKV ? 2 : 4) local_bwd_kernel(BwdArgs a) {
  extern __shared__ __align__(256) unsigned char smem[];
  unsigned char* ring = smem;
  uint64_t* inert_tab = reinterpret_cast<uint64_t*>(smem + kRing * kSlotBytes);  // [kMaskTiles], dQ pass

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, grp = lane >> 4;
  // XCD-aware order (as the forward): XCD x takes a contiguous range.
  const int64_t nx = gridDim.x, nyz = (int64_t)gridDim.y * gridDim.z;
  const int64_t total = nx * nyz;
  int64_t lin = blockIdx.x + nx * (blockIdx.y + (int64_t)gridDim.y * blockIdx.z);
  {
    const int64_t x = lin % 8, q8 = total / 8, r8 = total % 8;
    lin = x * q8 + min(x, r8) + lin / 8;
  }
  const int parts = DKV ? a.parts : 1;
  const int part = (int)(lin % parts);
  const int64_t blk = lin % nx / parts;
  const int h = (int)((lin / nx) % gridDim.y);
  const int64_t b = lin / (nx * gridDim.y);
  const int G = a.G, Hq = a.Hq;
  const int64_t L = a.L, W = a.W;
  const int cw = 16 * wave + col;

  // ---- this lane's column: operands, per-column values, visible row range
  u32x4_t X1[4], X2[4];
  bool cok;
  int64_t rlo, rhi;           // visible rows [rlo, rhi] (tile-row units)
  float lse2_c = 0.f, d_c = 0.f;
  int64_t cq = 0, cj = 0;
  int cg = 0;
  if constexpr (!DKV) {
    const int QB = 128 / G;
    cq = blk * QB + cw / G;
    cg = cw % G;
    cok = cw < QB * G && cq < L;
    rlo = max(cq - W, (int64_t)0);
    rhi = min(cq + W, L - 1);
    const int64_t row = ((b * L + cq) * Hq + (int64_t)h * G + cg) * 128;
    float dsum = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const u32x4_t z = {0u, 0u, 0u, 0u};
      X1[j] = z;
      X2[j] = z;
      u32x4_t o = z;
      if (cok) {
        X1[j] = *reinterpret_cast<const u32x4_t*>(a.q + row + 32 * j + 8 * grp);
        X2[j] = *reinterpret_cast<const u32x4_t*>(a.dout + row + 32 * j + 8 * grp);
        o = *reinterpret_cast<const u32x4_t*>(a.out + row + 32 * j + 8 * grp);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
        dsum += bf16_lo(X2[j][e]) * bf16_lo(o[e]) + bf16_hi(X2[j][e]) * bf16_hi(o[e]);
    }
    d_c = across4_sum(dsum);
    const float lse = cok ? a.lse[(b * L + cq) * Hq + (int64_t)h * G + cg] : 0.f;
    lse2_c = lse * kLog2e;
    if (cok && grp == 0) {
      const int64_t ridx = (b * a.Hkv + h) * a.row_pitch + cq * G + cg;
      a.lse_rows[ridx] = lse2_c;
      a.d_rows[ridx] = d_c;
    }
  } else {
    cj = blk * 128 + cw;
    cok = cj < L;
    rlo = G * max(cj - W, (int64_t)0);
    rhi = G * min(cj + W, L - 1) + G - 1;
    const int64_t row = ((b * L + (cok ? cj : 0)) * a.Hkv + h) * 128;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const u32x4_t z = {0u, 0u, 0u, 0u};
      X1[j] = z;
      X2[j] = z;
      if (cok) {
        X1[j] = *reinterpret_cast<const u32x4_t*>(a.k + row + 32 * j + 8 * grp);
        X2[j] = *reinterpret_cast<const u32x4_t*>(a.v + row + 32 * j + 8 * grp);
      }
    }
  }
  if (!cok) {
    rlo = 1;  // nothing visible
    rhi = 0;
  }

  // ---- the workgroup's row tiles: the union of its columns' windows (of
  // which a part takes its share), and this wave's rows
  int64_t lo_all, hi_all;
  int64_t wlo = 0, whi = -1;   // rows some column of the wave sees
  int64_t flo = 0, fhi = -1;   // rows all of them see
  if constexpr (!DKV) {
    const int QB = 128 / G;
    const int64_t q0 = blk * QB, q1 = min(q0 + QB, L) - 1;
    lo_all = max(q0 - W, (int64_t)0);
    hi_all = min(q1 + W, L - 1);
    const int64_t a0 = q0 + 16 * wave / G, a1 = min(q0 + (16 * wave + 15) / G, q1);
    if (16 * wave < QB * G && a0 < L) {
      wlo = max(a0 - W, (int64_t)0);
      whi = min(a1 + W, L - 1);
      flo = max(a1 - W, (int64_t)0);
      fhi = min(a0 + W, L - 1);
    }
  } else {
    const int64_t j0 = blk * 128, j1 = min(j0 + 128, L) - 1;
    lo_all = G * max(j0 - W, (int64_t)0);
    hi_all = G * min(j1 + W, L - 1) + G - 1;
    const int64_t a0 = j0 + 16 * wave, a1 = min(a0 + 15, L - 1);
    if (a0 < L) {
      wlo = G * max(a0 - W, (int64_t)0);
      whi = G * min(a1 + W, L - 1) + G - 1;
      flo = G * max(a1 - W, (int64_t)0);
      fhi = G * min(a0 + W, L - 1) + G - 1;
    }
  }
  const int64_t tall = hi_all / 64 - lo_all / 64 + 1;
  const int64_t t0 = lo_all / 64 + tall * part / parts;
  const int ntiles = (int)(lo_all / 64 + tall * (part + 1) / parts - t0);
  const bool tab = !DKV && ntiles <= kMaskTiles;

  // ---- the stream: row s of (b, h) is row (s / RG) RH + h RG + s % RG of the
  // tensors.  Instruction n of a wave fills rows 8 wave + 4 n + (lane >> 4) of
  // the tile; rows past the last repeat it (nothing sees them).
  const int RG = DKV ? G : 1, RH = DKV ? Hq : a.Hkv;
  const uint16_t* const xa = (DKV ? a.q : a.k) + (b * L * RH + (int64_t)h * RG) * 128;
  const uint16_t* const xb = (DKV ? a.dout : a.v) + (b * L * RH + (int64_t)h * RG) * 128;
  int ri[2], rg[2];            // position and head of each instruction's first row
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const int s = __builtin_amdgcn_readfirstlane((int)(t0 * 64) + 8 * wave + 4 * n);
    ri[n] = s / RG;
    rg[n] = s % RG;
  }
  const int step_i = 64 / RG, step_g = 64 % RG;
  // The next tile into slot s.
  auto issue_tile = [&](int s) {
    unsigned char* dst = ring + s * kSlotBytes + 2048 * wave;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const int last = (int)L - 1;
      const int i0 = __builtin_amdgcn_readfirstlane(min(ri[n], last));
      const int v = rg[n] + grp;
      const int di = (v >= RG) + (v >= 2 * RG) + (v >= 3 * RG);
      const bool in = ri[n] + di <= last;
      const uint32_t row = in ? (uint32_t)di * (uint32_t)RH + (uint32_t)(v - di * RG)
                              : (uint32_t)(last - i0) * (uint32_t)RH + (uint32_t)(RG - 1);
      const uint32_t off = 256u * row + 16u * ((uint32_t)col ^ swizzle(8u * wave + 4u * n + grp));
      const int64_t left = ((int64_t)(last - i0) * RH + RG) * 256;
      const int bytes = left < 0xfffffff0ll ? (int)(uint32_t)left : -16;
      const __amdgpu_buffer_rsrc_t ra = row_rsrc(xa + (int64_t)i0 * RH * 128, bytes);
      const __amdgpu_buffer_rsrc_t rb = row_rsrc(xb + (int64_t)i0 * RH * 128, bytes);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void_t*)(dst + 1024 * n), 16, off, 0, 0,
                                               0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rb, (lds_void_t*)(dst + kTileBytes + 1024 * n), 16, off, 0, 0, 0);
      ri[n] += step_i;
      rg[n] += step_g;
      if (rg[n] >= RG) {
        rg[n] -= RG;
        ++ri[n];
      }
    }
  };
  if constexpr (!DKV) {
    if (tab)
      for (int t = wave; t < ntiles; t += kWaves) {
        const uint64_t bits = inert_bits(a, b, t0 + t);
        if (lane == 0) lds_write_u64(lds_addr(&inert_tab[t]), bits);
      }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    asm volatile("" : "+v"(X1[j]));
    asm volatile("" : "+v"(X2[j]));
  }
  if (ntiles > 0) issue_tile(0);

  f32x4_t acc3[8], acc4[8];
#pragma unroll
  for (int td = 0; td < 8; ++td) {
    acc3[td] = zero4();
    acc4[td] = zero4();
  }
  const float c = a.scale_log2;
  // This lane's operand rows (row col, part 4 kq + grp: kq flips bits 6, 7)
  // and transposed reads (row 4 grp + (col >> 2), dims 4 (col & 3) ..: the dim
  // tile flips bits 5..7), within a slot.
  const bool any = rhi >= rlo;
  const uint32_t span = (uint32_t)(rhi - rlo);
  const uint32_t arow = 256u * col + 16u * ((uint32_t)grp ^ swizzle(col));
  const uint32_t rt = 4u * grp + (col >> 2);
  const uint32_t trow = 256u * rt + 16u * (((col >> 1) & 1u) ^ swizzle(rt)) + 8u * (col & 1u);

  for (int t = 0; t < ntiles; ++t) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const int64_t r0 = (t0 + t) * 64;
    const bool seen = r0 + 63 >= wlo && r0 <= whi;  // wave-uniform
    // per-row values of the dK/dV pass, issued before the next tile's DMA so
    // that their wait does not wait for it
    f32x4_t lse2_r[4], d_r[4];
    if constexpr (DKV) {
      const int64_t rb = (b * a.Hkv + h) * a.row_pitch + r0 + 4 * grp;
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        lse2_r[mt] = *reinterpret_cast<const f32x4_t*>(a.lse_rows + rb + 16 * mt);
        d_r[mt] = *reinterpret_cast<const f32x4_t*>(a.d_rows + rb + 16 * mt);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (t + 1 < ntiles) issue_tile((t + 1) % kRing);
    asm volatile("" ::: "memory");
    const uint32_t sbase = lds_addr(ring + (t % kRing) * kSlotBytes);
    uint64_t inert = 0ull;
    if constexpr (!DKV) inert = uniform_u64(tab ? lds_read_u64(lds_addr(&inert_tab[t]))
                                                : inert_bits(a, b, t0 + t));
    if (!seen) continue;

    // P and dS of the visible rows: row r0 + 16 mt + 4 grp + r lies in
    // [rlo, rhi] (one unsigned compare; none where every column sees the whole
    // tile); the dQ pass drops inert key rows from dS (their k' = 0 adds
    // nothing).
    const int rel = (int)r0 + 4 * grp - (int)rlo;
    const bool plain = r0 >= flo && r0 + 63 <= fhi && inert == 0;  // wave-uniform
    const uint32_t at = sbase + arow, tt = sbase + trow;
    auto rows32 = [&](auto hc) {
      constexpr int hh = decltype(hc)::value;
      constexpr int kRead = DKV ? 8 : 4;
      f32x4_t S[2], dP[2];
      S[0] = S[1] = dP[0] = dP[1] = zero4();
      // product o: part kq = o >> 2, S (o & 2 == 0) or dP, rows 16 (o & 1) ..;
      // kRead operand reads in flight
      auto operand = [&](int o) {
        return lds_read16((at ^ (64u * (o >> 2))) + 4096u * (2 * hh + (o & 1)) +
                          ((o & 2) ? (uint32_t)kTileBytes : 0u));
      };
      u32x4_t x[16];
#pragma unroll
      for (int o = 0; o < kRead; ++o) x[o] = operand(o);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int o = 0; o < 16; ++o) {
        if (o & 2)
          dP[o & 1] = mfma_bf16_16x16x32(x[o], X2[o >> 2], dP[o & 1]);
        else
          S[o & 1] = mfma_bf16_16x16x32(x[o], X1[o >> 2], S[o & 1]);
        if (o + kRead < 16) x[o + kRead] = operand(o + kRead);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float l2 = DKV ? lse2_r[2 * hh + m][r] : lse2_c;
          const float dd = DKV ? d_r[2 * hh + m][r] : d_c;
          const float p = exp2_hw(__builtin_fmaf(S[m][r], c, -l2));
          S[m][r] = p;
          dP[m][r] = p * (dP[m][r] - dd);
        }
      const uint32_t dead = (uint32_t)(inert >> (32 * hh)) >> (4 * grp);
      if (!plain) {
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const bool vis = any & ((uint32_t)(rel + 32 * hh + 16 * m + r) <= span);
            if constexpr (DKV) S[m][r] = vis ? S[m][r] : 0.f;
            const bool live = DKV ? vis : vis & (((dead >> (16 * m + r)) & 1u) == 0u);
            dP[m][r] = live ? dP[m][r] : 0.f;
          }
      }
      u32x4_t Pb, Sb;  // the B operands: element 4 m + r is row 32 hh + 16 m + 4 grp + r
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        Sb[2 * m] = pack_bf16x2(dP[m][0], dP[m][1]);
        Sb[2 * m + 1] = pack_bf16x2(dP[m][2], dP[m][3]);
        if constexpr (DKV) {
          Pb[2 * m] = pack_bf16x2(S[m][0], S[m][1]);
          Pb[2 * m + 1] = pack_bf16x2(S[m][2], S[m][3]);
        }
      }
      // product o: dims 16 (o >> DKV) .., of A^T . dS^T or (o & 1) B^T . P^T;
      // kRead / 2 operands (two reads each) in flight
      constexpr int N = DKV ? 16 : 8, kT = kRead / 2;
      auto transposed = [&](int o) {
        const uint32_t ad = (tt ^ (32u * (DKV ? o >> 1 : o))) + 8192u * hh +
                            (DKV && (o & 1) ? (uint32_t)kTileBytes : 0u);
        const u32x2_t y0 = read_transposed(ad), y1 = read_transposed(ad + 4096u);
        return u32x4_t{y0[0], y0[1], y1[0], y1[1]};
      };
      u32x4_t y[N];
#pragma unroll
      for (int o = 0; o < kT; ++o) y[o] = transposed(o);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int o = 0; o < N; ++o) {
        if (DKV && (o & 1))
          acc3[o >> 1] = mfma_bf16_16x16x32(y[o], Pb, acc3[o >> 1]);
        else
          acc4[DKV ? o >> 1 : o] = mfma_bf16_16x16x32(y[o], Sb, acc4[DKV ? o >> 1 : o]);
        if (o + kT < N) y[o + kT] = transposed(o + kT);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    rows32(std::integral_constant<int, 0>{});
    rows32(std::integral_constant<int, 1>{});
  }

  // ---- outputs (fp32): the lane holds dims 16 td + 4 grp .. + 3 of its column
  if (!cok) return;
  if constexpr (!DKV) {
    float* dst = a.dq + ((b * L + cq) * Hq + (int64_t)h * G + cg) * 128;
#pragma unroll
    for (int td = 0; td < 8; ++td) {
      f32x4_t o = acc4[td];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] *= a.scale;
      *reinterpret_cast<f32x4_t*>(dst + 16 * td + 4 * grp) = o;
    }
  } else {
    const bool dead = key_inert(a, b, cj);  // dk = dK' m, dv = dV' m
    const int64_t n = a.B * L * a.Hkv * 128;
    const int64_t at = ((b * L + cj) * a.Hkv + h) * 128;
    float* dk = (parts > 1 ? a.partial + (int64_t)part * 2 * n : a.dk) + at;
    float* dv = (parts > 1 ? a.partial + ((int64_t)part * 2 + 1) * n : a.dv) + at;
#pragma unroll
    for (int td = 0; td < 8; ++td) {
      f32x4_t ok = acc4[td], ov = acc3[td];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        ok[e] = dead ? 0.f : ok[e] * a.scale;
        ov[e] = dead ? 0.f : ov[e];
      }
      *reinterpret_cast<f32x4_t*>(dk + 16 * td + 4 * grp) = ok;
      *reinterpret_cast<f32x4_t*>(dv + 16 * td + 4 * grp) = ov;
    }
  }
}

// dk and dv of a dK/dV pass in parts: n4 vectors of each, added in order.
__global__ void __launch_bounds__(256)
    local_bwd_sum_kernel(const float* __restrict__ partial, int parts, int64_t n4,
                         float* __restrict__ dk, float* __restrict__ dv) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= 2 * n4) return;
  const f32x4_t* src = reinterpret_cast<const f32x4_t*>(partial) + e;
  f32x4_t s = src[0];
  for (int p = 1; p < parts; ++p) {
    const f32x4_t x = src[(int64_t)p * 2 * n4];
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] += x[i];
  }
  reinterpret_cast<f32x4_t*>(e < n4 ? dk : dv)[e < n4 ? e : e - n4] = s;
}

struct BwdPlan {
  int64_t row_pitch;        // L G rounded up to 64
  int max_parts;
  size_t lse, d, partial;   // workspace offsets
  size_t total;
};

int64_t key_blocks(int64_t B, int64_t L, int64_t Hkv) { return B * Hkv * ((L + 127) / 128); }

BwdPlan bwd_plan(int64_t B, int64_t L, int64_t Hkv, int64_t G) {
  BwdPlan p;
  p.row_pitch = (L * G + 63) / 64 * 64;
  const int64_t units = std::max<int64_t>(key_blocks(B, L, Hkv), 1);
  p.max_parts = (int)std::clamp<int64_t>(1024 / units, 1, kMaxParts);
  size_t o = 0;
  auto take = [&](size_t n) {
    const size_t at = o;
    o += (n + 255) & ~(size_t)255;
    return at;
  };
  p.lse = take((size_t)(B * Hkv * p.row_pitch) * 4);
  p.d = take((size_t)(B * Hkv * p.row_pitch) * 4);
  p.partial = take(p.max_parts > 1 ? (size_t)(p.max_parts * B * L * Hkv) * 1024 : 0);
  p.total = o;
  return p;
}

// Row parts of the dK/dV pass.  A workgroup (128 keys) has a CU to itself, so
// the launch takes ceil(units parts / 256) rounds of its tiles / parts, each
// with about 6 tiles' time around the loop; a part writes and reads back 2 KB
// per key row, a tile's time (2.3 us) for 10 MB.
// 5003 keys, window 1280 (160 workgroups of 295 tiles): 470 us in 3 parts and 14
// for their sum, 664 whole; 2 x 1984 keys, window 319: 103 + 8 us, 184 whole.
int pick_parts(const BwdPlan& p, int64_t B, int64_t L, int64_t Hkv, int64_t G, int64_t W) {
  const int64_t units = key_blocks(B, L, Hkv);
  const int64_t tiles = (G * std::min(L, 128 + 2 * std::min(W, L)) + 63) / 64;
  int best = 1;
  double least = 0.;
  for (int n = 1; n <= p.max_parts && (n == 1 || tiles / n >= 4); ++n) {
    const double rounds = (double)((units * n + 255) / 256);
    const double cost = rounds * ((double)((tiles + n - 1) / n) + 6.) +
                        (n > 1 ? 2. + n * (double)(B * L * Hkv) * 2048. / 1e7 : 0.);
    if (n == 1 || cost < least) {
      least = cost;
      best = n;
    }
  }
  return best;
}

}  // namespace

extern "C" int64_t mrsa_local_attention_bwd_workspace_bytes(int64_t batch, int64_t seq_len,
                                                            int64_t q_heads, int64_t kv_heads) {
  if (batch < 0 || seq_len < 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0)
    return -1;
  return (int64_t)bwd_plan(batch, seq_len, kv_heads, q_heads / kv_heads).total;
}

extern "C" int mrsa_local_attention_bwd(const void* q, const void* k, const void* v,
                                        const uint8_t* key_valid, const void* out,
                                        const float* lse, const void* grad_out, int64_t batch,
                                        int64_t seq_len, int64_t q_heads, int64_t kv_heads,
                                        int64_t head_dim, int64_t window, int64_t inert_chunk,
                                        float sm_scale, float* grad_q, float* grad_k,
                                        float* grad_v, void* workspace, int64_t workspace_bytes,
                                        void* stream) {
  if (batch < 0 || seq_len < 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0 ||
      head_dim <= 0 || window < 0 || inert_chunk < 0 || !(sm_scale > 0.f) ||
      sm_scale == __builtin_inff())
    return MRSA_ERR_INVALID_ARGUMENT;
  if (batch == 0 || seq_len == 0) return MRSA_OK;
  if (head_dim != 128) return MRSA_ERR_UNSUPPORTED;
  const int64_t G = q_heads / kv_heads;
  if (G > 128 || kv_heads > 65535 || batch > 65535) return MRSA_ERR_UNSUPPORTED;
  // rows and tiles are counted in 32 bits
  if ((seq_len * G + 63) / 64 >= 131072) return MRSA_ERR_UNSUPPORTED;
  if (!q || !k || !v || !out || !lse || !grad_out || !grad_q || !grad_k || !grad_v || !workspace)
    return MRSA_ERR_INVALID_ARGUMENT;
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out | (uintptr_t)grad_out |
       (uintptr_t)grad_q | (uintptr_t)grad_k | (uintptr_t)grad_v) % 16 != 0)
    return MRSA_ERR_INVALID_ARGUMENT;
  const BwdPlan p = bwd_plan(batch, seq_len, kv_heads, G);
  if (workspace_bytes < (int64_t)p.total || (uintptr_t)workspace % 256 != 0)
    return MRSA_ERR_INVALID_ARGUMENT;
  char* ws = (char*)workspace;
  hipStream_t s = (hipStream_t)stream;
  BwdArgs a;
  a.q = (const uint16_t*)q;
  a.k = (const uint16_t*)k;
  a.v = (const uint16_t*)v;
  a.out = (const uint16_t*)out;
  a.dout = (const uint16_t*)grad_out;
  a.lse = lse;
  a.key_valid = key_valid;
  a.B = batch;
  a.L = seq_len;
  a.Hq = (int)q_heads;
  a.Hkv = (int)kv_heads;
  a.G = (int)G;
  a.W = window;
  a.inert_chunk = inert_chunk;
  a.scale = sm_scale;
  a.scale_log2 = sm_scale * kLog2e;
  a.row_pitch = p.row_pitch;
  a.parts = pick_parts(p, batch, seq_len, kv_heads, G, window);
  a.partial = (float*)(ws + p.partial);
  a.lse_rows = (float*)(ws + p.lse);
  a.d_rows = (float*)(ws + p.d);
  a.dq = grad_q;
  a.dk = grad_k;
  a.dv = grad_v;
  const size_t ring = (size_t)kRing * kSlotBytes, smem = ring + kMaskTiles * 8;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(local_bwd_kernel<false>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
    return MRSA_ERR_LAUNCH;
  const int64_t QB = 128 / G;
  hipLaunchKernelGGL(local_bwd_kernel<false>,
                     dim3((unsigned)((seq_len + QB - 1) / QB), (unsigned)kv_heads, (unsigned)batch),
                     dim3(kThreads), smem, s, a);
  int st = mrsa_launch_status();
  if (st != MRSA_OK) return st;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(local_bwd_kernel<true>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)ring) != hipSuccess)
    return MRSA_ERR_LAUNCH;
  hipLaunchKernelGGL(local_bwd_kernel<true>,
                     dim3((unsigned)((seq_len + 127) / 128 * a.parts), (unsigned)kv_heads,
                          (unsigned)batch),
                     dim3(kThreads), ring, s, a);
  st = mrsa_launch_status();
  if (st != MRSA_OK || a.parts == 1) return st;
  const int64_t n4 = batch * seq_len * kv_heads * 32;
  hipLaunchKernelGGL(local_bwd_sum_kernel, dim3((unsigned)((2 * n4 + 255) / 256)), dim3(256), 0, s,
                     a.partial, a.parts, n4, grad_k, grad_v);
  return mrsa_launch_status();
}
