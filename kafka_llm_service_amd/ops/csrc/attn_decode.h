// Paged decode attention, one piece of one row's keys per workgroup (page layouts and the wave's step: attention.hip).
#pragma once
#include "common.h"

#include <type_traits>

namespace kafka {

constexpr int PAGE = 16;

struct AttnWorkItem {
  int q_start;  // first query token (row of q / out)
  int q_count;  // tokens in this tile
  int bt_row;   // block-table row used for the keys
  int kv_lo;    // first key position (inclusive)
  int kv_hi;    // last key position (exclusive)
  int split;    // -1: write normalized bf16 to out; >= 0: write partial #split
  int pad0, pad1;
};

// Reductions with the partner lane l ^ 32 on gfx950's v_permlane32_swap (one VALU op, no LDS crossbar round trip
// through ds_bpermute — which also queued behind the K/V fragment reads): swapping a register with itself leaves
// x[l] in one result and x[l ^ 32] in the other, so a symmetric op of the two is the xor-32 reduction on every lane.
// max as llvm.maximum (gfx950 v_maximum3_f32, 3 inputs, no NaN-quieting v_max x, x of each MFMA result that fmaxf
// costs in IEEE mode; attn_tile.hip t3_max)
__device__ __forceinline__ float vmax(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float xor32_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return vmax(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xor32_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int KPAGE8 = PAGE * 128 + 32;  // fp8 K page bytes per (block, kv head): data + K/V exponents
constexpr int VPAGE8 = PAGE * 128;
constexpr int KEXP8 = PAGE * 128, VEXP8 = PAGE * 128 + 16;

__device__ __forceinline__ float exp2i(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }

// 8 e4m3 bytes (two dwords) -> bf16x8 times `sc` (a power of two)
__device__ __forceinline__ bf16x8 dq8(uint32_t lo, uint32_t hi, float sc) {
  const bf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, sc, false);
  const bf16x2 b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, sc, true);
  const bf16x2 c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, sc, false);
  const bf16x2 d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, sc, true);
  return bf16x8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

template <int D>
struct WaveAcc {
  f32x16 o[D / 32];
  float m;
  float l;
};

// K/V fragments of one 32-key block for one wave (register-staged; the next block is prefetched while the
// current one is computed: loads for block i+1 are issued before the MFMAs of block i, so HBM/L2 latency hides
// under the QK^T / softmax / PV work instead of stalling every 32-key step).
template <int D>
struct KVFrag {
  bf16x8 k[D / 16];
  bf16x8 v[2][D / 32];
};

// fp8: 16-B unit j of the lane's key = A-fragments of k-steps 2j, 2j + 1; V^T rows as 8-B loads; the lane's key
// exponent (K) and its 8 keys' exponents per page (V)
template <int D>
struct KVFrag8 {
  u32x4 k[D / 32];
  u32x2 v[2][D / 32];
  int kexp;
  u32x2 vexp[2];
};

template <int D>
__device__ __forceinline__ void load_kv8(KVFrag8<D>& f, const uint8_t* __restrict__ k_cache,
                                         const uint8_t* __restrict__ v_cache, int Hkv, int kvh, int page0,
                                         int page1, int lane) {
  const int r = lane & 31, h = lane >> 5;
  const int kp = (r >> 4) ? page1 : page0;
  const uint8_t* kb = k_cache + ((int64_t)kp * Hkv + kvh) * KPAGE8;
#pragma unroll
  for (int j = 0; j < D / 32; ++j)
    f.k[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(kb + ((2 * j + h) * PAGE + (r & 15)) * 16));
  f.kexp = (int)*reinterpret_cast<const int8_t*>(kb + KEXP8 + (r & 15));
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2) {
    const int vp = s2 ? page1 : page0;
    const uint8_t* vb = v_cache + ((int64_t)vp * Hkv + kvh) * VPAGE8 + r * PAGE + 8 * h;
#pragma unroll
    for (int t = 0; t < D / 32; ++t) f.v[s2][t] = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(vb + 32 * t * PAGE));
    f.vexp[s2] = *reinterpret_cast<const u32x2*>(k_cache + ((int64_t)vp * Hkv + kvh) * KPAGE8 + VEXP8 + 8 * h);
  }
}

template <int D>
__device__ __forceinline__ void load_kv(KVFrag<D>& f, const bf16* __restrict__ k_cache,
                                        const bf16* __restrict__ v_cache, int Hkv, int kvh, int page0, int page1,
                                        int lane) {
  const int r = lane & 31, h = lane >> 5;
  const int kp = (r >> 4) ? page1 : page0;
  // chunk plane 2kk + h, key r & 15
  const bf16* kptr = k_cache + ((int64_t)kp * Hkv + kvh) * (PAGE * D) + (r & 15) * 8 + h * (PAGE * 8);
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) f.k[kk] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(kptr + kk * (2 * PAGE * 8)));
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2) {
    const int vp = s2 ? page1 : page0;
    const bf16* vptr = v_cache + ((int64_t)vp * Hkv + kvh) * (D * PAGE) + r * PAGE + 8 * h;
#pragma unroll
    for (int t = 0; t < D / 32; ++t) f.v[s2][t] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(vptr + 32 * t * PAGE));
  }
}

// Page ids of a decode piece staged in LDS: page i of the row at pages[i - pg0] (one ds_read instead of an L2 round
// trip in front of every K/V block load — the decode loop is bound by that dependent chain per wave, not by HBM)
struct LdsPages {
  const int* p;
  int pg0;
  __device__ __forceinline__ int operator[](int i) const { return p[i - pg0]; }
};

// Pages holding keys [key0, key0 + 32) (key0 32-aligned); the second page is only dereferenced below `end`.
template <typename BT>
__device__ __forceinline__ void block_pages(const BT& bt, int key0, int end, int& p0, int& p1) {
  p0 = bt[key0 >> 4];
  p1 = (key0 + 16 < end) ? bt[(key0 >> 4) + 1] : p0;
}

// Online softmax of one 32-key S^T tile (raw scores, lane = query column) + the P.V MFMAs.
//   * `masked` (wave-uniform) is false for interior blocks: no per-element range / causal test at all;
//   * the O / l rescale runs only when some row's running max moved (wave vote) — exact, and after the first few
//     blocks of a row it almost never fires;
//   * the softmax scale is folded into one FMA in front of exp2.
// acc.m is kept in the scaled log2 domain.
// VS (fp8 cache): P column scaled by the per-key V exponents vexp (lane half h: keys of page s2 in register order)
template <int D, bool VS = false>
__device__ __forceinline__ void softmax_pv(f32x16& s, bool masked, int key0, int lo, int hi, int limit,
                                           float scale_log2, const bf16x8 (&vf)[2][D / 32], WaveAcc<D>& acc,
                                           int lane, u32x2 ve0 = {0u, 0u}, u32x2 ve1 = {0u, 0u}) {
  const int h = lane >> 5;
  if (masked) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = key0 + (i & 3) + 8 * (i >> 2) + 4 * h;
      if (!((key >= lo) & (key < hi) & (key <= limit))) s[i] = -INFINITY;
    }
  }
  float ma = vmax(s[0], s[1]), mb = vmax(s[2], s[3]);
#pragma unroll
  for (int i = 4; i < 16; i += 4) {
    ma = vmax(vmax(ma, s[i]), s[i + 1]);
    mb = vmax(vmax(mb, s[i + 2]), s[i + 3]);
  }
  const float mx = xor32_max(vmax(ma, mb));
  const float m_new = vmax(acc.m, mx * scale_log2);
  const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
  if (!__all(m_new == acc.m)) {
    const float alpha = exp2f(acc.m - m_use);
    acc.l *= alpha;
#pragma unroll
    for (int t = 0; t < D / 32; ++t) acc.o[t] *= alpha;
  }
  acc.m = m_new;
  float psum = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float p = fast_exp2(fmaf(s[i], scale_log2, -m_use));
    s[i] = p;
    psum += p;
  }
  psum = xor32_sum(psum);
  acc.l += psum;
  if constexpr (VS) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t w0 = j < 4 ? ve0[0] : ve0[1], w1 = j < 4 ? ve1[0] : ve1[1];
      s[j] = ldexpf(s[j], __builtin_amdgcn_sbfe(w0, 8 * (j & 3), 8));
      s[8 + j] = ldexpf(s[8 + j], __builtin_amdgcn_sbfe(w1, 8 * (j & 3), 8));
    }
  }
  bf16x8 pf[2];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    pf[0][j] = (bf16)s[j];
    pf[1][j] = (bf16)s[8 + j];
  }
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
    for (int t = 0; t < D / 32; ++t) acc.o[t] = mfma32(vf[s2][t], pf[s2], acc.o[t]);
}

// One 32-key step for one wave on already-loaded fragments.
template <int D>
__device__ __forceinline__ void attn_compute(const KVFrag<D>& f, int key0, int lo, int hi, int limit,
                                             const bf16x8 (&qf)[D / 16], float scale_log2, WaveAcc<D>& acc,
                                             int lane, bool masked = true) {
  f32x16 s = {};
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) s = mfma32(f.k[kk], qf[kk], s);
  softmax_pv<D>(s, masked, key0, lo, hi, limit, scale_log2, f.v, acc, lane);
}

template <int D>
__device__ __forceinline__ void attn_compute8(const KVFrag8<D>& f, int key0, int lo, int hi, int limit,
                                              const bf16x8 (&qf)[D / 16], float scale_log2, WaveAcc<D>& acc,
                                              int lane, bool masked) {
  const float ks = exp2i(f.kexp);
  f32x16 s = {};
#pragma unroll
  for (int j = 0; j < D / 32; ++j) {
    s = mfma32(dq8(f.k[j][0], f.k[j][1], ks), qf[2 * j], s);
    s = mfma32(dq8(f.k[j][2], f.k[j][3], ks), qf[2 * j + 1], s);
  }
  bf16x8 vf[2][D / 32];
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
    for (int t = 0; t < D / 32; ++t) vf[s2][t] = dq8(f.v[s2][t][0], f.v[s2][t][1], 1.f);
  softmax_pv<D, true>(s, masked, key0, lo, hi, limit, scale_log2, vf, acc, lane, f.vexp[0], f.vexp[1]);
}

// Key blocks first, first+stride, ... < nblk (block b covers keys [base + 32 b, base + 32 b + 32)), software
// pipelined one block deep. The prefetch of the block after the last one is clamped to the last block (pad, don't
// branch: no divergent load, no extra waitcnt).
template <int D, bool FP8, typename BT = const int*>
__device__ __forceinline__ void attn_blocks(const void* __restrict__ k_cache, const void* __restrict__ v_cache,
                                            int Hkv, int kvh, const BT bt, int base, int first,
                                            int nblk, int stride, int end, int lo, int hi, int limit,
                                            const bf16x8 (&qf)[D / 16], float scale_log2, WaveAcc<D>& acc,
                                            int lane) {
  if (first >= nblk) return;
  using Frag = std::conditional_t<FP8, KVFrag8<D>, KVFrag<D>>;
  auto load = [&](Frag& f, int p0, int p1) {
    if constexpr (FP8)
      load_kv8<D>(f, static_cast<const uint8_t*>(k_cache), static_cast<const uint8_t*>(v_cache), Hkv, kvh, p0, p1,
                  lane);
    else
      load_kv<D>(f, static_cast<const bf16*>(k_cache), static_cast<const bf16*>(v_cache), Hkv, kvh, p0, p1, lane);
  };
  auto compute = [&](const Frag& f, int b) {
    const int key0 = base + 32 * b;
    const bool masked = (key0 < lo) | (key0 + 32 > hi) | (key0 + 31 > limit);
    if constexpr (FP8)
      attn_compute8<D>(f, key0, lo, hi, limit, qf, scale_log2, acc, lane, masked);
    else
      attn_compute<D>(f, key0, lo, hi, limit, qf, scale_log2, acc, lane, masked);
  };
  int p0, p1;
  Frag cur;
  block_pages(bt, base + 32 * first, end, p0, p1);
  load(cur, p0, p1);
  // (fp8: keeping two blocks in flight measured slower — 55.6 vs 52.0 us on the attn_bench decode case)
  for (int b = first; b < nblk; b += stride) {
    const int nb = (b + stride < nblk) ? b + stride : b;
    Frag nxt;
    block_pages(bt, base + 32 * nb, end, p0, p1);
    load(nxt, p0, p1);
    compute(cur, b);
    cur = nxt;
  }
}

template <int D>
__device__ __forceinline__ void load_q_frags(bf16x8 (&qf)[D / 16], const bf16* qrow, bool valid, int h) {
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) {
    if (valid) {
      qf[kk] = load_bf16x8(qrow + 16 * kk + 8 * h);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) qf[kk][j] = (bf16)0.f;
    }
  }
}

template <int D>
__device__ __forceinline__ void init_acc(WaveAcc<D>& acc) {
#pragma unroll
  for (int t = 0; t < D / 32; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc.o[t][i] = 0.f;
  acc.m = -INFINITY;
  acc.l = 0.f;
}

// ------------------------------------------------------------------------------------------------------------------
// Decode: grid (work items, Hkv), 256 threads. Requires G <= 8.
// A work item is one decode row's key range [lo, hi) — the whole per-thread suffix, or one of `nsplit` pieces of a
// long one (the host sizes pieces so every workgroup streams about the same bytes: one 3k-token history no longer
// holds the whole launch while the short ones have finished). Row b's partials live at slots [0, npre) (cascade
// prefix partials written by the tile kernel, for the row's prefix group) and npre + split (this piece).
struct DecodeItem {
  int b, lo, hi, split, nsplit, npre, pad0, pad1;
};

// LDS of one decode piece (4 waves' partial results + the fused merge's per-split weights)
constexpr int DEC_MAXPG = 2048;  // page ids of one decode piece staged in LDS (longer pieces read the table)
template <int D>
struct DecodeSmem {
  int pages[DEC_MAXPG];
  bf16 qs[8][D];  // bf16: the unit's G <= 8 query heads (B operand rows), read per block instead of held in VGPRs
  float sO[4][8][D];
  float sM[4][8];
  float sL[4][8];
  float sW[8][65];
  float sWt[8];
  int s_last;
  bf16 so[8][D];  // OST: the final bf16 rows, stored from here as 16-B sc1 stores
};

// the workgroup's G final rows from sm.so to out (every thread of the workgroup calls it)
template <int D>
__device__ __forceinline__ void store_rows_sc1(DecodeSmem<D>& sm, bf16* __restrict__ out, int64_t out_stride, int b,
                                               int kvh, int G) {
  __syncthreads();
  const int t = threadIdx.x;
  if (t < G * (D / 8)) {
    const int g = t / (D / 8), c = (t % (D / 8)) * 8;
    store16_slab(reinterpret_cast<float*>(out + (int64_t)b * out_stride + (int64_t)(kvh * G + g) * D + c),
                 *reinterpret_cast<const f32x4*>(&sm.so[g][c]));
  }
}

// The keys [lo, hi) of row b, kv head kvh: the four waves' sums, maxima and accumulators are in sm when it returns. Every thread of
// the workgroup calls it with the same arguments (it synchronises the workgroup).
template <int D, bool FP8>
__device__ __forceinline__ void decode_stream(DecodeSmem<D>& sm, const bf16* __restrict__ q, int64_t q_stride,
                                              const void* __restrict__ k_cache, const void* __restrict__ v_cache,
                                              int Hkv, int G, const int* __restrict__ block_tables, int bt_stride,
                                              int b, int kvh, int lo, int hi, float scale_log2) {
  constexpr bool OCC3 = !FP8;  // bf16: three workgroups per CU, Q in LDS, one K/V block per wave in flight
  auto& sO = sm.sO;
  auto& sM = sm.sM;
  auto& sL = sm.sL;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int r = lane & 31, h = lane >> 5;
  const int a0 = lo & ~31;
  const int nb = hi > lo ? (hi - a0 + 31) >> 5 : 0;
  const int* bt = block_tables + (int64_t)b * bt_stride;

  // the piece's page ids -> LDS (pages covering [a0, hi))
  const int pg0 = a0 >> 4;
  const int npg = nb > 0 ? ((hi - 1) >> 4) - pg0 + 1 : 0;
  const bool lds_pt = npg <= DEC_MAXPG;
  if (lds_pt)
    for (int i = threadIdx.x; i < npg; i += 256) sm.pages[i] = bt[pg0 + i];
  if constexpr (OCC3) {
    for (int i = threadIdx.x; i < G * (D / 8); i += 256) {
      const int g = i / (D / 8), c = i % (D / 8);
      *reinterpret_cast<bf16x8*>(&sm.qs[g][8 * c]) = load_bf16x8(q + (int64_t)b * q_stride + (int64_t)(kvh * G + g) * D + 8 * c);
    }
  }
  __syncthreads();
  WaveAcc<D> acc;
  init_acc<D>(acc);
  if constexpr (OCC3) {
    // Three waves per SIMD (VGPR budget 168): no Q fragments and no second K/V block in registers — each wave
    // has its one block in flight at a time, and 12 waves per CU (3 workgroups) keep the memory system fed;
    // more resident workgroups also cover each other's piece start / end.
    if (w < nb && !FP8) {
      const bool qrow = r < G;
      for (int bk = w; bk < nb; bk += 4) {
        const int key0 = a0 + 32 * bk;
        int p0, p1;
        if (lds_pt)
          block_pages(LdsPages{sm.pages, pg0}, key0, hi, p0, p1);
        else
          block_pages(bt, key0, hi, p0, p1);
        KVFrag<D> f;
        load_kv<D>(f, static_cast<const bf16*>(k_cache), static_cast<const bf16*>(v_cache), Hkv, kvh, p0, p1, lane);
        f32x16 sacc = {};
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) {
          bf16x8 qv = *reinterpret_cast<const bf16x8*>(&sm.qs[qrow ? r : 0][16 * kk + 8 * h]);
          if (!qrow) qv = bf16x8{};
          sacc = mfma32(f.k[kk], qv, sacc);
        }
        const bool masked = (key0 < lo) | (key0 + 32 > hi);
        softmax_pv<D>(sacc, masked, key0, lo, hi, 0x7fffffff, scale_log2, f.v, acc, lane);
      }
    }
  } else if (w < nb) {
    bf16x8 qf[D / 16];
    load_q_frags<D>(qf, q + (int64_t)b * q_stride + (int64_t)(kvh * G + r) * D, r < G, h);
    if (lds_pt)
      attn_blocks<D, FP8>(k_cache, v_cache, Hkv, kvh, LdsPages{sm.pages, pg0}, a0, w, nb, 4, hi, lo, hi, 0x7fffffff,
                          qf, scale_log2, acc, lane);
    else
      attn_blocks<D, FP8>(k_cache, v_cache, Hkv, kvh, bt, a0, w, nb, 4, hi, lo, hi, 0x7fffffff, qf, scale_log2, acc,
                          lane);
  }
  // cross-wave combine
  if (r < G) {
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const int d = 32 * t + 8 * i4 + 4 * h;
        f32x4 v = {acc.o[t][4 * i4 + 0], acc.o[t][4 * i4 + 1], acc.o[t][4 * i4 + 2], acc.o[t][4 * i4 + 3]};
        *reinterpret_cast<f32x4*>(&sO[w][r][d]) = v;
      }
    if (h == 0) {
      sM[w][r] = acc.m;
      sL[w][r] = acc.l;
    }
  }
  __syncthreads();
}

// the piece's partial row to slot ``slot``: 16-B write-through (sc1, agent-coherent) stores (4-B ones cost several times more per byte)
template <int D>
__device__ __forceinline__ void store_piece_sc1(DecodeSmem<D>& sm, int b, int kvh, int G, int Hq, int slot, int S_total,
                                                float* __restrict__ out_part, float* __restrict__ lse_part) {
  auto& sO = sm.sO;
  auto& sM = sm.sM;
  auto& sL = sm.sL;
  for (int idx4 = threadIdx.x; idx4 < G * D / 4; idx4 += 256) {
    const int g = idx4 / (D / 4), d0 = (idx4 % (D / 4)) * 4;
    float M = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) M = fmaxf(M, sM[i][g]);
    float L = 0.f;
    f32x4 O4 = {0.f, 0.f, 0.f, 0.f};
    if (M != -INFINITY) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float f = exp2f(sM[i][g] - M);
        L += f * sL[i][g];
#pragma unroll
        for (int j = 0; j < 4; ++j) O4[j] += f * sO[i][g][d0 + j];
      }
    }
    const int64_t pidx = ((int64_t)b * Hq + kvh * G + g) * S_total + slot;
    const float inv = L > 0.f ? 1.f / L : 0.f, lv = L > 0.f ? M + log2f(L) : -INFINITY;
    f32x4 ov4;
#pragma unroll
    for (int j = 0; j < 4; ++j) ov4[j] = L > 0.f ? O4[j] * inv : 0.f;
    store16_slab(out_part + pidx * D + d0, ov4);
    if (d0 == 0) __hip_atomic_store(lse_part + pidx, lv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// One decode piece: keys [lo, hi) of row b, kv head kvh, piece `split` of S, partial slots from split_offset. Every
// thread of the workgroup calls it with the same arguments (it synchronises the workgroup); returns when the
// piece's partial or final rows are written.
// OST: the final bf16 rows leave through LDS as 16-B sc1 stores (one instruction per 16 B of a row instead of one
// 8-B plain store per thread: the lines leave this XCD's L2, so the launch ends with no dirty output lines to write
// back; the o GEMM reads them on every XCD). Needs 16-B aligned rows (host-checked).
template <int D, bool FP8, bool OST = false>
__device__ __forceinline__ void decode_piece(DecodeSmem<D>& sm, const bf16* __restrict__ q, int64_t q_stride,
                                             const void* __restrict__ k_cache, const void* __restrict__ v_cache,
                                             int Hkv, int G, const int* __restrict__ block_tables, int bt_stride,
                                             int b, int kvh, int lo, int hi, int split, int S, int split_offset,
                                             float* __restrict__ out_part, float* __restrict__ lse_part, int S_total,
                                             float scale_log2, bf16* __restrict__ out, int64_t out_stride,
                                             int* __restrict__ tickets, const bf16* __restrict__ pre_bf16) {
  constexpr int MG = 32;       // prefix partials per load round trip of the fused merge
  auto& sO = sm.sO;
  auto& sM = sm.sM;
  auto& sL = sm.sL;
  auto& sW = sm.sW;
  auto& sWt = sm.sWt;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int Hq = Hkv * G;
  decode_stream<D, FP8>(sm, q, q_stride, k_cache, v_cache, Hkv, G, block_tables, bt_stride, b, kvh, lo, hi, scale_log2);
  if (out != nullptr && S == 1) {
    // Fused merge (one split per sequence): fold in the cascade-prefix partials [0, split_offset) written earlier
    // on the stream and write the final bf16 rows — no merge kernel, no partial round trip of this split.
    // Phase 1: wave w owns heads w, w + 4: lanes load the prefix lse values in parallel, wave-reduce the max and
    // the weight sum, and publish per-split weights in LDS. Phase 2: thread (g, 4 dims) sums weight x partial over
    // the splits with all loads of a group of 8 in flight.
    for (int g = w; g < G; g += 4) {
      float Ms = -INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i) Ms = fmaxf(Ms, sM[i][g]);
      float Ls = 0.f;
      if (Ms != -INFINITY) {
#pragma unroll
        for (int i = 0; i < 4; ++i) Ls += exp2f(sM[i][g] - Ms) * sL[i][g];
      }
      const float ls = Ls > 0.f ? Ms + log2f(Ls) : -INFINITY;
      const int64_t pbase = ((int64_t)b * Hq + kvh * G + g) * S_total;
      float lp = -INFINITY;
      if (lane < split_offset) lp = lse_part[pbase + lane];
      const float lv = lane < split_offset ? lp : (lane == split_offset ? ls : -INFINITY);
      float mx = lv;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
      const float wv = mx == -INFINITY ? 0.f : exp2f(lv - mx);
      float ws = wv;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) ws += __shfl_xor(ws, o, 64);
      if (lane <= split_offset) sW[g][lane] = wv;
      if (lane == 0) sWt[g] = ws;
    }
    __syncthreads();
    const int g = threadIdx.x >> 5, c = (threadIdx.x & 31) * 4;
    if (g < G) {
      // this workgroup's own (normalised) result for dims c..c+3
      float Ms = -INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i) Ms = fmaxf(Ms, sM[i][g]);
      f32x4 os = {0.f, 0.f, 0.f, 0.f};
      float Ls = 0.f;
      if (Ms != -INFINITY) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float f = exp2f(sM[i][g] - Ms);
          Ls += f * sL[i][g];
          os += *reinterpret_cast<const f32x4*>(&sO[i][g][c]) * f;
        }
      }
      f32x4 acc4 = Ls > 0.f ? os * (sW[g][split_offset] / Ls) : f32x4{0.f, 0.f, 0.f, 0.f};
      const int64_t pbase = ((int64_t)b * Hq + kvh * G + g) * S_total * D + c;
      int s2 = 0;
      // MG prefix partials per round trip (the cascade writes 32 per row: 2 round trips at MG = 16, 4 at 8)
      if (pre_bf16 != nullptr) {  // bf16 cascade partials (tile v3): half the bytes of the fp32 round trip
        const bf16* pb = pre_bf16 + pbase;
        for (; s2 + MG <= split_offset; s2 += MG) {
          bf16x4 v[MG];
#pragma unroll
          for (int j = 0; j < MG; ++j) v[j] = *reinterpret_cast<const bf16x4*>(pb + (s2 + j) * D);
#pragma unroll
          for (int j = 0; j < MG; ++j) {
            const float wj = sW[g][s2 + j];
            acc4 += f32x4{(float)v[j][0], (float)v[j][1], (float)v[j][2], (float)v[j][3]} * wj;
          }
        }
        for (; s2 < split_offset; ++s2) {
          const bf16x4 v = *reinterpret_cast<const bf16x4*>(pb + s2 * D);
          acc4 += f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]} * sW[g][s2];
        }
      } else {
        const float* pp = out_part + pbase;
        for (; s2 + MG <= split_offset; s2 += MG) {
          f32x4 v[MG];
#pragma unroll
          for (int j = 0; j < MG; ++j) v[j] = *reinterpret_cast<const f32x4*>(pp + (s2 + j) * D);
#pragma unroll
          for (int j = 0; j < MG; ++j) acc4 += v[j] * sW[g][s2 + j];
        }
        for (; s2 < split_offset; ++s2) {
          acc4 += *reinterpret_cast<const f32x4*>(pp + s2 * D) * sW[g][s2];
        }
      }
      const float inv = sWt[g] > 0.f ? 1.f / sWt[g] : 0.f;
      bf16x4 o4;
#pragma unroll
      for (int j = 0; j < 4; ++j) o4[j] = (bf16)(acc4[j] * inv);
      if constexpr (OST)
        *reinterpret_cast<bf16x4*>(&sm.so[g][c]) = o4;
      else
        *reinterpret_cast<bf16x4*>(out + (int64_t)b * out_stride + (int64_t)(kvh * G + g) * D + c) = o4;
    }
    if constexpr (OST) store_rows_sc1<D>(sm, out, out_stride, b, kvh, G);
    return;
  }
  if (out != nullptr) {
    // ticket merge: each split's partial row leaves write-through, and the last workgroup reads it back with 16-B sc1 loads
    // (ld4 below)
    store_piece_sc1<D>(sm, b, kvh, G, Hq, split_offset + split, S_total, out_part, lse_part);
  } else
  for (int idx = threadIdx.x; idx < G * D; idx += 256) {
    const int g = idx / D, d = idx % D;
    float M = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) M = fmaxf(M, sM[i][g]);
    float L = 0.f, O = 0.f;
    if (M != -INFINITY) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float f = exp2f(sM[i][g] - M);
        L += f * sL[i][g];
        O += f * sO[i][g][d];
      }
    }
    const int64_t pidx = ((int64_t)b * Hq + kvh * G + g) * S_total + split_offset + split;
    const float ov = L > 0.f ? O / L : 0.f, lv = L > 0.f ? M + log2f(L) : -INFINITY;
    if (out == nullptr) {
      out_part[pidx * D + d] = ov;
      if (d == 0) lse_part[pidx] = lv;
    } else {  // ticket merge: write-through (agent-coherent) stores, no L2-wide write-back fence needed
      __hip_atomic_store(out_part + pidx * D + d, ov, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (d == 0) __hip_atomic_store(lse_part + pidx, lv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (out == nullptr) return;
  // Ticket merge (S > 1, e.g. one long sequence spread over many workgroups): every split publishes its partial
  // with agent-coherent write-through stores (another XCD's workgroup may read it; a __threadfence release here
  // would write back the whole L2 from every workgroup), waits for them, takes a ticket, and the LAST of the S
  // workgroups of (b, kvh) merges all split_offset + S partials (agent-coherent loads) and writes the bf16 rows —
  // no merge kernel launch. The last one also re-arms the counter for the next launch.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    int* tk = tickets + b * Hkv + kvh;
    const int t = __hip_atomic_fetch_add(tk, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    sm.s_last = t == S - 1;
    if (t == S - 1) __hip_atomic_store(tk, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!sm.s_last) return;
  auto ld = [](const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  // 16-B agent-coherent loads (sc1: not served from this XCD's possibly stale L2) as compiler builtins over a buffer
  // of out_part, so hipcc's waitcnt pass tracks them (out_part < 2 GiB: host-checked)
  const auto prs = buf_rsrc(out_part);
  auto ld4 = [&](const float* p) { return load16_sc1(prs, (int)((p - out_part) * 4)); };
  const int n = split_offset + S;  // <= 64 (host-checked)
  for (int g = w; g < G; g += 4) {
    const int64_t pbase = ((int64_t)b * Hq + kvh * G + g) * S_total;
    const float lv = lane < n ? ld(lse_part + pbase + lane) : -INFINITY;
    float mx = lv;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    const float wv = mx == -INFINITY ? 0.f : exp2f(lv - mx);
    float ws = wv;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ws += __shfl_xor(ws, o, 64);
    if (lane < n) sW[g][lane] = wv;
    if (lane == 0) sWt[g] = ws;
  }
  __syncthreads();
  const int g = threadIdx.x >> 5, c = (threadIdx.x & 31) * 4;
  if (g < G) {
    f32x4 acc4 = {0.f, 0.f, 0.f, 0.f};
    const float* pp = out_part + ((int64_t)b * Hq + kvh * G + g) * S_total * D + c;
    const int p0 = pre_bf16 != nullptr ? split_offset : 0;  // first fp32 slot (the pieces, or every slot)
    // one round trip for the common row: the first PQ fp32 slots (agent-coherent loads) and MG bf16 prefix slots
    // are all in flight before the first wait (was: the prefix batch, then the pieces batch — two tail latencies)
    constexpr int PQ = 8;
    f32x4 pv[PQ];
#pragma unroll
    for (int j = 0; j < PQ; ++j) pv[j] = ld4(pp + min(p0 + j, n - 1) * D);
    int s0 = 0;
    if (pre_bf16 != nullptr) {  // the cascade's bf16 prefix partials, MG loads per round trip (as the one-piece path)
      const bf16* pb = pre_bf16 + ((int64_t)b * Hq + kvh * G + g) * S_total * D + c;
      for (; s0 + MG <= split_offset; s0 += MG) {
        bf16x4 v[MG];
#pragma unroll
        for (int j = 0; j < MG; ++j) v[j] = *reinterpret_cast<const bf16x4*>(pb + (s0 + j) * D);
#pragma unroll
        for (int j = 0; j < MG; ++j) {
          const float wj = sW[g][s0 + j];
          acc4 += f32x4{(float)v[j][0], (float)v[j][1], (float)v[j][2], (float)v[j][3]} * wj;
        }
      }
      for (; s0 < split_offset; ++s0) {
        const bf16x4 v = *reinterpret_cast<const bf16x4*>(pb + s0 * D);
        acc4 += f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]} * sW[g][s0];
      }
    }
#pragma unroll
    for (int j = 0; j < PQ; ++j)
      if (p0 + j < n) acc4 += pv[j] * sW[g][p0 + j];
    // rows with more pieces: groups of 16 with all loads in flight (the tail of the kernel: latency, not bandwidth)
    for (int s2 = p0 + PQ; s2 < n; s2 += 16) {
      f32x4 v[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) v[j] = ld4(pp + min(s2 + j, n - 1) * D);
#pragma unroll
      for (int j = 0; j < 16; ++j)
        if (s2 + j < n) acc4 += v[j] * sW[g][s2 + j];
    }
    const float inv = sWt[g] > 0.f ? 1.f / sWt[g] : 0.f;
    bf16x4 o4;
#pragma unroll
    for (int j = 0; j < 4; ++j) o4[j] = (bf16)(acc4[j] * inv);
    if constexpr (OST)
      *reinterpret_cast<bf16x4*>(&sm.so[g][c]) = o4;
    else
      *reinterpret_cast<bf16x4*>(out + (int64_t)b * out_stride + (int64_t)(kvh * G + g) * D + c) = o4;
  }
  if constexpr (OST) store_rows_sc1<D>(sm, out, out_stride, b, kvh, G);
}

}  // namespace kafka
