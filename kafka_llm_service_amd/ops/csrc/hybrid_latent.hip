// Latent attention of prompt portions on expanded keys and values, for gfx950 (bf16).
//
// A latent-attention layer caches one latent row c (and one rotated key part) per token; head h's key and value are
// W_uk,h c and W_uv,h c. A decoded token attends in the latent space (hybrid.hip): its cost is the cache, read once for all
// heads, and nothing per head is materialised. A portion of many rows is bound by its products instead, and there the
// latent space is the dear one: 2 (kv_rank + rot_dim) + 2 kv_rank multiply-adds per (row, key, head) against
// 2 (dim + rot_dim) + 2 vdim on the heads' own keys and values (2176 against 640 at 512 / 64 / 128 / 128), which cost one
// product of kv_rank x (dim + vdim) per key and head, however many rows follow.
//   latent_gather  the context's cache rows (all of it, or what the window reaches) one below the other: latents [M, kv_rank]
//                  for the two products K = C W_uk^T and V^T = W_uv C^T, rotated parts [M, rot_dim]
//   latent_rows    softmax attention of one head's rows against them
#include "chunk_common.h"

namespace kafka {
namespace hy {

using namespace chunk;

constexpr int LX_KEYS = 64;    // keys of a block; a portion's gathered rows start at a multiple of it
constexpr int LX_ROWS = 128;   // rows of a workgroup

// LDS operands are visible to the workgroup; global loads stay in flight
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// portion s: px[8 s ..] = (first row, rows, first position, first gathered key, first gathered row, block-table row, keys' end)
struct Portions {
  const int* px;
  const int* blocks;   // portion of every LX_KEYS gathered rows
  const int* tiles;    // [n][4] = (portion, first row in it, -, -)
};

__global__ __launch_bounds__(NT) void latent_gather_kernel(const bf16* __restrict__ cache, int R, int rd,
                                                           const int* __restrict__ bt, int bt_stride, Portions pt,
                                                           bf16* __restrict__ ck, bf16* __restrict__ kr) {
  const int s = pt.blocks[blockIdx.x];
  const int* px = pt.px + 8 * s;
  const int64_t m0 = (int64_t)blockIdx.x * LX_KEYS;
  const int j0 = px[3] + (int)(m0 - px[4]), end = px[6], Dk = R + rd, vecs = Dk >> 3;
  const int* btr = bt + (int64_t)px[5] * bt_stride;
  for (int u = threadIdx.x; u < LX_KEYS * vecs; u += NT) {
    const int r = u / vecs, d = (u - r * vecs) << 3, j = j0 + r;
    bf16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};   // (rows past the context: zeros, masked by every row)
    if (j < end) v = load_bf16x8(cache + ((int64_t)btr[j >> 4] * 16 + (j & 15)) * Dk + d);
    if (d < R) store_bf16x8(ck + (m0 + r) * R + d, v);
    else store_bf16x8(kr + (m0 + r) * rd + (d - R), v);
  }
}

// A workgroup takes 128 rows of one portion and one head, a wave 32 of them, and walks the keys 64 at a time through LDS (the
// next block's rows are in registers meanwhile):
//   scores   S^T = K Q^T, lane = row. The key rows lie in LDS with bits 2 and 3 of their numbers swapped, which leaves lane
//            half lh with keys 8 lh .. + 7 of every 16;
//   softmax  a row's maximum, sum and weights live in its two lanes, the accumulators are rescaled only when a row's maximum
//            has moved;
//   values   O^T += V^T P^T: the weights are the right operand as they lie in the registers, the left one is a channel's 8
//            consecutive keys.
// What bounds it: a wave's chain of scores, softmax and values (two waves per SIMD hide part of it), and half the LDS rate
// for the operands; K and V of a head come from its XCD's cache. 2048 fresh rows x 32 heads with
// the products around it 178 us (latent space: 1170), 8192 rows with a window of 1024 216 us alone, 0.6 PFLOP/s (4550).
// ND, NR: steps of 16 channels of a head's own and rotated key part; NV: tiles of 32 value channels.
template <int ND, int NR, int NV, bool GATE>
__global__ __launch_bounds__(NT, 2) void latent_rows_kernel(
    const bf16* __restrict__ q, int64_t q_t, int64_t q_h, const bf16* __restrict__ q_rot, int64_t qr_t, int64_t qr_h,
    const bf16* __restrict__ K, const bf16* __restrict__ kr, const bf16* __restrict__ Vt, int64_t M, Portions pt, int n_tiles,
    int H, float scale_log2e, int window, const float* __restrict__ sink, const bf16* __restrict__ gate, int64_t gs,
    bf16* __restrict__ out, int64_t os) {
  constexpr int NK = ND + NR, KS = 16 * NK + 8, VS = LX_KEYS + 8, KV = 2 * NK, D = 16 * ND, Dv = 32 * NV;
  constexpr int KF = LX_KEYS * KV / NT, VF = Dv * (LX_KEYS / 8) / NT;   // 16-byte pieces a thread moves per block
  static_assert(LX_KEYS * KV % NT == 0 && Dv * (LX_KEYS / 8) % NT == 0, "pieces");
  typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
  __shared__ __attribute__((aligned(16))) bf16 Ks[LX_KEYS * KS];
  __shared__ __attribute__((aligned(16))) bf16 Vs[Dv * VS];
  // workgroups go round the eight XCDs: a head's stay on one where the heads divide
  int h, tile;
  if (H % 8 == 0) {
    const int x = blockIdx.x & 7, k = blockIdx.x >> 3, hx = H >> 3;
    h = x + 8 * (k % hx);
    tile = k / hx;
  } else {
    h = blockIdx.x % H;
    tile = blockIdx.x / H;
  }
  const int* px = pt.px + 8 * pt.tiles[4 * tile];
  const int r0 = pt.tiles[4 * tile + 1], n = px[1], p0 = px[2], klo = px[3];
  const int64_t m0 = px[4];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, lr = lane & 31, lh = lane >> 5;
  const int r = r0 + 32 * w + lr;                 // this lane's row of the portion
  const int rc = min(r, n - 1), p = p0 + rc;
  const int64_t t = (int64_t)px[0] + rc;
  const int wmin = p0 + min(r0 + 32 * w, n - 1), wmax = p0 + min(r0 + 32 * w + 31, n - 1);   // the wave's positions
  const bool wave_live = r0 + 32 * w < n;
  const int tmax = p0 + min(r0 + LX_ROWS - 1, n - 1);
  bf16x8 qf[NK];
#pragma unroll
  for (int ks = 0; ks < NK; ++ks)
    qf[ks] = ks < ND ? load_bf16x8(q + t * q_t + (int64_t)h * q_h + 16 * ks + 8 * lh)
                     : load_bf16x8(q_rot + t * qr_t + (int64_t)h * qr_h + 16 * (ks - ND) + 8 * lh);
  bf16x8 kf[KF], vf[VF];
  auto fetch = [&](int kb) {
    const int64_t m = m0 + (int64_t)kb * LX_KEYS;
#pragma unroll
    for (int i = 0; i < KF; ++i) {
      const int u = tid + NT * i, row = u / KV, c = u - row * KV;
      kf[i] = c < 2 * ND ? load_bf16x8(K + (m + row) * ((int64_t)H * D) + (int64_t)h * D + 8 * c)
                         : load_bf16x8(kr + (m + row) * (16 * NR) + 8 * (c - 2 * ND));
    }
#pragma unroll
    for (int i = 0; i < VF; ++i) {
      const int u = tid + NT * i, ch = u >> 3, c = u & 7;
      vf[i] = load_bf16x8(Vt + ((int64_t)h * Dv + ch) * M + m + 8 * c);
    }
  };
  auto stash = [&]() {
#pragma unroll
    for (int i = 0; i < KF; ++i) {
      const int u = tid + NT * i, row = u / KV, c = u - row * KV;
      const int at = (row & ~12) | ((row & 4) << 1) | ((row & 8) >> 1);   // bits 2 and 3 swapped
      store_bf16x8(Ks + at * KS + 8 * c, kf[i]);
    }
#pragma unroll
    for (int i = 0; i < VF; ++i) {
      const int u = tid + NT * i, ch = u >> 3, c = u & 7;
      store_bf16x8(Vs + ch * VS + 8 * c, vf[i]);
    }
  };
  float m = -INFINITY, l = 0.f;
  f32x16 O[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int i = 0; i < 16; ++i) O[v][i] = 0.f;
  const int lo = window > 0 ? max(0, p0 + r0 - window + 1) : 0;   // first key the tile sees
  const int kb0 = max(0, lo - klo) / LX_KEYS, kb1 = (tmax - klo) / LX_KEYS + 1;
  fetch(kb0);
  for (int kb = kb0; kb < kb1; ++kb) {
    lds_barrier();   // (the block before has been read)
    stash();
    lds_barrier();
    if (kb + 1 < kb1) fetch(kb + 1);
    const int key0 = klo + kb * LX_KEYS;
    // (uniform per wave) blocks that none of its rows sees
    if (!wave_live || key0 > wmax || (window > 0 && key0 + LX_KEYS - 1 <= wmin - window)) continue;
    f32x16 S[2];
#pragma unroll
    for (int sb = 0; sb < 2; ++sb)
#pragma unroll
      for (int i = 0; i < 16; ++i) S[sb][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < NK; ++ks)
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
        S[sb] = mfma32(load_bf16x8(Ks + (32 * sb + lr) * KS + 16 * ks + 8 * lh), qf[ks], S[sb]);
    mfma_settle();
    float mx = -INFINITY;
    if (key0 + LX_KEYS - 1 > wmin || (window > 0 && key0 <= wmax - window)) {
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = key0 + 32 * sb + 16 * (i >> 3) + 8 * lh + (i & 7);
          S[sb][i] = key > p || (window > 0 && key <= p - window) ? -INFINITY : S[sb][i];
        }
    }
#pragma unroll
    for (int sb = 0; sb < 2; ++sb)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, S[sb][i]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * scale_log2e;   // (the scale is positive)
    const float mn = fmaxf(m, mx);
    const float base = mn == -INFINITY ? 0.f : mn;   // nothing visible yet: every weight is 2^-inf = 0
    if (__any(mx > m)) {
      const float corr = m == -INFINITY ? 0.f : fast_exp2(m - base);
      l *= corr;
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int i = 0; i < 16; ++i) O[v][i] *= corr;
    }
    m = mn;
#pragma unroll
    for (int sb = 0; sb < 2; ++sb) {
      bf16x8 pf[2];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float e = fast_exp2(S[sb][i] * scale_log2e - base);
        l += e;
        pf[i >> 3][i & 7] = (bf16)e;
      }
#pragma unroll
      for (int pg = 0; pg < 2; ++pg)
#pragma unroll
        for (int v = 0; v < NV; ++v)
          O[v] = mfma32(load_bf16x8(Vs + (32 * v + lr) * VS + 32 * sb + 16 * pg + 8 * lh), pf[pg], O[v]);
    }
  }
  mfma_settle();
  l += __shfl_xor(l, 32, 64);
  if (r >= n) return;
  if (sink != nullptr) l += fast_exp2(sink[h] * LOG2E - m);
  const float inv = 1.0f / l;
  bf16* op = out + t * os + (int64_t)h * Dv;
  const bf16* gp = GATE ? gate + t * gs + (int64_t)h * Dv : nullptr;
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const int c = 32 * v + 8 * i4 + 4 * lh;
      bf16x4 o, g;
      if (GATE) g = *reinterpret_cast<const bf16x4*>(gp + c);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float x = O[v][4 * i4 + e] * inv;
        if (GATE) x = x / (1.0f + expf(-(float)g[e]));
        o[e] = (bf16)x;
      }
      *reinterpret_cast<bf16x4*>(op + c) = o;
    }
}

}  // namespace hy
}  // namespace kafka

using namespace kafka::hy;

extern "C" {

int kafka_hy_latent_rows_ok(int R, int rd, int D, int Dv) {
  return R >= 32 && R % 32 == 0 && R <= 512 && (rd == 0 || rd == 64) && D == 128 && Dv == 128;
}

hipError_t kafka_hy_latent_gather(const void* cache, int R, int rd, const int* bt, int bt_stride, const int* px,
                                  const int* blocks, int n_blocks, void* ck, void* kr, hipStream_t st) {
  if (n_blocks <= 0) return hipSuccess;
  if (R % 8 || rd % 8) return hipErrorInvalidValue;
  latent_gather_kernel<<<n_blocks, NT, 0, st>>>((const bf16*)cache, R, rd, bt, bt_stride, Portions{px, blocks, nullptr},
                                                (bf16*)ck, (bf16*)kr);
  return hipGetLastError();
}

hipError_t kafka_hy_latent_rows(const void* q, int64_t q_t, int64_t q_h, const void* q_rot, int64_t qr_t, int64_t qr_h,
                                const void* K, const void* kr, const void* Vt, int64_t M, const int* px, const int* tiles,
                                int n_tiles, int H, int rd, float scale, int window, const float* sink, const void* gate,
                                int64_t gs, void* out, int64_t os, hipStream_t st) {
  if (n_tiles <= 0) return hipSuccess;
  if (!kafka_hy_latent_rows_ok(32, rd, 128, 128) || window < 0 || !(scale > 0.f) || M % LX_KEYS ||
      (int64_t)n_tiles * H > 0x7fffffff)
    return hipErrorInvalidValue;
  auto a = [&](auto k) {
    k<<<(unsigned)(n_tiles * H), NT, 0, st>>>((const bf16*)q, q_t, q_h, (const bf16*)q_rot, qr_t, qr_h, (const bf16*)K,
                                              (const bf16*)kr, (const bf16*)Vt, M, Portions{px, nullptr, tiles}, n_tiles, H,
                                              scale * LOG2E, window, sink, (const bf16*)gate, gs, (bf16*)out, os);
  };
  if (rd == 64) gate ? a(latent_rows_kernel<8, 4, 4, true>) : a(latent_rows_kernel<8, 4, 4, false>);
  else gate ? a(latent_rows_kernel<8, 0, 4, true>) : a(latent_rows_kernel<8, 0, 4, false>);
  return hipGetLastError();
}

}  // extern "C"
