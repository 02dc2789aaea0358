// Latent attention for gfx950 (bf16): prompt portions on expanded keys and values; single tokens at kv_rank 512.
//
// A latent-attention layer caches one latent row c (and one rotated key part) per token; head h's key and value are
// W_uk,h c and W_uv,h c. A decoded token attends in the latent space (latent_decode, for other ranks hybrid.hip): its cost is the
// cache, read once for all heads, and nothing per head is materialised. A portion of many rows is bound by its products
// instead, and there the latent space is the dear one: 2 (kv_rank + rot_dim) + 2 kv_rank multiply-adds per (row, key, head)
// against 2 (dim + rot_dim) + 2 vdim on the heads' own keys and values (2176 against 640 at 512 / 64 / 128 / 128), which cost
// one product of kv_rank x (dim + vdim) per key and head, however many rows follow.
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
// for the operands; K and V of a head come from its XCD's cache. With the gather and the products around it, operands from
// memory, 32 heads: 2048 fresh rows of 128 + 64 channels 192 us (in the latent space 626), 8192 rows of 128 + 0 with a window of
// 1024 310 (2120; this kernel alone 209 of them, 0.6 PFLOP/s).
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

// ---- attention in the latent space, kv_rank 512 ---------------------------------------------------------------------
// One workgroup (4 waves) per tile of 32 query rows = (token, head) pairs that read the same sequence and, with gridDim.z > 1,
// per range of its key blocks (partials for latent_merge, hybrid.hip). Keys go by in blocks of two pages. The cache rows of four
// blocks lie in LDS as they are, sent there without a register on the way (16-byte chunk c of key row k at chunk c ^ (k & 7)
// of its group of eight), and serve both products:
//   scores   wave w: S = Q K^T of 16 rows and the 16 keys of page w & 1 (16x16x32), Q in registers for the whole walk;
//   softmax  row maxima across lanes and, through LDS, waves; weights as bf16 in LDS, a lane's part of the row sums stays;
//   values   wave w owns 128 columns, lane n four of them: O += P V with eight keys' 8-byte pieces of the rows turned into
//            four operands by byte permutes.
// What bounds it: a block's chain of waits, softmax and products (1.5 us; Q's scores want 72 registers and one workgroup fits a
// CU), with many sequences the rows' way to the CUs as well. The walk for other ranks (hybrid.hip) reads keys in 32-byte pieces
// and the values from a second, transposed copy; here, with the launch's merge, 32 heads, operands from memory: 64 sequences x 1706
// keys 168 -> 70 us (126 MB; from a warm cache 131 -> 51), 16 sequences 93 -> 38, one 80 -> 28, one x 8000 136 -> 41.
// Rows past the tile's last position are masked as keys and zeroed as values: what a page holds there does not matter.
constexpr int LD_R = 512, LD_KEYS = 32, LD_SLOTS = 4;
constexpr int LD_RUN = 512;   // blocks whose page ids lie in LDS at a time (16k tokens)
constexpr int LD_PS = LD_KEYS + 8;

typedef __attribute__((address_space(3))) void ld_lds_t;
// 16 B per lane, 1 KiB to consecutive LDS bytes
__device__ __forceinline__ void ld_dma16(const void* g, void* lds) {
  __builtin_amdgcn_global_load_lds(g, (ld_lds_t*)lds, 16, 0, 0);
}
__device__ __forceinline__ f32x4 ld_mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// c[j] += a b[j] in the sums' own vector registers (the compiler keeps them in accumulation registers and moves them for every
// rescale). One statement, wait included: the compiler does not know that these products take eight passes, nor of a wait that
// stands elsewhere, and may copy a statement's outputs as soon as it ends.
__device__ __forceinline__ void ld_mfma32(f32x16 (&c)[4], bf16x8 a, const bf16x8 (&b)[4]) {
  asm volatile(
      "s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %4, %5, %0\n\tv_mfma_f32_32x32x16_bf16 %1, %4, %6, %1\n\t"
      "v_mfma_f32_32x32x16_bf16 %2, %4, %7, %2\n\tv_mfma_f32_32x32x16_bf16 %3, %4, %8, %3\n\ts_nop 11"
      : "+v"(c[0]), "+v"(c[1]), "+v"(c[2]), "+v"(c[3])
      : "v"(a), "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]));
}
// the value of the lane n places on in its 16
template <int N>
__device__ __forceinline__ float ld_ror(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + N, 0xf, 0xf, false));
}
typedef unsigned ld_u2 __attribute__((ext_vector_type(2)));
typedef unsigned ld_u4 __attribute__((ext_vector_type(4)));

template <int RD>
__global__ __launch_bounds__(256, 2) void latent_decode_kernel(
    const bf16* __restrict__ q_lat, int64_t ql_h, int64_t ql_t, const bf16* __restrict__ q_rot, int64_t qr_t, int64_t qr_h,
    const bf16* __restrict__ cache, const int* __restrict__ bt, int bt_stride, const int* __restrict__ items,
    const int64_t* __restrict__ positions, float scale_log2e, bf16* __restrict__ out, int64_t o_h, int64_t o_t, int H,
    float* __restrict__ po, float* __restrict__ pml, int T, int window, const float* __restrict__ sink) {
  constexpr int R = LD_R, Dk = R + RD, ROW = Dk * 2, CPK = Dk / 8, PAGE_B = 16 * ROW, SLOT = 2 * PAGE_B;
  constexpr int NP = PAGE_B / 2048, NKS = Dk / 32;   // 1-KiB pieces of a wave and block, steps of 32 channels
  __shared__ __attribute__((aligned(16))) unsigned char smem[LD_SLOTS * SLOT + 32 * LD_PS * 2 + (64 + 32 + 32) * 4 + 2 * LD_RUN * 4];
  bf16* Ps = reinterpret_cast<bf16*>(smem + LD_SLOTS * SLOT); // [32][LD_PS]
  float* mloc = reinterpret_cast<float*>(Ps + 32 * LD_PS);    // [2][32]
  float* corr_s = mloc + 64;                                  // [32]
  int* prow_s = reinterpret_cast<int*>(corr_s + 32);          // [32]
  int* pg_s = prow_s + 32;                                    // [2 LD_RUN]
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int k16 = lane & 15, g = lane >> 4, n32 = lane & 31, lh = lane >> 5, pw = w & 1, qt = w >> 1;
  const int t0 = items[4 * blockIdx.x], ntok = items[4 * blockIdx.x + 1], sg = items[4 * blockIdx.x + 2];
  const int h0 = blockIdx.y * 32, hpr = min(H - h0, 32), nrows = ntok * hpr;
  const int maxpos = (int)positions[t0 + ntok - 1], last = maxpos >> 4;
  const int* btr = bt + (int64_t)sg * bt_stride;
  const int nsplit = gridDim.z, nblocks = (maxpos >> 5) + 1;
  const int kbmin = window > 0 ? max(0, (int)positions[t0] - window + 1) >> 5 : 0;
  const int bps = (nblocks - kbmin + nsplit - 1) / nsplit;
  const int kb0 = kbmin + blockIdx.z * bps, kb1 = min(nblocks, kb0 + bps);

  // Q fragments (zeros for rows beyond the tile): lane holds row 16 qt + k16, channels 32 ks + 8 g ..
  bf16x8 aq[NKS];
  {
    const int r = 16 * qt + k16, rr = min(r, nrows - 1);
    const int64_t t = t0 + rr / hpr, h = h0 + rr % hpr;
    const bf16* ql = q_lat + h * ql_h + t * ql_t + 8 * g;
    const bf16* qr = RD ? q_rot + t * qr_t + h * qr_h + 8 * g : nullptr;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      aq[ks] = load_bf16x8(ks * 32 < R ? ql + 32 * ks : qr + (32 * ks - R));
      if (r >= nrows) aq[ks] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }
  int soff[NP];   // where the lane's 16 bytes of piece c of its half page come from
#pragma unroll
  for (int c = 0; c < NP; ++c) {
    const int p = 64 * (NP * qt + c) + lane, key = p / CPK, cc = p - key * CPK;
    soff[c] = key * ROW + 16 * ((cc & ~7) | ((cc ^ key) & 7));
  }
  auto issue = [&](int x) {   // wave w: half w >> 1 of page w & 1 of the run's block x
    const char* src = reinterpret_cast<const char*>(cache) + (int64_t)__builtin_amdgcn_readfirstlane(pg_s[2 * x + pw]) * PAGE_B;
    unsigned char* dst = smem + (x % LD_SLOTS) * SLOT + pw * PAGE_B + qt * (PAGE_B / 2);
#pragma unroll
    for (int c = 0; c < NP; ++c) ld_dma16(src + soff[c], dst + c * 1024);
  };
  if (threadIdx.x < 32) prow_s[threadIdx.x] = threadIdx.x < nrows ? (int)positions[t0 + threadIdx.x / hpr] : 0;
  lds_barrier();
  int prow[4];
  float m[4], lsum[4];
  f32x16 O[4];
  const int r0 = 16 * qt + 4 * g;   // the lane's first row of the scores
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    prow[i] = prow_s[r0 + i];
    m[i] = -INFINITY;
    lsum[i] = 0.f;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) O[j][i] = 0.f;
  const unsigned char* kbase[2];
#pragma unroll
  for (int o = 0; o < 2; ++o) kbase[o] = smem + pw * PAGE_B + k16 * ROW + 16 * ((4 * o + g) ^ (k16 & 7));
  const unsigned char* vbase[8];
#pragma unroll
  for (int k = 0; k < 8; ++k)
    vbase[k] = smem + (8 * lh + k) * ROW + 16 * (16 * w + 8 * (n32 >> 4) + (((n32 >> 1) & 7) ^ k)) + 8 * (n32 & 1);

  for (int run = kb0; run < kb1; run += LD_RUN) {
   const int nb = min(kb1 - run, LD_RUN);
   for (int i = threadIdx.x; i < 2 * nb; i += 256) pg_s[i] = btr[min(2 * run + i, last)];   // (past the last page: it again)
   lds_barrier();
#pragma unroll
   for (int x = 0; x < LD_SLOTS - 1; ++x)
     if (x < nb) issue(x);
   for (int x = 0; x < nb; ++x) {
    const int kb = run + x, so = (x % LD_SLOTS) * SLOT;
    // this wave's part of the block has landed (those of up to two more stay on their way), then everyone's; everyone has left
    // the block before, whose slot the third one from here takes
    if (x + 2 < nb)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NP) : "memory");
    else if (x + 1 < nb)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NP) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    if (x + LD_SLOTS - 1 < nb) issue(x + LD_SLOTS - 1);
    f32x4 s2[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {   // half of the reads in flight at a time
      bf16x8 kf[NKS / 2];
#pragma unroll
      for (int i = 0; i < NKS / 2; ++i) {
        const int ks = hf * (NKS / 2) + i;
        kf[i] = *reinterpret_cast<const bf16x8*>(kbase[ks & 1] + so + 128 * (ks >> 1));
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < NKS / 2; ++i) s2[i & 1] = ld_mfma16(aq[hf * (NKS / 2) + i], kf[i], s2[i & 1]);
    }
    const int key = kb * LD_KEYS + 16 * pw + k16;
    float s[4];
    f32x4 mx;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s[i] = (key <= prow[i] && (window == 0 || key > prow[i] - window)) ? (s2[0][i] + s2[1][i]) * scale_log2e : -INFINITY;
      float v = s[i];
      v = fmaxf(v, ld_ror<8>(v));
      v = fmaxf(v, ld_ror<4>(v));
      v = fmaxf(v, ld_ror<2>(v));
      mx[i] = fmaxf(v, ld_ror<1>(v));
    }
    if (k16 == 0) *reinterpret_cast<f32x4*>(mloc + 32 * pw + r0) = mx;
    lds_barrier();
    {
      const f32x4 ma = *reinterpret_cast<const f32x4*>(mloc + r0), mb = *reinterpret_cast<const f32x4*>(mloc + 32 + r0);
      f32x4 cr;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float mn = fmaxf(m[i], fmaxf(ma[i], mb[i]));
        // (a range that starts past a row's position leaves the row empty: no inf - inf)
        cr[i] = mn == -INFINITY ? 0.f : fast_exp2(m[i] - mn);
        const float p = mn == -INFINITY ? 0.f : fast_exp2(s[i] - mn);
        lsum[i] = lsum[i] * cr[i] + p;
        m[i] = mn;
        Ps[(r0 + i) * LD_PS + 16 * pw + k16] = (bf16)p;
      }
      if (pw == 0 && k16 == 0) *reinterpret_cast<f32x4*>(corr_s + r0) = cr;
    }
    lds_barrier();
    f32x4 cr[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) cr[x] = *reinterpret_cast<const f32x4*>(corr_s + 8 * x + 4 * lh);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) O[j][i] *= cr[i >> 2][i & 3];
    ld_u2 v[2][8];
    bf16x8 a[2];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      a[st] = *reinterpret_cast<const bf16x8*>(Ps + n32 * LD_PS + 16 * st + 8 * lh);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[st][k] = *reinterpret_cast<const ld_u2*>(vbase[k] + so + st * PAGE_B);
    }
    if (kb * LD_KEYS + LD_KEYS - 1 > maxpos) {
#pragma unroll
      for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (kb * LD_KEYS + 16 * st + 8 * lh + k > maxpos) v[st][k] = ld_u2{0u, 0u};
    }
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      bf16x8 b[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        ld_u4 p;
#pragma unroll
        for (int x4 = 0; x4 < 4; ++x4)
          p[x4] = __builtin_amdgcn_perm(v[st][2 * x4 + 1][j >> 1], v[st][2 * x4][j >> 1], j & 1 ? 0x07060302u : 0x05040100u);
        b[j] = __builtin_bit_cast(bf16x8, p);
      }
      ld_mfma32(O, a[st], b);
    }
   }
   lds_barrier();   // (the run's page ids, slots and corr_s are read until here)
  }
  // ---- row sums: across the lanes of a row, then the two pages
  {
    f32x4 l, mm;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v = lsum[i];
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
      l[i] = v;
      mm[i] = m[i];
    }
    if (k16 == 0) {
      *reinterpret_cast<f32x4*>(mloc + 32 * pw + r0) = l;
      if (pw == 0) *reinterpret_cast<f32x4*>(corr_s + r0) = mm;
    }
  }
  lds_barrier();
  const int c0 = 128 * w + 4 * n32;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = (i & 3) + 8 * (i >> 2) + 4 * lh;
    if (r >= nrows) continue;
    float l = mloc[r] + mloc[32 + r];
    const float mr = corr_s[r];
    const int64_t t = t0 + r / hpr, h = h0 + r % hpr;
    if (nsplit == 1) {
      if (sink != nullptr) l += fast_exp2(sink[h] * LOG2E - mr);
      const float inv = 1.0f / l;
      typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
      *reinterpret_cast<bf16x4*>(out + h * o_h + t * o_t + c0) =
          bf16x4{(bf16)(O[0][i] * inv), (bf16)(O[1][i] * inv), (bf16)(O[2][i] * inv), (bf16)(O[3][i] * inv)};
    } else {
      const int64_t row = ((int64_t)blockIdx.z * H + h) * T + t;
      if (w == 0 && n32 == 0) {
        pml[2 * row] = mr;
        pml[2 * row + 1] = l;
      }
      *reinterpret_cast<f32x4*>(po + row * R + c0) = f32x4{O[0][i], O[1][i], O[2][i], O[3][i]};
    }
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

int kafka_hy_latent_decode_ok(const void* cache, int R, int rd, const void* out, int64_t o_h, int64_t o_t) {
  return R == LD_R && (rd == 0 || rd == 64) && (reinterpret_cast<uintptr_t>(cache) & 15) == 0 &&
         (reinterpret_cast<uintptr_t>(out) & 7) == 0 && o_h % 4 == 0 && o_t % 4 == 0;
}

hipError_t kafka_hy_latent_decode(const void* q_lat, int64_t ql_h, int64_t ql_t, const void* q_rot, int64_t qr_t, int64_t qr_h,
                                  const void* cache, int rd, const int* bt, int bt_stride, const int* items, int n_items,
                                  const int64_t* positions, float scale_log2e, void* out, int64_t o_h, int64_t o_t, int H,
                                  int nsplit, float* po, float* pml, int T, int window, const float* sink, hipStream_t st) {
  auto a = [&](auto k) {
    k<<<dim3((unsigned)n_items, (unsigned)((H + 31) / 32), (unsigned)nsplit), 256, 0, st>>>(
        (const bf16*)q_lat, ql_h, ql_t, (const bf16*)q_rot, qr_t, qr_h, (const bf16*)cache, bt, bt_stride, items, positions,
        scale_log2e, (bf16*)out, o_h, o_t, H, po, pml, T, window, sink);
  };
  rd ? a(latent_decode_kernel<64>) : a(latent_decode_kernel<0>);
  return hipGetLastError();
}

}  // extern "C"
