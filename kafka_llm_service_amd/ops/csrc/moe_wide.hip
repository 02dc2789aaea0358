// Expert products of long steps on wave-tiled expert weights, and what surrounds them, for gfx950.
//
//   grouped_wide   Y = X_e W_e^T per expert segment of the routed entries, 128 rows x 256 columns a workgroup, for steps
//                  whose experts have many rows. The weights come in the wave-tiled order of the weight-streaming
//                  kernels (Wt[E][N/32][K/16][64][8]): a wave owns 64 columns and loads its operands straight from
//                  memory in 1 KB pieces; only the activations go through LDS (64-deep steps, double buffered, next
//                  step's loads in flight), where all four waves share them. Work items are ordered row tile first (up to 2048
//                  rows), then column tile, then the next rows, then expert, and every XCD takes one contiguous stretch of
//                  them: the row tiles of a column tile run side by side on one L2 and its weights leave memory once.
//                  Epilogues: silu(gate) * up or its clamped form on GLU-interleaved tiles (a wave holds both tiles of a
//                  pair), relu squared, the weighted combine into fp32 rows, or the weighted rows as they are (in entry
//                  order; their consumer gathers a token's rows through the sort's inverse, no atomics).
//   grouped_ring   the same on 256 x 256 tiles (lower ones for an expert's last rows), both operands through a ring in LDS
//   moe_sort       stable sort of (token, choice) entries by expert: every wave counts and then places its stretch of the
//                  entries 64 at a time, equal experts found by ballots over the bits of their ids; one workgroup, or for
//                  more than 4096 entries of up to 64 experts one per 2048 behind a launch that counts
//   narrow         fp32 products of bf16 rows with up to 64 bf16 weight rows (router logits, gate projections): 16 rows a
//                  workgroup, its 16 (or 8) waves split K, 16x16x32 products; with a bias, or followed in place by the
//                  choice of the k largest scores, a wave per row
#include <type_traits>

#include "moe_sort.h"
#include "ring.h"

namespace kafka {
namespace mw {

// ---- grouped products -------------------------------------------------------------------------------------------------
constexpr int BM = 128, BN = 256, BK = 64;
constexpr int KS = BK / 16;        // matrix steps per staged block
constexpr int MT = BM / 32;        // row tiles
constexpr int XL = BM * (BK / 8) / 256;

enum { EPI_GLU = 0, EPI_RELU2 = 1, EPI_COMBINE = 2, EPI_ROWS = 3 };

// 16-byte piece c (0 .. 7) of LDS row r
__device__ __forceinline__ int xoff(int r, int c) { return r * BK + 8 * (c ^ (r & 7)); }

// item -> (expert, row tile, column tile) over the experts' segments; false past the last item. Every wave does this.
__device__ __forceinline__ bool find_item(const int* expert_off, int E, int ntn, int BM, int& e, int& rt, int& nt) {
  const int lane = threadIdx.x & 63;
  // all items, in waves of 64 experts: the total first, then this workgroup's place
  int total = 0;
  for (int b = 0; b < E; b += 64) {
    int t = 0;
    if (b + lane < E) t = (expert_off[b + lane + 1] - expert_off[b + lane] + BM - 1) / BM * ntn;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
    total += t;
  }
  const int per = (total + 7) >> 3, k = blockIdx.x >> 3;
  const int item = (blockIdx.x & 7) * per + k;
  if (k >= per || item >= total) return false;
  int base = 0;
  for (int b = 0; b < E; b += 64) {
    int t = 0;
    if (b + lane < E) t = (expert_off[b + lane + 1] - expert_off[b + lane] + BM - 1) / BM * ntn;
    int incl = t;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(incl, o, 64);
      if (lane >= o) incl += u;
    }
    const unsigned long long hit = __ballot(base + incl > item);
    if (hit) {
      const int l = __builtin_ctzll(hit);
      const int before = base + __shfl(incl - t, l, 64), tiles = __shfl(t, l, 64) / ntn;
      e = __builtin_amdgcn_readfirstlane(b + l);
      const int i = __builtin_amdgcn_readfirstlane(item - before), ti = __builtin_amdgcn_readfirstlane(tiles);
      // row tiles of up to 2048 rows side by side, then the next column tile, then the next 2048 rows: what an XCD's 32
      // CUs work on at once is about as many rows as columns
      const int gr = 2048 / BM, g = i / (gr * ntn), j = i - g * gr * ntn, in_g = min(gr, ti - g * gr);
      nt = j / in_g;
      rt = g * gr + (j - nt * in_g);
      return true;
    }
    base += __shfl(incl, 63, 64);
  }
  return false;
}

template <bool GATHER, int EPI>
__global__ __launch_bounds__(256, 2) void grouped_wide_kernel(const bf16* __restrict__ X, int64_t ldx,
                                                              const bf16x8* __restrict__ Wt, int E, int N, int K,
                                                              const int* __restrict__ perm_tok,
                                                              const float* __restrict__ perm_w,
                                                              const int* __restrict__ expert_off,
                                                              bf16* __restrict__ Y, int64_t ldy,
                                                              float* __restrict__ out, int64_t ldo, float glu_limit,
                                                              float glu_alpha) {
  __shared__ __attribute__((aligned(16))) bf16 xs[2][BM * BK];
  int e, rt, nt;
  if (!find_item(expert_off, E, (N + BN - 1) / BN, BM, e, rt, nt)) return;   // (uniform)
  const int seg0 = expert_off[e] + rt * BM, rows = min(BM, expert_off[e + 1] - seg0);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r = lane & 31, h = lane >> 5;
  const int nb = (nt * 4 + w) * 2;                 // this wave's two 32-column tiles
  const bool active = nb < (N >> 5);               // (N is a multiple of 64: both or none)
  const bf16x8* wp = Wt + ((int64_t)e * (N >> 5) + (active ? nb : 0)) * (K >> 4) * 64 + lane;
  const int64_t wstep = (int64_t)(K >> 4) * 64;    // the second tile
  const int nk = K / BK;
  const bf16* xsrc[XL];
  int xdst[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int idx = tid + 256 * i, row = idx >> 3, c = idx & 7;
    const int ent = seg0 + min(row, rows - 1);     // rows past the segment reload a valid row, never stored
    xsrc[i] = X + (GATHER ? (int64_t)perm_tok[ent] : (int64_t)ent) * ldx + c * 8;
    xdst[i] = xoff(row, c);
  }
  bf16x8 xr[XL], wa[KS][2], wb[KS][2];
  auto load_x = [&](int ch) {
#pragma unroll
    for (int i = 0; i < XL; ++i) xr[i] = load_bf16x8(xsrc[i] + ch * BK);
  };
  auto store_x = [&](int buf) {
#pragma unroll
    for (int i = 0; i < XL; ++i) *reinterpret_cast<bf16x8*>(&xs[buf][xdst[i]]) = xr[i];
  };
  auto load_w = [&](bf16x8(&wv)[KS][2], int ch) {
#pragma unroll
    for (int t = 0; t < KS; ++t)
#pragma unroll
      for (int j = 0; j < 2; ++j) wv[t][j] = wp[(int64_t)(ch * KS + t) * 64 + j * wstep];
    __builtin_amdgcn_sched_barrier(0);             // (requested before this step's products)
  };
  f32x16 acc[MT][2];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mt][j][i] = 0.f;
  auto compute = [&](int buf, const bf16x8(&wv)[KS][2]) {
#pragma unroll
    for (int t = 0; t < KS; ++t)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const bf16x8 xf = *reinterpret_cast<const bf16x8*>(&xs[buf][xoff(mt * 32 + r, 2 * t + h)]);
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[mt][j] = mfma32(xf, wv[t][j], acc[mt][j]);
      }
  };
  load_x(0);
  load_w(wa, 0);
  store_x(0);
  __syncthreads();
  for (int ch = 0; ch < nk; ch += 2) {               // (nk is even; the last step's prefetch repeats a block)
    load_x(ch + 1);
    load_w(wb, ch + 1);
    compute(0, wa);
    store_x(1);
    __syncthreads();
    const int nx = min(ch + 2, nk - 1);
    load_x(nx);
    load_w(wa, nx);
    compute(1, wb);
    store_x(0);
    __syncthreads();
  }
  // the last products' results are complete before anything reads them behind a branch
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 15");
  __builtin_amdgcn_sched_barrier(0);
  if (!active) return;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int m = mt * 32 + (i & 3) + 8 * (i >> 2) + 4 * h;
      if (m >= rows) continue;
      const int ent = seg0 + m;
      if constexpr (EPI == EPI_COMBINE) {
        float* o = out + (int64_t)perm_tok[ent] * ldo + nb * 32 + r;
        const float pw = perm_w[ent];
        atomicAdd(o, pw * acc[mt][0][i]);
        atomicAdd(o + 32, pw * acc[mt][1][i]);
      } else if constexpr (EPI == EPI_ROWS) {
        bf16* y = Y + (int64_t)ent * ldy + nb * 32 + r;
        const float pw = perm_w[ent];
        y[0] = (bf16)(pw * acc[mt][0][i]);
        y[32] = (bf16)(pw * acc[mt][1][i]);
      } else if constexpr (EPI == EPI_RELU2) {
        bf16* y = Y + (int64_t)ent * ldy + nb * 32 + r;
        const float a = fmaxf(acc[mt][0][i], 0.f), b = fmaxf(acc[mt][1][i], 0.f);
        y[0] = (bf16)(a * a);
        y[32] = (bf16)(b * b);
      } else {
        float g = acc[mt][0][i], u = acc[mt][1][i], al = 1.0f;
        if (glu_limit > 0.f) {   // (uniform) the clamped form
          g = fminf(g, glu_limit);
          u = fminf(fmaxf(u, -glu_limit), glu_limit) + 1.0f;
          al = glu_alpha;
        }
        Y[(int64_t)ent * ldy + (nb >> 1) * 32 + r] = (bf16)(times_sigmoid(g, al * g) * u);
      }
    }
}

// ---- the same on 256 x 256 tiles through a ring in LDS ---------------------------------------------------------------
// Four waves of 128 x 128 (ring.h; one workgroup per CU): an operand byte read from LDS feeds four products instead of the two of
// the kernel above, and a byte from the cache twice as many. Results
// leave in 16-byte pieces. An expert's last rows go on a tile of 64 or 128 rows where they fit one (the weights' way is then what it
// takes, a third of a whole tile). What bounds it: the card lowers its clock to 1.9 - 2.0 GHz under these products, and the last
// round of the chip.
// Measured, us, stages of 32 and 64 bytes of a row a store / units of 64 and results in whole cache lines (random routing
// and values): 32768 entries of 16 experts, 4096 -> 5376 relu2 1132 / 1077, 5376 -> 4096 rows 1123 / 1084; 3800 of 8, 4096 -> 2 x 14336 glu 750 /
// 732, 14336 -> 4096 rows 360 / 350, combined 382 / 375; 5386 of 8, 4096 -> 2 x 4608 glu 366 / 353, 4608 -> 4096 rows 196 / 188, combined 243 / 233.
struct RingArgs {
  const bf16* X;
  int64_t ldx;
  const bf16x8* Wt;
  int N, K;
  const int* perm_tok;
  const float* perm_w;
  bf16* Y;
  int64_t ldy;
  float* out;
  int64_t ldo;
  float glu_limit, glu_alpha;
};

// rows (at most 32 MT) entries from seg0 on of expert e, 256 columns from 256 nt on
template <int MT, bool GATHER, int EPI>
__device__ __forceinline__ void ring_tile(const RingArgs& A, char* smem, int e, int seg0, int rows, int nt) {
  using R = ring::Ring<MT, 8, EPI != EPI_COMBINE>;   // (sums added to memory: lanes along the columns of a row)
  const int N = A.N, K = A.K;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, q = lane >> 4;
  const int nb = nt * 8 + 4 * (w & 1);             // this wave's first 32-column tile (N is a multiple of 128)
  unsigned xo[R::PX], wo[R::WR];
#pragma unroll
  for (int u = 0; u < R::PX; ++u) {
    const int row = R::xrow(w, u, lane), m = min(row, rows - 1);   // rows past the segment reload a valid row, never stored
    const unsigned at = GATHER ? (unsigned)A.perm_tok[seg0 + m] : (unsigned)m;
    xo[u] = at * (unsigned)(A.ldx * 2) + R::xbyte(row, u, lane);
  }
#pragma unroll
  for (int u = 0; u < R::WR; ++u)                  // (tiles past N reload the last, never stored)
    wo[u] = (unsigned)(min(nt * 8 + R::wtile(w, u), (N >> 5) - 1) * (K >> 4) + R::wblock(w, u)) * 1024u;
  ring::f32x4v acc[MT][8];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < 8; ++b) acc[a][b] = ring::f32x4v{0.f, 0.f, 0.f, 0.f};
  R::multiply(acc, smem, R::xbuffer(GATHER ? A.X : A.X + (int64_t)seg0 * A.ldx), xo,
              ring::buffer(A.Wt + (int64_t)e * (N >> 5) * (K >> 4) * 64), R::wlane(lane), wo, K / R::BK, lane, w);
  if (nb >= (N >> 5)) return;
  if constexpr (EPI == EPI_COMBINE) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = 16 * (MT * (w >> 1) + mt) + 4 * q + i;
        if (m >= rows) continue;
        const float pw = A.perm_w[seg0 + m];
        float* o = A.out + (int64_t)A.perm_tok[seg0 + m] * A.ldo + nb * 32 + r;
#pragma unroll
        for (int j = 0; j < 8; ++j) atomicAdd(o + 16 * j, pw * acc[mt][j][i]);
      }
  } else {
    bf16* const y = A.Y + (int64_t)seg0 * A.ldy + (EPI == EPI_GLU ? nb * 16 : nb * 32);
    const int tiles = EPI == EPI_GLU ? ((N >> 5) - nb) / 2 : (N >> 5) - nb;
    float pw[MT];
    if constexpr (EPI == EPI_ROWS) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) pw[mt] = A.perm_w[seg0 + min(16 * (MT * (w >> 1) + mt) + r, rows - 1)];
    }
    auto value = [&](auto mc, auto c, int i) {
      constexpr int mt = decltype(mc)::value, t = decltype(c)::value * (EPI == EPI_GLU ? 2 : 1);
      const float v = acc[mt][2 * t + (i >> 2)][i & 3];
      if constexpr (EPI == EPI_ROWS) {
        return pw[mt] * v;
      } else if constexpr (EPI == EPI_RELU2) {
        const float a = fmaxf(v, 0.f);
        return a * a;
      } else {                                       // tiles of 32: gate, up, gate, up
        float g = v, u = acc[mt][(2 * t + 2 + (i >> 2)) & 7][i & 3], al = 1.0f;
        if (A.glu_limit > 0.f) {                     // (uniform) the clamped form
          g = fminf(g, A.glu_limit);
          u = fminf(fmaxf(u, -A.glu_limit), A.glu_limit) + 1.0f;
          al = A.glu_alpha;
        }
        return times_sigmoid(g, al * g) * u;
      }
    };
    R::template rows_bf16<EPI == EPI_GLU ? 2 : 4>(y, A.ldy, rows, tiles, lane, w, value);
  }
}

template <bool GATHER, int EPI>
__global__ __launch_bounds__(256, 1) void grouped_ring_kernel(const bf16* __restrict__ X, int64_t ldx,
                                                              const bf16x8* __restrict__ Wt, int E, int N, int K,
                                                              const int* __restrict__ perm_tok,
                                                              const float* __restrict__ perm_w,
                                                              const int* __restrict__ expert_off,
                                                              bf16* __restrict__ Y, int64_t ldy,
                                                              float* __restrict__ out, int64_t ldo, float glu_limit,
                                                              float glu_alpha) {
  constexpr int BM = ring::Ring<8, 8, true>::BM;
  __shared__ __attribute__((aligned(1024))) char smem[ring::Ring<8, 8, true>::LDS];
  int e, rt, nt;
  if (!find_item(expert_off, E, (N + 255) / 256, BM, e, rt, nt)) return;   // (uniform)
  const int seg0 = expert_off[e] + rt * BM, rows = min(BM, expert_off[e + 1] - seg0);
  const RingArgs A{X, ldx, Wt, N, K, perm_tok, perm_w, Y, ldy, out, ldo, glu_limit, glu_alpha};
  // an expert's last rows on a lower tile where they fit one: the weights' way is then what it takes, a third of a whole tile
  // (22 rows an expert, us, whole / low tile of the combined product: 8 experts 2304 -> 2048 46 / 22, 4608 -> 4096 85 / 64, 64 of 768 -> 2048 50 / 40)
  if (rows > 224) ring_tile<8, GATHER, EPI>(A, smem, e, seg0, rows, nt);
  else if (rows > 192) ring_tile<7, GATHER, EPI>(A, smem, e, seg0, rows, nt);
  else if (rows > 160) ring_tile<6, GATHER, EPI>(A, smem, e, seg0, rows, nt);
  else if (rows > 128) ring_tile<5, GATHER, EPI>(A, smem, e, seg0, rows, nt);
  else if (rows > 64) ring_tile<4, GATHER, EPI>(A, smem, e, seg0, rows, nt);
  else ring_tile<2, GATHER, EPI>(A, smem, e, seg0, rows, nt);
}

// ---- stable sort by expert --------------------------------------------------------------------------------------------
constexpr int SORT_MAXE = 512;

// lanes of the wave whose (valid) entry has this lane's expert
__device__ __forceinline__ unsigned long long same_expert(int e, bool valid, int bits) {
  unsigned long long m = __ballot(valid);
  for (int b = 0; b < bits; ++b) {
    const unsigned long long s = __ballot((e >> b) & 1);
    m &= ((e >> b) & 1) ? s : ~s;
  }
  return m;
}

__global__ __launch_bounds__(SORT_NT) void moe_sort_few_kernel(const float* __restrict__ topk_w, const int* __restrict__ topk_e,
                                                               int n, int k, int E, int bits, int bm,
                                                               int* __restrict__ perm_tok, float* __restrict__ perm_w,
                                                               int* __restrict__ expert_off, int* __restrict__ tile_off,
                                                               int* __restrict__ inv, const int* __restrict__ counts, int parts,
                                                               float* __restrict__ zero, int64_t nzero) {
  __shared__ int cnt[SORT_W][64];
  if ((int)blockIdx.x >= parts) {
    clear(zero, nzero, blockIdx.x - parts, gridDim.x - parts);
    return;
  }
  const int lo = parts > 1 ? blockIdx.x * SORT_PART : 0, hi = parts > 1 ? min(n, lo + SORT_PART) : n;
  sort_few_experts(topk_w, topk_e, lo, hi, k, E, bits, bm, perm_tok, perm_w, expert_off, tile_off, inv, counts, blockIdx.x,
                   parts, cnt);
}

// how many of the part's entries go to expert `lane`
__global__ __launch_bounds__(SORT_NT) void moe_sort_count_kernel(const int* __restrict__ topk_e, int n, int E, int bits,
                                                                 int* __restrict__ counts) {
  __shared__ int cnt[SORT_W][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, lo = blockIdx.x * SORT_PART;
  const int c = sort_count(topk_e, sort_stretch(lo, min(n, lo + SORT_PART), w), bits);
  cnt[w][lane] = lane < E ? c : 0;
  __syncthreads();
  if (w > 0) return;
  int tot = 0;
#pragma unroll
  for (int i = 0; i < SORT_W; ++i) tot += cnt[i][lane];
  counts[64 * blockIdx.x + lane] = tot;
}

// more experts: a counter in LDS per wave and expert
__global__ __launch_bounds__(SORT_NT) void moe_sort_kernel(const float* __restrict__ topk_w,
                                                           const int* __restrict__ topk_e, int n, int k, int E, int bits,
                                                           int bm, int* __restrict__ perm_tok,
                                                           float* __restrict__ perm_w, int* __restrict__ expert_off,
                                                           int* __restrict__ tile_off, int* __restrict__ inv) {
  __shared__ int cnt[SORT_W][SORT_MAXE];
  __shared__ int sum[2][SORT_W];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  for (int i = tid; i < SORT_W * E; i += SORT_NT) cnt[i / E][i % E] = 0;
  const int per = ((n + SORT_W - 1) / SORT_W + 63) / 64 * 64;   // a wave's stretch of the entries
  const int i0 = w * per, i1 = min(n, i0 + per);
  constexpr int PF = 8;
  __syncthreads();
  for (int b0 = i0; b0 < i1; b0 += 64 * PF) {
    int ev[PF];
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      const int i = b0 + 64 * p + lane;
      ev[p] = i < i1 ? topk_e[i] : 0;
    }
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      const bool valid = b0 + 64 * p + lane < i1;
      const unsigned long long m = same_expert(ev[p], valid, bits);
      if (valid && __builtin_ctzll(m) == lane) cnt[w][ev[p]] += __builtin_popcountll(m);
      __builtin_amdgcn_wave_barrier();
    }
  }
  __syncthreads();
  // per expert: counts -> exclusive sums over the waves; then exclusive sums over the experts (and their row tiles)
  int tot = 0;
  if (tid < E)
    for (int i = 0; i < SORT_W; ++i) {
      const int c = cnt[i][tid];
      cnt[i][tid] = tot;
      tot += c;
    }
  int a = tid < E ? tot : 0, t = tid < E ? (tot + bm - 1) / bm : 0;
  const int a0 = a;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(a, o, 64), v = __shfl_up(t, o, 64);
    if (lane >= o) {
      a += u;
      t += v;
    }
  }
  if (lane == 63) {
    sum[0][w] = a;
    sum[1][w] = t;
  }
  __syncthreads();
  for (int i = 0; i < w; ++i) {
    a += sum[0][i];
    t += sum[1][i];
  }
  if (tid < E) {
    expert_off[tid + 1] = a;
    tile_off[tid + 1] = t;
    for (int i = 0; i < SORT_W; ++i) cnt[i][tid] += a - a0;
    if (tid == 0) expert_off[0] = tile_off[0] = 0;
  }
  __syncthreads();
  for (int b0 = i0; b0 < i1; b0 += 64 * PF) {
    int ev[PF];
    float wv[PF];
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      const int i = b0 + 64 * p + lane;
      ev[p] = i < i1 ? topk_e[i] : 0;
      wv[p] = i < i1 ? topk_w[i] : 0.f;
    }
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      const int i = b0 + 64 * p + lane;
      const bool valid = i < i1;
      const unsigned long long m = same_expert(ev[p], valid, bits);
      const int at = valid ? cnt[w][ev[p]] : 0;
      __builtin_amdgcn_wave_barrier();             // (every lane has read before the first of an expert moves it on)
      if (valid) {
        const int pos = at + __builtin_popcountll(m & ((1ull << lane) - 1));
        perm_tok[pos] = i / k;
        perm_w[pos] = wv[p];
        if (inv != nullptr) inv[i] = pos;
        if (__builtin_ctzll(m) == lane) cnt[w][ev[p]] = at + __builtin_popcountll(m);
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// ---- narrow products --------------------------------------------------------------------------------------------------
constexpr int NR_ROWS = 16, NR_MAXN = 64, NR_MAXK = 16;
// waves of a workgroup and row length of their parts in LDS, TN: tiles of 16 weight rows
__host__ __device__ constexpr int nr_waves(int TN) { return TN <= 2 ? 16 : 8; }
__host__ __device__ constexpr int nr_ld(int TN) { return 16 * TN + 1; }
typedef float f32x4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4v mfma16(bf16x8 a, bf16x8 b, f32x4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// z[row][n] = x[row] . w[n] for 16 rows, the waves' parts summed through LDS -> z in part[0]. A wave's operands go through LDS of its
// own (ring), ST steps at a time, so that a load takes whole cache lines of a row: straight to the registers each took half a line of
// 16 rows, and what a CU takes in is what these products wait for. A row's 16-byte pieces are turned by its number, so that reading a
// fragment meets all banks. us, K = 4096, before / now: 16 columns 16 rows 9.0 / 4.3, 2048 9.6 / 6.0, 8192 18.8 / 14.8; 32 columns 12.4 /
// 5.4, 13.1 / 7.5, 27.1 / 18.2; 64 columns 20.6 / 8.4, 21.4 / 9.6, 40.8 / 24.3; the choice and sort of 16 rows, 16 experts 13.4 / 8.8.
constexpr int nr_steps(int TN) { return TN == 1 ? 4 : 2; }
constexpr int nr_ring(int TN) { return (1 + TN) * NR_ROWS * 64 * nr_steps(TN); }   // bytes a wave
typedef __attribute__((address_space(3))) void nr_lds_t;
template <int TN>
__device__ __forceinline__ void narrow_product(const bf16* __restrict__ x, int64_t xs, int64_t T, const bf16* __restrict__ wt,
                                               int N, int K, float (*part)[NR_ROWS][nr_ld(TN)]) {
  constexpr int ST = nr_steps(TN), ROW = 64 * ST, PCS = 4 * ST, TILE = NR_ROWS * ROW;   // bytes and 16-byte pieces of a row
  constexpr int NW = nr_waves(TN), PF = TN <= 2 ? 8 : 4;   // steps of a wave in a run
  __shared__ __attribute__((aligned(16))) unsigned char ring[NW * nr_ring(TN)];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, q = lane >> 4;
  unsigned char* const my = ring + w * nr_ring(TN);
  f32x4v acc[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) acc[j] = f32x4v{0.f, 0.f, 0.f, 0.f};
  const int ns = K / 32;
  for (int s0 = w * PF; s0 < ns; s0 += NW * PF) {
#pragma unroll
    for (int h = 0; h < PF; h += ST) {
#pragma unroll
      for (int i = 0; i < TILE / 1024; ++i) {
        const int row = i * (64 / PCS) + lane / PCS, at = min((s0 + h) * 32 + ((lane ^ row) & (PCS - 1)) * 8, K - 8);
        const int64_t t = min((int64_t)blockIdx.x * NR_ROWS + row, T - 1);
        __builtin_amdgcn_global_load_lds(x + t * xs + at, (nr_lds_t*)(my + i * 1024), 16, 0, 0);
#pragma unroll
        for (int j = 0; j < TN; ++j)
          __builtin_amdgcn_global_load_lds(wt + (int64_t)min(16 * j + row, N - 1) * K + at,
                                           (nr_lds_t*)(my + (1 + j) * TILE + i * 1024), 16, 0, 0);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      bf16x8 a[ST], b[ST][TN];
#pragma unroll
      for (int p = 0; p < ST; ++p) {
        const unsigned char* f = my + r * ROW + (((4 * p + q) ^ r) & (PCS - 1)) * 16;
        a[p] = *reinterpret_cast<const bf16x8*>(f);
        if (s0 + h + p >= ns) a[p] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < TN; ++j) b[p][j] = *reinterpret_cast<const bf16x8*>(f + (1 + j) * TILE);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (read, before the next loads land there)
#pragma unroll
      for (int p = 0; p < ST; ++p)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[j] = mfma16(a[p], b[p][j], acc[j]);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 15");
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) part[w][4 * q + i][16 * j + r] = acc[j][i];
  __syncthreads();
  for (int i = threadIdx.x; i < NR_ROWS * 16 * TN; i += 64 * NW) {
    const int row = i / (16 * TN), n = i - row * 16 * TN;
    float z = 0.f;
#pragma unroll
    for (int k = 0; k < NW; ++k) z += part[k][row][n];
    part[0][row][n] = z;
  }
  __syncthreads();
}

template <int TN>
__global__ __launch_bounds__(64 * nr_waves(TN)) void narrow_linear_kernel(const bf16* __restrict__ x, int64_t xs,
                                                            const bf16* __restrict__ wt, const float* __restrict__ bias,
                                                            int N, int K, float* __restrict__ out, int64_t os,
                                                            int64_t T) {
  __shared__ float part[nr_waves(TN)][NR_ROWS][nr_ld(TN)];
  narrow_product<TN>(x, xs, T, wt, N, K, part);
  for (int i = threadIdx.x; i < NR_ROWS * N; i += 64 * nr_waves(TN)) {
    const int row = i / N, n = i - row * N;
    const int64_t t = (int64_t)blockIdx.x * NR_ROWS + row;
    if (t < T) out[t * os + n] = part[0][row][n] + (bias != nullptr ? bias[n] : 0.f);
  }
}

// lane exchange within 16 lanes: the neighbour, the pair's neighbour, the mirrored half, the mirrored 16
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <typename OP>
__device__ __forceinline__ float row16(float v, OP op) {
  v = op(v, dpp<0xB1>(v));
  v = op(v, dpp<0x4E>(v));
  v = op(v, dpp<0x141>(v));
  return op(v, dpp<0x140>(v));
}

// what a routing launch of up to NR_ROWS rows does beside: the stable sort of its choices by expert, and clearing the experts' sums
struct RouteSort {
  int bits, bm;
  int *perm_tok, *expert_off, *tile_off;
  float *perm_w, *zero;
  int64_t nzero;
};

// softmax over all N experts, the k largest (ties: the lower index), their scores as weights (norm: divided by their sum)
// times scale; lane = expert: up to 16 live in the first 16 lanes (the others run along), exchanges without LDS (1.3 us of 16 rows).
// SORT: one workgroup, with the sort (a launch of its own: 4.7 us of 16 rows) and, in further ones, the clearing
template <int TN, bool SORT>
__global__ __launch_bounds__(64 * nr_waves(TN)) void narrow_route_kernel(const bf16* __restrict__ x, int64_t xs,
                                                           const bf16* __restrict__ wt, int N, int K, int k, bool norm,
                                                           float scale, float* __restrict__ tw, int* __restrict__ te,
                                                           int64_t T, RouteSort so) {
  __shared__ float part[nr_waves(TN)][NR_ROWS][nr_ld(TN)];
  if (SORT && blockIdx.x > 0) {
    clear(so.zero, so.nzero, blockIdx.x - 1, gridDim.x - 1);
    return;
  }
  narrow_product<TN>(x, xs, T, wt, N, K, part);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll 1
  for (int row = w; row < NR_ROWS; row += nr_waves(TN)) {
    const int64_t t = (int64_t)blockIdx.x * NR_ROWS + row;
    if (t >= T) break;   // (uniform)
    const float z = lane < N ? part[0][row][lane] : -INFINITY;
    const float mx = TN == 1 ? row16(z, [](float a, float b) { return fmaxf(a, b); }) : wave_max(z);
    const float ex = lane < N ? expf(z - mx) : 0.f;
    const float s = ex / (TN == 1 ? row16(ex, [](float a, float b) { return a + b; }) : wave_sum(ex));
    float c = lane < N ? s : -1.f, mine = 0.f, sum = 0.f;
    int me = 0;
    for (int j = 0; j < k; ++j) {
      float bv = c;
      int bi = lane;
      auto take = [&](float ov, int oi) {
        if (ov > bv || (ov == bv && oi < bi)) {
          bv = ov;
          bi = oi;
        }
      };
      if constexpr (TN == 1) {
        take(dpp<0xB1>(bv), __float_as_int(dpp<0xB1>(__int_as_float(bi))));
        take(dpp<0x4E>(bv), __float_as_int(dpp<0x4E>(__int_as_float(bi))));
        take(dpp<0x141>(bv), __float_as_int(dpp<0x141>(__int_as_float(bi))));
        take(dpp<0x140>(bv), __float_as_int(dpp<0x140>(__int_as_float(bi))));
      } else {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
          const float ov = __shfl_xor(bv, o, 64);
          take(ov, __shfl_xor(bi, o, 64));
        }
      }
      if (lane == j) {
        mine = bv;
        me = bi;
      }
      if (lane == bi) c = -1.f;
      sum += bv;
    }
    if (lane < k) {
      tw[t * k + lane] = (norm ? mine / sum : mine) * scale;
      te[t * k + lane] = me;
    }
  }
  if constexpr (SORT) {
    static_assert(nr_waves(TN) == SORT_W, "the sort's waves");
    __shared__ int cnt[SORT_W][64];
    __syncthreads();   // (the sort reads what other threads of the workgroup wrote)
    sort_few_experts(tw, te, 0, (int)T * k, k, N, so.bits, so.bm, so.perm_tok, so.perm_w, so.expert_off, so.tile_off, nullptr, nullptr,
                     0, 1, cnt);
  }
}

}  // namespace mw
}  // namespace kafka

using namespace kafka;
using namespace kafka::mw;

extern "C" {

int kafka_moe_sort_max_e() { return SORT_MAXE; }

// workgroups of a sort (its scratch: 64 counts each): one up to 4096 entries, where a second launch costs what it saves
int kafka_moe_sort_parts(int n, int E) { return E > 64 || n <= 2 * SORT_PART ? 1 : (n + SORT_PART - 1) / SORT_PART; }

// zero: nzero 16-byte pieces that the launch clears (up to 64 experts)
hipError_t kafka_launch_moe_sort(const float* topk_w, const int* topk_e, int n, int k, int E, int bm, int* perm_tok,
                                 float* perm_w, int* expert_off, int* tile_off, int* inv, int* counts, float* zero, int64_t nzero,
                                 hipStream_t st) {
  if (n < 1) return hipSuccess;
  if (E < 1 || (zero != nullptr && E > 64) || E > SORT_MAXE || k < 1 || bm < 1) return hipErrorInvalidValue;
  int bits = 0;
  while ((1 << bits) < E) ++bits;
  if (E > 64) {
    moe_sort_kernel<<<1, SORT_NT, 0, st>>>(topk_w, topk_e, n, k, E, bits, bm, perm_tok, perm_w, expert_off, tile_off, inv);
    return hipGetLastError();
  }
  const int parts = counts != nullptr ? kafka_moe_sort_parts(n, E) : 1;
  if (parts > 1) moe_sort_count_kernel<<<parts, SORT_NT, 0, st>>>(topk_e, n, E, bits, counts);
  moe_sort_few_kernel<<<parts + (zero != nullptr ? clear_blocks(nzero) : 0), SORT_NT, 0, st>>>(
      topk_w, topk_e, n, k, E, bits, bm, perm_tok, perm_w, expert_off, tile_off, inv, counts, parts, zero, nzero);
  return hipGetLastError();
}

// epi: 0 gate_up -> silu(gate) * up (or clamped) into Y [n_ent][N / 2], 1 relu squared into Y [n_ent][N], 2 combine into
// out [T][N], 3 weighted rows into Y [n_ent][N]
hipError_t kafka_launch_grouped_wide(const bf16* X, int64_t ldx, const bf16* Wt, int E, int N, int K,
                                     const int* perm_tok, const float* perm_w, const int* expert_off, int n_ent,
                                     int gather, int epi, bf16* Y, int64_t ldy, float* out, int64_t ldo,
                                     float glu_limit, float glu_alpha, int bm, int64_t xrows, hipStream_t st) {
  if (n_ent < 1 || E < 1) return hipSuccess;
  // what the ring kernel addresses with 32 bits (all rows of X where they are gathered, a tile's otherwise, and an expert's weights)
  // and stores in 16-byte pieces
  const bool ring_ok = N % 128 == 0 && (gather ? xrows : 256) * ldx * 2 < (int64_t)0xffff0000 &&
                       (int64_t)N * K * 2 < (int64_t)0xffff0000 &&
                       (epi == EPI_COMBINE || (ldy % 8 == 0 && reinterpret_cast<uintptr_t>(Y) % 16 == 0));
  if (bm == 0) {
    // Which tiles, from the mean rows r of an expert. Few rows: the ring kernel's low tiles, up to 96 rows (an expert of more than 128
    // takes a whole tile) in the first product and 128 in the second. us, 128-row kernel / ring: 8 experts 2048 -> 2 x 2304 40 rows 37 / 27,
    // 90 40 / 31, 110 42 / 50; 4096 -> 2 x 4608 40 rows 147 / 143, 90 152 / 156, 110 150 / 182; 4608 -> 4096 rows 77 / 67, 95 / 83 combined, 110 87 / 88;
    // 16 experts 1536 -> 4096 combined 40 rows 42 / 37, 110 72 / 57; 64 experts 4096 -> 2 x 1536 4 rows 269 / 264, 40 282 / 275, 1536 -> 4096 combined 40
    // rows 164 / 160, 110 249 / 220; 256 of them 4 rows 529 / 540, 40 672 / 673, 110 939 / 888. Very short rows of many tiles wait for a tile's start,
    // which two workgroups a CU hide: 256 experts 512 -> 2048 combined 4 rows 103 / 115, 22 125 / 136, 40 152 / 155; 16 experts 22 rows 19 / 12.
    // Beyond, by rounds: one is 256 tiles of 256 x 256 or 512 of 128 x 256, the same products; the ring
    // kernel does them 1.4 times as fast, but in whole rounds, the other one's last round thins out (a quarter of one on
    // average); a mean of 128 rows is 1.6 tiles of 128: 2048 -> 2 x 2304 280 rows 63 / 99, 600 rows 100 / 100, 1300 rows 218 / 208;
    // 4096 -> 2 x 14336 140 rows 454 / 428, 600 rows 1143 / 1025.
    const int64_t r = ((int64_t)n_ent + E - 1) / E, ct = (N + BN - 1) / BN * (int64_t)E;
    const bool low = r <= (epi == EPI_GLU || epi == EPI_RELU2 ? 96 : 128) && (K >= 768 || r >= 32 || ct <= 512);
    const double ring_rounds = (double)(((r + 255) / 256 * ct + 255) / 256) / 1.4;
    const double wide_rounds = (r <= 128 ? r / 128.0 + 0.6 : (double)((r + 127) / 128)) * ct / 512 + 0.25;
    bm = ring_ok && (low || ring_rounds < wide_rounds) ? 256 : 128;
  }
  if ((bm != 128 && bm != 256) || (bm == 256 && N % 128)) return hipErrorInvalidValue;
  if (bm == 256 && !ring_ok) bm = 128;
  if (N % 64 || K % (2 * BK) || N < 64 || K < 2 * BK || epi < 0 || epi > 3 || (epi == EPI_COMBINE) != (out != nullptr) ||
      (epi != EPI_COMBINE) != (Y != nullptr))
    return hipErrorInvalidValue;
  const int64_t items = ((int64_t)n_ent / bm + E) * ((N + BN - 1) / BN);   // an upper bound over all routings
  if (items > 0x0fffffff) return hipErrorInvalidValue;
  const unsigned grid = (unsigned)((items + 7) / 8 * 8);
  const auto* wt = reinterpret_cast<const bf16x8*>(Wt);
  auto a = [&](auto kern) {
    kern<<<grid, 256, 0, st>>>(X, ldx, wt, E, N, K, perm_tok, perm_w, expert_off, Y, ldy, out, ldo, glu_limit, glu_alpha);
  };
#define GW_BM(G, EPI) (bm == 256 ? a(grouped_ring_kernel<G, EPI>) : a(grouped_wide_kernel<G, EPI>))
#define GW_EPI(G)                                       \
  do {                                                  \
    if (epi == EPI_GLU) GW_BM(G, EPI_GLU);              \
    else if (epi == EPI_RELU2) GW_BM(G, EPI_RELU2);     \
    else if (epi == EPI_ROWS) GW_BM(G, EPI_ROWS);       \
    else GW_BM(G, EPI_COMBINE);                         \
  } while (0)
  if (gather) GW_EPI(true); else GW_EPI(false);
#undef GW_EPI
#undef GW_BM
  return hipGetLastError();
}

// bf16 rows and weights in 16-byte pieces, up to 64 weight rows
int kafka_narrow_ok(int N, int K, int64_t xs) { return N >= 1 && N <= NR_MAXN && K >= 32 && K % 32 == 0 && xs % 8 == 0; }
int kafka_narrow_max_k() { return NR_MAXK; }

hipError_t kafka_launch_narrow_linear(const bf16* x, int64_t xs, const bf16* w, const float* bias, int N, int K,
                                      float* out, int64_t os, int64_t T, hipStream_t st) {
  if (T <= 0) return hipSuccess;
  if (!kafka_narrow_ok(N, K, xs)) return hipErrorInvalidValue;
  const unsigned g = (unsigned)((T + NR_ROWS - 1) / NR_ROWS);
  auto a = [&](auto kern, int tn) { kern<<<g, 64 * nr_waves(tn), 0, st>>>(x, xs, w, bias, N, K, out, os, T); };
  if (N <= 16) a(narrow_linear_kernel<1>, 1);
  else if (N <= 32) a(narrow_linear_kernel<2>, 2);
  else if (N <= 48) a(narrow_linear_kernel<3>, 3);
  else a(narrow_linear_kernel<4>, 4);
  return hipGetLastError();
}

hipError_t kafka_launch_narrow_route(const bf16* x, int64_t xs, const bf16* w, int N, int K, int k, int norm, float scale,
                                     float* tw, int* te, int64_t T, hipStream_t st) {
  if (T <= 0) return hipSuccess;
  if (!kafka_narrow_ok(N, K, xs) || k < 1 || k > N || k > NR_MAXK) return hipErrorInvalidValue;
  const unsigned g = (unsigned)((T + NR_ROWS - 1) / NR_ROWS);
  auto a = [&](auto kern, int tn) {
    kern<<<g, 64 * nr_waves(tn), 0, st>>>(x, xs, w, N, K, k, norm != 0, scale, tw, te, T, RouteSort{});
  };
  if (N <= 16) a(narrow_route_kernel<1, false>, 1);
  else if (N <= 32) a(narrow_route_kernel<2, false>, 2);
  else if (N <= 48) a(narrow_route_kernel<3, false>, 3);
  else a(narrow_route_kernel<4, false>, 4);
  return hipGetLastError();
}

// rows and experts whose routing takes the sort along
int kafka_narrow_sort_ok(int N, int64_t T) { return N <= 32 && T <= NR_ROWS; }

hipError_t kafka_launch_narrow_route_sort(const bf16* x, int64_t xs, const bf16* w, int N, int K, int k, int norm, float scale,
                                          float* tw, int* te, int64_t T, int bm, int* perm_tok, float* perm_w, int* expert_off,
                                          int* tile_off, float* zero, int64_t nzero, hipStream_t st) {
  if (T <= 0) return hipSuccess;
  if (!kafka_narrow_ok(N, K, xs) || !kafka_narrow_sort_ok(N, T) || k < 1 || k > N || k > NR_MAXK || bm < 1) return hipErrorInvalidValue;
  RouteSort so{0, bm, perm_tok, expert_off, tile_off, perm_w, zero, nzero};
  while ((1 << so.bits) < N) ++so.bits;
  const unsigned g = 1 + (zero != nullptr ? clear_blocks(nzero) : 0);
  auto a = [&](auto kern) { kern<<<g, SORT_NT, 0, st>>>(x, xs, w, N, K, k, norm != 0, scale, tw, te, T, so); };
  if (N <= 16) a(narrow_route_kernel<1, true>);
  else a(narrow_route_kernel<2, true>);
  return hipGetLastError();
}

}  // extern "C"
