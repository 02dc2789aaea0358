// Tile attention v3 for gfx950: the cascade prefix pass (all decode rows of a batch against the shared system
// prompt's KV, `shared_prefix_decode_attention`) and chunked / causal prefill
// (`prefill_flash_attention`). Same work items, page layouts and outputs as attn_prefill_kernel (attention.hip);
// selected as tile variant 3 (ops.tile_rows(3) = 256 rows).
//
// Structure (one workgroup = 4 or 8 waves, two waves per SIMD, 128 or 256 query rows of one KV head):
//   * each wave owns 32 query rows (one 32-row MFMA block). A wave is a pipeline over 64-key tiles (4 pages): between the products
//     of the next tile's keys stand the exponentials of this one, between the products of this one's values the rest of
//     them and the next one's maxima, each product behind the LDS reads of the eight fragments after it. Waves of a SIMD
//     are mostly at the same place, so what stood one after the other in a wave (products, then softmax, then products,
//     reads in front of each) did so on the SIMD. What bounds it now: LDS, 32 KB of fragments a wave and tile (8 waves, 4096
//     rows of 32 heads against 8192 keys, 497 us: without the reads 389, without the exponentials 480, without the
//     copies 464), and the clock that the card holds. (64 rows a wave on one wave per SIMD halve the reads, but 256 + 256
//     registers did not hold it without scratch in the loop: 574 us.);
//   * K/V arrive by LDS-DMA (1 KiB per wave-instruction), 16 KB each per tile, into 2 or 3 slots for each: the keys run a
//     tile ahead of the values, and both slots that a step has read are filled again in its middle, behind its one counted
//     `s_waitcnt vmcnt` and one `s_barrier`;
//   * the DMA destination is lane-linear, so layouts are chosen on the SOURCE side: a K page (plane-major, see
//     rope_kv.hip) is copied verbatim — its plane-major order already makes the A-fragment reads of a 16-lane
//     ds_read_b128 group hit 16 distinct bank slots; the V^T page is copied with the 16-B halves of rows 8..15 of
//     every 16-row group swapped (source lane permutation L ^ ((L >> 4) & 1)), which makes the V^T fragment reads
//     conflict-free too (linear destination, permuted source, same permutation on the read);
//   * softmax in the S^T layout (lane = query column: row max / sum are lane-local plus one permlane32 swap) with a
//     deferred rescale (T13): O and l are rescaled only when some row's max grew by more than 2^THR, so the 64-wide
//     O rescale almost never runs.
#pragma once
#include "common.h"

#include <type_traits>

namespace kafka {

namespace tile3 {
constexpr int PAGE = 16;
constexpr int D = 128;
constexpr int TK = 64;                  // keys per tile (4 pages)
constexpr int KBYTES = TK * D * 2;      // K part of a ring slot
constexpr int SLOT = 2 * KBYTES;        // K + V
constexpr int MAXPG = 2048;             // page ids of an item's key range staged in LDS
template <int NSLOT>
constexpr int lds_bytes() { return NSLOT * SLOT + MAXPG * 4 + 64; }
constexpr float THR = 24.f;             // deferred-rescale threshold (log2 domain): P <= 2^THR, fp32-safe
}  // namespace tile3

struct TileItem {
  int q_start, q_count, bt_row, kv_lo, kv_hi, split, alt, pad1;
};

// Second partial buffer of a launch (fp32 [rows, Hq, S, D] + lse [rows, Hq, S]) for the items flagged `alt`: the
// cascade's prefix pass also serves the new-turn prefill rows of the step, whose prefix partials join their own
// suffix tiles' partials (merged by attn_merge) instead of the decode rows' bf16 slots. Row = token - tok_off.
struct AltPart {
  float* part = nullptr;
  float* lse = nullptr;
  int S = 0;
  int tok_off = 0;
};

typedef __attribute__((address_space(3))) void lds_void_t;

// N pieces of 1 KiB from g on (uniform; lane_bytes: this lane's 16 bytes of a piece) to lds on. Buffer loads: the immediate moves both sides, and
// the compiler knows that they leave the waits for LDS reads alone (behind global_load_lds, a FLAT form, it waits for every read there is)
template <int N, int AUX, int C = 0>
__device__ __forceinline__ void dma_pieces(const bf16* g, int lane_bytes, char* lds) {
  if constexpr (C < N) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(buf_rsrc(g), (lds_void_t*)lds, 16, lane_bytes, 0, 1024 * C, AUX);
    dma_pieces<N, AUX, C + 1>(g, lane_bytes, lds);
  }
}

// max without fmaxf's NaN-quieting: IEEE-mode v_max_f32 needs each MFMA result canonicalised first (a v_max x, x
// per value: 3 VALU ops per pair of scores); llvm.maximum lowers to gfx950's v_maximum3_f32, 3 inputs per op, no
// canonicalisation (it propagates NaN instead of dropping it: a NaN score poisons its row either way)
__device__ __forceinline__ float t3_max(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float t3_xor32_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return t3_max(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float t3_xor32_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <int N>
__device__ __forceinline__ void t3_wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// raw barrier, opaque to the compiler's memory model: no vmcnt(0) drain of the DMAs in flight (a __syncthreads()
// would emit one), and no LDS access is moved across it
__device__ __forceinline__ void t3_barrier() { asm volatile("s_barrier" ::: "memory"); }

// diagnostic-build stamp (ABL == 8): the 100 MHz constant clock, comparable across CUs and XCDs
__device__ __forceinline__ uint64_t t3_rt() {
  uint64_t t;
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_memrealtime %0\n\ts_waitcnt lgkmcnt(0)" : "=s"(t)::"memory");
  __builtin_amdgcn_sched_barrier(0);
  return t;
}

// s_waitcnt vmcnt(n * DPT) for a wave-uniform n in [0, 2] (the count is an immediate)
template <int DPT>
__device__ __forceinline__ void t3_wait_tiles(int n) {
  if (n >= 2)
    t3_wait_vmcnt<2 * DPT>();
  else if (n == 1)
    t3_wait_vmcnt<DPT>();
  else
    t3_wait_vmcnt<0>();
}

// ABL = 8 (diagnostic build, KAFKA_TILE_ABL=8, benchmarks/attn_tile_stamps.py): workgroup phase stamps on the 100 MHz
// clock, every launch in the cascade's form (8 waves, three slots); the full kernel runs and lse_part is overwritten with
// u64 [entry, prologue done, first tile landed, loop done, epilogue done, 0, 0, 0] per workgroup blockIdx.y * Hkv + blockIdx.x.
// PST = 1: the bf16 prefix partials are stored sc1 (16-B stores whose lines leave this XCD's L2: the reader, the
// suffix decode's merge, runs on any XCD, and the launch ends with fewer dirty lines to write back)
// PST = 2: as 1, and fp32 partials and every lse as well: a workgroup of the same launch reads them (attn_mixed.hip)
// One work item on key/value head kvh: NW waves (32 NW query rows), NSLOT ring slots of smem (lds_bytes<NSLOT>()). Every thread of
// the workgroup calls it with the same arguments.
template <int ABL, int KVAUX, int PST, int NW, int NSLOT>
__device__ __forceinline__ void tile_item(char* smem, const TileItem it, int kvh, const bf16* __restrict__ q,
                                          int64_t q_stride, const bf16* __restrict__ k_cache,
                                          const bf16* __restrict__ v_cache, int Hkv, int G,
                                          const int* __restrict__ block_tables, int bt_stride,
                                          const int* __restrict__ q_limit, bf16* __restrict__ out, int64_t out_stride,
                                          float* __restrict__ out_part, float* __restrict__ lse_part, int S_total,
                                          float scale_log2, int part_bf16, const AltPart& ap) {
  using namespace tile3;
  constexpr int RB = 1;                   // 32-row MFMA blocks per wave
  constexpr int DPT = 32 / NW;            // LDS-DMA instructions per wave per tile (16 K + 16 V pieces per tile)
  int* s_pages = reinterpret_cast<int*>(smem + NSLOT * SLOT);
  int* s_hi = s_pages + MAXPG;

  uint64_t ph[5] = {0, 0, 0, 0, 0};
  if constexpr (ABL == 8) ph[0] = t3_rt();
  // an item flagged alt without an alt buffer (host bug) would write row B + q of the main buffer, past its end:
  // dropped (workgroup-uniform), as the decode kernel drops malformed items
  if (it.alt != 0 && ap.part == nullptr) return;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, h = lane >> 5;
  const int Hq = Hkv * G;

  // ---- rows of this wave: R = 64 w + 32 rb + r -> token R / G, head kvh G + R % G
  int token[RB], head[RB], limit[RB];
  bool valid[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int R = 32 * RB * w + 32 * rb + r;
    const int tok = R / G;
    valid[rb] = tok < it.q_count;
    token[rb] = it.q_start + tok;
    head[rb] = kvh * G + R % G;
  }
  // prologue loads that depend only on the work item go out together (one round trip): the item's page ids and the
  // causal limits; Q fragments (B operand of S^T = K . Q^T: lane (r, h) holds Q[row r][16 kk + 8 h + j]) follow the
  // first DMAs
  const int lo0 = it.kv_lo;
  const int pg00 = (lo0 & ~63) >> 4;
  const int npg_all0 = ((it.kv_hi + 15) >> 4) - pg00;
  const int npg0 = min(npg_all0, 2048);
  const int* bt0 = block_tables + (int64_t)it.bt_row * bt_stride;
  constexpr int PPT = MAXPG / (64 * NW);  // page ids per thread
  int pgv[PPT];
#pragma unroll
  for (int k = 0; k < PPT; ++k) {
    const int i = tid + k * (64 * NW);
    pgv[k] = i < npg0 ? bt0[pg00 + i] : 0;
  }
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) limit[rb] = valid[rb] ? q_limit[token[rb]] : -1;
  bf16x8 qf[RB][D / 16];
  auto load_q = [&]() {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const bf16* qrow = q + (int64_t)token[rb] * q_stride + (int64_t)head[rb] * D + 8 * h;
#pragma unroll
      for (int kk = 0; kk < D / 16; ++kk) {
        if (valid[rb]) {
          qf[rb][kk] = load_bf16x8(qrow + 16 * kk);
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) qf[rb][kk][j] = (bf16)0.f;
        }
      }
    }
  };
  // (Q fragments are loaded after the first K/V tiles' DMAs are issued: those are the critical path — Q loads issued
  // ahead of them delayed the first tile, -0.6 % on the headline, profiles/r04/bench_ab_tile_prologue.jsonl)
  // per-block wave-uniform bounds: keys past hi_b are masked for every row of the block, keys <= wmin_b for none
  int hi_b[2], wmin_b[2];  // (RB == 1: block 1 mirrors block 0)
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    int mx = limit[rb], mn = valid[rb] ? limit[rb] : 0x7fffffff;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      mx = max(mx, __shfl_xor(mx, o, 64));
      mn = min(mn, __shfl_xor(mn, o, 64));
    }
    hi_b[rb] = min(it.kv_hi, mx + 1);
    wmin_b[rb] = mn;
  }
  if constexpr (RB == 1) {
    hi_b[1] = hi_b[0];
    wmin_b[1] = wmin_b[0];
  }
  // (a block without valid rows does not make tiles edges: its rows are never written)
  const int hi_e = min(hi_b[0] > 0 ? hi_b[0] : 0x7fffffff, hi_b[1] > 0 ? hi_b[1] : 0x7fffffff);
  const int lo = it.kv_lo;
  const int base = lo & ~(TK - 1);
  const int pg0 = base >> 4;
  const int npg_all = ((it.kv_hi + 15) >> 4) - pg0;
  const int npg = min(npg_all, MAXPG);
#pragma unroll
  for (int k = 0; k < PPT; ++k) {
    const int i = tid + k * (64 * NW);
    if (i < npg) s_pages[i] = pgv[k];
  }
  if (lane == 0) s_hi[w] = max(hi_b[0], hi_b[1]);
  __syncthreads();
  if constexpr (ABL == 8) ph[1] = t3_rt();
  int hi_wg = s_hi[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) hi_wg = max(hi_wg, s_hi[i]);
  // (the host never builds an item spanning more than MAXPG pages; a violating item yields NaN rows)
  const bool fits = npg_all <= MAXPG;
  const int ntiles = (fits && hi_wg > lo) ? (hi_wg - base + TK - 1) / TK : 0;

  const int jf = (lo > base && ntiles > 0) ? 1 : 0;  // (= j0 below)
  auto tile_of = [&](int i) { return i < ntiles - jf ? i + jf : 0; };
  // ---- DMA: keys and values have NSLOT slots each; group g is the keys of processing index g (tile t(g)) and the values of g - 1, which are
  // needed a tile later: wave w copies page w of both
  const int pw = (w * 4) / NW, c0 = (w % (NW / 4)) * (DPT / 2);   // its page of the tile, its 1-KiB pieces of K and of V
  const int kl = 16 * lane, vl = 16 * (lane ^ ((lane >> 4) & 1));
  auto page_of = [&](int i) { return s_pages[min(4 * tile_of(min(i, ntiles - 1)) + pw, npg - 1)]; };
  auto issue = [&](int g, int kpage, int vpage) {
    char* const kd = smem + (g % NSLOT) * KBYTES + pw * 4096 + c0 * 1024;
    char* const vd = smem + (NSLOT + (g + NSLOT - 1) % NSLOT) * KBYTES + pw * 4096 + c0 * 1024;
    if (g < ntiles || g == 1) dma_pieces<DPT / 2, KVAUX>(k_cache + ((int64_t)kpage * Hkv + kvh) * (tile3::PAGE * D) + c0 * 512, kl, kd);
    if (g > 0) dma_pieces<DPT / 2, KVAUX>(v_cache + ((int64_t)vpage * Hkv + kvh) * (tile3::PAGE * D) + c0 * 512, vl, vd);
  };
  int last_page = 0;                                 // of the keys of the group that was issued last: the next one's values'
  if (ntiles > 0) {
    last_page = __builtin_amdgcn_readfirstlane(page_of(0));
    issue(0, last_page, 0);
  }
  load_q();                                          // (the first products take the rows and the first keys, no more)
  if (ntiles > 0) {
#pragma unroll
    for (int g = 1; g < NSLOT; ++g) {
      const int pg = __builtin_amdgcn_readfirstlane(page_of(g));
      if (g <= ntiles) issue(g, pg, last_page);
      last_page = pg;
    }
  }

  // Running state per row block: O^T accumulators; this lane's half of the row sums (of the rounded weights, as the products take them: two a
  // dot product; as products with ones they were an eighth of the matrix cores' work); the running max m (exp2 domain).
  // (Folding -m into the QK^T accumulator init would save the per-score FMA too, but needs Q prescaled by
  // scale * log2(e) in bf16: +0.4 % relative score error, 0.037 abs on a peaked row vs 0.02 tolerance — rejected.)
  f32x16 o[RB][D / 32];
  float m[RB], ls[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[rb][t][i] = 0.f;
    ls[rb] = 0.f;
    m[rb] = -INFINITY;
  }

  // Processing order: the interior tiles first, then the edge tiles (range ends, causal diagonal): online softmax does not care about key
  // order. Index i -> tile t(i): tiles j0 .. ntiles-1, then tile 0 when it starts below lo.
  const int j0 = (lo > base && ntiles > 0) ? 1 : 0;
  const int wmin_all = min(wmin_b[0], wmin_b[1]);
  const int clean_end = min(hi_e, wmin_all == 0x7fffffff ? 0x7fffffff : wmin_all + 1);  // keys below: no mask
  const int j_e = clean_end > base ? min(ntiles, (clean_end - base) / TK) : 0;
  const int n_int = max(0, j_e - j0);

  // The loop is a pipeline over tiles within the wave: step j multiplies the keys of tile j + 1 between the exponentials of tile j, then
  // the values of tile j between the rest of them and the maxima of tile j + 1. The eight fragments ahead of a product are on their way from LDS
  // (fr): 16 of keys (kb = f & 1, depth f >> 1), 16 of values (32 keys' half, 16 keys, 32 columns).
  const char* const Kl = smem + (r >> 4) * 4096 + (h * 16 + (r & 15)) * 16;                 // [slot][page 4][plane 16][key 16][16 B]
  const char* const Vl = smem + NSLOT * KBYTES + r * 32 + 16 * (h ^ ((r >> 3) & 1));        // [slot][page 4][d 128][2 x 16 B] (halves swapped)
  bf16x8 fr[8];
  f32x16 sa[RB][2], sb[RB][2];
  auto kfrag = [&](const char* k, int f) { return *reinterpret_cast<const bf16x8*>(k + (f & 1) * 8192 + (f >> 1) * 512); };
  auto vfrag = [&](const char* v, int f) { return *reinterpret_cast<const bf16x8*>(v + (f >> 2) * 4096 + (f & 3) * 1024); };
  auto kslot = [&](int i) { return Kl + (i % NSLOT) * KBYTES; };
  auto vslot = [&](int i) { return Vl + (i % NSLOT) * KBYTES; };
  auto mask = [&](f32x16(&s)[RB][2], int i) {        // wave-uniform per 32-key half: range edges and the causal diagonal
    const int key0 = base + TK * tile_of(i);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const int k0 = key0 + 32 * kb;
        if ((k0 < lo) | (k0 + 32 > hi_b[rb]) | (k0 + 31 > wmin_b[rb])) {
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const int key = k0 + (e & 3) + 8 * (e >> 2) + 4 * h;
            if (!((key >= lo) & (key < hi_b[rb]) & (key <= limit[rb]))) s[rb][kb][e] = -INFINITY;
          }
        }
      }
  };
  // deferred rescale, rare: only when a row's max passed m + THR (or at its first finite scores)
  auto rescale = [&](const float (&mx)[RB]) {
    float smax[RB];
    bool need = false;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      smax[rb] = t3_xor32_max(mx[rb]) * scale_log2;
      need = need | !(smax[rb] <= m[rb] + THR);
    }
    if (__any(need)) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const float mn = fmaxf(m[rb], smax[rb]);
        const float alpha = (mn == -INFINITY) ? 1.f : exp2f(m[rb] - mn);
#pragma unroll
        for (int t = 0; t < D / 32; ++t) o[rb][t] *= alpha;
        ls[rb] *= alpha;
        m[rb] = mn;
      }
    }
  };
  int next_page = 0;                                 // page of the keys of the group that is issued next, on its way from LDS
  // every wave has read the keys of tile j + 1 and the values of tile j, and group j + 2 has landed: their slots are filled again
  auto meet = [&](int j) {
    __builtin_amdgcn_s_waitcnt(0xC07F);              // lgkmcnt(0): this wave's reads of those slots
    t3_wait_tiles<DPT>(min(NSLOT - 2, max(0, ntiles - 1 - (j + 2))));
    t3_barrier();
    const int g = j + 1 + NSLOT;
    if (g <= ntiles) {
      const int pg = __builtin_amdgcn_readfirstlane(next_page);
      issue(g, pg, last_page);
      last_page = pg;
      next_page = page_of(g + 1);
    }
  };
  // step j: s the scores of tile j, sn those of the next one (unless LAST)
  auto tile_step = [&](auto last_c, int j, f32x16(&s)[RB][2], f32x16(&sn)[RB][2]) {
    constexpr bool LAST = decltype(last_c)::value;
    const f32x16 zero = {};
    const char *kc = kslot(j + 1), *vc = vslot(j);
    float mu[RB];
    bf16x8 pf[RB][2], pg[RB][2];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) mu[rb] = (m[rb] == -INFINITY) ? 0.f : m[rb];
    auto prob = [&](int rb, float x) { return (bf16)fast_exp2(fmaf(x, scale_log2, -mu[rb])); };
    auto add = [&](int rb, const bf16x8& p) {        // the row sums' share of eight weights
      const bf16x2 one = {(bf16)1.f, (bf16)1.f};
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        const bf16x2 two = {p[i], p[i + 1]};
        ls[rb] = __builtin_amdgcn_fdot2_f32_bf16(two, one, ls[rb], false);
      }
    };
    if constexpr (LAST) {
#pragma unroll
      for (int p = 0; p < 8; ++p) fr[p] = vfrag(vc, p);
#pragma unroll
      for (int p = 0; p < 16; ++p)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) pf[rb][p >> 3][p & 7] = prob(rb, s[rb][0][p]);
    } else {
#pragma unroll
      for (int p = 0; p < 16; ++p) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
          sn[rb][p & 1] = mfma32(fr[p & 7], qf[rb][p >> 1], p < 2 ? zero : sn[rb][p & 1]);
          pf[rb][p >> 3][p & 7] = prob(rb, s[rb][0][p]);
        }
        fr[p & 7] = p < 8 ? kfrag(kc, p + 8) : vfrag(vc, p - 8);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int p = 0; p < 8; ++p) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        o[rb][p & 3] = mfma32(fr[p], pf[rb][p >> 2], o[rb][p & 3]);
        pg[rb][p >> 2][2 * (p & 3)] = prob(rb, s[rb][1][2 * p]);
        pg[rb][p >> 2][2 * (p & 3) + 1] = prob(rb, s[rb][1][2 * p + 1]);
        if ((p & 3) == 0) add(rb, pf[rb][p >> 2]);
      }
      fr[p] = vfrag(vc, p + 8);
      __builtin_amdgcn_sched_barrier(0);
    }
    float ma[RB], mb[RB];
    const char* kn = kslot(j + 2);
    if constexpr (!LAST) {
      // (the compiler would move the exponentials to the products that take them)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) asm volatile("" : "+v"(pg[rb][0]), "+v"(pg[rb][1]));
      meet(j);
      if (j + 1 >= n_int) mask(sn, j + 1);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        ma[rb] = t3_max(sn[rb][0][0], sn[rb][1][0]);
        mb[rb] = t3_max(sn[rb][0][1], sn[rb][1][1]);
      }
    }
#pragma unroll
    for (int p = 0; p < 8; ++p) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        o[rb][p & 3] = mfma32(fr[p], pg[rb][p >> 2], o[rb][p & 3]);
        if (!LAST && p > 0) {
          ma[rb] = t3_max(t3_max(ma[rb], sn[rb][0][2 * p]), sn[rb][1][2 * p]);
          mb[rb] = t3_max(t3_max(mb[rb], sn[rb][0][2 * p + 1]), sn[rb][1][2 * p + 1]);
        }
        if ((p & 3) == 0) add(rb, pg[rb][p >> 2]);
      }
      if constexpr (!LAST) fr[p] = kfrag(kn, p);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!LAST) {
      float mx[RB];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) mx[rb] = t3_max(ma[rb], mb[rb]);
      rescale(mx);
    }
  };
  if (ntiles > 0) {
    t3_wait_vmcnt<DPT>();                            // (group 1 is whole whatever there is: its keys are the last ones' again where they are past them)
    t3_barrier();
    if constexpr (ABL == 8) ph[2] = t3_rt();
    next_page = page_of(NSLOT);
#pragma unroll
    for (int p = 0; p < 8; ++p) fr[p] = kfrag(Kl, p);
#pragma unroll
    for (int p = 0; p < 16; ++p) {
      const f32x16 zero = {};
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) sa[rb][p & 1] = mfma32(fr[p & 7], qf[rb][p >> 1], p < 2 ? zero : sa[rb][p & 1]);
      if (p < 8) fr[p] = kfrag(Kl, p + 8);
    }
    meet(-1);
#pragma unroll
    for (int p = 0; p < 8; ++p) fr[p] = kfrag(kslot(1), p);
    if (n_int < 1) mask(sa, 0);
    float mx[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      mx[rb] = t3_max(sa[rb][0][0], sa[rb][1][0]);
#pragma unroll
      for (int i = 1; i < 16; ++i) mx[rb] = t3_max(t3_max(mx[rb], sa[rb][0][i]), sa[rb][1][i]);
    }
    rescale(mx);
    int j = 0;
    for (; j + 2 < ntiles; j += 2) {
      tile_step(std::false_type{}, j, sa, sb);
      tile_step(std::false_type{}, j + 1, sb, sa);
    }
    if (j + 1 < ntiles) {
      tile_step(std::false_type{}, j, sa, sb);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        sa[rb][0] = sb[rb][0];
        sa[rb][1] = sb[rb][1];
      }
      ++j;
    }
    tile_step(std::true_type{}, j, sa, sb);
  }
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) ls[rb] = t3_xor32_sum(ls[rb]);

  if constexpr (ABL == 8) ph[3] = t3_rt();
  // ---- epilogue: through a per-wave LDS transpose (the keys' slots are idle: every wave has read the last ones before it passed the last
  // meeting, and nothing more is on its way there), so every store instruction writes whole 128-B lines
  const bool part = it.split >= 0;
  const bool alt = part && it.alt != 0 && ap.part != nullptr;  // (workgroup-uniform)
  float* const opart = alt ? ap.part : out_part;
  float* const lpart = alt ? ap.lse : lse_part;
  const int Sx = alt ? ap.S : S_total, toff = alt ? ap.tok_off : 0;
  const bool pbf = part_bf16 && !alt;
  char* slab = smem + w * (4096 * RB);
  const int cc = lane & 7;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    if (!__any(valid[rb])) continue;  // wave-uniform
    const float ll = fits ? ls[rb] : __builtin_nanf("");
    const float inv = ll > 0.f ? 1.f / ll : (fits ? 0.f : ll);
    if (ABL != 8 && part && valid[rb] && h == 0) {
      float* lp = lpart + ((int64_t)(token[rb] - toff) * Hq + head[rb]) * Sx + it.split;
      const float lv = ll > 0.f ? m[rb] + log2f(ll) : (fits ? -INFINITY : ll);
      if constexpr (PST == 2) __hip_atomic_store(lp, lv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else *lp = lv;
    }
    const int R0 = 32 * RB * w + 32 * rb;
    const int nvalid = it.q_count * G - R0;
    char* sl = slab + rb * 4096;
    auto flush = [&](int rd) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int row = (lane >> 3) + 8 * k;
        const f32x4 v = *reinterpret_cast<const f32x4*>(sl + row * 128 + 16 * (cc ^ (row & 7)));
        if (row < nvalid) {
          const int R2 = R0 + row, tok2 = it.q_start + R2 / G, head2 = kvh * G + R2 % G;
          f32x4* dst;
          if (PST && pbf) {
            float* d = reinterpret_cast<float*>(reinterpret_cast<bf16*>(out_part) +
                                                (((int64_t)tok2 * Hq + head2) * S_total + it.split) * D + 64 * rd + 8 * cc);
            store16_slab(d, v);  // (common.h: asm store + its hazard wait state)
            continue;
          }
          if (part && !pbf)
            dst = reinterpret_cast<f32x4*>(opart + (((int64_t)(tok2 - toff) * Hq + head2) * Sx + it.split) * D +
                                           32 * rd + 4 * cc);
          else if (part)  // bf16 partial (O / l in [-max|v|, max|v|]: half the bytes of the cascade round trip)
            dst = reinterpret_cast<f32x4*>(reinterpret_cast<bf16*>(out_part) +
                                           (((int64_t)tok2 * Hq + head2) * S_total + it.split) * D + 64 * rd + 8 * cc);
          else
            dst = reinterpret_cast<f32x4*>(out + (int64_t)tok2 * out_stride + (int64_t)head2 * D + 64 * rd + 8 * cc);
          if constexpr (PST == 2) store16_slab(reinterpret_cast<float*>(dst), v);
          else *dst = v;
        }
      }
    };
    if (part && !pbf) {
#pragma unroll
      for (int rd = 0; rd < 4; ++rd) {
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          const int c = 2 * i4 + h;
          const f32x4 v = {o[rb][rd][4 * i4] * inv, o[rb][rd][4 * i4 + 1] * inv, o[rb][rd][4 * i4 + 2] * inv,
                           o[rb][rd][4 * i4 + 3] * inv};
          *reinterpret_cast<f32x4*>(sl + r * 128 + 16 * (c ^ (r & 7))) = v;
        }
        flush(rd);
      }
    } else {
#pragma unroll
      for (int rd = 0; rd < 2; ++rd) {
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
          for (int i4 = 0; i4 < 4; ++i4) {
            bf16x4 v;
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) v[jj] = (bf16)(o[rb][2 * rd + tt][4 * i4 + jj] * inv);
            *reinterpret_cast<bf16x4*>(sl + r * 128 + 16 * ((4 * tt + i4) ^ (r & 7)) + 8 * h) = v;
          }
        flush(rd);
      }
    }
  }
  if constexpr (ABL == 8) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    ph[4] = t3_rt();
    if (tid == 0) {
      uint64_t* dst = reinterpret_cast<uint64_t*>(lse_part) + ((int64_t)blockIdx.y * Hkv + blockIdx.x) * 8;
#pragma unroll
      for (int k = 0; k < 5; ++k) dst[k] = ph[k];
    }
  }
}

}  // namespace kafka
