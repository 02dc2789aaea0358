// The cascade's prefix tiles and the decode pieces of a step in one launch (gfx950, bf16 pages).
//
// The prefix pass (query rows of many sequences against the keys that they share) is bound by the matrix cores and LDS, the
// decode pieces (every row's own keys) by memory: one after the other each leaves idle what the other waits for. Here a workgroup is either a
// tile of 128 query rows (attn_tile.h, four waves, two ring slots) or a decode piece (attn_decode.h), two workgroups a CU; the
// tiles come first in the grid, so that the first round of the chip is about one tile and one piece on every CU.
//
// Every tile and every piece leaves its partial (tiles bf16, or fp32 for a new turn's rows; pieces fp32; with their log-sum-exp) write-through
// and then counts itself in at each of its (row, kv head) counters. The last workgroups of the grid merge: each waits until its rows' counters
// have reached the number of their parts, reads these agent-coherently, writes the final rows and sets the counters back to zero. Workgroups are
// dispatched in the grid's order, so whatever they wait for is running or done when they start, and waits for nothing itself; the wait is
// bounded all the same: a row past it is not a number, here and in every launch on the same counters, whose parts of before may yet come.
// So counters are a step's own (or cleared before the launch). (Merged by whichever part comes last instead: a tile that comes last has up to 128 rows
// of heads to merge alone, 20 - 40 us; 64 rows of 1344 keys 82 -> 85 us, 30 rows 54 -> 77.)
//
// us of a layer's attention, tile and decode launch / this one (Llama-3-8B heads, 18000 shared keys; caches not resident): 64 rows of 1344
// keys 84 / 67, 96 of 900 99 / 75, 30 of 1344 53 / 47, 64 of 400 48 / 45, 64 of 5000 210 / 186. The first moves 370 MB: 5.5 TB/s, where the
// decode kernel alone reaches 6.4; the rest is the merges at its end (5 us) and tiles that go on beside the last pieces.
#include "attn_decode.h"
#include "attn_tile.h"

namespace kafka {

namespace mixed {
constexpr int NW = 4, NSLOT = 2, ROWS = 32 * NW;             // a tile's waves, ring slots, query rows
constexpr int TILE_LDS = tile3::lds_bytes<NSLOT>();
constexpr int MAXS = 64;                                     // parts of a row
constexpr int PRE = 16;                                      // row_parts: a row's parts, and above this bit those that tiles left in bf16
constexpr int LOST = -(1 << 30);                             // a counter whose row was given up: parts that come later leave it below zero
}  // namespace mixed

// a row's parts: [rows, Hq, S, 128] and lse [rows, Hq, S]
struct MixedParts {
  const float* part;
  const bf16* pre;     // the first npre of them, or nullptr
  const float* lse;
  int S;
};

// Final row at ``o`` of row x head ``row`` from its n parts, the first npre of them bf16, by 16 lanes of 8 dimensions. Everything it reads
// was written by other workgroups of this launch: agent-coherent loads, the first sixteen parts asked for beside the log-sum-exps.
__device__ __forceinline__ void mixed_merge_row(const MixedParts& m, int64_t row, int npre, int n, bf16* o) {
  constexpr int D = 128, U = 16;
  const int l = threadIdx.x & 15;
  const int64_t base = row * m.S;
  const auto prs = buf_rsrc(m.part), brs = buf_rsrc(m.pre);   // (both under 2 GiB: host-checked)
  f32x4 v[U], p[2][2];
  auto load_pre = [&](int s0) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s0 + u < npre) v[u] = load16_sc1(brs, (int)(((base + s0 + u) * D + 8 * l) * 2));
  };
  auto load_part = [&](int s0) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (s0 + u < n) p[u][h] = load16_sc1(prs, (int)(((base + s0 + u) * D + 8 * l + 4 * h) * 4));
  };
  float w[mixed::MAXS / 16];
  float mx = -INFINITY;
#pragma unroll
  for (int k = 0; k < mixed::MAXS / 16; ++k)
    w[k] = 16 * k + l < n ? __hip_atomic_load(m.lse + base + 16 * k + l, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : -INFINITY;
  load_pre(0);
  load_part(npre);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int k = 0; k < mixed::MAXS / 16; ++k) mx = t3_max(mx, w[k]);   // (a part that is not a number makes its row one)
#pragma unroll
  for (int x = 8; x > 0; x >>= 1) mx = t3_max(mx, __shfl_xor(mx, x, 16));
  float sum = 0.f;
#pragma unroll
  for (int k = 0; k < mixed::MAXS / 16; ++k) {
    w[k] = mx == -INFINITY ? 0.f : exp2f(w[k] - mx);
    sum += w[k];
  }
#pragma unroll
  for (int x = 8; x > 0; x >>= 1) sum += __shfl_xor(sum, x, 16);
  auto weight = [&](int s) {                         // of part s (the same for the 16 lanes)
    float x = w[0];
#pragma unroll
    for (int k = 1; k < mixed::MAXS / 16; ++k) x = (s >> 4) == k ? w[k] : x;
    return __shfl(x, s & 15, 16);
  };
  float acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = 0.f;
  for (int s0 = 0; s0 < npre;) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s0 + u < npre) {
        const float ws = weight(s0 + u);
        const bf16x8 x = __builtin_bit_cast(bf16x8, v[u]);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] += ws * (float)x[j];
      }
    s0 += U;
    if (s0 < npre) load_pre(s0);
  }
  for (int s0 = npre; s0 < n;) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (s0 + u < n) {
        const float ws = weight(s0 + u);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] += ws * p[u][j >> 2][j & 3];
      }
    s0 += 2;
    if (s0 < n) load_part(s0);
  }
  const float inv = sum > 0.f ? 1.f / sum : sum == 0.f ? 0.f : sum;
  bf16x8 r;
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = (bf16)(acc[j] * inv);
  store16_slab(reinterpret_cast<float*>(o + 8 * l), __builtin_bit_cast(f32x4, r));
}

// grid (Hkv, tiles + pieces + merges): the heads of an item are consecutive workgroups, dealt to different XCDs, as in the launches of
// their own
__global__ __launch_bounds__(256, 2) void attn_mixed_kernel(const TileItem* __restrict__ titems, int n_tiles,
                                                            const DecodeItem* __restrict__ ditems, int n_pieces,
                                                            const int* __restrict__ row_parts, int n_rows,
                                                            const bf16* __restrict__ q, int64_t q_stride,
                                                            const bf16* __restrict__ k_cache,
                                                            const bf16* __restrict__ v_cache, int Hkv, int G,
                                                            const int* __restrict__ block_tables, int bt_stride,
                                                            const int* __restrict__ q_limit, int B,
                                                            float* __restrict__ part, float* __restrict__ lse,
                                                            bf16* __restrict__ pre, int S_total, float scale_log2,
                                                            bf16* __restrict__ out, int64_t out_stride,
                                                            int* __restrict__ counters, int polls, AltPart ap) {
  using namespace mixed;
  __shared__ __attribute__((aligned(16))) char smem[TILE_LDS];
  static_assert(sizeof(DecodeSmem<128>) <= TILE_LDS, "a piece's LDS is a tile's");
  const int kvh = blockIdx.x, tid = threadIdx.x, y = blockIdx.y, Hq = Hkv * G;
  auto count = [&](int row) {
    __hip_atomic_fetch_add(counters + (int64_t)row * Hkv + kvh, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  if (y < n_tiles) {                                 // (workgroup-uniform)
    const TileItem it = titems[y];
    // a malformed item (host bug) is dropped instead of indexing out of bounds (workgroup-uniform)
    if (it.q_count < 1 || it.q_count * G > ROWS || it.q_start < 0 || it.split < 0 || it.q_start + it.q_count > (it.alt ? n_rows : B) ||
        it.split >= (it.alt ? ap.S : S_total) || (it.alt && it.q_start < ap.tok_off))
      return;
    // (the launch's other row tiles read the same keys: the loads keep the default policy)
    tile_item<0, 0, 2, NW, NSLOT>(smem, it, kvh, q, q_stride, k_cache, v_cache, Hkv, G, block_tables, bt_stride, q_limit, nullptr,
                                  0, reinterpret_cast<float*>(pre), lse, S_total, scale_log2, 1, ap);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid < it.q_count && row_parts[it.q_start + tid] != 0) count(it.q_start + tid);
    return;
  }
  if (y < n_tiles + n_pieces) {
    const DecodeItem it = ditems[y - n_tiles];
    const int b = it.b, split = it.split, np = it.nsplit, npre = it.npre;
    if (b < 0 || b >= B || split < 0 || split >= np || npre < 0 || npre + np > S_total) return;   // (uniform; as above)
    DecodeSmem<128>& sm = *reinterpret_cast<DecodeSmem<128>*>(smem);
    decode_stream<128, false>(sm, q, q_stride, k_cache, v_cache, Hkv, G, block_tables, bt_stride, b, kvh, it.lo, it.hi, scale_log2);
    store_piece_sc1<128>(sm, b, kvh, G, Hq, npre + split, S_total, part, lse);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) count(b);
    return;
  }
  // rows of 16 / G tokens, 16 lanes per (row, head)
  const int tw = 16 / G, row0 = (y - n_tiles - n_pieces) * tw;
  int* s_ok = reinterpret_cast<int*>(smem);
  if (tid < tw) {
    const int row = row0 + tid;
    int n = row < n_rows ? row_parts[row] & ((1 << PRE) - 1) : 0;
    if (n > 0) {
      // (parts that do not fit, a host bug: nothing of them is read. Rows between the decode rows and the new turns' have none.)
      const bool fits = n <= min(MAXS, row < B ? S_total : ap.S) && (row < B || row >= ap.tok_off);
      int* c = counters + (int64_t)row * Hkv + kvh;
      int left = fits ? polls : 0, got = 0;
      while (left > 0 && (got = __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) >= 0 && got < n) {
        --left;
        __builtin_amdgcn_s_sleep(8);
      }
      const bool ok = left > 0 && got >= n;
      __hip_atomic_store(c, ok ? 0 : LOST, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      n = ok ? n : -1;
    }
    s_ok[tid] = n;
  }
  __syncthreads();
  const int i = tid >> 4, row = row0 + i / G, head = kvh * G + i % G, n = s_ok[i / G];
  if (n == 0) return;
  bf16* const o = out + (int64_t)row * out_stride + (int64_t)head * 128;
  if (n < 0) {
#pragma unroll
    for (int j = 0; j < 8; ++j) o[8 * (tid & 15) + j] = (bf16)__builtin_nanf("");
  } else if (row < B) {
    mixed_merge_row(MixedParts{part, pre, lse, S_total}, (int64_t)row * Hq + head, min(row_parts[row] >> PRE, n), n, o);
  } else {
    mixed_merge_row(MixedParts{ap.part, nullptr, ap.lse, ap.S}, (int64_t)(row - ap.tok_off) * Hq + head, 0, n, o);
  }
}

// titems: int32 [n_tiles, 8] as attn_tile.h, ditems [n_pieces, 8] as attn_decode.h; row_parts [n_rows]: parts of every row that this launch
// merges (0: none of it; the parts of a row of new turns are tiles flagged alt), and above bit 16 those that tiles leave in bf16.
// counters: [n_rows, Hkv] zeros, zeros again behind it but for rows that were given up. polls: looks at a counter (of about a us) before that.
extern "C" hipError_t kafka_launch_attn_mixed(const int* titems, int n_tiles, const int* ditems, int n_pieces,
                                             const int* row_parts, int n_rows, const bf16* q, int64_t q_stride,
                                             const void* k_cache, const void* v_cache, int Hkv, int G,
                                             const int* block_tables, int bt_stride, const int* q_limit, int B,
                                             float* part, float* lse, bf16* pre, int S_total, float scale, bf16* out,
                                             int64_t out_stride, int* counters, int polls, float* alt_part, float* alt_lse, int alt_S,
                                             int alt_tok_off, hipStream_t st) {
  if (n_tiles + n_pieces == 0 || n_rows == 0) return hipSuccess;
  if (G < 1 || G > 8 || 16 % G || n_tiles < 0 || n_pieces < 0 || n_rows < B) return hipErrorInvalidValue;
  const int n_merge = (n_rows + 16 / G - 1) / (16 / G);
  if ((int64_t)n_tiles + n_pieces + n_merge > 65535) return hipErrorInvalidValue;
  if (!part || !lse || !pre || !out || !counters || out_stride % 8 || reinterpret_cast<uintptr_t>(out) % 16 || S_total < 1 ||
      (n_rows > B && (!alt_part || alt_tok_off < B || alt_tok_off > n_rows)))
    return hipErrorInvalidValue;
  attn_mixed_kernel<<<dim3(Hkv, n_tiles + n_pieces + n_merge), 256, 0, st>>>(
      reinterpret_cast<const TileItem*>(titems), n_tiles, reinterpret_cast<const DecodeItem*>(ditems), n_pieces, row_parts, n_rows, q,
      q_stride, static_cast<const bf16*>(k_cache), static_cast<const bf16*>(v_cache), Hkv, G, block_tables, bt_stride, q_limit, B, part,
      lse, pre, S_total, scale * 1.4426950408889634f, out, out_stride, counters, polls, AltPart{alt_part, alt_lse, alt_S, alt_tok_off});
  return hipGetLastError();
}

}  // namespace kafka
