// Tile attention (attn_tile.h) as a launch of its own: the cascade prefix pass and chunked / causal prefill.
#include "attn_tile.h"

#include <cstdlib>

namespace kafka {

// An item (256 query rows) is 8 / NW workgroups of one key/value head. Prompts: two of four waves and two ring slots each, two workgroups
// a CU, whose waves do not wait for each other and whose halves of a causal item end where their own rows do; 4096 rows of 32 heads
// against 8192 keys, us, 8 waves 497, two of 4 482; on another card before the loop was a pipeline, 8 waves, / now 489 / 466, behind
// 4096 of the keys 408 / 374.
// A cascade's prefix pass (few row tiles, keys from memory) reads the keys once an item: 8 waves, three slots (4: 30.9 vs 29.9 us per
// cascade launch, profiles/r05/cascade/cascade_nslot_*.jsonl). So do a few short portions behind long histories of their own, whose keys
// come from memory in many short parts: from eight parts a row on, where there are items for more than half the CUs (fewer leave CUs to
// the second half). Two and four portions of 60 tokens behind 3000, 8 key/value heads, a step of four layers, two of 4 / 8 waves:
// 706 / 689 and 871 / 844; with four parts (eight portions) 1164 / 1167, on fewer CUs (one portion) 556 / 567.
template <int ABL, int KVAUX, int PST, int NW, int NSLOT>
__global__ __launch_bounds__(64 * NW, 2) void attn_tile_kernel(const TileItem* __restrict__ items,
                                                               const bf16* __restrict__ q, int64_t q_stride,
                                                               const bf16* __restrict__ k_cache,
                                                               const bf16* __restrict__ v_cache, int Hkv, int G,
                                                               const int* __restrict__ block_tables, int bt_stride,
                                                               const int* __restrict__ q_limit, bf16* __restrict__ out,
                                                               int64_t out_stride, float* __restrict__ out_part,
                                                               float* __restrict__ lse_part, int S_total,
                                                               float scale_log2, int part_bf16, AltPart ap) {
  __shared__ __attribute__((aligned(16))) char smem[tile3::lds_bytes<NSLOT>()];
  TileItem it = items[blockIdx.y];
  const int share = blockIdx.x / Hkv, tok = 32 * NW / G;
  it.q_start += share * tok;
  it.q_count = min(it.q_count - share * tok, NW == 8 ? it.q_count : tok);
  if (it.q_count <= 0) return;
  tile_item<ABL, KVAUX, PST, NW, NSLOT>(smem, it, blockIdx.x - share * Hkv, q, q_stride, k_cache, v_cache, Hkv, G, block_tables,
                                        bt_stride, q_limit, out, out_stride, out_part, lse_part, S_total, scale_log2, part_bf16, ap);
}

// Host launcher (bf16 KV only; the fp8 cache keeps tile variant 0). Items: int32 [n, 8] as attn_prefill_kernel.
extern "C" hipError_t kafka_launch_attn_tile(const void* items, int n_items, const bf16* q, int64_t q_stride,
                                            const void* k_cache, const void* v_cache, int Hkv, int G, int D,
                                            const int* block_tables, int bt_stride, const int* q_limit, bf16* out,
                                            int64_t out_stride, float* out_part, float* lse_part, int S_total,
                                            float scale, int part_bf16, float* alt_part, float* alt_lse, int alt_S,
                                            int alt_tok_off, hipStream_t st) {
  if (n_items == 0) return hipSuccess;
  if (D != 128 || G < 1 || G > 32 || (256 % G) != 0 || n_items > 65535) return hipErrorInvalidValue;
  const float scale_log2 = scale * 1.4426950408889634f;
  static const bool stamps = [] {  // diagnostic build (benchmarks/attn_tile_stamps.py)
    const char* e = getenv("KAFKA_TILE_ABL");
    return e && atoi(e) == 8;
  }();
  // The cascade prefix pass (bf16 partials) reads each K / V tile of the shared prefix once per KV head and 256 query
  // rows (one workgroup at the headline's 64 streams): its DMAs go nt (aux = 2), +0.9 % on the headline
  // (profiles/r05/cascade/bench_ab_kv_nt.jsonl). Prefill launches keep the default policy: their query tiles re-read
  // the same keys.
  // Its bf16 partials are stored sc1 (16-B stores that leave this XCD's L2: +0.2..0.6 %, bench_ab_part_sc1.jsonl).
  auto go = [&](auto kern, int shares) {
    kern<<<dim3(Hkv * shares, n_items), 512 / shares, 0, st>>>(
        reinterpret_cast<const TileItem*>(items), q, q_stride, static_cast<const bf16*>(k_cache), static_cast<const bf16*>(v_cache), Hkv, G,
        block_tables, bt_stride, q_limit, out, out_stride, out_part, lse_part, S_total, scale_log2, part_bf16,
        AltPart{alt_part, alt_lse, alt_S, alt_tok_off});
  };
  if (stamps) go(attn_tile_kernel<8, 0, 0, 8, 3>, 1);
  else if (part_bf16) go(attn_tile_kernel<0, 2, 1, 8, 3>, 1);
  else if (out_part != nullptr && S_total >= 8 && n_items * Hkv > 128) go(attn_tile_kernel<0, 0, 0, 8, 3>, 1);
  else go(attn_tile_kernel<0, 0, 0, 4, 2>, 2);
  return hipGetLastError();
}

}  // namespace kafka
