// Stable sort of a step's routed entries by expert, one workgroup of 1024 threads or one per part of the entries (moe.hip,
// moe_wide.hip).
#pragma once
#include "common.h"

namespace kafka {
namespace mw {

constexpr int SORT_NT = 1024, SORT_W = SORT_NT / 64;

// Up to 64 experts: lane e counts expert e, in registers. A wave takes a stretch of the entries, 16 x 64 at a time: the ballots of
// the expert numbers' bits give the count of lane e's expert as well as an entry's rank among its equals; the waves' counts meet in
// LDS once, between the two walks. One workgroup is bound by its latencies and, past some thousand entries, by the scattered stores
// of one CU: then SORT_PART entries go to a workgroup each, counted by a launch in front (counts [parts][64]). us before (a counter in
// LDS per wave and expert, read and written for every 64 entries) / now: 64 entries 7 / 4, 4000 10 / 8, 19800 34 / 11, 32768 40 / 10.
constexpr int SORT_PART = 2048;

// The sums that the experts add to are cleared by further workgroups of the same launch, beside the sort's latencies (a launch
// of its own: 4.5 us of 128 rows of 4096, 26 of 2805).
__device__ __forceinline__ void clear(float* __restrict__ p, int64_t pieces, int block, int blocks) {
  typedef float f32x4c __attribute__((ext_vector_type(4)));
  for (int64_t i = (int64_t)block * SORT_NT + threadIdx.x; i < pieces; i += (int64_t)blocks * SORT_NT)
    reinterpret_cast<f32x4c*>(p)[i] = f32x4c{0.f, 0.f, 0.f, 0.f};
}
inline int clear_blocks(int64_t pieces) {   // four pieces a thread
  const int64_t b = (pieces + 4 * SORT_NT - 1) / (4 * SORT_NT);
  return (int)(b < 2048 ? b : 2048);
}

struct Stretch {
  int i0, i1;
};
__device__ __forceinline__ Stretch sort_stretch(int lo, int hi, int w) {
  const int per = ((hi - lo + SORT_W - 1) / SORT_W + 63) / 64 * 64;
  return {lo + w * per, min(hi, lo + (w + 1) * per)};
}

// entries of expert `lane` in the wave's stretch
__device__ __forceinline__ int sort_count(const int* topk_e, Stretch st, int bits) {
  constexpr int PF = 16;
  const int lane = threadIdx.x & 63;
  int mine = 0;
  for (int b0 = st.i0; b0 < st.i1; b0 += 64 * PF) {
    int ev[PF];
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      const int i = b0 + 64 * p + lane;
      ev[p] = i < st.i1 ? topk_e[i] : 0;
    }
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      unsigned long long m = __ballot(b0 + 64 * p + lane < st.i1);
      if (m == 0) break;   // (uniform)
      for (int b = 0; b < bits; ++b) {
        const unsigned long long s = __ballot((ev[p] >> b) & 1);
        m &= (lane >> b) & 1 ? s : ~s;
      }
      mine += __popcll(m);
    }
  }
  return mine;
}

// the workgroup's entries lo .. hi - 1 of n; parts == 1: counted here, else `counts` holds every part's and this is part `part`
__device__ __forceinline__ void sort_few_experts(const float* topk_w, const int* topk_e, int lo, int hi, int k, int E, int bits,
                                                 int bm, int* __restrict__ perm_tok, float* __restrict__ perm_w,
                                                 int* __restrict__ expert_off, int* __restrict__ tile_off,
                                                 int* __restrict__ inv, const int* counts, int part, int parts,
                                                 int (*cnt)[64]) {
  constexpr int PF = 16;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const Stretch st = sort_stretch(lo, hi, w);
  const int mine = sort_count(topk_e, st, bits);
  cnt[w][lane] = lane < E ? mine : 0;
  __syncthreads();
  int pre = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < SORT_W; ++i) {
    const int c = cnt[i][lane];
    pre += i < w ? c : 0;
    tot += c;
  }
  if (parts > 1) {
    tot = 0;
#pragma unroll 8
    for (int b = 0; b < parts; ++b) {
      const int c = counts[64 * b + lane];
      pre += b < part ? c : 0;
      tot += c;
    }
  }
  int a = tot, t = (tot + bm - 1) / bm;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(a, o, 64), v = __shfl_up(t, o, 64);
    if (lane >= o) {
      a += u;
      t += v;
    }
  }
  if (part == 0 && w == 0 && lane < E) {
    expert_off[lane + 1] = a;
    tile_off[lane + 1] = t;
    if (lane == 0) expert_off[0] = tile_off[0] = 0;
  }
  int base = a - tot + pre;   // where the wave's next entry of expert `lane` goes
  for (int b0 = st.i0; b0 < st.i1; b0 += 64 * PF) {
    int ev[PF];
    float wv[PF];
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      const int i = b0 + 64 * p + lane;
      ev[p] = i < st.i1 ? topk_e[i] : 0;
      wv[p] = i < st.i1 ? topk_w[i] : 0.f;
    }
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      const int i = b0 + 64 * p + lane;
      const unsigned long long valid = __ballot(i < st.i1);
      if (valid == 0) break;   // (uniform)
      unsigned long long m = valid, same = valid;
      for (int b = 0; b < bits; ++b) {
        const unsigned long long s = __ballot((ev[p] >> b) & 1);
        m &= (lane >> b) & 1 ? s : ~s;
        same &= (ev[p] >> b) & 1 ? s : ~s;
      }
      const int pos = __shfl(base, ev[p], 64) + __popcll(same & ((1ull << lane) - 1));
      if (i < st.i1) {
        perm_tok[pos] = i / k;
        perm_w[pos] = wv[p];
        if (inv != nullptr) inv[i] = pos;
      }
      base += __popcll(m);
    }
  }
}

}  // namespace mw
}  // namespace kafka
