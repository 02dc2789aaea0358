// Values of a step's rows into their pages, key after key for every column: v[page][column][16 keys] (gfx950).
//
// Stored row by row these are two-byte stores, a line each: 22 of 36 us of 4099 rows of 40 heads of 128. Here the 16 rows
// of a page that the step writes whole share it: the wave of a row takes a sixteenth of the columns of all 16 rows, turns them round
// in LDS and stores 16-byte pieces; a row of a page that it does not write whole goes one by one.
#pragma once
#include "common.h"

namespace kafka {
namespace pv {

constexpr int COLS = 64;                                   // columns turned at once
typedef bf16 Turn[16][COLS + 8];

// the slots of the rows around row t (asked for before anything waits), lane l: row t - 15 + l
__device__ __forceinline__ int64_t near(const int64_t* __restrict__ slots, int t, int T, int lane) {
  return slots[min(max(t - 15 + min(lane, 30), 0), T - 1)];
}

// Wave of row t in place slot >= 0 of v, which starts 16-byte aligned as the rows' C values at x do (C of a row in any
// number, strides of rows a multiple of 8). POS(key): where in a column's 16 the key of a page goes.
template <class Pos>
__device__ __forceinline__ void store(const bf16* __restrict__ x, int64_t xs, int C, int t, int T, int64_t slot, int64_t around,
                                      bf16* __restrict__ v, Turn& turn, int lane, Pos pos) {
  const int off = (int)(slot & 15), first = t - off, part = C / 16;
  const bool mine = lane >= 15 - off && lane < 31 - off;   // the page's rows, if the 16 from its first one on are its own
  const bool whole = first >= 0 && first + 16 <= T && C % 128 == 0 && __ballot(!mine || around == slot + (lane - 15)) == ~0ull;
  bf16* page = v + (slot >> 4) * (int64_t)C * 16;
  if (!whole) {
    const int at = pos(off);
    for (int u = lane * 8; u < C; u += 512) {
      const bf16x8 r = load_bf16x8(x + t * xs + u);
#pragma unroll
      for (int j = 0; j < 8; ++j) page[(u + j) * 16 + at] = r[j];
    }
    return;
  }
  for (int c0 = off * part; c0 < (off + 1) * part; c0 += COLS) {
    const int nc = min(COLS, (off + 1) * part - c0);       // (a multiple of 8)
    bf16x8 r[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) r[i] = load_bf16x8(x + (int64_t)(first + 8 * i + (lane >> 3)) * xs + c0 + min((lane & 7) * 8, nc - 8));
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // (the turn before has been read)
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < 2; ++i) *reinterpret_cast<bf16x8*>(&turn[8 * i + (lane >> 3)][(lane & 7) * 8]) = r[i];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (lane < nc) {
      bf16x8 o[2];
#pragma unroll
      for (int k = 0; k < 16; ++k) o[pos(k) >> 3][pos(k) & 7] = turn[k][lane];
#pragma unroll
      for (int i = 0; i < 2; ++i) store_bf16x8(page + (c0 + lane) * 16 + 8 * i, o[i]);
    }
  }
}

}  // namespace pv
}  // namespace kafka
