// What the kernels that run a recurrence in chunks of 128 tokens on the matrix cores share (hybrid_memory.hip,
// hybrid_ssd.hip): tile sizes, the split of an fp32 factor into bf16 parts, the workgroup order, transposed tiles.
#pragma once
#include "common.h"

namespace kafka {
namespace chunk {

constexpr int NT = 256;
constexpr float LOG2E = 1.4426950408889634f;
constexpr int CH = 128;         // tokens per chunk
constexpr int VSL = 64;         // value columns of a workgroup
constexpr int LDJ = CH + 8;     // row length of a transposed tile in LDS
constexpr int DS = 128;         // key channels staged at a time
constexpr int LDD = DS + 8;     // row length of a tile of an entry state's part in LDS

// v = a + b + c with bf16 parts that hold all its bits
struct Split {
  bf16x8 p[3];
};
__device__ __forceinline__ Split split3(const float (&v)[8]) {
  Split s;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const bf16 a = (bf16)v[e];
    const float r = v[e] - (float)a;
    const bf16 b = (bf16)r;
    s.p[0][e] = a;
    s.p[1][e] = b;
    s.p[2][e] = (bf16)(r - (float)b);
  }
  return s;
}

// results of matrix products are complete before anything behind a branch reads them
__device__ __forceinline__ void mfma_settle() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 15");
  __builtin_amdgcn_sched_barrier(0);
}

// which (chunk, head, value slice): a (chunk, head)'s slices run on one XCD (workgroups go round the eight XCDs)
__device__ __forceinline__ bool chunk_item(int items, int slices, int& item, int& slice) {
  const int lin = blockIdx.x, xcd = lin & 7, k = lin >> 3;
  item = (k / slices) * 8 + xcd;
  slice = k % slices;
  return item < items;
}
__host__ __device__ __forceinline__ int chunk_grid(int items, int slices) { return (items + 7) / 8 * 8 * slices; }

// rows row0 .. row0 + 127 (past n: the last one), columns c0 .. c0 + nc - 1 of the head's part at col -> tile[column][row].
// A wave moves 4 x 8 columns of 16 x 4 rows: 64 bytes in a run from memory, pairs of banks in LDS (all columns of 8 x 4 rows: eight on one bank).
__device__ __forceinline__ void stage_transposed(const bf16* src, int64_t stride, int n, int c0, int nc, int ncols,
                                                 bf16* tile, int tid) {
  const int cgs = nc >> 3, blocks = (cgs + 3) >> 2;
  for (int u = tid; u < blocks * CH; u += NT) {
    const int q = u >> 6, half = q >= blocks, cg = 4 * (q - half * blocks) + (u & 3), rq = 16 * half + ((u >> 2) & 15), c = c0 + 8 * cg;
    if (cg >= cgs) continue;
    bf16x8 x[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      x[k] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
      if (c < ncols) x[k] = load_bf16x8(src + (int64_t)min(4 * rq + k, n - 1) * stride + c);
    }
    typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const bf16x4 y = {x[0][e], x[1][e], x[2][e], x[3][e]};
      *reinterpret_cast<bf16x4*>(tile + (8 * cg + e) * LDJ + 4 * rq) = y;
    }
  }
}

// channels 0 .. nd - 1 (nd <= DS) of VSL fp32 rows (past nv: zeros) in three bf16 parts -> buf[part][row][channel]. All of a thread's
// loads go out together.
__device__ __forceinline__ void stage_split(const float* src, int64_t stride, int nd, int nv, bf16* buf, int tid) {
  typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
  constexpr int RQ = DS / 4, NU = VSL * RQ / NT;
  static_assert(NT % RQ == 0 && VSL * RQ % NT == 0, "whole rows");
  const int v = tid / RQ, d = 4 * (tid % RQ);
  if (d >= nd) return;
  f32x4 x[NU];
#pragma unroll
  for (int k = 0; k < NU; ++k) {
    const int r = v + k * (NT / RQ);
    x[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (r < nv) x[k] = *reinterpret_cast<const f32x4*>(src + r * stride + d);
  }
#pragma unroll
  for (int k = 0; k < NU; ++k) {
    bf16x4 p[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bf16 a = (bf16)x[k][e];
      const float rr = x[k][e] - (float)a;
      const bf16 b = (bf16)rr;
      p[0][e] = a;
      p[1][e] = b;
      p[2][e] = (bf16)(rr - (float)b);
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x4*>(buf + (i * VSL + v + k * (NT / RQ)) * LDD + d) = p[i];
  }
}

}  // namespace chunk
}  // namespace kafka
