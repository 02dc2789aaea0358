// Matrix products of long steps: a tile of 32 MT x 32 NT through a ring of 32-deep stages in LDS (gfx950).
//
// Four waves of 16 MT x 16 NT (2 x 2). Activations and weights arrive by LDS-DMA: four stages of weights, and three units of
// activations, each of two stages: 128 bytes of a row are a whole cache line, 64 would ask for every line twice (5 - 9 % of the
// expert products of 8192 rows). Two stages are in flight while one is multiplied, one counted wait and one barrier per
// stage; a wave reads a stage's fragments while it multiplies the one before. The pieces are buffer loads: a lane's place is
// one register, the stage an offset in a scalar register, so that a piece costs one instruction beside the products instead of the four of
// 64-bit addresses. The next stage's reads stand in the first three quarters of the products (the last ones land before the
// stage ends), the pieces between them. 16x16x32 products: the matrix cores alone reach 1.89 PFLOP/s on them at one wave
// per SIMD, 1.47 on 32x32x16.
//
// Weights are wave-tiled (Wt[N/32][K/16][64][8]): a piece is a whole 1 KB tile of 32 columns x 16. With SWAP the products are
// taken with the weights first, so that a lane holds sums of one row and of columns in a run; the columns of a tile are laid out in LDS
// such (by the lanes' places in the source) that the run is 8 long over a pair of fragments: results leave in 16-byte pieces
// instead of 2-byte ones. The activations' 16-byte pieces are permuted at the source so that eight neighbouring rows of a
// fragment lie in different banks.
#pragma once
#include "common.h"

namespace kafka {
namespace ring {

typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_t;
constexpr int BK = 32, KB = BK / 16;
constexpr int LGKM0 = 0xC07F;   // s_waitcnt lgkmcnt(0) alone, in a form that the compiler counts too

// c += a b in an accumulation register: left to itself the compiler moves sums between the two register files in the loop.
// (Operands come from LDS, so their waits are the compiler's; two products on one sum are MT NT products apart.)
__device__ __forceinline__ void mfma16(f32x4v& c, bf16x8 a, bf16x8 b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

template <int N>
__device__ __forceinline__ void vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <bool B>
struct Full {
  static constexpr bool value = B;
};

// all of the 4 GB behind p, as a buffer: the places in it are the caller's to keep in bounds
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, -1, 0x00020000);
}

// WNT: weights that one row tile reads are asked for past the caches' retention (nt), so that the activations, which every column
// tile reads, stay in the L2s: 222 rows of 4096 -> 28672 64 -> 61 us, of 14336 -> 4096 in eight splits 41 -> 36.
template <int MT_, int NT_, bool SWAP_, bool WNT = false>
struct Ring {
  static constexpr int MT = MT_, NT = NT_;
  static constexpr bool SWAP = SWAP_;
  static constexpr int BM = 32 * MT, BN = 32 * NT;
  static constexpr int NX = 3, NW = 4, XU = BM * 2 * BK * 2, WS = BN * BK * 2, LDS = NX * XU + NW * WS;   // bytes
  // 1 KB pieces a wave moves: of a unit of activations (the first DO of them in an odd step, DE in the even one after it), of a stage of weights
  static constexpr int PX = MT, DO = (PX + 1) / 2, DE = PX / 2, DW = BN / 64;
  static constexpr int NM = MT * NT, NR = MT + NT;                  // products and fragments of a stage
  static constexpr int RST = NM * 3 / 4 / NR > 0 ? NM * 3 / 4 / NR : 1, DST = NM * 3 / 4 / (DO + DW);
  static_assert(BN % 64 == 0 && 1 + (DO + DW - 1) * DST < NM && (NR - 1) * RST < NM && LDS <= 163840, "ring");

  // what a lane adds to a weight piece's place: its 16 bytes of the tile
  static __device__ __forceinline__ unsigned wlane(int lane) {
    const int l = lane & 31;
    return ((lane & 32) + (SWAP ? 8 * ((l & 15) >> 2) + 4 * (l >> 4) + (l & 3) : l)) * 16;
  }
  // row of the tile whose 16 bytes a lane moves in wave w's u-th piece of a unit (u < PX), and where in the row's 128 bytes they start
  static __device__ __forceinline__ int xrow(int w, int u, int lane) { return 8 * (PX * w + u) + (lane >> 3); }
  static __device__ __forceinline__ int xbyte(int row, int lane) { return 16 * ((lane & 7) ^ (row & 7)); }
  // (32-column tile, 16-deep block) of wave w's u-th weight piece
  static __device__ __forceinline__ int wtile(int w, int u) { return (DW * w + u) / KB; }
  static __device__ __forceinline__ int wblock(int w, int u) { return (DW * w + u) % KB; }

  // acc += the tile's products over nst stages (even, at least 4). xo: byte offsets of this lane's activation pieces in xr, wo: of
  // this wave's weight pieces in wr (behind which wl is the lane's), both at the first stage.
  static __device__ __forceinline__ void multiply(f32x4v (&acc)[MT][NT], char* smem, __amdgpu_buffer_rsrc_t xr,
                                                  const unsigned (&xo)[PX], __amdgpu_buffer_rsrc_t wr, unsigned wl,
                                                  const unsigned (&wo)[DW], int nst, int lane, int w) {
    const int r = lane & 15, q = lane >> 4;
    char* const wsm = smem + NX * XU;
    auto xpiece = [&](int v, int slot, int u) {      // u-th piece of unit v
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_t*)(smem + slot * XU + (PX * w + u) * 1024), 16, xo[u],
                                               v * (4 * BK), 0, 0);
    };
    auto wpiece = [&](int s, int u) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_t*)(wsm + (s & (NW - 1)) * WS + (DW * w + u) * 1024), 16, wl,
                                               wo[u] + s * (KB * 1024), 0, WNT ? 2 : 0);
    };
    // what step s asks for: weights of stage s + 4, a half (the second where s is even) of the unit of stage s + 4 or s + 5
    auto piece = [&](int s, int odd, int slot, int u) {
      const int dx = odd ? DO : DE;
      if (u < dx) xpiece((s + 4 + odd) >> 1, slot, (odd ? 0 : DO) + u);
      else wpiece(s + 4, u - dx);
    };
    // where this lane's fragments lie: rows 16 i + r, 8-deep piece q of the stage's half of a unit; columns 16 j + r, piece q of
    // tile j / 2
    const int xrw = (16 * MT * (w >> 1) + r) * (4 * BK), xa0 = xrw + 16 * (q ^ (r & 7)), xa1 = xrw + 16 * ((4 + q) ^ (r & 7));
    const int wa = (NT / 2 * (w & 1) * KB + (q >> 1)) * 1024 + ((q & 1) * 32 + r) * 16;
    auto read = [&](bf16x8(&an)[MT], bf16x8(&bn)[NT], const char* xb, const char* wb, int i) {
      if (i < NT)
        bn[i < NT ? i : 0] = *reinterpret_cast<const bf16x8*>(wb + (i >> 1) * KB * 1024 + (i & 1) * 256);
      else
        an[i < NT ? 0 : i - NT] = *reinterpret_cast<const bf16x8*>(xb + (i - NT) * 16 * 4 * BK);
    };
    // all that was asked for up to step s - 3 has arrived, everywhere: stage s + 1 is there, stage s read
    auto turn = [&](int s) {
      if (s <= nst - 5) vmcnt<PX + 2 * DW>();
      else if (s == nst - 4) vmcnt<DE + 2 * DW>();   // (an even step's, and the weights alone)
      else if (s == nst - 3) vmcnt<DW>();
      else vmcnt<0>();
      asm volatile("s_barrier" ::: "memory");
    };
    bf16x8 a0[MT], b0[NT], a1[MT], b1[NT];
#pragma unroll
    for (int u = 0; u < PX; ++u) xpiece(0, 0, u);
#pragma unroll
    for (int u = 0; u < DW; ++u) wpiece(0, u);
#pragma unroll
    for (int u = 0; u < DO + DW; ++u) piece(-3, 1, 1, u);
#pragma unroll
    for (int u = 0; u < DE + DW; ++u) piece(-2, 0, 1, u);
#pragma unroll
    for (int u = 0; u < DO + DW; ++u)
      if (u >= DO || nst > 4) piece(-1, 1, 2, u);
    if (nst > 4) vmcnt<PX + DO + 3 * DW>();
    else vmcnt<PX + 3 * DW>();
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int i = 0; i < NR; ++i) read(a0, b0, smem + xa0, wsm + wa, i);
    int slot = 0;                                    // of the pair's unit
    // ``full``: whole pieces (s + 5 < nst for an odd s), no conditions in the way. Pairs: odd is a constant.
    auto step = [&](auto full, auto is_odd, int s, const bf16x8(&a)[MT], const bf16x8(&b)[NT], bf16x8(&an)[MT],
                    bf16x8(&bn)[NT]) {
      constexpr bool load = decltype(full)::value;
      constexpr int odd = decltype(is_odd)::value ? 1 : 0, DX = odd ? DO : DE, DPS = DX + DW;
      const int next = slot == NX - 1 ? 0 : slot + 1, third = next == NX - 1 ? 0 : next + 1;
      const int to = odd ? slot : third;             // the unit that step s fills
      __builtin_amdgcn_s_waitcnt(LGKM0);             // (this stage's fragments)
      const bool more = load || s + 1 < nst;
      if constexpr (load) {
        vmcnt<PX + 2 * DW>();
        asm volatile("s_barrier" ::: "memory");
      } else {
        if (more) turn(s);
#pragma unroll
        for (int u = 0; u < DPS; ++u)
          if (s + 4 + (u < DX ? odd : 0) < nst) piece(s, odd, to, u);
      }
      const char* xb = smem + (odd ? next * XU + xa0 : slot * XU + xa1);
      const char* wb = wsm + ((s + 1) & (NW - 1)) * WS + wa;
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        if (load && m % DST == 1 % DST && m / DST < DPS) piece(s, odd, to, m / DST);
        if (more && m % RST == 0 && m / RST < NR) read(an, bn, xb, wb, m / RST);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (SWAP) mfma16(acc[m / NT][m % NT], b[m % NT], a[m / NT]);
        else mfma16(acc[m / NT][m % NT], a[m / NT], b[m % NT]);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (odd) slot = next;
    };
    int s = 0;
    for (; s + 6 < nst; s += 2) {
      step(Full<true>(), Full<false>(), s, a0, b0, a1, b1);
      step(Full<true>(), Full<true>(), s + 1, a1, b1, a0, b0);
    }
    for (; s < nst; s += 2) {
      step(Full<false>(), Full<false>(), s, a0, b0, a1, b1);
      step(Full<false>(), Full<true>(), s + 1, a1, b1, a0, b0);
    }
    // the last products' results are complete before anything reads them behind a branch
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 15");
    __builtin_amdgcn_sched_barrier(0);
  }
};

}  // namespace ring
}  // namespace kafka
