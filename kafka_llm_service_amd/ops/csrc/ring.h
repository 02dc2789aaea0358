// Matrix products of long steps: a tile of 32 MT x 32 NT through a ring of 64-deep units in LDS (gfx950).
//
// Four waves of 16 MT x 16 NT (2 x 2), one a SIMD. Activations and weights arrive by LDS-DMA, as many units of each as LDS holds (256 x 256:
// two of activations and three of weights; these come from further away). A unit is multiplied in two halves of 32: while a wave multiplies one it
// reads the other's fragments, and what it does not read any more is filled again at once. Where the second half has been read stands
// the one place per unit at which the waves meet (the turn): behind it all have read this unit and the next one has arrived.
// The next unit's pieces are asked for between the products that follow, evenly over three quarters of a unit, activations first.
//
// With one wave a SIMD the matrix cores wait for whatever the wave does beside the products (16 cycles each, room for three further
// instructions). Hence: buffer loads, a lane's place one register, the unit an offset in a scalar register, a piece's place within
// four an immediate that the memory's and the LDS side's address share (so the scalar registers change once for four pieces);
// no conditions between the products; fragments a few products before they are needed. Of 16384 deep 256 x 256 tiles the
// loop takes 2.2 k cycles a unit, 2.05 k of them products (32-deep stages with a turn each, before: 2.6 k). The card lowers its clock under
// these products (random values 1.8 - 2.0 GHz, zeros 2.4), so that a sixth of the cycles is worth half of that: us, before /
// now, 8192 rows of 4096 -> 4096 204 / 189, 5376 -> 4096 256 / 239, 2048 rows of 4096 -> 28672 387 / 362, 14336 -> 4096 255 / 230, 222 rows of
// 4096 -> 28672 on 224 x 128 61 / 56, 600 of 4096 -> 4096 on 128 x 192 48.7 / 45.1; 128 x 128 as before (within 2 %: what the L2s give).
// 16x16x32 products: the matrix cores alone reach 2.1 PFLOP/s on them under random values, 1.84 on 32x32x16, and 2.13 where
// one operand of a product is always the one before's (rows of a tile there and back); 2.45 of zeros on either.
// 128 bytes of a row are a whole cache line; 64 would ask for every line twice.
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
constexpr int LGKM0 = 0xC07F;   // s_waitcnt lgkmcnt(0) alone, in a form that the compiler counts too

// c += a b in an accumulation register: left to itself the compiler moves sums between the two register files in the loop.
// (Operands come from LDS, so their waits are the compiler's; two products on one sum are MT NT products apart; the zeros that
// the sums begin with are written well before.)
__device__ __forceinline__ void mfma16(f32x4v& c, bf16x8 a, bf16x8 b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

template <int N>
__device__ __forceinline__ void vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <int I>
struct Num {
  static constexpr int value = I;
};

// f(Num<0>()), f(Num<1>()) ... f(Num<N - 1>())
template <int N, int I = 0, typename F>
__device__ __forceinline__ void each(F&& f) {
  if constexpr (I < N) {
    f(Num<I>());
    each<N, I + 1>(f);
  }
}

// all of the 4 GB behind p, as a buffer: the places in it are the caller's to keep in bounds
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, -1, 0x00020000);
}

// WNT: weights that one row tile reads are asked for past the caches' retention (nt), so that the activations, which every column
// tile reads, stay in the L2s: 222 rows of 4096 -> 28672 64 -> 61 us, of 14336 -> 4096 in eight splits 41 -> 36. OCC workgroups share a CU's LDS.
template <int MT_, int NT_, bool SWAP_, bool WNT = false, int OCC = 1>
struct Ring {
  static constexpr int MT = MT_, NT = NT_;
  static constexpr bool SWAP = SWAP_;
  static constexpr int BK = 64, BM = 32 * MT, BN = 32 * NT, XU = BM * BK * 2, WU = BN * BK * 2;   // bytes of a unit
  // units of activations and of weights in LDS: as many as fit, of weights one more if that fits
  static constexpr int ROOM = 163840 / OCC, MOST = 5, FIT = ROOM / (XU + WU);
  static constexpr int NX = FIT < MOST ? FIT : MOST, NW = NX < MOST && NX * XU + (NX + 1) * WU <= ROOM ? NX + 1 : NX,
                       LDS = NX * XU + NW * WU;
  // 1 KB pieces that a wave moves of a unit; weight pieces that follow each other in memory (within a column tile)
  static constexpr int PX = MT, PW = NT, P = PX + PW, WRUN = NT % 4 == 0 ? 4 : 2, WR = PW / WRUN;
  // products and fragments of half a unit; products from one fragment's read to the next one's and from one piece to the next; products
  // of the first half in front of the turn (its reads, and six products for the last one to arrive)
  static constexpr int NM = MT * NT, NR = MT + NT;
  static constexpr int RST = NM * 3 / 4 / NR > 0 ? NM * 3 / 4 / NR : 1, DST = 2 * NM * 3 / 4 / P > 0 ? 2 * NM * 3 / 4 / P : 1;
  static constexpr int READ = (NR - 1) * RST + 1, TURN = READ + 6 < NM ? READ + 6 : NM;
  static_assert(BN % 64 == 0 && READ <= NM && 1 + (P - 1) * DST < 2 * NM && NX >= 2 && LDS <= ROOM, "ring");

  // what a lane adds to a weight piece's place: its 16 bytes of the tile
  static __device__ __forceinline__ unsigned wlane(int lane) {
    const int l = lane & 31;
    return ((lane & 32) + (SWAP ? 8 * ((l & 15) >> 2) + 4 * (l >> 4) + (l & 3) : l)) * 16;
  }
  // row of the tile whose 16 bytes a lane moves in wave w's u-th piece of a unit (u < PX), and where in xbuffer(the row's 128 bytes) they
  // start: pieces u % 4 apart share an address register, the load's immediate moves both sides by 1 KB a piece
  static __device__ __forceinline__ int xrow(int w, int u, int lane) { return 8 * (PX * w + u) + (lane >> 3); }
  static __device__ __forceinline__ int xbyte(int row, int u, int lane) {
    return 16 * ((lane & 7) ^ (row & 7)) + 3072 - 1024 * (u & 3);
  }
  static __device__ __forceinline__ __amdgpu_buffer_rsrc_t xbuffer(const bf16* p) {
    return buffer(reinterpret_cast<const char*>(p) - 3072);
  }
  // (32-column tile, 16-deep block) of wave w's g-th run of weight pieces
  static __device__ __forceinline__ int wtile(int w, int g) { return (PW * w + WRUN * g) / 4; }
  static __device__ __forceinline__ int wblock(int w, int g) { return (PW * w + WRUN * g) % 4; }

  // acc (zeros) += the tile's products over nu units (at least 2). xo: byte offsets of this lane's activation pieces in xr (an xbuffer), wo: of
  // this wave's runs of weight pieces in wr (behind which wl is the lane's), both at the first unit.
  static __device__ __forceinline__ void multiply(f32x4v (&acc)[MT][NT], char* smem, __amdgpu_buffer_rsrc_t xr,
                                                  const unsigned (&xo)[PX], __amdgpu_buffer_rsrc_t wr, unsigned wl,
                                                  const unsigned (&wo)[WR], int nu, int lane, int w) {
    const int r = lane & 15, q = lane >> 4;
    char* const wsm = smem + NX * XU;
    // a piece of unit v, into a slot
    auto xpiece = [&](auto piece, int v, int slot) {
      constexpr int u = decltype(piece)::value;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_t*)(smem + slot * XU + (PX * w + (u & ~3)) * 1024), 16, xo[u],
                                               v * (2 * BK), 1024 * (u & 3), 0);
    };
    auto wpiece = [&](auto piece, int v, int slot) {
      constexpr int u = decltype(piece)::value, g = u / WRUN;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_t*)(wsm + slot * WU + (PW * w + WRUN * g) * 1024), 16, wl, wo[g] + v * 4096,
                                               1024 * (u % WRUN), WNT ? 2 : 0);
    };
    // where this lane's fragments lie: rows 16 i + r, 8-deep piece q of a half; columns 16 j + r, piece q of tile j / 2
    const int xrw = (16 * MT * (w >> 1) + r) * (2 * BK), xa0 = xrw + 16 * (q ^ (r & 7)), xa1 = xrw + 16 * ((4 + q) ^ (r & 7));
    const int wa = (NT / 2 * (w & 1) * 4 + (q >> 1)) * 1024 + ((q & 1) * 32 + r) * 16;
    auto read = [&](bf16x8(&an)[MT], bf16x8(&bn)[NT], const char* xb, const char* wb, int i) {
      if (i < NT)
        bn[i < NT ? i : 0] = *reinterpret_cast<const bf16x8*>(wb + (i >> 1) * 4096 + (i & 1) * 256);
      else
        an[i < NT ? 0 : i - NT] = *reinterpret_cast<const bf16x8*>(xb + (i - NT) * 16 * (2 * BK));
    };
    bf16x8 a0[MT], b0[NT], a1[MT], b1[NT];
    int v = 0, xs = 0, ws = 0;                       // the unit, its slots
    // products FROM .. TO of a half (a, b), AT products behind the turn, between them: the other half's reads (from xb, wb), the pieces
    // of activations (XL) and weights (WL) that fill the unit's slots
    auto part = [&](auto from, auto to, auto at, auto rd, auto xl, auto wld, const bf16x8(&a)[MT], const bf16x8(&b)[NT],
                    bf16x8(&an)[MT], bf16x8(&bn)[NT], const char* xb, const char* wb) {
      constexpr int FROM = decltype(from)::value, TO = decltype(to)::value, AT = decltype(at)::value;
      constexpr bool RD = decltype(rd)::value != 0, XL = decltype(xl)::value != 0, WL = decltype(wld)::value != 0;
      each<TO - FROM>([&](auto k) {
        constexpr int m = FROM + decltype(k)::value, t = AT + decltype(k)::value, i = m / NT,
                      j = i & 1 ? NT - 1 - m % NT : m % NT;
        if constexpr (t % DST == 1 % DST && t / DST < PX) {
          if constexpr (XL) xpiece(Num<t / DST>(), v + NX, xs);
        } else if constexpr (t % DST == 1 % DST && t / DST < P) {
          if constexpr (WL) wpiece(Num<t / DST - PX>(), v + NW, ws);
        }
        if constexpr (RD && m % RST == 0 && m / RST < NR) read(an, bn, xb, wb, m / RST);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (SWAP) mfma16(acc[i][j], b[j], a[i]);
        else mfma16(acc[i][j], a[i], b[j]);
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    constexpr Num<0> no, zero;
    constexpr Num<1> yes;
    constexpr Num<NM> all;
    constexpr Num<TURN> turn;
    constexpr Num<2 * NM> never;                     // (no piece has its place there)
    // behind the turn: the rest of unit v, then the first products of unit v + 1
    auto unit = [&](auto xl, auto wld) {
      const int xn = xs == NX - 1 ? 0 : xs + 1, wn = ws == NW - 1 ? 0 : ws + 1;
      const char *xb = smem + xn * XU, *wb = wsm + wn * WU + wa;
      part(turn, all, zero, no, xl, wld, a0, b0, a1, b1, xb, wb);
      part(zero, all, Num<NM - TURN>(), yes, xl, wld, a1, b1, a0, b0, xb + xa0, wb);
      __builtin_amdgcn_s_waitcnt(LGKM0);
      part(zero, turn, Num<2 * NM - TURN>(), yes, xl, wld, a0, b0, a1, b1, xb + xa1, wb + 2048);
      xs = xn;
      ws = wn;
      ++v;
    };
    each<NW>([&](auto first) {
      constexpr int f = decltype(first)::value;
      if (f < 2 || f < nu) {
        if constexpr (f < NX) each<PX>([&](auto u) { xpiece(u, f, f); });
        each<PW>([&](auto u) { wpiece(u, f, f); });
      }
    });
    __builtin_amdgcn_sched_barrier(0);
    // the zeros are in the accumulation registers while the first pieces are on their way: the compiler would write them in front of the first
    // product of each, and knows of no wait between the two
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) asm volatile("" : "+a"(acc[i][j]));
    __builtin_amdgcn_sched_barrier(0);
    if (nu >= NW) vmcnt<NX * PX + NW * PW - P>();
    else vmcnt<0>();
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int i = 0; i < NR; ++i) read(a0, b0, smem + xa0, wsm + wa, i);
    __builtin_amdgcn_s_waitcnt(LGKM0);
    part(zero, turn, never, yes, no, no, a0, b0, a1, b1, smem + xa1, wsm + wa + 2048);
    // The turn waits for unit v + 1: of what was asked for since, NX - 2 units of activations and NW - 2 of weights may be under way. (Loops
    // one after the other and no branches in one: the sums would move between registers where those meet.)
    constexpr int AWAY = (NX - 2) * PX + (NW - 2) * PW;
    for (; v + NW < nu;) {
      __builtin_amdgcn_s_waitcnt(LGKM0);
      vmcnt<AWAY>();
      asm volatile("s_barrier" ::: "memory");
      unit(yes, yes);
    }
    if constexpr (NX < NW)
      for (; v + NX < nu;) {                         // (once: the last unit of activations)
        __builtin_amdgcn_s_waitcnt(LGKM0);
        vmcnt<AWAY>();
        asm volatile("s_barrier" ::: "memory");
        unit(yes, no);
      }
    for (; v + 1 < nu;) {
      __builtin_amdgcn_s_waitcnt(LGKM0);
      const int left = nu - 2 - v;                   // units behind the next one
      if (NW > 2 && left == 1) vmcnt<(NX > 2 ? 1 : 0) * PX + PW>();
      else if (NW > 3 && left == 2) vmcnt<(NX > 3 ? 2 : NX - 2) * PX + 2 * PW>();
      else vmcnt<0>();
      asm volatile("s_barrier" ::: "memory");
      unit(no, no);
    }
    __builtin_amdgcn_s_waitcnt(LGKM0);
    part(turn, all, never, no, no, no, a0, b0, a1, b1, smem, smem);
    part(zero, all, never, no, no, no, a1, b1, a0, b0, smem, smem);
    // the last products' results are complete before anything reads them behind a branch
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 15");
    __builtin_amdgcn_sched_barrier(0);
  }

  // The tile's results (SWAP). A lane holds eight columns in a run of one row, 16 rows x 4 runs a fragment; pairs of lanes (rows m, m + 1) trade
  // pieces, so that a store takes eight rows of 128 bytes, whole cache lines, where 16 rows of 64 would take every line twice. Each kind of
  // result is code of its own in one run: with the choice between them inside the loops a workgroup jumped through 60 KB of instructions
  // that no cache held (256 x 256 bf16: 18.6 k cycles, 4.3 k so; 8192 rows of 4096 -> 4096 193 -> 181 us).
  static __device__ __forceinline__ void trade(int odd, const f32x4v& p0, const f32x4v& p1, f32x4v& even_row, f32x4v& odd_row) {
    f32x4v got;
#pragma unroll
    for (int i = 0; i < 4; ++i)                      // (the neighbouring lane's)
      got[i] = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, odd ? p0[i] : p1[i]), 0xB1, 0xf, 0xf, true));
    even_row = odd ? got : p0;
    odd_row = odd ? p1 : got;
  }
  // value(mt, t, i): column i of the run in the wave's t-th 32-column tile of results; y: row 0, the wave's first column; rows, tiles: how many there are
  template <int TILES, typename V>
  static __device__ __forceinline__ void rows_bf16(bf16* y, int64_t ld, int rows, int tiles, int lane, int w, V&& value) {
    const int r = lane & 15, q = lane >> 4, odd = r & 1;
    auto run = [&](auto mt, auto t) {
      bf16x8 o;
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = (bf16)value(mt, t, i);
      return __builtin_bit_cast(f32x4v, o);
    };
    each<MT>([&](auto mt) {
      const int m = 16 * (MT * (w >> 1) + decltype(mt)::value) + (r & ~1);
      bf16* const p = y + m * ld + 8 * q;
      each<TILES / 2>([&](auto pair) {
        constexpr int t = 2 * decltype(pair)::value;
        f32x4v a, b;
        trade(odd, run(mt, Num<t>()), run(mt, Num<t + 1>()), a, b);
        if (t + odd < tiles) {
          bf16* const c = p + 32 * (t + odd);
          if (m < rows) *reinterpret_cast<f32x4v*>(c) = a;
          if (m + 1 < rows) *reinterpret_cast<f32x4v*>(c + ld) = b;
        }
      });
      if constexpr (TILES % 2) {
        const f32x4v a = run(mt, Num<TILES - 1>());
        if (TILES - 1 < tiles && m + odd < rows) *reinterpret_cast<f32x4v*>(p + odd * ld + 32 * (TILES - 1)) = a;
      }
    });
  }
  // the sums themselves; column(t): where the wave's t-th tile begins in a row of p
  template <typename F>
  static __device__ __forceinline__ void rows_f32(const f32x4v (&acc)[MT][NT], float* p, int64_t ld, int rows, int tiles, int lane,
                                                  int w, F&& column) {
    const int r = lane & 15, q = lane >> 4, odd = r & 1;
    each<MT>([&](auto mt) {
      constexpr int i = decltype(mt)::value;
      const int m = 16 * (MT * (w >> 1) + i) + (r & ~1);
      each<NT / 2>([&](auto tile) {
        constexpr int t = decltype(tile)::value;
        f32x4v a, b;
        trade(odd, acc[i][2 * t], acc[i][2 * t + 1], a, b);
        if (t < tiles) {
          float* const c = p + m * ld + column(t) + 8 * q + 4 * odd;
          if (m < rows) *reinterpret_cast<f32x4v*>(c) = a;
          if (m + 1 < rows) *reinterpret_cast<f32x4v*>(c + ld) = b;
        }
      });
    });
  }
};

}  // namespace ring
}  // namespace kafka
