// Dense products of long steps on wave-tiled weights: Y[M, N] = X[M, K] W[N, K]^T, bf16, fp32 sums (gfx950).
//
// Tiles of 128 - 256 rows and columns (ring.h), K split over workgroups into fp32 slabs where a step has few rows: the host
// picks by a model of the launch (ops.tile_plan). What bounds it: a whole round of 256 x 256 tiles takes 1.2 - 1.35 us per 64 of K
// (1.6 - 1.8 PFLOP/s, the card's clock under the values) and about 10 us for its start and its results; smaller tiles are bound by what the L2s
// give the CUs, 65 - 75 GB/s each whatever the tile (17 - 19 TB/s): 192 x 192 0.79 us per 64 of K, 256 x 128 0.69, 128 x 128 (two workgroups a CU)
// 0.43 each. So a tile is as large as leaves no round of the chip half empty, and sizes between 128 and 256 pay: 2048 rows of 4096 -> 6144 on
// 256 x 256 95 us, on 256 x 192 74. Tried: workgroups that go on to their next tiles with the ring kept full (0.5 - 1.8 % of two to seven rounds:
// the card lowers its clock by what the gaps were); K begun at another place for every column tile (0 - 2 %); two of the four waves moving the
// weights alone, eight stages ahead (3 % more: their latency is not what a step of 136 - 256 rows waits for).
#include "ring.h"

namespace kafka {
namespace tg {

enum { OUT_BF16 = 0, OUT_SLAB = 1, OUT_GLU = 2, OUT_SLAB_GLU = 3, OUT_RELU2 = 4, OUT_GELU = 5 };

struct TileArgs {
  const bf16* X;
  int64_t ldx;
  const bf16x8* Wt;
  int M, N, K, S;
  bf16* Y;
  int64_t ldy;
  float* P;
  int mode;
};

// rows (at most 32 MT) rows from row0 on, 32 NT columns from tile nt on, split sp
template <int MT, int NT, int OCC, bool WNT>
__device__ __forceinline__ void tile(const TileArgs& A, char* smem, int sp, int nt, int row0, int rows) {
  using R = ring::Ring<MT, NT, true, WNT, OCC>;
  const int N = A.N, K = A.K, mode = A.mode;
  const int64_t ldx = A.ldx, ldy = A.ldy;
  // K in units of 64, split as evenly as they go
  const int units = K >> 6, u0 = (int)((int64_t)units * sp / A.S), u1 = (int)((int64_t)units * (sp + 1) / A.S);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  unsigned xo[R::PX], wo[R::WR];
#pragma unroll
  for (int u = 0; u < R::PX; ++u) {            // rows past M reload the last, never stored
    const int row = R::xrow(w, u, lane);
    xo[u] = (unsigned)min(row, rows - 1) * (unsigned)(ldx * 2) + R::xbyte(row, u, lane);
  }
#pragma unroll
  for (int u = 0; u < R::WR; ++u)                  // (tiles past N reload the last, never stored)
    wo[u] = (unsigned)(min(nt * NT + R::wtile(w, u), (N >> 5) - 1) * (K >> 4) + R::wblock(w, u)) * 1024u;
  ring::f32x4v acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = ring::f32x4v{0.f, 0.f, 0.f, 0.f};
  R::multiply(acc, smem, R::xbuffer(A.X + (int64_t)row0 * ldx + 64 * u0), xo, ring::buffer(A.Wt + (int64_t)u0 * 4 * 64),
              R::wlane(lane), wo, u1 - u0, lane, w);
  const int nb = nt * NT + NT / 2 * (w & 1), nall = N >> 5;   // this wave's first tile of 32 columns, all of them
  if (nb >= nall) return;
  auto sum = [&](auto m, auto c, int i) { return acc[decltype(m)::value][2 * decltype(c)::value + (i >> 2)][i & 3]; };
  if (mode == OUT_SLAB || mode == OUT_SLAB_GLU) {
    float* const p = A.P + ((int64_t)sp * A.M + row0) * N;
    // (gate | up order of interleaved tiles)
    if (mode == OUT_SLAB) R::rows_f32(acc, p, N, rows, nall - nb, lane, w, [&](int t) { return (nb + t) * 32; });
    else R::rows_f32(acc, p, N, rows, nall - nb, lane, w, [&](int t) { return (((nb + t) & 1) ? N >> 1 : 0) + ((nb + t) >> 1) * 32; });
    return;
  }
  bf16* const y = A.Y + (int64_t)row0 * ldy;
  if (mode == OUT_BF16) {
    R::template rows_bf16<NT / 2>(y + nb * 32, ldy, rows, nall - nb, lane, w, sum);
  } else if (mode == OUT_RELU2) {
    R::template rows_bf16<NT / 2>(y + nb * 32, ldy, rows, nall - nb, lane, w, [&](auto m, auto c, int i) {
      const float a = sum(m, c, i), p = a < 0.f ? 0.f : a;   // (not a number stays)
      return p * p;
    });
  } else if constexpr (NT % 4 == 0) {                        // tiles of 32: gate, up, gate, up
    auto gated = [&](auto m, auto c, int i, bool gelu) {
      constexpr int t = 2 * decltype(c)::value;
      return gate_act(sum(m, ring::Num<t>(), i), gelu) * sum(m, ring::Num<t + 1>(), i);
    };
    if (mode == OUT_GLU)
      R::template rows_bf16<NT / 4>(y + nb * 16, ldy, rows, (nall - nb) / 2, lane, w, [&](auto m, auto c, int i) { return gated(m, c, i, false); });
    else
      R::template rows_bf16<NT / 4>(y + nb * 16, ldy, rows, (nall - nb) / 2, lane, w, [&](auto m, auto c, int i) { return gated(m, c, i, true); });
  }
}

// A last row tile of at most LOW rows is one of that height: its weights' way is then what it takes, a third of a whole tile. The whole tiles are
// dealt out first, evenly, then those, to each XCD what it has fewer of the others. us, before / now: 4099 rows of 4096 -> 28672 698 / 669,
// of 4096 -> 4096 152 / 112, of 14336 -> 4096 504 / 376; 2060 rows of 4096 -> 4096 on 256 x 128 87 / 65. (Dealt out evenly by themselves, an XCD
// had 65 tiles for its 64 places in two rounds: 1024 rows of 4096 -> 18560 on 160 x 256 142, so 129.) One row tile alone, WNT, has a height
// that fits; tiles of 128 rows are low enough.
constexpr int LOW = 64;
template <int MT>
__device__ constexpr int low_rows(int M) {
  return MT > 4 && M > 32 * MT && M % (32 * MT) <= LOW ? M % (32 * MT) : 0;
}

// MT, NT: 16-row and 16-column parts of a wave's tile (2 x 2 waves); OCC workgroups on a CU; WNT: of one row tile
template <int MT, int NT, int OCC, bool WNT>
__global__ __launch_bounds__(256, OCC) void tile_gemm_kernel(const TileArgs A) {
  using R = ring::Ring<MT, NT, true, WNT, OCC>;
  using L = ring::Ring<LOW / 32, NT, true, WNT, OCC>;
  constexpr bool HAS_LOW = MT > 4 && !WNT;
  __shared__ __attribute__((aligned(1024))) char smem[HAS_LOW && L::LDS > R::LDS ? L::LDS : R::LDS];
  // item -> (split, rows, columns): an XCD takes one contiguous stretch of them: of a split the row tiles of up to 2048 rows
  // side by side, then the next column tile, so that its weights leave memory once
  const int low = HAS_LOW ? low_rows<MT>(A.M) : 0, rts = low ? A.M / R::BM : (A.M + R::BM - 1) / R::BM;
  const int nts = (A.N + R::BN - 1) / R::BN, tiles = rts * nts, total = tiles * A.S;
  const int all = low ? nts * A.S : 0, per = (total + 7) >> 3, both = (total + all + 7) >> 3;   // low tiles; of an XCD: whole tiles, tiles
  const int k8 = blockIdx.x >> 3, x8 = blockIdx.x & 7, whole = max(0, min(per, total - x8 * per));
  if (k8 < whole) {                                  // (uniform)
    const int item = x8 * per + k8;
    constexpr int GR = 2048 / R::BM;
    const int sp = item / tiles, it = item - sp * tiles, g = it / (GR * nts), j = it - g * GR * nts, in_g = min(GR, rts - g * GR);
    const int nt = j / in_g, row0 = (g * GR + j - nt * in_g) * R::BM;
    tile<MT, NT, OCC, WNT>(A, smem, sp, nt, row0, min(R::BM, A.M - row0));
  } else if constexpr (HAS_LOW) {
    const int item = x8 * both - min(x8 * per, total) + k8 - whole;
    if (k8 >= both || item >= all) return;
    tile<LOW / 32, NT, OCC, WNT>(A, smem, item / nts, item % nts, rts * R::BM, low);
  }
}

// act: 1, 3 W tiled as gate, up pairs (silu or gelu(gate) * up into Y, slabs in gate | up order), 2 relu squared into Y
extern "C" hipError_t kafka_launch_tile_gemm(const bf16* X, int64_t ldx, const bf16* Wt, int M, int N, int K, int mt, int nt,
                                             int splits, int act, bf16* Y, int64_t ldy, float* P, hipStream_t st) {
  if (M <= 0) return hipSuccess;
  const bool glu = act & 1;
  if (act < 0 || act > 3 || (act == 2 && P)) return hipErrorInvalidValue;
  if (glu && Y && nt % 4) return hipErrorInvalidValue;   // (a wave holds whole gate, up pairs)
  if (N < 32 || N % 32 || K % 64 || splits < 1 || K / 64 < 2 * splits || ldx % 8 || (glu && N % 64)) return hipErrorInvalidValue;
  if ((Y != nullptr) == (P != nullptr) || (Y && (splits != 1 || ldy % 8 || reinterpret_cast<uintptr_t>(Y) % 16)))
    return hipErrorInvalidValue;
  if (reinterpret_cast<uintptr_t>(X) % 16 || 256 * ldx * 2 > (int64_t)0xffff0000 || (int64_t)N * K * 2 > (int64_t)0xffff0000)
    return hipErrorInvalidValue;
  const int mode = P ? (glu ? OUT_SLAB_GLU : OUT_SLAB) : (act == 1 ? OUT_GLU : act == 2 ? OUT_RELU2 : act == 3 ? OUT_GELU : OUT_BF16);
  const TileArgs A{X, ldx, reinterpret_cast<const bf16x8*>(Wt), M, N, K, splits, Y, ldy, P, mode};
  const int64_t nts = (int64_t)((N + 32 * nt - 1) / (32 * nt)) * splits;
  if ((M + 32 * mt - 1) / (32 * mt) * nts > 0x0fffffff) return hipErrorInvalidValue;
  auto a = [&](auto kern) {
    const int64_t total = (M + 32 * mt - 1) / (32 * mt) * nts;   // (the low tiles among them)
    kern<<<(unsigned)((total + 7) / 8 * 8), 256, 0, st>>>(A);
  };
  // 128 x 128: two workgroups share a CU and its LDS, with two units of activations and three of weights each. Where each has a CU to itself five of
  // both fit, which long loops without splits on 96 workgroups and more are the faster for (us, sharing / alone: 96 - 256 workgroups of K = 2048 17.4 - 19.6 /
  // 14.9 - 17.9, of 7168 57 / 48, 1000 rows of 4096 -> 4096 37.0 / 35.9); 64 - 72 of them take 13.8 / 14.3, and short loops wait for all that is asked
  // for in front of them (splits of 512 10.8 - 14 / 11.7 - 15, of 896 - 1024 16.4 - 19 / 17.1 - 20, of 3584 as long).
  const int64_t wgs = (M + 127) / 128 * nts;
  if (mt == 4 && nt == 4 && splits == 1 && K >= 2048 && wgs >= 96 && wgs <= 256) {
    if (M <= 128) a(tile_gemm_kernel<4, 4, 1, true>);
    else a(tile_gemm_kernel<4, 4, 1, false>);
    return hipGetLastError();
  }
#define TILE(MT, NT, OCC)                                        \
  if (mt == MT && nt == NT) {                                    \
    if (M <= 32 * MT) a(tile_gemm_kernel<MT, NT, OCC, true>);    \
    else a(tile_gemm_kernel<MT, NT, OCC, false>);                \
    return hipGetLastError();                                    \
  }
  TILE(8, 8, 1)
  TILE(8, 4, 1)
  TILE(8, 6, 1)
  TILE(7, 8, 1)
  TILE(7, 6, 1)
  TILE(7, 4, 1)
  TILE(6, 8, 1)
  TILE(6, 6, 1)
  TILE(5, 8, 1)
  TILE(5, 4, 1)
  TILE(4, 6, 1)
  TILE(4, 8, 1)
  TILE(4, 4, 2)
#undef TILE
  return hipErrorInvalidValue;
}

}  // namespace tg
}  // namespace kafka
