// Small products of bf16 rows with row-major weights: Y[b][m][n] = sum_k X[b][m][k] W[b][n][k], fp32 sums, bf16 or fp32 results
// (gfx950). Gates and routers (few columns, long rows), low-rank projections (short rows, many columns) and the products of
// latent attention's heads (a small product per head): what has neither a tiled copy nor the size for one.
//
// What bounds it: a round trip to memory, a launch, and with long rows what a CU takes in: 16 waves share K, and their operands come
// through LDS in whole cache lines of a row (straight to the registers a load takes half a line of 16 rows). us, K = 4096, before / now:
// 8 columns 16 rows 7.5 / 4.1, 2048 8.1 / 5.8, 8192 15.6 / 14.0; 64 columns 64 rows 9.1 / 4.8, 300 9.4 / 5.6, 2048 17.1 / 10.3, 4096 32 / 20.4; 32 columns
// 4096 rows 17.2 / 12.3. The library's call costs the host 17 us and this one 3, which is what steps of few rows wait for.
// us, library on the GPU / this kernel: 64 columns of K = 4096, 64 rows 7.6 / 4.8, 2048 15.2 / 10.3, 4096 15.9 / 20.4; 8 columns of 1900 rows
// 15.3 / 5.8, with the call 18.8, 8192 21 / 14; 32 columns of 1900 rows 20 / 6.3; 4096 columns of
// K = 64, 64 rows 3.6 / 3.3, 300 5.4 / 4.7, 900 5.8 / 8.4; 2048 of K = 16, 64 rows 4.0 / 2.8, 4096 10.1 / 8.9; 8192 of K = 128, 128 rows
// 4.7 / 4.6, 300 6.3 / 9.8; 32 heads of 128 -> 512, 64 rows 4.6 / 4.6, 128 5.5 / 7.9, of 512 -> 128, 64 rows 8.6 / 4.7, 300 15.3 / 16.1.
#include "common.h"

namespace kafka {
namespace sg {

typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_t;
struct Strides {
  int64_t xb, xm, wb, wn, yb, ym;
};
// what a product's rows meet. GELU_GATE: gelu(sum) * emb[tok[m]][n] (rows outside the table: NaN). SIGMOID_GATE: the sum as bf16, times
// sigmoid(emb[m][b * rows + n]), head b's part of a row of gates (a launch of its own: 4.0 us of 64 rows of 32 heads of 128).
enum { NO_GATE, GELU_GATE, SIGMOID_GATE };
struct Gate {
  const int64_t* tok;
  const bf16* emb;
  int64_t stride, rows;
};

// A wave: 16 rows x 16 NT columns over its share of K. KW waves of a workgroup share K (their sums meet in LDS), the other
// 4 / KW (KW up to 4) take further columns. Products are taken with the weights first: a lane holds four columns of one row.
template <int NT, int KW, bool F32, int GATE = NO_GATE>
__global__ __launch_bounds__(64 * (KW > 4 ? KW : 4)) void small_gemm_kernel(const bf16* __restrict__ X, const bf16* __restrict__ W,
                                                                            int M, int N, int K, const float* __restrict__ bias,
                                                                            void* __restrict__ Y, Strides st, Gate gate) {
  constexpr int NW = KW > 4 ? KW : 4, CW = NW / KW;   // waves; column parts
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, q = lane >> 4;
  const int kw = w % KW, m0 = blockIdx.x * 16, n0 = (blockIdx.y * CW + w / KW) * 16 * NT, b = blockIdx.z;
  // shares of K in whole steps of 32
  const int steps = (K + 31) >> 5, s0 = steps * kw / KW, s1 = steps * (kw + 1) / KW;
  const bf16* x = X + b * st.xb + (int64_t)min(m0 + r, M - 1) * st.xm + 8 * q;
  const bf16* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) wp[t] = W + b * st.wb + (int64_t)min(n0 + 16 * t + r, N - 1) * st.wn + 8 * q;
  f32x4v acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4v{0.f, 0.f, 0.f, 0.f};
  const bf16x8 zero = {};
  auto step = [&](int s, bool in) {
    const bf16x8 xv = in ? load_bf16x8(x + 32 * s) : zero;
#pragma unroll
    for (int t = 0; t < NT; ++t)
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(in ? load_bf16x8(wp[t] + 32 * s) : zero, xv, acc[t], 0, 0, 0);
  };
  const int whole = min(s1, K >> 5);                 // (a last step of 8, 16 or 24: the lanes past K bring zeros)
  int s = s0;
  if constexpr (KW == 16) {
    // ST steps at a time through LDS of the wave's own, a load whole cache lines of a row; a row's 16-byte pieces turned by its number
    constexpr int ST = NT == 1 ? 4 : 2, ROW = 64 * ST, PCS = 4 * ST, TILE = 16 * ROW;   // bytes and pieces of a row
    __shared__ __attribute__((aligned(16))) unsigned char ring[NW * (1 + NT) * TILE];
    unsigned char* const my = ring + w * (1 + NT) * TILE;
    for (; s + ST <= whole; s += ST) {
#pragma unroll
      for (int i = 0; i < TILE / 1024; ++i) {
        const int row = i * (64 / PCS) + lane / PCS, at = 32 * s + ((lane ^ row) & (PCS - 1)) * 8;
        __builtin_amdgcn_global_load_lds(X + b * st.xb + (int64_t)min(m0 + row, M - 1) * st.xm + at, (lds_t*)(my + i * 1024), 16, 0, 0);
#pragma unroll
        for (int t = 0; t < NT; ++t)
          __builtin_amdgcn_global_load_lds(W + b * st.wb + (int64_t)min(n0 + 16 * t + row, N - 1) * st.wn + at,
                                           (lds_t*)(my + (1 + t) * TILE + i * 1024), 16, 0, 0);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      bf16x8 xv[ST], wv[ST][NT];
#pragma unroll
      for (int j = 0; j < ST; ++j) {
        const unsigned char* f = my + r * ROW + (((4 * j + q) ^ r) & (PCS - 1)) * 16;
        xv[j] = *reinterpret_cast<const bf16x8*>(f);
#pragma unroll
        for (int t = 0; t < NT; ++t) wv[j][t] = *reinterpret_cast<const bf16x8*>(f + (1 + t) * TILE);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (read, before the next loads land there)
#pragma unroll
      for (int j = 0; j < ST; ++j)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[j][t], xv[j], acc[t], 0, 0, 0);
    }
  }
  constexpr int U = 4;                               // steps whose loads are in flight together
  for (; KW < 16 && s + U <= whole; s += U) {
    bf16x8 xv[U], wv[U][NT];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      xv[j] = load_bf16x8(x + 32 * (s + j));
#pragma unroll
      for (int t = 0; t < NT; ++t) wv[j][t] = load_bf16x8(wp[t] + 32 * (s + j));
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < U; ++j)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[j][t], xv[j], acc[t], 0, 0, 0);
  }
  for (; s < whole; ++s) step(s, true);
  if (s < s1) step(s, 32 * s + 8 * q < K);
  if constexpr (KW > 1) {
    __shared__ f32x4v part[NW][NT][64];
#pragma unroll
    for (int t = 0; t < NT; ++t) part[w][t][lane] = acc[t];
    __syncthreads();
    if (kw) return;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 1; j < KW; ++j) acc[t] += part[w + j][t][lane];
  }
  const int m = m0 + r;
  if (m >= M) return;
  const int64_t tok = GATE == GELU_GATE ? gate.tok[m] : 0;
  const bool known = tok >= 0 && tok < gate.rows;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int n = n0 + 16 * t + 4 * q;               // (N is a multiple of 4)
    if (n >= N) continue;
    const int64_t at = b * st.yb + (int64_t)m * st.ym + n;
    if constexpr (F32) {
      if (bias) acc[t] += *reinterpret_cast<const f32x4v*>(bias + n);
      *reinterpret_cast<f32x4v*>(reinterpret_cast<float*>(Y) + at) = acc[t];
    } else {
      bf16x4 o, g;
      if constexpr (GATE == SIGMOID_GATE) g = *reinterpret_cast<const bf16x4*>(gate.emb + m * gate.stride + b * gate.rows + n);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (GATE == SIGMOID_GATE)
          o[i] = (bf16)((float)(bf16)acc[t][i] * (1.0f / (1.0f + expf(-(float)g[i]))));
        else if constexpr (GATE == GELU_GATE)
          o[i] = known ? (bf16)(gate_act(acc[t][i], true) * (float)gate.emb[tok * gate.stride + n + i]) : (bf16)__builtin_nanf("");
        else
          o[i] = (bf16)acc[t][i];
      }
      *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16*>(Y) + at) = o;
    }
  }
}

extern "C" hipError_t kafka_launch_small_gemm(const bf16* X, const bf16* W, int B, int M, int N, int K, int64_t xb, int64_t xm,
                                              int64_t wb, int64_t wn, const float* bias, int f32, void* Y, int64_t yb, int64_t ym,
                                              const int64_t* tok, const bf16* emb, int64_t emb_stride, int64_t emb_rows,
                                              hipStream_t st) {
  // tok: a gelu gate; emb alone: a sigmoid gate of rows emb_stride apart, a head's part emb_rows wide
  const Gate gate{tok, emb, emb_stride, emb_rows};
  const bool sig = tok == nullptr && emb != nullptr;
  if (sig && (f32 || bias || emb_stride % 4 || emb_rows % 4 || reinterpret_cast<uintptr_t>(emb) % 8)) return hipErrorInvalidValue;
  if (tok != nullptr && (f32 || bias || B != 1 || K < 1024)) return hipErrorInvalidValue;
  if (B < 1 || M < 1 || N < 1) return hipSuccess;
  const uintptr_t ya = reinterpret_cast<uintptr_t>(Y);
  if (N % 4 || K < 8 || K % 8 || xb % 8 || xm % 8 || wb % 8 || wn % 8 || yb % 4 || ym % 4 || reinterpret_cast<uintptr_t>(X) % 16 ||
      reinterpret_cast<uintptr_t>(W) % 16 || ya % (f32 ? 16 : 8) || B > 65535 ||
      (bias && (!f32 || reinterpret_cast<uintptr_t>(bias) % 16)) || (N + 15) / 16 > 65535)
    return hipErrorInvalidValue;
  const Strides s{xb, xm, wb, wn, yb, ym};
  const int rows = (M + 15) / 16;
  auto go = [&](auto kern, int nt, int kw) {
    const int cols = 16 * nt * (kw >= 4 ? 1 : 4 / kw);
    kern<<<dim3(rows, (N + cols - 1) / cols, B), 64 * (kw > 4 ? kw : 4), 0, st>>>(X, W, M, N, K, bias, Y, s, gate);
    return hipGetLastError();
  };
  // Long K: 16 waves share it, a workgroup per 16 columns (64 columns of 4096 in one workgroup of 8 waves 9.0 us at 64 rows, so 4.8);
  // in between 4 waves; short K: a wave takes 64 columns alone.
  // Gates of more rows than one round of such workgroups: 32 columns each, one round again. us at 2048 rows of 64 columns, the library and the gate's
  // launch / 16 columns / 32: K = 4096 21.6 / 11.0 / 8.9, 2048 11.5 / 7.9 / 6.6; 3000 rows (two rounds)
  // of K = 4096 18.5, 17.1 on 32 columns, of 2048 11.8, 12.1.
  if (tok != nullptr)
    return N > 32 && (int64_t)rows * ((N + 15) / 16) > 256 ? go(small_gemm_kernel<2, 16, false, GELU_GATE>, 2, 16)
                                                           : go(small_gemm_kernel<1, 16, false, GELU_GATE>, 1, 16);
  if (sig)
    return K >= 1024  ? go(small_gemm_kernel<1, 16, false, SIGMOID_GATE>, 1, 16)
           : K >= 256 ? go(small_gemm_kernel<2, 4, false, SIGMOID_GATE>, 2, 4)
                      : go(small_gemm_kernel<4, 1, false, SIGMOID_GATE>, 4, 1);
  if (K >= 1024) return f32 ? go(small_gemm_kernel<1, 16, true>, 1, 16) : go(small_gemm_kernel<1, 16, false>, 1, 16);
  if (K >= 256) return f32 ? go(small_gemm_kernel<2, 4, true>, 2, 4) : go(small_gemm_kernel<2, 4, false>, 2, 4);
  return f32 ? go(small_gemm_kernel<4, 1, true>, 4, 1) : go(small_gemm_kernel<4, 1, false>, 4, 1);
}

}  // namespace sg
}  // namespace kafka
