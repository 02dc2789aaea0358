// RMSNorm, fused residual-add + RMSNorm, and SwiGLU activation for gfx950.
//
// All three are HBM-bound streaming ops: one workgroup per token row, 16-byte (bf16x8) loads per lane, the
// row kept in registers between the reduction and the scale pass (one HBM read + one write per element),
// fp32 accumulation. The residual add is fused into the norm so the decoder layer reads the residual
// stream once per sub-block instead of three times.
//
// Split-K slab inputs: the decode GEMM (wstream_gemm.hip) leaves its output as S fp32 partial slabs
// P[S][T][n]; every kernel here can take such a slab instead of a bf16 input and sums the S partials while
// loading (load_in8 in common.h), so the split-K combine costs no launch of its own.
#include <cstdlib>

#include "common.h"

namespace kafka {

// y = x * rsqrt(mean(x^2) + eps) * w     (x: [T, d] with row stride, out: [T, d] contiguous)
// If RESID: r = x + r (rounded to bf16, written back to r), y = norm(r) * w.
template <int NV, bool RESID, int NT = 256, bool SC1 = false>
__global__ __launch_bounds__(NT) void rmsnorm_kernel(bf16* __restrict__ out, int64_t out_stride,
                                                       const bf16* __restrict__ x, const float* __restrict__ xp,
                                                       int S, int64_t ps, int64_t x_stride,
                                                       bf16* __restrict__ resid, int64_t r_stride,
                                                       const bf16* __restrict__ w, int d, float eps) {
  __shared__ float red[NT / 64];
  const int64_t row = blockIdx.x;
  const int nvec = d >> 3;
  float v[NV][8];
  float ss = 0.f;
  // the weight loads go out with the row loads (not after the reduction: one HBM round trip instead of two)
  bf16x8 wv[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int vi = threadIdx.x + i * NT;
    if (vi < nvec) wv[i] = load_bf16x8(w + vi * 8);
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int vi = threadIdx.x + i * NT;
    if (vi < nvec) {
      load_in8(v[i], x, xp, S, ps, row * x_stride + vi * 8);
      if constexpr (RESID) {
        const bf16x8 b = load_bf16x8(resid + row * r_stride + vi * 8);
        bf16x8 s;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          s[j] = (bf16)(v[i][j] + (float)b[j]);
          v[i][j] = (float)s[j];
        }
        if constexpr (SC1)
          store16_slab(reinterpret_cast<float*>(resid + row * r_stride + vi * 8), __builtin_bit_cast(f32x4, s));
        else
          store_bf16x8(resid + row * r_stride + vi * 8, s);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) ss += v[i][j] * v[i][j];
    }
  }
  ss = block_sum<NT>(ss, red);
  const float r = rsqrtf(ss / (float)d + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int vi = threadIdx.x + i * NT;
    if (vi < nvec) {
      bf16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (bf16)(v[i][j] * r * (float)wv[i][j]);
      if constexpr (SC1)
        store16_slab(reinterpret_cast<float*>(out + row * out_stride + vi * 8), __builtin_bit_cast(f32x4, o));
      else
        store_bf16x8(out + row * out_stride + vi * 8, o);
    }
  }
}

// out[t, :] = silu(x[t, :F]) * x[t, F:]   (x: [T, 2F] row stride xs (bf16 or slabs), out: [T, F] contiguous)
// SLABS: load_in8's choice by the number of slabs stands out of the way of bf16 rows, whose two loads otherwise wait for each other on
// twice the registers: 4099 rows of 2 x 14336 66 -> 53 us (6.6 TB/s, partly from the memory-side cache).
template <bool SLABS>
__global__ __launch_bounds__(256) void silu_mul_kernel(bf16* __restrict__ out, const bf16* __restrict__ x,
                                                        const float* __restrict__ xp, int S, int64_t ps,
                                                        int64_t xs, int F, bool gelu) {
  const int64_t row = blockIdx.y;
  const int nvec = F >> 3;
  for (int vi = blockIdx.x * 256 + threadIdx.x; vi < nvec; vi += gridDim.x * 256) {
    float g[8], u[8];
    if constexpr (SLABS) {
      load_in8(g, nullptr, xp, S, ps, row * xs + vi * 8);
      load_in8(u, nullptr, xp, S, ps, row * xs + F + vi * 8);
    } else {
      const bf16x8 a = load_bf16x8(x + row * xs + vi * 8), b = load_bf16x8(x + row * xs + F + vi * 8);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        g[j] = (float)a[j];
        u[j] = (float)b[j];
      }
    }
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = (bf16)(gate_act(g[j], gelu) * u[j]);
    store_bf16x8(out + row * (int64_t)F + vi * 8, o);
  }
}

template <bool RESID>
static hipError_t launch_rmsnorm_t(bf16* out, int64_t os, const bf16* x, const float* xp, int S, int64_t ps,
                                   int64_t xs, bf16* r, int64_t rs, const bf16* w, int T, int d, float eps,
                                   hipStream_t st) {
  const int nvec = d / 8;
  const int nv = (nvec + 255) / 256;
  dim3 grid(T), block(256);
  if (T == 0) return hipSuccess;
  // outputs (normalised rows and the in-place residual) as 16-B sc1 stores — the lines leave this XCD's L2, so the
  // launch ends with none of them dirty (+2.1 % on the headline with RoPE's, profiles/r06/ab/); KAFKA_SC1_NORM=0 keeps
  // plain stores. Needs 16-B aligned rows. common.h "Store / load scopes"
  static const bool sc1 = [] {
    const char* e = getenv("KAFKA_SC1_NORM");
    return e == nullptr || e[0] != '0';
  }();
  if (nvec <= 512 && nvec > 256) {  // e.g. d = 4096: one 16-B vector per thread, twice the loads in flight per row
    if (sc1 && os % 8 == 0 && rs % 8 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0 &&
        (!RESID || reinterpret_cast<uintptr_t>(r) % 16 == 0))
      rmsnorm_kernel<1, RESID, 512, true><<<grid, 512, 0, st>>>(out, os, x, xp, S, ps, xs, r, rs, w, d, eps);
    else
      rmsnorm_kernel<1, RESID, 512><<<grid, 512, 0, st>>>(out, os, x, xp, S, ps, xs, r, rs, w, d, eps);
    return hipGetLastError();
  }
  switch (nv) {
    case 1: rmsnorm_kernel<1, RESID><<<grid, block, 0, st>>>(out, os, x, xp, S, ps, xs, r, rs, w, d, eps); break;
    case 2: rmsnorm_kernel<2, RESID><<<grid, block, 0, st>>>(out, os, x, xp, S, ps, xs, r, rs, w, d, eps); break;
    case 3:
    case 4: rmsnorm_kernel<4, RESID><<<grid, block, 0, st>>>(out, os, x, xp, S, ps, xs, r, rs, w, d, eps); break;
    default: rmsnorm_kernel<8, RESID><<<grid, block, 0, st>>>(out, os, x, xp, S, ps, xs, r, rs, w, d, eps); break;
  }
  return hipGetLastError();
}

// ---- rows picked by an index ---------------------------------------------------------------------------------------------
// The two ends of a step: the tokens' rows of the embedding with the first layer's norm, and the rows whose logits are asked for with
// the last one's. Three launches of torch's gathers (3 - 11 us each for a few rows: its small-index kernel walks the
// index) beside two norms become two launches. A row outside the table comes out as NaN.
// us a step of one row 455 -> 450, of 64 rows 829 -> 822, 29 rows on the small cache 744 -> 733.
template <int NV, int NT, bool EMBED>
__global__ __launch_bounds__(NT) void rows_norm_kernel(bf16* __restrict__ out, int64_t out_stride, const bf16* __restrict__ x,
                                                       int64_t x_stride, const float* __restrict__ xp, int S, int64_t ps,
                                                       bf16* __restrict__ resid, int64_t r_stride,
                                                       const int64_t* __restrict__ idx, int64_t n_src,
                                                       const bf16* __restrict__ w, int d, float eps) {
  __shared__ float red[NT / 64];
  const int64_t row = blockIdx.x, src = idx[row];
  const bool in = src >= 0 && src < n_src;
  const int64_t from = in ? src : 0;
  const int nvec = d >> 3;
  float v[NV][8];
  float ss = in ? 0.f : __builtin_nanf("");
  bf16x8 wv[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int vi = threadIdx.x + i * NT;
    if (vi < nvec) wv[i] = load_bf16x8(w + vi * 8);
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int vi = threadIdx.x + i * NT;
    if (vi < nvec) {
      load_in8(v[i], x, xp, S, ps, from * x_stride + vi * 8);
      if constexpr (EMBED) {   // the row itself begins the residual stream
        bf16x8 s;
#pragma unroll
        for (int j = 0; j < 8; ++j) s[j] = in ? (bf16)v[i][j] : (bf16)__builtin_nanf("");
        store_bf16x8(resid + row * r_stride + vi * 8, s);
      } else {
        const bf16x8 b = load_bf16x8(resid + from * r_stride + vi * 8);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] = (float)(bf16)(v[i][j] + (float)b[j]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) ss += v[i][j] * v[i][j];
    }
  }
  ss = block_sum<NT>(ss, red);
  const float r = rsqrtf(ss / (float)d + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int vi = threadIdx.x + i * NT;
    if (vi < nvec) {
      bf16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (bf16)(v[i][j] * r * (float)wv[i][j]);
      store_bf16x8(out + row * out_stride + vi * 8, o);
    }
  }
}

// embed: resid[i] = x[idx[i]], out[i] = norm(resid[i]); else out[i] = norm(x[idx[i]] + resid[idx[i]]), x bf16 or S slabs xp
extern "C" hipError_t kafka_launch_rows_norm(bf16* out, int64_t os, const bf16* x, int64_t xs, const float* xp, int S, int64_t ps,
                                             bf16* resid, int64_t rs, const int64_t* idx, int64_t n_src, const bf16* w, int n,
                                             int d, float eps, int embed, hipStream_t st) {
  if (n == 0) return hipSuccess;
  const int nvec = d / 8;
  auto go = [&](auto kern, int nt) {
    kern<<<n, nt, 0, st>>>(out, os, x, xs, xp, S, ps, resid, rs, idx, n_src, w, d, eps);
    return hipGetLastError();
  };
  if (nvec <= 512 && nvec > 256) return embed ? go(rows_norm_kernel<1, 512, true>, 512) : go(rows_norm_kernel<1, 512, false>, 512);
  if (nvec <= 256) return embed ? go(rows_norm_kernel<1, 256, true>, 256) : go(rows_norm_kernel<1, 256, false>, 256);
  if (nvec <= 1024) return embed ? go(rows_norm_kernel<4, 256, true>, 256) : go(rows_norm_kernel<4, 256, false>, 256);
  return embed ? go(rows_norm_kernel<8, 256, true>, 256) : go(rows_norm_kernel<8, 256, false>, 256);
}

// out[i] = src[idx[i]] in 16-byte pieces, a workgroup per row and 16 KB. ALSO 1: the rows a second time, 2: fp32 rows in bf16 as well. (A
// copy or conversion of its own: 4.7 us of 64 rows of 4096 fp32, 11 us of 2048 - 2805.)
template <int ALSO>
__global__ __launch_bounds__(256) void gather_rows_kernel(char* __restrict__ out, int64_t out_bytes, const char* __restrict__ src,
                                                          int64_t src_bytes, const int64_t* __restrict__ idx, int64_t n_src,
                                                          int row_bytes, char* __restrict__ also, int64_t also_bytes) {
  typedef int i32x4 __attribute__((ext_vector_type(4)));
  const int64_t s = idx[blockIdx.x];
  const bool in = s >= 0 && s < n_src;
  const char* from = src + (in ? s : 0) * src_bytes;
  char* to = out + (int64_t)blockIdx.x * out_bytes;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int at = ((int)blockIdx.y * 1024 + i * 256 + (int)threadIdx.x) * 16;
    if (at < row_bytes) {
      i32x4 v = *reinterpret_cast<const i32x4*>(from + at);
      if (!in) v = i32x4{-1, -1, -1, -1};   // (NaN as fp32 and as bf16)
      *reinterpret_cast<i32x4*>(to + at) = v;
      if constexpr (ALSO == 1) *reinterpret_cast<i32x4*>(also + (int64_t)blockIdx.x * also_bytes + at) = v;
      if constexpr (ALSO == 2) {
        const f32x4 f = __builtin_bit_cast(f32x4, v);
        *reinterpret_cast<bf16x4*>(also + (int64_t)blockIdx.x * also_bytes + at / 2) = bf16x4{(bf16)f[0], (bf16)f[1], (bf16)f[2], (bf16)f[3]};
      }
    }
  }
}

// also: nullptr, or rows of the same type (also_half 0), or bf16 rows of fp32 ones (1)
extern "C" hipError_t kafka_launch_gather_rows(void* out, int64_t out_bytes, const void* src, int64_t src_bytes, const int64_t* idx,
                                               int64_t n_src, int n, int row_bytes, void* also, int64_t also_bytes, int also_half,
                                               hipStream_t st) {
  if (n == 0) return hipSuccess;
  auto a = [&](auto k) {
    k<<<dim3(n, (row_bytes + 16383) / 16384), 256, 0, st>>>((char*)out, out_bytes, (const char*)src, src_bytes, idx, n_src, row_bytes,
                                                            (char*)also, also_bytes);
  };
  if (also == nullptr) a(gather_rows_kernel<0>);
  else if (also_half) a(gather_rows_kernel<2>);
  else a(gather_rows_kernel<1>);
  return hipGetLastError();
}

// Bytes of pinned host memory (dst and src at whole 8-byte pieces) into device memory, 16 KB a workgroup, eight loads of a
// thread in flight. Bound by the host link. A copy engine takes the queue from the kernels and gives it back, which is
// most of the time of a step's plan (about 20 us before the first kernel); this is one more kernel of the queue: a step of four Llama
// layers takes 727 -> 715 us with 29 sequences of 7900 tokens, 764 -> 756 with 64 behind a shared prompt. The loads are of system scope, because the host
// writes the same memory again a few steps later and a cache that holds the old bytes must not answer.
__global__ __launch_bounds__(256) void host_copy_kernel(char* __restrict__ dst, const char* src, int64_t n) {
  const int64_t n8 = n / 8, first = (int64_t)blockIdx.x * 2048 + threadIdx.x;
  const uint64_t* from = reinterpret_cast<const uint64_t*>(src);
  uint64_t v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int64_t at = first + i * 256;
    if (at < n8) v[i] = __hip_atomic_load(from + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int64_t at = first + i * 256;
    if (at < n8) reinterpret_cast<uint64_t*>(dst)[at] = v[i];
  }
  const int64_t tail = n8 * 8 + threadIdx.x;
  if (blockIdx.x == 0 && tail < n)
    dst[tail] = __hip_atomic_load(src + tail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

extern "C" hipError_t kafka_launch_host_copy(void* dst, const void* src, int64_t n, hipStream_t st) {
  if (n == 0) return hipSuccess;
  host_copy_kernel<<<(unsigned)((n + 16383) / 16384), 256, 0, st>>>((char*)dst, (const char*)src, n);
  return hipGetLastError();
}

extern "C" hipError_t kafka_launch_rmsnorm(bf16* out, int64_t os, const bf16* x, int64_t xs, const bf16* w, int T, int d,
                          float eps, hipStream_t st) {
  return launch_rmsnorm_t<false>(out, os, x, nullptr, 0, 0, xs, nullptr, 0, w, T, d, eps, st);
}

extern "C" hipError_t kafka_launch_fused_add_rmsnorm(bf16* out, int64_t os, const bf16* x, int64_t xs, bf16* resid, int64_t rs,
                                    const bf16* w, int T, int d, float eps, hipStream_t st) {
  return launch_rmsnorm_t<true>(out, os, x, nullptr, 0, 0, xs, resid, rs, w, T, d, eps, st);
}

// fused add + RMSNorm whose x input is S fp32 split-K slabs [S][T][d] (row stride d, slab stride ps)
extern "C" hipError_t kafka_launch_fused_add_rmsnorm_slab(bf16* out, int64_t os, const float* xp, int S, int64_t ps,
                                                         bf16* resid, int64_t rs, const bf16* w, int T, int d,
                                                         float eps, hipStream_t st) {
  return launch_rmsnorm_t<true>(out, os, nullptr, xp, S, ps, d, resid, rs, w, T, d, eps, st);
}

extern "C" hipError_t kafka_launch_silu_mul(bf16* out, const bf16* x, int64_t xs, int T, int F, int gelu, hipStream_t st) {
  if (T == 0) return hipSuccess;
  const int nvec = F / 8;
  int gx = (nvec + 255) / 256;
  if (gx > 64) gx = 64;
  silu_mul_kernel<false><<<dim3(gx, T), dim3(256), 0, st>>>(out, x, nullptr, 0, 0, xs, F, gelu != 0);
  return hipGetLastError();
}

// SwiGLU over S fp32 split-K slabs [S][T][2F]
extern "C" hipError_t kafka_launch_silu_mul_slab(bf16* out, const float* xp, int S, int64_t ps, int T, int F,
                                                int gelu, hipStream_t st) {
  if (T == 0) return hipSuccess;
  const int nvec = F / 8;
  int gx = (nvec + 255) / 256;
  if (gx > 64) gx = 64;
  silu_mul_kernel<true><<<dim3(gx, T), dim3(256), 0, st>>>(out, nullptr, xp, S, ps, 2 * (int64_t)F, F, gelu != 0);
  return hipGetLastError();
}

}  // namespace kafka
