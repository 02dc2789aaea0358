// Kernels for decoders with hyper-connected residual streams, windowed softmax attention with sinks and group-limited
// routing, for gfx950.
//
// Every kernel is built for bf16 and for fp32 activations; the residual streams and their mixing, norm statistics,
// rotation, attention scores and weights, router scores and the value mix are fp32 in both. Sizes are run-time values
// with no alignment assumptions.
//
//   stream_step         one pass over S residual streams [S][T][d] (fp32): the write of a sublayer's output (all
//                       streams at once from the old ones: x_r <- sum_s M[s][r] x_s + b_r y), the next sublayer's read
//                       u = sum_s a_s x_s with its RMS norm, and the plain sum - every part optional. One workgroup
//                       per row; a row's columns are loaded in one round, and its read values stay in registers
//                       between the statistics and the scaling.
//   swish_clamp_mul     g' sigmoid(alpha g') (u' + 1) with g' = min(g, limit), u' = clamp(u, -limit, limit)
//   qk_norm_rope_store  RMS norm over the whole q and the whole k projection, rotation of dimension pairs (2i, 2i + 1),
//                       value mix with an earlier layer's values, paged key / transposed value store
//   window_attn         softmax attention with a sliding window and a sink logit; one wave per (row, head): lane = key
//                       for the scores (the query row broadcast from LDS), online softmax over 64-key blocks, then
//                       lane = value channel reading its channel's 16 consecutive tokens of a transposed page; a
//                       row's keys are visited in order, whatever the batch
//   window_attn_rows    the same attention on the matrix cores (bf16): 32 (token, head) rows of one key/value head, scores
//                       transposed so that rows are lanes - maxima, sums and weights stay in a lane's registers. Prompt portions: a
//                       wave each, no LDS and no barriers; decoded tokens: keys over the waves of a workgroup, and over several
//                       workgroups with a merge pass
//   window_attn_tile    the same for long portions of 128 channels, four items on one walk over keys in LDS
//   moe_topk_grouped    softmax or sigmoid scores, choice among the best groups (by their largest score or the sum of
//                       their two largest) by corrected score, weights normalised or as they are, times a scale
#include "common.h"

#include <type_traits>

namespace kafka {
namespace hs {

template <typename T>
__device__ __forceinline__ float ldf(const T* p) { return (float)(*p); }
template <typename T>
__device__ __forceinline__ void stf(T* p, float v) { *p = (T)v; }
// element i of a bf16 or fp32 array chosen at run time (uniform over the launch)
__device__ __forceinline__ float ldx(const void* p, bool f32, int64_t i) {
  return f32 ? reinterpret_cast<const float*>(p)[i] : (float)reinterpret_cast<const bf16*>(p)[i];
}

constexpr int NT = 256;
constexpr int PAGE = 16;
constexpr float LOG2E = 1.4426950408889634f;

// Workgroup barrier for LDS hand-overs that leaves global loads (a prefetched next block) in flight: __syncthreads()
// would drain them as well. This wave's LDS reads and writes are complete (lgkmcnt 0) before it arrives.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// ---- residual streams ----------------------------------------------------------------------------------------------
constexpr int SMAX = 16;   // streams
// columns of a row a thread keeps in registers (all S streams of each): rows up to NT * stream_nv(S) wide are loaded in
// one round of independent loads, written once, and their read values wait in registers for the row's mean square;
// wider rows walk the rest column by column and recompute the read values from the streams just written
__host__ __device__ constexpr int stream_nv(int S) { return S <= 4 ? 16 : S <= 8 ? 8 : 4; }

template <int S>
__global__ __launch_bounds__(NT) void stream_step_kernel(float* __restrict__ xs, int64_t s_stride, int64_t t_stride,
                                                         const void* __restrict__ y, int64_t ys, bool y_f32,
                                                         const void* __restrict__ y2, int64_t y2s, bool y2_f32,
                                                         const float* __restrict__ row_scale,
                                                         const float* __restrict__ mix, const float* __restrict__ wr,
                                                         const float* __restrict__ rd, const float* __restrict__ nw,
                                                         float eps, void* __restrict__ out, int64_t os, bool out_f32,
                                                         float* __restrict__ total, int64_t ts, int d, bool center) {
  constexpr int NV = stream_nv(S);
  __shared__ float red[NT / 64];
  __shared__ float cM[SMAX * SMAX], cb[SMAX], ca[SMAX];
  const int64_t t = blockIdx.x;
  for (int i = threadIdx.x; i < S * S; i += NT)
    if (mix != nullptr) cM[i] = mix[i];
  if (threadIdx.x < S) {
    if (wr != nullptr) cb[threadIdx.x] = wr[threadIdx.x];
    if (rd != nullptr) ca[threadIdx.x] = rd[threadIdx.x];
  }
  __syncthreads();
  float* xr = xs + t * t_stride;
  const float rs2 = y2 != nullptr ? row_scale[t] : 0.f;
  // new stream values of one column from the old ones and the sublayer's output
  auto write = [&](float (&x)[S], float yv) {
    float nx[S];
#pragma unroll
    for (int r = 0; r < S; ++r) {
      float v = cb[r] * yv;
#pragma unroll
      for (int s = 0; s < S; ++s) v += cM[s * S + r] * x[s];
      nx[r] = v;
    }
#pragma unroll
    for (int s = 0; s < S; ++s) x[s] = nx[s];
  };
  auto read = [&](const float (&x)[S]) {
    float u = 0.f;
#pragma unroll
    for (int s = 0; s < S; ++s) u += ca[s] * x[s];
    return u;
  };
  float xv[NV][S], yv[NV];
  float acc = 0.f, accs = 0.f;   // sum of squares and plain sum of the read values
  // the register part: every load of the row's first NT * NV columns is issued before anything is stored
#pragma unroll
  for (int it = 0; it < NV; ++it) {
    const int i = threadIdx.x + it * NT;
    yv[it] = 0.f;
    if (i < d) {
#pragma unroll
      for (int s = 0; s < S; ++s) xv[it][s] = xr[s * s_stride + i];
      if (mix != nullptr) {
        yv[it] = ldx(y, y_f32, t * ys + i);
        if (y2 != nullptr) yv[it] += rs2 * ldx(y2, y2_f32, t * y2s + i);
      }
    }
  }
#pragma unroll
  for (int it = 0; it < NV; ++it) {
    const int i = threadIdx.x + it * NT;
    if (i < d) {
      if (mix != nullptr) {
        write(xv[it], yv[it]);
#pragma unroll
        for (int s = 0; s < S; ++s) xr[s * s_stride + i] = xv[it][s];
      }
      if (total != nullptr) {
        float v = 0.f;
#pragma unroll
        for (int s = 0; s < S; ++s) v += xv[it][s];
        total[t * ts + i] = v;
      }
      if (rd != nullptr) {
        const float u = read(xv[it]);
        acc += u * u;
        accs += u;
        yv[it] = u;  // (the sublayer output is used up: its register keeps the read value)
      }
    }
  }
  for (int i = threadIdx.x + NV * NT; i < d; i += NT) {
    float x[S];
#pragma unroll
    for (int s = 0; s < S; ++s) x[s] = xr[s * s_stride + i];
    if (mix != nullptr) {
      float v = ldx(y, y_f32, t * ys + i);
      if (y2 != nullptr) v += rs2 * ldx(y2, y2_f32, t * y2s + i);
      write(x, v);
#pragma unroll
      for (int s = 0; s < S; ++s) xr[s * s_stride + i] = x[s];
    }
    if (total != nullptr) {
      float v = 0.f;
#pragma unroll
      for (int s = 0; s < S; ++s) v += x[s];
      total[t * ts + i] = v;
    }
    if (rd != nullptr) {
      const float u = read(x);
      acc += u * u;
      accs += u;
    }
  }
  if (rd == nullptr) return;
  // a centred norm takes the row's mean off first and measures the deviations in a second pass over the read values
  float mean = 0.f;
  if (center) {
    mean = block_sum<NT>(accs, red) / (float)d;
    acc = 0.f;
#pragma unroll
    for (int it = 0; it < NV; ++it) {
      const int i = threadIdx.x + it * NT;
      if (i < d) acc += (yv[it] - mean) * (yv[it] - mean);
    }
    for (int i = threadIdx.x + NV * NT; i < d; i += NT) {
      float x[S];
#pragma unroll
      for (int s = 0; s < S; ++s) x[s] = xr[s * s_stride + i];
      const float u = read(x) - mean;
      acc += u * u;
    }
  }
  const float rs = 1.0f / sqrtf(block_sum<NT>(acc, red) / (float)d + eps);
  auto store = [&](int i, float u) {
    const float v = (u - mean) * rs * nw[i];
    if (out_f32) reinterpret_cast<float*>(out)[t * os + i] = v;
    else reinterpret_cast<bf16*>(out)[t * os + i] = (bf16)v;
  };
#pragma unroll
  for (int it = 0; it < NV; ++it) {
    const int i = threadIdx.x + it * NT;
    if (i < d) store(i, yv[it]);
  }
  for (int i = threadIdx.x + NV * NT; i < d; i += NT) {  // (this thread's own writes of the first pass)
    float x[S];
#pragma unroll
    for (int s = 0; s < S; ++s) x[s] = xr[s * s_stride + i];
    store(i, read(x));
  }
}

template <typename AT>
__global__ void swish_clamp_mul_kernel(const AT* __restrict__ gu, int64_t gs, AT* __restrict__ out, int64_t os, int64_t T,
                                       int F, float limit, float alpha) {
  const int64_t n = T * F;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = i / F;
    const int f = (int)(i - t * F);
    const float g = fminf(ldf(gu + t * gs + f), limit);
    const float u = fminf(fmaxf(ldf(gu + t * gs + F + f), -limit), limit);
    stf(out + t * os + f, g / (1.0f + expf(-alpha * g)) * (u + 1.0f));
  }
}

// the same on bf16 rows whose sizes, strides and bases are multiples of 8 elements: 8 gate and 8 up values per thread step
__global__ void swish_clamp_mul_vec8_kernel(const bf16* __restrict__ gu, int64_t gs, bf16* __restrict__ out, int64_t os,
                                            int64_t T, int F, float limit, float alpha) {
  const int F8 = F >> 3;
  const int64_t n = T * F8;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = i / F8;
    const int f = (int)(i - t * F8) << 3;
    const bf16x8 gv = load_bf16x8(gu + t * gs + f), uv = load_bf16x8(gu + t * gs + F + f);
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float g = fminf((float)gv[j], limit);
      const float u = fminf(fmaxf((float)uv[j], -limit), limit);
      o[j] = (bf16)(g / (1.0f + expf(-alpha * g)) * (u + 1.0f));
    }
    store_bf16x8(out + t * os + f, o);
  }
}

// ---- attention inputs ------------------------------------------------------------------------------------------------
// one workgroup per row of the fused projection [q (H D) | k (G D) | v (G Dv)]
template <typename AT>
__global__ __launch_bounds__(NT) void qk_norm_rope_store_kernel(
    const AT* __restrict__ qkv, int64_t qs, int H, int G, int D, int Dv, const float* __restrict__ qw,
    const float* __restrict__ kw, float eps, const int64_t* __restrict__ positions, const float* __restrict__ cos_sin,
    int dims, const AT* __restrict__ vf, int64_t vfs, int vf_off, float lam, AT* __restrict__ kc, AT* __restrict__ vt,
    const int64_t* __restrict__ slots, AT* __restrict__ q_out, int64_t qos) {
  __shared__ float red[NT / 64];
  const int64_t t = blockIdx.x;
  const int Cq = H * D, Ck = G * D, Cv = G * Dv;
  const AT* row = qkv + t * qs;
  float sq = 0.f, sk = 0.f;
  for (int i = threadIdx.x; i < Cq; i += NT) {
    const float v = ldf(row + i);
    sq += v * v;
  }
  for (int i = threadIdx.x; i < Ck; i += NT) {
    const float v = ldf(row + Cq + i);
    sk += v * v;
  }
  const float rq = 1.0f / sqrtf(block_sum<NT>(sq, red) / (float)Cq + eps);
  const float rk = 1.0f / sqrtf(block_sum<NT>(sk, red) / (float)Ck + eps);
  const int half = dims >> 1;
  const float* cs = dims > 0 ? cos_sin + positions[t] * dims : nullptr;
  const int64_t slot = slots[t];
  // element i of a normed projection, rotated with its pair partner when it lies in a head's first `dims` dimensions
  auto elem = [&](const AT* src, const float* w, float r, int i) {
    const float a = ldf(src + i) * r * w[i];
    const int dh = i % D;
    if (dh >= dims) return a;
    const int ip = (dh & 1) ? i - 1 : i + 1;  // the pair partner within the head
    const float b = ldf(src + ip) * r * w[ip];
    const float c = cs[dh >> 1], s = cs[half + (dh >> 1)];
    return (dh & 1) ? a * c + b * s : a * c - b * s;
  };
  for (int i = threadIdx.x; i < Cq; i += NT) stf(q_out + t * qos + i, elem(row, qw, rq, i));
  if (slot < 0) return;
  AT* kd = kc + slot * Ck;
  for (int i = threadIdx.x; i < Ck; i += NT) stf(kd + i, elem(row + Cq, kw, rk, i));
  AT* vd = vt + (slot / PAGE) * (int64_t)Cv * PAGE + (slot % PAGE);
  for (int i = threadIdx.x; i < Cv; i += NT) {
    float v = ldf(row + Cq + Ck + i);
    if (vf != nullptr) v = (1.0f - lam) * v + lam * ldf(vf + t * vfs + vf_off + i);
    stf(vd + (int64_t)i * PAGE, v);
  }
}

// ---- windowed softmax attention with a sink -----------------------------------------------------------------------
// sigmoid of a head's raw gate: a factor on the head's whole output
template <typename T>
__device__ __forceinline__ float head_gate(const T* p) { return 1.0f / (1.0f + expf(-ldf(p))); }

constexpr int WA_MAXD = 1024;  // query / key size (the query row sits in LDS as fp32)
constexpr int WA_NV = 8;      // value size up to 64 * WA_NV

template <typename AT>
__global__ __launch_bounds__(NT) void window_attn_kernel(const AT* __restrict__ q, int64_t qs,
                                                         const AT* __restrict__ kc, const AT* __restrict__ vt,
                                                         const int* __restrict__ bt, int bt_stride,
                                                         const int* __restrict__ tok_seg,
                                                         const int64_t* __restrict__ positions, int H, int G, int D,
                                                         int Dv, int Ck, int kstep, float scale_log2e, int window,
                                                         const float* __restrict__ sink,
                                                         const AT* __restrict__ gate, int64_t gs,
                                                         AT* __restrict__ out, int64_t os, int64_t pairs,
                                                         float out_scale) {
  // D: size of a query row and of the key it meets; key/value head g's key starts at column g * kstep of a key row of
  // Ck columns (kstep = D: one key head per key/value head; kstep = 0, D = Ck: every query row meets the whole key row)
  __shared__ float qsh[NT / 64][WA_MAXD];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t pair = (int64_t)blockIdx.x * (NT / 64) + wave;
  if (pair >= pairs) return;  // whole waves leave; nothing below synchronises across waves
  const int64_t t = pair / H;
  const int h = (int)(pair - t * H);
  const int g = h / (H / G);
  const int64_t p = positions[t];
  const int* pages = bt + (int64_t)tok_seg[t] * bt_stride;
  float* qw = qsh[wave];
  for (int i = lane; i < D; i += 64) qw[i] = ldf(q + t * qs + (int64_t)h * D + i) * scale_log2e;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int Cv = G * Dv;
  float acc[WA_NV];
#pragma unroll
  for (int i = 0; i < WA_NV; ++i) acc[i] = 0.f;
  // the sink is a term of the denominator without a value: the running maximum and sum start from it
  float m = -INFINITY, l = 0.f;
  if (sink != nullptr) {
    m = sink[h] * LOG2E;
    l = 1.f;
  }
  const int64_t lo = window > 0 ? (p - window + 1 > 0 ? p - window + 1 : 0) : 0;  // first visible key
  for (int64_t j0 = lo & ~(int64_t)(PAGE - 1); j0 <= p; j0 += 64) {
    const int64_t j = j0 + lane;
    float s = -INFINITY;
    if (j <= p && j >= lo) {
      const AT* kr = kc + ((int64_t)pages[j / PAGE] * PAGE + (j % PAGE)) * Ck + (int64_t)g * kstep;
      float dot = 0.f;
      for (int i = 0; i < D; ++i) dot += qw[i] * ldf(kr + i);
      s = dot;
    }
    const float mn = fmaxf(m, wave_max(s));  // finite: the block holds a visible key (j0 <= p and j0 + 63 >= lo)
    const float corr = fast_exp2(m - mn);    // 0 while m is -inf
    const float w = fast_exp2(s - mn);       // 0 for masked keys
    l = l * corr + wave_sum(w);
    m = mn;
    const int nk = (int)((p - j0 + 1 < 64) ? (p - j0 + 1) : 64);  // keys of this block up to the row's own
#pragma unroll
    for (int i = 0; i < WA_NV; ++i) acc[i] *= corr;
    for (int pg = 0; pg * PAGE < nk; ++pg) {
      const int64_t page = pages[(j0 >> 4) + pg];
      const int ne = (nk - pg * PAGE < PAGE) ? nk - pg * PAGE : PAGE;
      float wk[PAGE];
#pragma unroll
      for (int e = 0; e < PAGE; ++e) wk[e] = __shfl(w, pg * PAGE + e, 64);
#pragma unroll
      for (int i = 0; i < WA_NV; ++i) {
        const int v = lane + 64 * i;
        if (v < Dv) {
          const AT* vp = vt + (page * Cv + (int64_t)g * Dv + v) * PAGE;
          float a = acc[i];
#pragma unroll
          for (int e = 0; e < PAGE; ++e)
            if (e < ne) a += wk[e] * ldf(vp + e);
          acc[i] = a;
        }
      }
    }
  }
  float inv = out_scale / l;
  if (gate != nullptr) inv *= head_gate(gate + t * gs + h);
#pragma unroll
  for (int i = 0; i < WA_NV; ++i) {
    const int v = lane + 64 * i;
    if (v < Dv) stf(out + t * os + (int64_t)h * Dv + v, acc[i] * inv);
  }
}

// ---- windowed softmax attention on the matrix cores (bf16) --------------------------------------------------------
// An item is 32 query rows = (token, query head) pairs of consecutive tokens of one segment for one key/value head
// (floor(32 / rep) tokens, rep = H / G query heads per key/value head). A wave walks keys 32 at a time:
//   scores   S^T = K Q^T: lane = row, a lane's 16 registers = its half of the block's keys. The key rows are loaded with
//            bits 2 and 3 of their numbers swapped, which leaves lane half lh with keys 8 lh .. + 7 of each page;
//   softmax  a row's maximum, sum and weights live in its two lanes; the accumulators are rescaled only when a row's
//            maximum has moved;
//   values   O^T += V^T P^T: the weights are the right operand as they lie in the registers, the left one is a channel's
//            8 consecutive tokens of a transposed page (16 bytes).
// Keys ahead of the row or behind its window count as -inf; scores, maxima, sums and accumulators are fp32; the sink joins the
// denominator once, at the end. Needs 16-token pages, D % 16 == 0, at most 32 query heads per key/value head. NKS, NVT: steps of 16
// key channels and tiles of 32 value channels held in registers (queries past D are zero).
//   prompt portions: a wave per item, no LDS and no barriers; the four waves of a workgroup are neighbouring items (the same
//     keys, from the cache), a key/value head's workgroups go to one XCD where there are eight of them, the items with the most
//     keys first.
//   SPLIT, decoded tokens: a workgroup per item (one key/value head's side by side), its blocks of keys dealt to the four waves in turn, the waves' maxima, sums and
//     accumulators met in LDS at the end. With gridDim.z > 1 the item's blocks are dealt to that many workgroups in contiguous
//     ranges; each leaves its unnormalised accumulators in po [z][T][H Dv] and (row maximum, row sum) in pml [z][T][H][2] for
//     window_merge. What bounds it: the round trips of a block, which is why no wave waits for another in the walk: with the scores
//     of 128 keys shared through LDS, three barriers a block and the values asked for behind them, us (operands from memory, with the
//     merge; before / now): 16 sequences x 1700 keys, 32 heads over 8, 38 / 28, 64 sequences 102 / 86 (4.6 TB/s), one x 8000 28 / 19, 128 x
//     300 43 / 34; 32 over 2, 128 x 1700, 70 / 44; 64 channels, 64 x 1700, 65 / 46; 256 channels, 16 over 4, 16 x 1700 52 / 34. Two
//     blocks in flight a wave (one wave a SIMD) 31, 84, 21, 48, 47, 47, 37; past the caches' retention 42, 110, 28, 42 (a line
//     of keys is four loads).
constexpr int WM_ROWS = 32;

template <int NKS, int NVT, bool SPLIT>
__global__ __launch_bounds__(256, NKS * 4 + NVT * 16 <= 96 ? 2 : 1) void window_attn_rows_kernel(
    const bf16* __restrict__ q, int64_t qs, const bf16* __restrict__ kc, const bf16* __restrict__ vt,
    const int* __restrict__ bt, int bt_stride, const int* __restrict__ items, int n_items,
    const int64_t* __restrict__ positions, int H, int G, int D, int Dv, int Ck, int kstep, float scale_log2e, int window,
    const float* __restrict__ sink, const bf16* __restrict__ gate, int64_t gs, bf16* __restrict__ out, int64_t os,
    float out_scale, int tok_lim, bool vec4, float* __restrict__ po, float* __restrict__ pml, int64_t T) {
  constexpr int STEP = SPLIT ? 4 : 1;   // blocks from a wave's one to its next
  const int lane = threadIdx.x & 63, lr = lane & 31, lh = lane >> 5, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int item = __builtin_amdgcn_readfirstlane(
      SPLIT ? (int)(blockIdx.x % (unsigned)n_items) : n_items - 1 - ((int)blockIdx.y * (int)(blockDim.x >> 6) + (int)(threadIdx.x >> 6)));
  if (item < 0) return;   // whole waves leave; nothing below synchronises across waves unless SPLIT
  const int t0 = items[4 * item], ntok = items[4 * item + 1], sg = items[4 * item + 2];   // (uniform)
  if (SPLIT ? ntok > tok_lim : ntok < tok_lim) return;   // (an item of the other form)
  const int g = SPLIT ? blockIdx.x / (unsigned)n_items : blockIdx.x, rep = H / G, nks = D >> 4, nrows = ntok * rep;
  const bool live = lr < nrows;
  const int row = min(lr, nrows - 1), h = g * rep + row % rep;
  const int64_t t = t0 + row / rep;
  const int p = (int)positions[t], minpos = (int)positions[t0], maxpos = (int)positions[t0 + ntok - 1];
  const int* btr = bt + (int64_t)sg * bt_stride;
  const int Cv = G * Dv;
  bf16x8 qf[NKS], kf[NKS];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) {
    qf[ks] = load_bf16x8(q + t * qs + (int64_t)h * D + 16 * min(ks, nks - 1) + 8 * lh);
    if (ks >= nks) qf[ks] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
  }
  const int krow = (lr & 19) | ((lr & 4) << 1) | ((lr & 8) >> 1);   // bits 2 and 3 swapped
  // the two pages of a block (past the item's last position: the last valid one, masked below)
  const int lastpg = maxpos >> 4;
  auto page_of = [&](int kb, int pg) { return btr[min(2 * kb + pg, lastpg)]; };
  auto fetch_keys = [&](int pa, int pb) {
    const bf16* kp = kc + ((int64_t)(krow & 16 ? pb : pa) * PAGE + (krow & 15)) * Ck + (int64_t)g * kstep + 8 * lh;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) kf[ks] = load_bf16x8(kp + 16 * min(ks, nks - 1));
  };
  float m = -INFINITY, l = 0.f;
  f32x16 O[NVT];
#pragma unroll
  for (int v = 0; v < NVT; ++v)
#pragma unroll
    for (int i = 0; i < 16; ++i) O[v][i] = 0.f;
  int kb0 = window > 0 ? max(0, minpos - window + 1) >> 5 : 0, kb1 = (maxpos >> 5) + 1;
  if constexpr (SPLIT) {   // of the z-th of gridDim.z ranges, every fourth
    const int per = (kb1 - kb0 + (int)gridDim.z - 1) / (int)gridDim.z;
    kb0 += (int)blockIdx.z * per;
    kb1 = min(kb1, kb0 + per);
    kb0 += w;
  }
  int pa = page_of(kb0, 0), pb = page_of(kb0, 1), na = page_of(kb0 + STEP, 0), nb = page_of(kb0 + STEP, 1);
  fetch_keys(pa, pb);
  for (int kb = kb0; kb < kb1; kb += STEP) {
    const int fa = page_of(kb + 2 * STEP, 0), fb = page_of(kb + 2 * STEP, 1);   // (two blocks ahead)
    bf16x8 vf[2][NVT];
#pragma unroll
    for (int pg = 0; pg < 2; ++pg) {
      const bf16* vp = vt + ((int64_t)(pg ? pb : pa) * Cv + (int64_t)g * Dv) * PAGE + 8 * lh;
#pragma unroll
      for (int v = 0; v < NVT; ++v) vf[pg][v] = load_bf16x8(vp + (int64_t)min(32 * v + lr, Dv - 1) * PAGE);
    }
    f32x16 S;
#pragma unroll
    for (int i = 0; i < 16; ++i) S[i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) S = mfma32(kf[ks], qf[ks], S);
    fetch_keys(na, nb);
    pa = na;
    pb = nb;
    na = fa;
    nb = fb;
    float s[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = S[i] * scale_log2e;
    // (uniform) a block that every row sees whole needs no mask
    if (32 * kb + 31 > minpos || (window > 0 && 32 * kb <= maxpos - window)) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = 32 * kb + 16 * (i >> 3) + 8 * lh + (i & 7);
        if (key > p || (window > 0 && key <= p - window)) s[i] = -INFINITY;
      }
    }
    float mx = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mn = fmaxf(m, mx);
    const float base = mn == -INFINITY ? 0.f : mn;   // nothing visible yet: every weight is 2^-inf = 0
    if (__any(mx > m)) {
      const float corr = m == -INFINITY ? 0.f : fast_exp2(m - base);
      l *= corr;
#pragma unroll
      for (int v = 0; v < NVT; ++v)
#pragma unroll
        for (int i = 0; i < 16; ++i) O[v][i] *= corr;
    }
    m = mn;
    bf16x8 pf[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float e = fast_exp2(s[i] - base);
      l += e;
      pf[i >> 3][i & 7] = (bf16)e;
    }
#pragma unroll
    for (int pg = 0; pg < 2; ++pg)
#pragma unroll
      for (int v = 0; v < NVT; ++v) O[v] = mfma32(vf[pg][v], pf[pg], O[v]);
  }
  // the last products' results are complete before anything reads them behind a branch
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 15");
  __builtin_amdgcn_sched_barrier(0);
  l += __shfl_xor(l, 32, 64);
  if constexpr (SPLIT) {
    constexpr int LO = 32 * NVT + 4;
    __shared__ __attribute__((aligned(16))) float part[4 * WM_ROWS * LO];   // [wave][row]
    __shared__ float ml[4][WM_ROWS][2];
    if (live) {
      if (lh == 0) {
        ml[w][lr][0] = m;
        ml[w][lr][1] = l;
      }
#pragma unroll
      for (int v = 0; v < NVT; ++v)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4)
          *reinterpret_cast<f32x4*>(part + (w * WM_ROWS + lr) * LO + 32 * v + 8 * i4 + 4 * lh) =
              f32x4{O[v][4 * i4], O[v][4 * i4 + 1], O[v][4 * i4 + 2], O[v][4 * i4 + 3]};
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nrows * Dv; i += 256) {
      const int r = i / Dv, c = i - r * Dv, hr = g * rep + r % rep;
      const int64_t tr = t0 + r / rep;
      const float mn = fmaxf(fmaxf(ml[0][r][0], ml[1][r][0]), fmaxf(ml[2][r][0], ml[3][r][0]));
      // (a range may lie wholly outside a row's window: then mn is -inf and the row stays empty)
      float o = 0.f, lt = 0.f;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float f = ml[k][r][0] == -INFINITY ? 0.f : fast_exp2(ml[k][r][0] - mn);
        lt += f * ml[k][r][1];
        o += f * part[(k * WM_ROWS + r) * LO + c];
      }
      if (gridDim.z == 1) {
        if (sink != nullptr) lt += fast_exp2(sink[hr] * LOG2E - mn);
        float inv = out_scale / lt;
        if (gate != nullptr) inv *= head_gate(gate + tr * gs + hr);
        out[tr * os + (int64_t)hr * Dv + c] = (bf16)(o * inv);
      } else {
        const int64_t at = ((int64_t)blockIdx.z * T + tr) * H + hr;
        if (c == 0) {
          pml[2 * at] = mn;
          pml[2 * at + 1] = lt;
        }
        po[at * Dv + c] = o;
      }
    }
    return;
  }
  if (!live) return;
  if (sink != nullptr) l += fast_exp2(sink[h] * LOG2E - m);
  float inv = out_scale / l;
  if (gate != nullptr) inv *= head_gate(gate + t * gs + h);
  bf16* op = out + t * os + (int64_t)h * Dv;
#pragma unroll
  for (int v = 0; v < NVT; ++v)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const int c = 32 * v + 8 * i4 + 4 * lh;
      if (vec4) {
        typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
        if (c < Dv) {
          const bf16x4 o = {(bf16)(O[v][4 * i4] * inv), (bf16)(O[v][4 * i4 + 1] * inv), (bf16)(O[v][4 * i4 + 2] * inv),
                            (bf16)(O[v][4 * i4 + 3] * inv)};
          *reinterpret_cast<bf16x4*>(op + c) = o;
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c + e < Dv) op[c + e] = (bf16)(O[v][4 * i4 + e] * inv);
      }
    }
}

// ---- the same for long portions, 128 channels: four items share their keys in LDS ------------------------------------------
// A workgroup takes four neighbouring items of one key/value head, a wave each (as above: S^T = K Q^T, the weights stay in
// registers, O^T += V^T P^T), and walks the union of their keys 64 at a time; two workgroups share a CU. Chunk c (16 bytes) of key row k lies
// at c ^ k of its page, the halves of channels 8 .. 15 of every 16 in a V^T page are swapped: every operand read meets all banks once. Items
// of different segments go one segment after the other, the rest of the workgroup helps loading. The accumulators are rescaled only
// when a row's maximum has grown by more than 2^WT_THR.
// A wave is a pipeline over the tiles, as in attn_tile.h: the next tile's products with the keys stand between this one's exponentials, its
// products with the values between the rest of them and the next maxima, and eight fragments are on their way from LDS at any time. K and V^T
// pages have two slots each, without a register on the way (buffer loads); the keys run a tile ahead, and both slots that a step has read are
// filled again in its middle, where the waves meet.
// What bounds it: LDS (32 KB of fragments a wave and tile) and the clock. us in a step, products and softmax of a tile one after the other and
// eight waves a workgroup / now: 8192 fresh rows x 32 heads over 8 594 / 518 (1.06 PFLOP/s), 1100, 843 and 862 rows, 32 over 2, 48.4 / 43.2. (Before
// that a wave's operands came through the caches, twice as long.)
constexpr int WT_WAVES = 4, WT_KEYS = 64, WT_SLOTS = 2, WT_RUN = 512;   // WT_RUN: tiles whose page ids lie in LDS at a time
constexpr int WT_KB = WT_KEYS * 256, WT_PIECES = 16 / WT_WAVES;         // bytes of a tile's keys; 1-KiB pieces of them that a wave copies
constexpr float WT_THR = 8.f;
// Items (those that it works on, not the single tokens between them) x key/value heads from which it runs: a wave each on 256 CUs, fewer leave
// whole CUs idle that the form above still uses. us there / here, 32 heads over 2 or 8, one portion, behind 3000 keys, three portions, ten behind
// 200: 500 waves 15 / 15, 74 / 58, 8.6 / 12.5, 11 / 17; 1000 waves 32 / 24, 132 / 71, 16 / 16, 17 / 19; 1150 42 / 27, 196 / 87, 22 / 16, 25 / 23;
// 1280 48 / 30, 203 / 92, 27 / 19, 28 / 19. The line is that of eight waves a workgroup, which were even at 1200 - 1500; with four it is ahead
// from 1000 - 1150 on, and behind long histories well below that.
constexpr int WT_MIN_WAVES = 1280;

typedef __attribute__((address_space(3))) void wt_lds_t;
// pieces C .. of a page from g on (uniform), this lane's bytes of each less 1 KiB a piece, which the immediate adds on both sides
template <int C = 0>
__device__ __forceinline__ void wt_dma(const char* g, const int (&at)[WT_PIECES], unsigned char* lds) {
  if constexpr (C < WT_PIECES) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(buf_rsrc(g), (wt_lds_t*)lds, 16, at[C], 0, 1024 * C, 0);
    wt_dma<C + 1>(g, at, lds);
  }
}
__device__ __forceinline__ float wt_max(float a, float b) { return __builtin_elementwise_maximum(a, b); }

__global__ __launch_bounds__(64 * WT_WAVES, 2) void window_attn_tile_kernel(
    const bf16* __restrict__ q, int64_t qs, const bf16* __restrict__ kc, const bf16* __restrict__ vt,
    const int* __restrict__ bt, int bt_stride, const int* __restrict__ items, int n_items,
    const int64_t* __restrict__ positions, int H, int G, int Ck, int kstep, float scale_log2e, int window,
    const float* __restrict__ sink, const bf16* __restrict__ gate, int64_t gs, bf16* __restrict__ out, int64_t os,
    float out_scale, int min_tok, bool vec4) {
  constexpr int D = 128, Dv = 128, NKS = 8, NVT = 4;
  __shared__ __attribute__((aligned(16))) unsigned char smem[2 * WT_SLOTS * WT_KB + 4 * WT_RUN * 4 + WT_WAVES * 16];
  int* pg_s = reinterpret_cast<int*>(smem + 2 * WT_SLOTS * WT_KB);   // [4 WT_RUN]
  int4* who = reinterpret_cast<int4*>(pg_s + 4 * WT_RUN);            // [waves] (segment or -1, first tile, end tile, last page)
  const int lane = threadIdx.x & 63, lr = lane & 31, lh = lane >> 5, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int item = n_items - 1 - ((int)blockIdx.y * WT_WAVES + w);
  int t0 = 0, ntok = 0, sg = -1;
  if (item >= 0) {
    t0 = items[4 * item];
    ntok = items[4 * item + 1];
    sg = ntok >= min_tok ? items[4 * item + 2] : -1;
  }
  const bool mine = sg >= 0;   // (uniform per wave)
  const int g = blockIdx.x, rep = H / G, nrows = max(ntok, 1) * rep, Cv = G * Dv;
  const int row = min(lr, nrows - 1), h = g * rep + row % rep;
  const int64_t t = t0 + row / rep;
  int p = -1, minpos = 0, maxpos = -1;
  bf16x8 qf[NKS];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) qf[ks] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
  if (mine) {
    p = (int)positions[t];
    minpos = (int)positions[t0];
    maxpos = (int)positions[t0 + ntok - 1];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) qf[ks] = load_bf16x8(q + t * qs + (int64_t)h * D + 16 * ks + 8 * lh);
  }
  const int jb = window > 0 ? max(0, minpos - window + 1) / WT_KEYS : 0, je = maxpos / WT_KEYS + 1;   // tiles of this wave
  if (lane == 0) who[w] = int4{sg, jb, je, maxpos >> 4};
  const int krow = (lr & 19) | ((lr & 4) << 1) | ((lr & 8) >> 1), kk = krow & 15;   // bits 2 and 3 swapped
  int kat[NKS];             // operands' places in a slot
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) kat[ks] = (krow >> 4) * 4096 + kk * 256 + 16 * ((2 * ks + lh) ^ kk);
  const int vat = WT_SLOTS * WT_KB + lr * 32 + 16 * (lh ^ ((lr >> 3) & 1));
  // wave w copies WT_PIECES 1-KiB pieces of K and of V^T of page pw of a tile
  constexpr int PW = 4 / WT_PIECES;                 // waves of a page
  const int pw = w / PW, c0 = (w % PW) * WT_PIECES;
  int ksrc[WT_PIECES], vsrc[WT_PIECES];
#pragma unroll
  for (int c = 0; c < WT_PIECES; ++c) {
    const int k = 4 * (c0 + c) + (lane >> 4);
    ksrc[c] = k * Ck * 2 + 16 * ((lane & 15) ^ k) - 1024 * c;   // (Ck >= 128: not below zero)
    vsrc[c] = c0 * 1024 + (lane ^ ((lane >> 4) & 1)) * 16;
  }
  // group i of the run: the keys of tile i and the values of tile i - 1
  auto page_of = [&](int i, int n) { return pg_s[4 * min(i, n - 1) + pw]; };
  auto issue = [&](int i, int n, int64_t kpage, int64_t vpage) {
    unsigned char* const dst = smem + pw * 4096 + c0 * 1024;
    if (i < n)
      wt_dma(reinterpret_cast<const char*>(kc + kpage * PAGE * Ck + (int64_t)g * kstep), ksrc, dst + (i % WT_SLOTS) * WT_KB);
    if (i > 0)
      wt_dma(reinterpret_cast<const char*>(vt + (vpage * Cv + (int64_t)g * Dv) * PAGE), vsrc,
             dst + (WT_SLOTS + (i + WT_SLOTS - 1) % WT_SLOTS) * WT_KB);
  };
  float m = -INFINITY, l = 0.f;
  f32x16 O[NVT], sa[2], sb[2];
#pragma unroll
  for (int v = 0; v < NVT; ++v)
#pragma unroll
    for (int i = 0; i < 16; ++i) O[v][i] = 0.f;
  bf16x8 fr[8];             // fragments on their way: 16 of keys (32-key half f & 1, depth f >> 1), 16 of values (page f >> 2, channels f & 3)
  auto kfrag = [&](const unsigned char* k, int f) { return *reinterpret_cast<const bf16x8*>(k + kat[f >> 1] + (f & 1) * 8192); };
  auto vfrag = [&](const unsigned char* v, int f) { return *reinterpret_cast<const bf16x8*>(v + vat + (f >> 2) * 4096 + (f & 3) * 1024); };
  __builtin_amdgcn_s_waitcnt(0x0F70);   // (vmcnt(0): left open, the queries' loads are waited for, with the tiles', in every step)
  lds_barrier();
  for (int a = 0; a < WT_WAVES;) {   // (uniform) waves a .. b - 1 walk one segment
    const int4 wa = who[a];
    const int seg = __builtin_amdgcn_readfirstlane(wa.x);
    int b = a + 1, lo = __builtin_amdgcn_readfirstlane(wa.y), hi = __builtin_amdgcn_readfirstlane(wa.z),
        lastpg = __builtin_amdgcn_readfirstlane(wa.w);
    for (; b < WT_WAVES; ++b) {
      const int4 wb = who[b];
      if (__builtin_amdgcn_readfirstlane(wb.x) != seg) break;
      lo = min(lo, __builtin_amdgcn_readfirstlane(wb.y));
      hi = max(hi, __builtin_amdgcn_readfirstlane(wb.z));
      lastpg = max(lastpg, __builtin_amdgcn_readfirstlane(wb.w));
    }
    const bool on = w >= a && w < b;
    a = b;
    if (seg < 0) continue;
    const int* btr = bt + (int64_t)seg * bt_stride;
    for (int run = lo; run < hi; run += WT_RUN) {
      const int n = min(hi - run, WT_RUN);
      for (int i = threadIdx.x; i < 4 * n; i += 64 * WT_WAVES) pg_s[i] = btr[min(4 * run + i, lastpg)];   // (past the last page: it again)
      lds_barrier();
      int last_page = 0, next_page = 0;              // of the keys of the group issued last; of the next one's, on its way
#pragma unroll
      for (int i = 0; i < WT_SLOTS; ++i) {
        const int pg = __builtin_amdgcn_readfirstlane(page_of(i, n));
        if (i <= n) issue(i, n, pg, last_page);
        last_page = pg;
      }
      next_page = page_of(WT_SLOTS, n);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      lds_barrier();
      // this wave's reads of the keys of tile j + 1 and the values of tile j are done, group j + 2 has landed; then everyone's: the slots are
      // filled again
      auto meet = [&](int j) {
        static_assert(WT_SLOTS == 2, "the wait");
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
        const int i = j + 1 + WT_SLOTS;
        if (i <= n) {
          const int pg = __builtin_amdgcn_readfirstlane(next_page);
          issue(i, n, pg, last_page);
          last_page = pg;
          next_page = page_of(i + 1, n);
        }
      };
      // step j: CUR: tile j, whose scores S holds, is this wave's; NXT: tile j + 1 is, its scores go to T
      auto step = [&](auto cur_c, auto nxt_c, int j, f32x16(&S)[2], f32x16(&T)[2]) {
        constexpr bool CUR = decltype(cur_c)::value, NXT = decltype(nxt_c)::value;
        const unsigned char *kc1 = smem + ((j + 1) % WT_SLOTS) * WT_KB, *kc2 = smem + ((j + 2) % WT_SLOTS) * WT_KB,
                            *vc = smem + (max(j, 0) % WT_SLOTS) * WT_KB;
        const float base = m == -INFINITY ? 0.f : m;   // nothing visible yet: every weight is 2^-inf = 0
        bf16x8 pf[2], pg[2];
        auto prob = [&](float x) {
          const float e = fast_exp2(fmaf(x, scale_log2e, -base));
          l += e;
          return (bf16)e;
        };
        if constexpr (!CUR && NXT) {
#pragma unroll
          for (int f = 0; f < 8; ++f) fr[f] = kfrag(kc1, f);
        }
        if constexpr (CUR && !NXT) {
#pragma unroll
          for (int f = 0; f < 8; ++f) fr[f] = vfrag(vc, f);
#pragma unroll
          for (int i = 0; i < 16; ++i) pf[i >> 3][i & 7] = prob(S[0][i]);
        }
        if constexpr (NXT) {
#pragma unroll
          for (int f = 0; f < 16; ++f) {
            const f32x16 zero = {};
            T[f & 1] = mfma32(fr[f & 7], qf[f >> 1], f < 2 ? zero : T[f & 1]);
            if (f < 8) fr[f] = kfrag(kc1, f + 8);
            else if (CUR) fr[f - 8] = vfrag(vc, f - 8);
            if (CUR) pf[f >> 3][f & 7] = prob(S[0][f]);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        if constexpr (CUR) {
#pragma unroll
          for (int f = 0; f < 8; ++f) {
            O[f & 3] = mfma32(fr[f], pf[f >> 2], O[f & 3]);
            fr[f] = vfrag(vc, f + 8);
            pg[f >> 2][2 * (f & 3)] = prob(S[1][2 * f]);
            pg[f >> 2][2 * (f & 3) + 1] = prob(S[1][2 * f + 1]);
            __builtin_amdgcn_sched_barrier(0);
          }
          // (the compiler would move the exponentials to the products that take them)
          asm volatile("" : "+v"(pg[0]), "+v"(pg[1]));
        }
        meet(j);
        float ma = 0.f, mb = 0.f;
        if constexpr (NXT) {
          const int key0 = (run + j + 1) * WT_KEYS;
          // (uniform) a tile that every row sees whole needs no mask
          if (key0 + WT_KEYS - 1 > minpos || (window > 0 && key0 <= maxpos - window)) {
#pragma unroll
            for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
              for (int i = 0; i < 16; ++i) {
                const int key = key0 + 32 * s2 + 16 * (i >> 3) + 8 * lh + (i & 7);
                if (key > p || (window > 0 && key <= p - window)) T[s2][i] = -INFINITY;
              }
          }
          ma = wt_max(T[0][0], T[1][0]), mb = wt_max(T[0][1], T[1][1]);
        }
#pragma unroll
        for (int f = 0; f < 8; ++f) {
          if constexpr (CUR) O[f & 3] = mfma32(fr[f], pg[f >> 2], O[f & 3]);
          if constexpr (NXT) {
            fr[f] = kfrag(kc2, f);                     // (past the run's last tile: not used)
            if (f > 0) {
              ma = wt_max(wt_max(ma, T[0][2 * f]), T[1][2 * f]);
              mb = wt_max(wt_max(mb, T[0][2 * f + 1]), T[1][2 * f + 1]);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (NXT) {
          float mx = wt_max(ma, mb);
          const auto r2 = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
          mx = wt_max(__uint_as_float(r2[0]), __uint_as_float(r2[1])) * scale_log2e;   // (the scale is positive)
          if (__any(!(mx <= m + WT_THR))) {
            const float mn = fmaxf(m, mx);
            const float corr = mn == -INFINITY ? 1.f : fast_exp2(m - mn);
            l *= corr;
#pragma unroll
            for (int v = 0; v < NVT; ++v) O[v] *= corr;
            m = mn;
          }
        }
      };
      const int first = on ? max(jb - run, 0) : n, end = on ? min(je - run, n) : 0;   // this wave's tiles of the run
      int j = -1;
      if (first < end) {
        for (; j + 1 < first; ++j) meet(j);
        step(std::false_type{}, std::true_type{}, j, sb, sa);
        ++j;
        for (; j + 2 < end; j += 2) {
          step(std::true_type{}, std::true_type{}, j, sa, sb);
          step(std::true_type{}, std::true_type{}, j + 1, sb, sa);
        }
        if (j + 1 < end) {
          step(std::true_type{}, std::true_type{}, j, sa, sb);
          sa[0] = sb[0];
          sa[1] = sb[1];
          ++j;
        }
        step(std::true_type{}, std::false_type{}, j, sa, sb);
        ++j;
      }
      for (; j < n; ++j) meet(j);
      lds_barrier();   // (the run's page ids and slots have been read)
    }
  }
  // the last products' results are complete before anything reads them behind a branch
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 15");
  __builtin_amdgcn_sched_barrier(0);
  l += __shfl_xor(l, 32, 64);
  if (!mine || lr >= nrows) return;
  if (sink != nullptr) l += fast_exp2(sink[h] * LOG2E - m);
  float inv = out_scale / l;
  if (gate != nullptr) inv *= head_gate(gate + t * gs + h);
  bf16* op = out + t * os + (int64_t)h * Dv;
#pragma unroll
  for (int v = 0; v < NVT; ++v)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const int c = 32 * v + 8 * i4 + 4 * lh;
      typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
      const bf16x4 o = {(bf16)(O[v][4 * i4] * inv), (bf16)(O[v][4 * i4 + 1] * inv), (bf16)(O[v][4 * i4 + 2] * inv),
                        (bf16)(O[v][4 * i4 + 3] * inv)};
      if (vec4) {
        *reinterpret_cast<bf16x4*>(op + c) = o;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) op[c + e] = o[e];
      }
    }
}

// out[t][h] = sum_z 2^(m_z - m) O_z / (sum_z 2^(m_z - m) l_z + 2^(sink_h - m)) over the (at most 64) key-range splits: lane z holds
// split z's maximum and sum, four splits' partials are in flight at a time
__global__ __launch_bounds__(64) void window_merge_kernel(const float* __restrict__ po, const float* __restrict__ pml, int nsplit,
                                                          int64_t T, int H, int Dv, const float* __restrict__ sink,
                                                          const bf16* __restrict__ gate, int64_t gs, bf16* __restrict__ out,
                                                          int64_t os, float out_scale) {
  const int64_t th = blockIdx.x;  // t * H + h
  const int64_t t = th / H;
  const int h = (int)(th - t * H), lane = threadIdx.x;
  const int64_t zs = T * H;
  const float mz = lane < nsplit ? pml[2 * (lane * zs + th)] : -INFINITY;
  const float lz = lane < nsplit ? pml[2 * (lane * zs + th) + 1] : 0.f;
  float mx = mz;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  const float wz = mz == -INFINITY ? 0.f : fast_exp2(mz - mx);
  float den = wz * lz;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) den += __shfl_xor(den, o, 64);
  if (sink != nullptr) den += fast_exp2(sink[h] * LOG2E - mx);
  float inv = out_scale / den;
  if (gate != nullptr) inv *= head_gate(gate + t * gs + h);
  for (int d0 = 0; d0 < Dv; d0 += 128) {
    float a[2] = {0.f, 0.f};
#pragma unroll 4
    for (int z = 0; z < nsplit; ++z) {
      const float f = __shfl(wz, z, 64);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int d = d0 + lane + 64 * k;
        const float v = d < Dv ? po[(z * zs + th) * Dv + d] : 0.f;
        a[k] += f == 0.f ? 0.f : f * v;
      }
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int d = d0 + lane + 64 * k;
      if (d < Dv) out[t * os + (int64_t)h * Dv + d] = (bf16)(a[k] * inv);
    }
  }
}

// ---- group-limited router ------------------------------------------------------------------------------------------
constexpr int GR_MAXE = 512;  // experts (8 per lane)
constexpr int GR_MAXK = 16;
constexpr int GR_MAXG = 64;   // groups (one per lane)

struct RouteForm {
  bool sigmoid;   // scores: sigmoid of each logit, else softmax over all experts
  bool top2;      // a group's score: the sum of its two largest c (groups of one: that one), else its largest c
  bool norm;      // weights: divided by (their sum + eps), else as they are
  float scale;    // factor on the weights
};

// one wave per row of fp32 logits [T, >= E]: s = softmax over the E experts or sigmoid; c = s + correction (when given);
// the `keep` groups (of `groups` equal runs of neighbouring experts) with the largest group score stay, the others' c
// count as -inf; the k largest c are chosen (ties: the lower index); weights from s of the chosen (RouteForm). With
// `gate` the logit in column E goes through a sigmoid.
// PL: experts a lane holds. One for up to 64 of them: every walk over a lane's experts, a division each, is an eighth as long (us: 64 rows x
// 8 experts in 4 groups 10.6 -> 7.9, 64 in 8 18.8 -> 13.9, 2805 x 8 13.0 -> 9.2).
template <int PL>
__global__ __launch_bounds__(NT) void moe_topk_grouped_kernel(const float* __restrict__ logits, int64_t ls, int E,
                                                              int k, const float* __restrict__ corr, int groups,
                                                              int keep, float eps, float* __restrict__ tw,
                                                              int* __restrict__ te, float* __restrict__ gate,
                                                              int64_t T, RouteForm form) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * (NT / 64) + wave;
  if (t >= T) return;
  float sc[PL], c[PL];
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    const int e = lane + 64 * i;
    sc[i] = e < E ? logits[t * ls + e] : -INFINITY;
    mx = fmaxf(mx, sc[i]);
  }
  if (form.sigmoid) {
#pragma unroll
    for (int i = 0; i < PL; ++i) sc[i] = 1.0f / (1.0f + expf(-sc[i]));   // (0 past E)
  } else {
    mx = wave_max(mx);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < PL; ++i) {
      sc[i] = lane + 64 * i < E ? expf(sc[i] - mx) : 0.f;
      sum += sc[i];
    }
    sum = wave_sum(sum);
#pragma unroll
    for (int i = 0; i < PL; ++i) sc[i] = sc[i] / sum;
  }
  const int gsz = E / groups;
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    const int e = lane + 64 * i;
    c[i] = e < E ? (corr != nullptr ? sc[i] + corr[e] : sc[i]) : -INFINITY;
  }
  if (keep < groups) {
    // lane g holds group g's score
    float gs = -INFINITY;
    for (int g = 0; g < groups; ++g) {
      float v = -INFINITY;
#pragma unroll
      for (int i = 0; i < PL; ++i) {
        const int e = lane + 64 * i;
        if (e < E && e / gsz == g) v = fmaxf(v, c[i]);
      }
      v = wave_max(v);
      if (form.top2 && gsz > 1) {   // the second largest: one holder of the largest (the lowest index) left out
        int hold = 0x7fffffff;
#pragma unroll
        for (int i = 0; i < PL; ++i) {
          const int e = lane + 64 * i;
          if (e < E && e / gsz == g && c[i] == v) hold = min(hold, e);
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) hold = min(hold, __shfl_xor(hold, o, 64));
        float v2 = -INFINITY;
#pragma unroll
        for (int i = 0; i < PL; ++i) {
          const int e = lane + 64 * i;
          if (e < E && e / gsz == g && e != hold) v2 = fmaxf(v2, c[i]);
        }
        v += wave_max(v2);
      }
      if (lane == g) gs = v;
    }
    unsigned long long kept = 0ull;
    for (int j = 0; j < keep; ++j) {
      float bv = gs;
      int bi = lane < groups ? lane : 0x7fffffff;
      if (lane >= groups || ((kept >> lane) & 1ull)) { bv = -INFINITY; bi = 0x7fffffff; }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(bv, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        if (oi != 0x7fffffff && (bi == 0x7fffffff || ov > bv || (ov == bv && oi < bi))) { bv = ov; bi = oi; }
      }
      kept |= 1ull << bi;
    }
#pragma unroll
    for (int i = 0; i < PL; ++i) {
      const int e = lane + 64 * i;
      if (e < E && !((kept >> (e / gsz)) & 1ull)) c[i] = -INFINITY;
    }
  }
  float val[GR_MAXK];
  float wsum = 0.f;
  unsigned taken = 0u;  // this lane's experts already chosen (bit i: expert lane + 64 i)
  for (int j = 0; j < k; ++j) {
    float bv = -INFINITY;
    int bi = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < PL; ++i) {
      const int e = lane + 64 * i;
      if (e < E && !((taken >> i) & 1u) && (bi == 0x7fffffff || c[i] > bv)) { bv = c[i]; bi = e; }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(bv, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (oi != 0x7fffffff && (bi == 0x7fffffff || ov > bv || (ov == bv && oi < bi))) { bv = ov; bi = oi; }
    }
    float mine = 0.f;
#pragma unroll
    for (int i = 0; i < PL; ++i)
      if (bi == lane + 64 * i) {
        taken |= 1u << i;
        mine = sc[i];
      }
    const float sv = __shfl(mine, bi & 63, 64);
    if (j < GR_MAXK) val[j] = sv;
    wsum += sv;
    if (lane == 0) te[t * k + j] = bi;
  }
  if (lane == 0) {
    const float inv = (form.norm ? 1.0f / (wsum + eps) : 1.0f) * form.scale;
    for (int j = 0; j < k; ++j) tw[t * k + j] = val[j] * inv;
    if (gate != nullptr) gate[t] = 1.0f / (1.0f + expf(-logits[t * ls + E]));
  }
}

static inline int ew_grid(int64_t n) { return (int)std::min<int64_t>((n + 255) / 256, 65535 * 4); }

}  // namespace hs
}  // namespace kafka

using namespace kafka::hs;

#define DISPATCH_AT(f32, ...)             \
  if (f32) {                              \
    using AT = float;                     \
    __VA_ARGS__;                          \
  } else {                                \
    using AT = bf16;                      \
    __VA_ARGS__;                          \
  }

extern "C" {

int kafka_hy_stream_max() { return SMAX; }

hipError_t kafka_hy_stream_step(float* xs, int64_t s_stride, int64_t t_stride, int S, const void* y, int64_t ys,
                                int y_f32, const void* y2, int64_t y2s, int y2_f32, const float* row_scale,
                                const float* mix, const float* wr, const float* rd, const float* nw, float eps,
                                void* out, int64_t os, int out_f32, float* total, int64_t ts, int64_t T, int d,
                                int center, hipStream_t st) {
  if (T <= 0 || d <= 0) return hipSuccess;
  if (S < 1 || S > SMAX) return hipErrorInvalidValue;
  auto a = [&](auto k) {
    k<<<(unsigned)T, NT, 0, st>>>(xs, s_stride, t_stride, y, ys, y_f32 != 0, y2, y2s, y2_f32 != 0, row_scale, mix, wr,
                                  rd, nw, eps, out, os, out_f32 != 0, total, ts, d, center != 0);
  };
  switch (S) {
    case 1: a(stream_step_kernel<1>); break;
    case 2: a(stream_step_kernel<2>); break;
    case 3: a(stream_step_kernel<3>); break;
    case 4: a(stream_step_kernel<4>); break;
    case 5: a(stream_step_kernel<5>); break;
    case 6: a(stream_step_kernel<6>); break;
    case 7: a(stream_step_kernel<7>); break;
    case 8: a(stream_step_kernel<8>); break;
    case 9: a(stream_step_kernel<9>); break;
    case 10: a(stream_step_kernel<10>); break;
    case 11: a(stream_step_kernel<11>); break;
    case 12: a(stream_step_kernel<12>); break;
    case 13: a(stream_step_kernel<13>); break;
    case 14: a(stream_step_kernel<14>); break;
    case 15: a(stream_step_kernel<15>); break;
    default: a(stream_step_kernel<16>); break;
  }
  return hipGetLastError();
}

hipError_t kafka_hy_swish_clamp_mul(int f32, const void* gu, int64_t gs, void* out, int64_t os, int64_t T, int F,
                                    float limit, float alpha, hipStream_t st) {
  if (T <= 0 || F <= 0) return hipSuccess;
  if (!f32 && F % 8 == 0 && gs % 8 == 0 && os % 8 == 0 && (reinterpret_cast<uintptr_t>(gu) & 15) == 0 &&
      (reinterpret_cast<uintptr_t>(out) & 15) == 0) {
    swish_clamp_mul_vec8_kernel<<<ew_grid(T * (F / 8)), 256, 0, st>>>((const bf16*)gu, gs, (bf16*)out, os, T, F, limit,
                                                                      alpha);
    return hipGetLastError();
  }
  DISPATCH_AT(f32, {
    swish_clamp_mul_kernel<AT><<<ew_grid(T * F), 256, 0, st>>>((const AT*)gu, gs, (AT*)out, os, T, F, limit, alpha);
  });
  return hipGetLastError();
}

hipError_t kafka_hy_qk_norm_rope_store(int f32, const void* qkv, int64_t qs, int H, int G, int D, int Dv,
                                       const float* qw, const float* kw, float eps, const int64_t* positions,
                                       const float* cos_sin, int dims, const void* vf, int64_t vfs, int vf_off,
                                       float lam, void* kc, void* vt, const int64_t* slots, void* q_out, int64_t qos,
                                       int64_t T, hipStream_t st) {
  if (T <= 0) return hipSuccess;
  if (dims < 0 || dims % 2 || dims > D || (dims > 0 && cos_sin == nullptr)) return hipErrorInvalidValue;
  DISPATCH_AT(f32, {
    qk_norm_rope_store_kernel<AT><<<(unsigned)T, NT, 0, st>>>((const AT*)qkv, qs, H, G, D, Dv, qw, kw, eps, positions,
                                                              cos_sin, dims, (const AT*)vf, vfs, vf_off, lam, (AT*)kc,
                                                              (AT*)vt, slots, (AT*)q_out, qos);
  });
  return hipGetLastError();
}

int kafka_hy_window_attn_max_d() { return WA_MAXD; }
int kafka_hy_window_attn_max_dv() { return 64 * WA_NV; }

hipError_t kafka_hy_window_attn(int f32, const void* q, int64_t qs, const void* kc, const void* vt, const int* bt,
                                int bt_stride, const int* tok_seg, const int64_t* positions, int H, int G, int D,
                                int Dv, float scale, int window, const float* sink, const void* gate, int64_t gs,
                                void* out, int64_t os, int64_t T, int shared_keys, float out_scale, hipStream_t st) {
  // shared_keys: D is the whole key row's size and every query row meets all G key heads of a token at once
  if (T <= 0) return hipSuccess;
  if (D > WA_MAXD || Dv > 64 * WA_NV || G < 1 || H % G || window < 0) return hipErrorInvalidValue;
  const int64_t pairs = T * H;
  const int grid = (int)((pairs + NT / 64 - 1) / (NT / 64));
  const int Ck = shared_keys ? D : G * D, kstep = shared_keys ? 0 : D;
  DISPATCH_AT(f32, {
    window_attn_kernel<AT><<<grid, NT, 0, st>>>((const AT*)q, qs, (const AT*)kc, (const AT*)vt, bt, bt_stride, tok_seg,
                                                positions, H, G, D, Dv, Ck, kstep, scale * LOG2E, window, sink,
                                                (const AT*)gate, gs, (AT*)out, os, pairs, out_scale);
  });
  return hipGetLastError();
}

// bf16 shapes the matrix-core kernel takes (else the per-wave kernel above runs)
int kafka_hy_window_attn_mfma_ok(int page, int D, int Dv, int rep) {
  return page == PAGE && D >= 16 && D % 16 == 0 && D <= 256 && Dv >= 1 && Dv <= 256 && rep >= 1 && rep <= WM_ROWS;
}

hipError_t kafka_hy_window_attn_mfma(const void* q, int64_t qs, const void* kc, const void* vt, const int* bt,
                                     int bt_stride, const int* items, int n_items, const int64_t* positions, int H,
                                     int G, int D, int Dv, float scale, int window, const float* sink,
                                     const void* gate, int64_t gs, void* out, int64_t os, int nsplit, float* po,
                                     float* pml, int64_t T, int shared_keys, float out_scale, int max_tok, int min_rows_tok,
                                     int tile_items, hipStream_t st) {
  // items of up to max_tok tokens here (0: none), those of at least min_rows_tok tokens a wave each (0: none), about tile_items of
  // which have something to share (window_attn_tile)
  if (n_items <= 0) return hipSuccess;
  const int Ck = shared_keys ? D : G * D, kstep = shared_keys ? 0 : D;
  if (G < 1 || H % G || window < 0 || !kafka_hy_window_attn_mfma_ok(PAGE, D, Dv, H / G)) return hipErrorInvalidValue;
  if (nsplit < 1 || nsplit > 64 || (nsplit > 1 && (po == nullptr || pml == nullptr))) return hipErrorInvalidValue;
  if (min_rows_tok > 0) {
    const bool vec4 = Dv % 4 == 0 && os % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 7) == 0;
    const int waves = (int64_t)n_items * G >= 2048 ? 4 : (int64_t)n_items * G >= 1024 ? 2 : 1;
    const int64_t gy = (n_items + waves - 1) / waves;
    if (gy > 65535) return hipErrorInvalidValue;
    const dim3 gr((unsigned)G, (unsigned)gy);
    auto b = [&](auto k) {
      k<<<gr, 64 * waves, 0, st>>>((const bf16*)q, qs, (const bf16*)kc, (const bf16*)vt, bt, bt_stride, items, n_items,
                                   positions, H, G, D, Dv, Ck, kstep, scale * LOG2E, window, sink, (const bf16*)gate, gs,
                                   (bf16*)out, os, out_scale, min_rows_tok, vec4, nullptr, nullptr, T);
    };
    const bool al = ((reinterpret_cast<uintptr_t>(kc) | reinterpret_cast<uintptr_t>(vt)) & 15) == 0;
    if (D == 128 && Dv == 128 && al && scale > 0.f && (int64_t)tile_items * G >= WT_MIN_WAVES) {
      window_attn_tile_kernel<<<dim3((unsigned)G, (unsigned)((n_items + WT_WAVES - 1) / WT_WAVES)), 64 * WT_WAVES, 0, st>>>(
          (const bf16*)q, qs, (const bf16*)kc, (const bf16*)vt, bt, bt_stride, items, n_items, positions, H, G, Ck, kstep,
          scale * LOG2E, window, sink, (const bf16*)gate, gs, (bf16*)out, os, out_scale, min_rows_tok, vec4);
    } else if (D <= 64) {
      if (Dv <= 64) b(window_attn_rows_kernel<4, 2, false>);
      else if (Dv <= 128) b(window_attn_rows_kernel<4, 4, false>);
      else b(window_attn_rows_kernel<4, 8, false>);
    } else if (D <= 128) {
      if (Dv <= 64) b(window_attn_rows_kernel<8, 2, false>);
      else if (Dv <= 128) b(window_attn_rows_kernel<8, 4, false>);
      else b(window_attn_rows_kernel<8, 8, false>);
    } else {
      if (Dv <= 64) b(window_attn_rows_kernel<16, 2, false>);
      else if (Dv <= 128) b(window_attn_rows_kernel<16, 4, false>);
      else b(window_attn_rows_kernel<16, 8, false>);
    }
  }
  if (max_tok <= 0) return hipGetLastError();
  if (nsplit > 1 && min_rows_tok > 0) return hipErrorInvalidValue;   // (the merge pass takes every row)
  const dim3 grid((unsigned)n_items * (unsigned)G, 1, (unsigned)nsplit);
  auto a = [&](auto k) {
    k<<<grid, 256, 0, st>>>((const bf16*)q, qs, (const bf16*)kc, (const bf16*)vt, bt, bt_stride, items, n_items, positions, H, G, D,
                            Dv, Ck, kstep, scale * LOG2E, window, sink, (const bf16*)gate, gs, (bf16*)out, os, out_scale, max_tok,
                            false, po, pml, T);
  };
  auto by_dv = [&](auto k2, auto k4, auto k8) { Dv <= 64 ? a(k2) : Dv <= 128 ? a(k4) : a(k8); };
  if (D <= 64)
    by_dv(window_attn_rows_kernel<4, 2, true>, window_attn_rows_kernel<4, 4, true>, window_attn_rows_kernel<4, 8, true>);
  else if (D <= 128)
    by_dv(window_attn_rows_kernel<8, 2, true>, window_attn_rows_kernel<8, 4, true>, window_attn_rows_kernel<8, 8, true>);
  else
    by_dv(window_attn_rows_kernel<16, 2, true>, window_attn_rows_kernel<16, 4, true>, window_attn_rows_kernel<16, 8, true>);
  if (nsplit > 1)
    window_merge_kernel<<<(unsigned)(T * H), 64, 0, st>>>(po, pml, nsplit, T, H, Dv, sink, (const bf16*)gate, gs,
                                                          (bf16*)out, os, out_scale);
  return hipGetLastError();
}

int kafka_hy_grouped_router_max_e() { return GR_MAXE; }
int kafka_hy_grouped_router_max_k() { return GR_MAXK; }
int kafka_hy_grouped_router_max_g() { return GR_MAXG; }

hipError_t kafka_hy_moe_topk_grouped(const float* logits, int64_t ls, int E, int k, const float* corr, int groups,
                                     int keep, float eps, float* tw, int* te, float* gate, int64_t T, int sigmoid,
                                     int top2, int norm, float scale, hipStream_t st) {
  if (T <= 0) return hipSuccess;
  if (E > GR_MAXE || k > GR_MAXK || k < 1 || groups < 1 || groups > GR_MAXG || E % groups || keep < 1 ||
      keep > groups || k > keep * (E / groups))
    return hipErrorInvalidValue;
  const int grid = (int)((T + NT / 64 - 1) / (NT / 64));
  auto a = [&](auto kern) {
    kern<<<grid, NT, 0, st>>>(logits, ls, E, k, corr, groups, keep, eps, tw, te, gate, T, RouteForm{sigmoid != 0, top2 != 0, norm != 0, scale});
  };
  if (E <= 64) a(moe_topk_grouped_kernel<1>);
  else a(moe_topk_grouped_kernel<GR_MAXE / 64>);
  return hipGetLastError();
}

}  // extern "C"
