// The Mamba-2 state-space recurrence of long segments on the matrix cores, for gfx950.
//
// Per head, with a decay exponent a_t = -exp(A_log) dt_t <= 0, dt_t = softplus(raw + bias):
//   S_t = e^(a_t) S_(t-1) + dt_t B_t x_t^T,   y_t = S_t^T C_t + D x_t      (B, C shared by the heads of a group)
// In chunks of 128 tokens, with c_t the running sum of the chunk's a:
//   y_t = e^(c_t) S_0^T C_t + sum_{j <= t} e^(c_t - c_j) dt_j (B_j . C_t) x_j + D x_t
//   U   = sum_j e^(c_end - c_j) dt_j B_j x_j^T,   S' = e^(c_end) S_0 + U
// No exponent is positive. Three launches:
//   ssd_state   U^T of every chunk in parallel
//   ssd_carry   the chunks' entry states in order (in place of U), the sequence's state advanced
//   ssd_out     the rows of every chunk in parallel
// x, B and C are bf16; every fp32 factor of a product (B times its weight, the weights of the rows, the entry state) is
// split into three bf16 parts that hold all its bits, one matrix product each, fp32 accumulation - as exact as the fp32
// multiply-adds of the token-by-token kernels. The running sums are formed in fp64 and kept as two floats, so that the
// difference of two of them is good to its own last bit however long the chunk's sum has become. A token's exponent is held
// at SSD_FLOOR or above: every decay over such a token is zero in fp32 either way, and the sums stay finite where A or dt do not.
//
// What bounds it: a workgroup is a chain of loads, LDS exchanges and products, so as many of them on a CU as LDS allows: three, when the
// registers are held to 168 (left to itself the compiler uses 200 and two fit). Beside that the chunks' contributions and entry
// states through memory (67 MB written, read and written by the carry, read at 2048 tokens x 128 heads of 128 x 64). Measured there,
// one layer of a step: 45 + 25 + 71 us; with two workgroups on a CU, the entry state loaded piece by piece, the sums formed twice
// and the carry an element a thread 50 + 33 + 99. The token-by-token form in two passes over chunks of 256 took 2 x 1196 + 87 us.
#include "chunk_common.h"

namespace kafka {
namespace hy {

using namespace chunk;

struct SsdIn {
  const bf16* xbc;      // rows [x heads | B groups | C groups]
  int64_t xs;
  const bf16* dt;       // raw step sizes [T, >= heads]
  int64_t ds;
  const float* dt_bias;
  const float* A_log;
  int H, P, N, G;
  const int* vseg;      // [chunks][4] = (first row, rows, -, -)
  float* U;             // [chunks][H][P][N]: own contribution, then entry state
  float* dec;           // [chunks][H]: e^(c_end)
  float* sums;          // [chunks][H][3][CH]: what ssd_sums finds
};

constexpr double SSD_FLOOR = -1000.0;   // (e^-1000 is far below the smallest fp32 number)

// The chunk's step sizes and running sums (times log2 e, as a float and what the float leaves out) by one wave; rows past n:
// dt = 0, the sum stays. They are kept (unless nullptr) for ssd_out, whose waves would wait for them (9 of its 100 us).
__device__ __forceinline__ void ssd_sums(const SsdIn& in, int row0, int n, int h, int lane, float* dt_s, float* ch_s,
                                         float* cl_s, float* keep) {
  const float A = -expf(in.A_log[h]), bias = in.dt_bias[h];
  double c[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int t = 64 * k + lane;
    float dt = 0.f;
    double a = 0.0;
    if (t < n) {
      const float raw = (float)in.dt[(int64_t)(row0 + t) * in.ds + h] + bias;
      dt = raw > 20.f ? raw : log1pf(expf(raw));
      a = (double)A * (double)dt;
    }
    dt_s[t] = dt;
    if (keep) keep[t] = dt;
    c[k] = a < SSD_FLOOR ? SSD_FLOOR : a;   // (NaN stays NaN)
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const double u = __shfl_up(c[k], o, 64);
      if (lane >= o) c[k] += u;
    }
  }
  c[1] += __shfl(c[0], 63, 64);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const double v = c[k] * 1.4426950408889634;
    const float hi = (float)v;
    const float lo = (float)(v - (double)hi);
    ch_s[64 * k + lane] = hi;
    cl_s[64 * k + lane] = lo;
    if (keep) {
      keep[CH + 64 * k + lane] = hi;
      keep[2 * CH + 64 * k + lane] = lo;
    }
  }
}

// 2^(c_a - c_b) of two running sums
__device__ __forceinline__ float ssd_decay(float ha, float la, float hb, float lb) {
  return fast_exp2((ha - hb) + (la - lb));
}

__global__ __launch_bounds__(NT, 3) void ssd_state_kernel(SsdIn in, int n_chunks, int slices) {
  __shared__ __attribute__((aligned(16))) bf16 Bt[DS * LDJ];
  __shared__ __attribute__((aligned(16))) bf16 Xt[VSL * LDJ];
  __shared__ __attribute__((aligned(16))) float f_s[CH];
  __shared__ float ch_s[CH], cl_s[CH];
  int item, slice;
  if (!chunk_item(n_chunks * in.H, slices, item, slice)) return;   // (uniform)
  const int ch = item / in.H, h = item - ch * in.H, v0 = slice * VSL;
  const int row0 = in.vseg[4 * ch], n = in.vseg[4 * ch + 1];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, lr = lane & 31, lh = lane >> 5;
  const int P = in.P, N = in.N, H = in.H, grp = h / (H / in.G);
  const bf16* rows = in.xbc + (int64_t)row0 * in.xs;
  if (w == 0) ssd_sums(in, row0, n, h, lane, f_s, ch_s, cl_s, slice == 0 ? in.sums + (int64_t)item * 3 * CH : nullptr);
  stage_transposed(rows + (int64_t)h * P, in.xs, n, v0, VSL, P, Xt, tid);
  for (int db = 0; db < N; db += DS) {
    if (db) __syncthreads();
    stage_transposed(rows + (int64_t)H * P + (int64_t)grp * N, in.xs, n, db, min(DS, N - db), N, Bt, tid);
    __syncthreads();
    if (db == 0) {   // the weight of every row, once
      if (tid < CH) f_s[tid] *= ssd_decay(ch_s[CH - 1], cl_s[CH - 1], ch_s[tid], cl_s[tid]);
      __syncthreads();
    }
    const int d = 32 * w + lr;   // (of this block; waves and lanes past N compute on what LDS holds and store nothing)
    f32x16 acc[2];
#pragma unroll
    for (int vt = 0; vt < 2; ++vt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[vt][i] = 0.f;
#pragma unroll 2
    for (int ks = 0; ks < CH / 16; ++ks) {
      const int j = 16 * ks + 8 * lh;
      const bf16x8 bv = *reinterpret_cast<const bf16x8*>(Bt + d * LDJ + j);
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = f_s[j + e] * (float)bv[e];
      const Split s = split3(x);
#pragma unroll
      for (int vt = 0; vt < 2; ++vt) {
        const bf16x8 vf = *reinterpret_cast<const bf16x8*>(Xt + (32 * vt + lr) * LDJ + j);
#pragma unroll
        for (int k = 0; k < 3; ++k) acc[vt] = mfma32(vf, s.p[k], acc[vt]);
      }
    }
    mfma_settle();
    if (db + d < N) {
      float* Up = in.U + ((int64_t)item * P + v0) * N + db + d;
#pragma unroll
      for (int vt = 0; vt < 2; ++vt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int v = 32 * vt + (i & 3) + 8 * (i >> 2) + 4 * lh;
          if (v0 + v < P) Up[(int64_t)v * N] = acc[vt][i];
        }
    }
  }
  if (slice == 0 && tid == 0) in.dec[item] = fast_exp2(ch_s[CH - 1] + cl_s[CH - 1]);
}

// grid (blocks of 4 NT elements of P * N, H, segments): cs[r] = (first chunk, chunks, first position, state slot). A thread owns four
// neighbouring elements of the state; the next chunks' contributions are in flight while PF are added up.
__global__ __launch_bounds__(NT) void ssd_carry_kernel(SsdIn in, const int* __restrict__ cs, float* __restrict__ state) {
  const int r = blockIdx.z, h = blockIdx.y, N = in.N, P = in.P, H = in.H;
  const int first = cs[4 * r], last = first + cs[4 * r + 1], p0 = cs[4 * r + 2], slot = cs[4 * r + 3];
  const int64_t i = 4 * ((int64_t)blockIdx.x * NT + threadIdx.x);   // element p * N + d (N is a multiple of 16)
  if (i >= (int64_t)P * N) return;
  const int p = (int)(i / N), d = (int)(i - (int64_t)p * N);
  float* st = state + (((int64_t)slot * H + h) * N + d) * P + p;
  float* el = in.U + (int64_t)h * P * N + i;
  const int64_t step = (int64_t)H * P * N;
  f32x4 S = {0.f, 0.f, 0.f, 0.f};
  if (p0 > 0)
#pragma unroll
    for (int e = 0; e < 4; ++e) S[e] = st[(int64_t)e * P];
  auto at = [&](int c) { return reinterpret_cast<f32x4*>(el + (int64_t)c * step); };
  constexpr int PF = 4;
  f32x4 u[PF];
#pragma unroll
  for (int k = 0; k < PF; ++k)
    if (first + k < last) u[k] = *at(first + k);
  for (int c0 = first; c0 < last; c0 += PF) {
    f32x4 nx[PF];
#pragma unroll
    for (int k = 0; k < PF; ++k)
      if (c0 + PF + k < last) nx[k] = *at(c0 + PF + k);
#pragma unroll
    for (int k = 0; k < PF; ++k)
      if (c0 + k < last) {
        *at(c0 + k) = S;                       // the chunk's entry state
        S = in.dec[(int64_t)(c0 + k) * H + h] * S + u[k];
      }
#pragma unroll
    for (int k = 0; k < PF; ++k) u[k] = nx[k];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) st[(int64_t)e * P] = S[e];
}

// NKS: 16-channel steps of a head's state rows held in registers (N <= 16 NKS; the steps past N multiply by zeros)
template <int NKS>
__global__ __launch_bounds__(NT, NKS <= 8 ? 3 : 2) void ssd_out_kernel(SsdIn in, int n_chunks, int slices, const float* __restrict__ Dp,
                                                     float* __restrict__ y, int64_t ys) {
  // one buffer, first for the entry state's three parts [3][VSL][DS + 8], then for the x columns [VSL][LDJ]
  typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
  __shared__ __attribute__((aligned(16))) bf16 buf[3 * VSL * LDD];
  __shared__ float sum_s[3 * CH];
  const float *dt_s = sum_s, *ch_s = sum_s + CH, *cl_s = sum_s + 2 * CH;
  int item, slice;
  if (!chunk_item(n_chunks * in.H, slices, item, slice)) return;   // (uniform)
  const int ch = item / in.H, h = item - ch * in.H, v0 = slice * VSL;
  const int row0 = in.vseg[4 * ch], n = in.vseg[4 * ch + 1];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, lr = lane & 31, lh = lane >> 5;
  const int P = in.P, N = in.N, H = in.H, nks = N >> 4, grp = h / (H / in.G);
  const bf16* rows = in.xbc + (int64_t)row0 * in.xs;
  const bf16* Bc = rows + (int64_t)H * P + (int64_t)grp * N + 8 * lh;
  for (int i = tid; i < 3 * CH; i += NT) sum_s[i] = in.sums[(int64_t)item * 3 * CH + i];
  const int t = 32 * w + lr;                       // this lane's row
  const bf16* crow = Bc + (int64_t)in.G * N + (int64_t)min(t, n - 1) * in.xs;
  bf16x8 qf[NKS], kf[NKS];
  auto fetch_keys = [&](int jt) {
    const bf16* krow = Bc + (int64_t)min(32 * jt + lr, n - 1) * in.xs;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) kf[ks] = load_bf16x8(krow + 16 * min(ks, nks - 1));
  };
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) {
    qf[ks] = load_bf16x8(crow + 16 * min(ks, nks - 1));
    if (ks >= nks) qf[ks] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
  }
  f32x16 acc[2];
#pragma unroll
  for (int vt = 0; vt < 2; ++vt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[vt][i] = 0.f;
  // ---- the entry state: acc = S_0^T C
  for (int db = 0; db < N; db += DS) {
    const int nd = min(DS, N - db);
    if (db) __syncthreads();
    stage_split(in.U + ((int64_t)item * P + v0) * N + db, N, nd, P - v0, buf, tid);
    __syncthreads();
    if (32 * w < n) {   // (uniform per wave)
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        const int d = 16 * ks - db;   // (uniform) the step's channels in this block
        if (d >= 0 && d < nd) {
#pragma unroll
          for (int vt = 0; vt < 2; ++vt)
#pragma unroll
            for (int k = 0; k < 3; ++k)
              acc[vt] = mfma32(*reinterpret_cast<const bf16x8*>(buf + (k * VSL + 32 * vt + lr) * LDD + d + 8 * lh),
                               qf[ks], acc[vt]);
        }
      }
      mfma_settle();
    }
  }
  fetch_keys(0);
  __syncthreads();
  stage_transposed(rows + (int64_t)h * P, in.xs, n, v0, VSL, P, buf, tid);
  __syncthreads();
  if (32 * w >= n) return;   // (uniform per wave; no barrier follows)
  const float th = ch_s[t], tl = cl_s[t], g0 = fast_exp2(th + tl), Dh = Dp[h];
  unsigned odd = 0;   // (two values a word: a full exponent carries)
#pragma unroll
  for (int vt = 0; vt < 2; ++vt)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
      const u32x4 x = *reinterpret_cast<const u32x4*>(buf + (32 * vt + lr) * LDJ + 32 * w + 16 * lh + 8 * e);
#pragma unroll
      for (int i = 0; i < 4; ++i) odd |= (x[i] & 0x7f807f80u) + 0x00800080u;
    }
  if (__any(odd & 0x80008000u)) {
    // (uniform per wave, never with finite inputs) In the products below a row has the weight 0 for the rows behind it in its
    // tile, and 0 times what is not finite is not 0. A tile that holds such values is summed row by row, up to the row itself.
    if (t >= n) return;
    const bf16 *ct = crow - 8 * lh, *b0 = Bc - 8 * lh;
    const float* Uh = in.U + ((int64_t)item * P + v0 + 32 * lh) * N;
    const int nv = min(32, P - v0 - 32 * lh);   // this lane's columns
    float yv[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      float a = 0.f;
      if (i < nv)
        for (int d = 0; d < N; ++d) a += Uh[(int64_t)i * N + d] * (float)ct[d];
      yv[i] = a * g0;
    }
    for (int j = 0; j <= t; ++j) {
      float wj = 0.f;
      for (int d = 0; d < N; ++d) wj += (float)b0[(int64_t)j * in.xs + d] * (float)ct[d];
      wj *= ssd_decay(th, tl, ch_s[j], cl_s[j]) * dt_s[j];
#pragma unroll
      for (int i = 0; i < 32; ++i) yv[i] += wj * (float)buf[(32 * lh + i) * LDJ + j];
    }
#pragma unroll
    for (int i = 0; i < 32; ++i)
      if (i < nv)
        y[(int64_t)(row0 + t) * ys + (int64_t)h * P + v0 + 32 * lh + i] = yv[i] + Dh * (float)buf[(32 * lh + i) * LDJ + t];
    return;
  }
#pragma unroll
  for (int vt = 0; vt < 2; ++vt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[vt][i] *= g0;
  // ---- the chunk's own rows: 32 at a time, M^T = B C^T (this lane's row: column), its weights split for X^T M^T
  for (int jt = 0; jt <= w; ++jt) {
    f32x16 M;
#pragma unroll
    for (int i = 0; i < 16; ++i) M[i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) M = mfma32(kf[ks], qf[ks], M);
    mfma_settle();
    if (jt < w) fetch_keys(jt + 1);
    float wt[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int j = 32 * jt + (i & 3) + 8 * (i >> 2) + 4 * lh;
      wt[i] = j <= t ? M[i] * (ssd_decay(th, tl, ch_s[j], cl_s[j]) * dt_s[j]) : 0.f;
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {   // 16 rows: this half's are 4 lh .. + 3 and 8 + 4 lh .. + 3
      const float x[8] = {wt[8 * s], wt[8 * s + 1], wt[8 * s + 2], wt[8 * s + 3],
                          wt[8 * s + 4], wt[8 * s + 5], wt[8 * s + 6], wt[8 * s + 7]};
      const Split sp = split3(x);
#pragma unroll
      for (int vt = 0; vt < 2; ++vt) {
        const bf16* vp = buf + (32 * vt + lr) * LDJ + 32 * jt + 16 * s + 4 * lh;
        const bf16x4 lo = *reinterpret_cast<const bf16x4*>(vp), hi = *reinterpret_cast<const bf16x4*>(vp + 8);
        const bf16x8 vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
        for (int k = 0; k < 3; ++k) acc[vt] = mfma32(vf, sp.p[k], acc[vt]);
      }
    }
  }
  mfma_settle();
  if (t >= n) return;
  const bf16* xr = rows + (int64_t)t * in.xs + (int64_t)h * P + v0;
  float* op = y + (int64_t)(row0 + t) * ys + (int64_t)h * P + v0;
#pragma unroll
  for (int vt = 0; vt < 2; ++vt)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const int v = 32 * vt + 8 * i4 + 4 * lh;
      if (v0 + v < P) {
        const bf16x4 xv = *reinterpret_cast<const bf16x4*>(xr + v);
        f32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = acc[vt][4 * i4 + e] + Dh * (float)xv[e];
        *reinterpret_cast<f32x4*>(op + v) = o;
      }
    }
}

}  // namespace hy
}  // namespace kafka

using namespace kafka::hy;

extern "C" {

int kafka_hy_ssd_chunk() { return CH; }
// bf16 rows whose x, B and C parts start at multiples of 8 elements
int kafka_hy_ssd_ok(int H, int P, int N, int G, int64_t xs) {
  return H >= 1 && G >= 1 && H % G == 0 && N >= 16 && N % 16 == 0 && N <= 256 && P >= 8 && P % 8 == 0 && xs % 8 == 0;
}
// floats of scratch per (chunk, head)
int64_t kafka_hy_ssd_scratch(int P, int N) { return (int64_t)P * N + 1 + 3 * CH; }

// the segments of cs in chunks (vseg: all their chunks in order)
hipError_t kafka_hy_ssd_scan(const void* xbc, int64_t xs, const void* dt, int64_t ds, const float* dt_bias,
                             const float* A_log, const float* Dp, int H, int P, int N, int G, const int* vseg, int n_chunks,
                             const int* cs, int R, float* scratch, float* state, float* y, int64_t ys, hipStream_t st) {
  if (R <= 0 || n_chunks <= 0) return hipSuccess;
  if (!kafka_hy_ssd_ok(H, P, N, G, xs) || R > 65535 || H > 65535 || ys % 4) return hipErrorInvalidValue;
  const int64_t items = (int64_t)n_chunks * H;
  const int slices = (P + VSL - 1) / VSL;
  if ((items + 8) * slices > 0x7fffffff) return hipErrorInvalidValue;
  SsdIn in{(const bf16*)xbc, xs, (const bf16*)dt, ds, dt_bias, A_log, H, P, N, G, vseg, scratch, scratch + items * P * N,
           scratch + items * ((int64_t)P * N + 1)};
  const unsigned g = (unsigned)chunk_grid((int)items, slices);
  ssd_state_kernel<<<g, NT, 0, st>>>(in, n_chunks, slices);
  ssd_carry_kernel<<<dim3((unsigned)(((int64_t)P * N + 4 * NT - 1) / (4 * NT)), H, R), NT, 0, st>>>(in, cs, state);
  if (N <= 64) ssd_out_kernel<4><<<g, NT, 0, st>>>(in, n_chunks, slices, Dp, y, ys);
  else if (N <= 128) ssd_out_kernel<8><<<g, NT, 0, st>>>(in, n_chunks, slices, Dp, y, ys);
  else ssd_out_kernel<16><<<g, NT, 0, st>>>(in, n_chunks, slices, Dp, y, ys);
  return hipGetLastError();
}

}  // extern "C"
