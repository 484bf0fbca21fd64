// Mixer frontend and readout of the SolveDelta layer on MI355X:
//   * causal depthwise conv4 + SiLU with initial / final state
//     (reference: causallsso/model.py:119-136, CPU semantics :146-164);
//   * the KDA decay gate  log_decay = -exp(log_rate[h]) * softplus(raw + bias[h, c])
//     (reference: causallsso/model.py:375-390);
//   * the sigmoid-gated RMSNorm feeding the output projection
//     (reference: causallsso/ops/norm_gate.py:20-43 definition, :46-150 owner).
// Forward and backward of each; parameter-gradient reductions are two-stage
// (per-workgroup partials in the caller's workspace, then one reduction kernel),
// so results are deterministic.  All arithmetic is FP32; bf16 in / out.
#include <hip/hip_runtime.h>

#include "sd_common.cuh"
#include "sd_internal.h"
#include "../../include/solvedelta_mixer.h"

namespace sd {

// These kernels' element work is transcendental: an IEEE division costs ten vector
// instructions and log1pf thirty, which, not HBM, bounded the decay gate and the
// convolution.  The quotients here have denominators in [1, 3], so they take the
// hardware's reciprocal and one residual (Newton) step instead.
// sigmoid(a) from t = e^{-|a|}: 1 / (1 + t) or t / (1 + t)
__device__ __forceinline__ float sigm_t(float a, float t) {
  const float n = a < 0.f ? t : 1.f, s = 1.f + t, r = __builtin_amdgcn_rcpf(s), q = n * r;
  return __builtin_fmaf(__builtin_fmaf(-s, q, n), r, q);
}
__device__ __forceinline__ float sigm(float a) { return sigm_t(a, __expf(-fabsf(a))); }
__device__ __forceinline__ float silu(float a) { return a * sigm(a); }
// softplus(x) = max(x, 0) + log(1 + t), t = e^{-|x|}: log(1 + t) = 2 atanh(z) with
// z = t / (2 + t) <= 1/3, by its series through z^17 (the next term is below
// 2e-10 of the sum).  z's residual, with what the sum 2 + t rounded off, is added
// to the small terms, so the result is rounded once.  Above torch's threshold of
// 20 it rounds to x as torch's does.
__device__ __forceinline__ float softplus_t(float x, float t) {
  const float s = 2.f + t, r = __builtin_amdgcn_rcpf(s), z = t * r, y = z * z, zz = z + z;
  const float e = __builtin_fmaf(-z, t - (s - 2.f), __builtin_fmaf(-s, z, t));  // t - (2 + t) z
  float p = 1.f / 17.f;
  p = __builtin_fmaf(p, y, 1.f / 15.f);
  p = __builtin_fmaf(p, y, 1.f / 13.f);
  p = __builtin_fmaf(p, y, 1.f / 11.f);
  p = __builtin_fmaf(p, y, 1.f / 9.f);
  p = __builtin_fmaf(p, y, 1.f / 7.f);
  p = __builtin_fmaf(p, y, 1.f / 5.f);
  p = __builtin_fmaf(p, y, 1.f / 3.f);
  const float l = zz + __builtin_fmaf(zz * y, p, (r + r) * e);
  return x > 0.f ? x + l : l;
}

// VEC (1, 2, 4 or 8) neighbouring bf16 channels of one token, kept packed until used:
// one access of 2 VEC bytes.
template <int VEC> struct BfV;
template <> struct BfV<1> {
  __bf16 v;
  __device__ __forceinline__ void get(float (&x)[1]) const { x[0] = bf2f(v); }
};
template <> struct BfV<2> {
  unsigned v;
  __device__ __forceinline__ void get(float (&x)[2]) const {
    x[0] = __uint_as_float(v << 16);
    x[1] = __uint_as_float(v & 0xffff0000u);
  }
};
template <> struct BfV<4> {
  uint2 v;
  __device__ __forceinline__ void get(float (&x)[4]) const {
    x[0] = __uint_as_float(v.x << 16);
    x[1] = __uint_as_float(v.x & 0xffff0000u);
    x[2] = __uint_as_float(v.y << 16);
    x[3] = __uint_as_float(v.y & 0xffff0000u);
  }
};
template <> struct BfV<8> {
  uint4 v;
  __device__ __forceinline__ void get(float (&x)[8]) const {
    const unsigned u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = __uint_as_float(u[i] << 16);
      x[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
    }
  }
};
template <int VEC>
__device__ __forceinline__ BfV<VEC> ldv(const __bf16* p) {
  return *reinterpret_cast<const BfV<VEC>*>(p);
}
template <int VEC>
__device__ __forceinline__ void stv(__bf16* p, const float (&x)[VEC]) {
  typedef __bf16 V __attribute__((ext_vector_type(VEC)));
  V v;
#pragma unroll
  for (int c = 0; c < VEC; ++c) v[c] = f2bf(x[c]);
  *reinterpret_cast<V*>(p) = v;
}

// ---------------------------------------------------------------------------
// conv4 + SiLU.  One thread per (channel, batch row, CONV_TC-token chunk): the
// chunk's inputs (plus the 3-token halo) are loaded into registers up front so
// the loads overlap, then the window slides through registers.  xs[-3..-1] is
// the initial state (zeros when absent); y_t = silu(sum_k w_k xs[t-3+k]).
// ---------------------------------------------------------------------------
constexpr int CONV_TC = 32;

struct ConvArgs {
  int B, T, D;
  const __bf16* __restrict__ x;
  long long sb, st;
  const float* __restrict__ w;       // [D][4]
  const __bf16* __restrict__ init;   // [B][D][3] or null
};

__device__ __forceinline__ float conv_x(const ConvArgs& a, int b, int t, int d) {
  if (t >= a.T) return 0.f;
  if (t >= 0) return bf2f(a.x[(long long)b * a.sb + (long long)t * a.st + d]);
  if (!a.init) return 0.f;
  return bf2f(a.init[((long long)b * a.D + d) * 3 + (t + 3)]);
}

// xs[t0 - 3 + j] for j < N: every load reads a clamped, valid token and is
// issued before the first use (a guarded load would branch and wait for the
// loads before it); tokens past T read 0, and the three halo tokens of the
// first chunk come from the initial state (zeros when absent).
template <int N>
__device__ __forceinline__ void conv_window(const ConvArgs& a, int b, int t0, int d, float (&xv)[N]) {
  const __bf16* xb = a.x + (long long)b * a.sb + d;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int t = t0 - 3 + j, tc = t < 0 ? 0 : (t < a.T ? t : a.T - 1);
    xv[j] = keep_if(t < a.T, bf2f(xb[(long long)tc * a.st]));
  }
  if (t0 == 0) {
#pragma unroll
    for (int j = 0; j < 3; ++j)
      xv[j] = a.init ? bf2f(a.init[((long long)b * a.D + d) * 3 + j]) : 0.f;
  }
}

__global__ __launch_bounds__(NTHREADS) void k_conv_fwd(ConvArgs a, __bf16* __restrict__ y,
                                                       __bf16* __restrict__ fin) {
  const int d = blockIdx.x * NTHREADS + threadIdx.x, b = blockIdx.z;
  if (d >= a.D) return;
  const int t0 = blockIdx.y * CONV_TC;
  const float w0 = a.w[d * 4], w1 = a.w[d * 4 + 1], w2 = a.w[d * 4 + 2], w3 = a.w[d * 4 + 3];
  float xv[CONV_TC + 3];
  conv_window(a, b, t0, d, xv);
#pragma unroll
  for (int j = 0; j < CONV_TC; ++j) {
    const int t = t0 + j;
    const float acc = w0 * xv[j] + w1 * xv[j + 1] + w2 * xv[j + 2] + w3 * xv[j + 3];
    if (t < a.T) y[((long long)b * a.T + t) * a.D + d] = f2bf(silu(acc));
  }
  if (fin && t0 + CONV_TC >= a.T) {  // the chunk that holds the last token writes the state
    __bf16* f = fin + ((long long)b * a.D + d) * 3;
    f[0] = f2bf(conv_x(a, b, a.T - 3, d));
    f[1] = f2bf(conv_x(a, b, a.T - 2, d));
    f[2] = f2bf(conv_x(a, b, a.T - 1, d));
  }
}

// Backward.  da_t = dy_t silu'(a_t);  dx_s = sum_k w_k da_{s+3-k} (+ dfinal);
// dw_k = sum_t da_t xs[t-3+k];  dinit_j = sum_{k<=j} w_k da_{j-k} (+ dfinal).
// Thread (d, b, chunk) recomputes a_t for t in [t0, t0 + CONV_TC + 3) from
// register-resident inputs (zero beyond T), so every dx of its chunk is local.
__global__ __launch_bounds__(NTHREADS) void k_conv_bwd(ConvArgs a, const __bf16* __restrict__ dy,
                                                       const __bf16* __restrict__ dfin,
                                                       __bf16* __restrict__ dx,
                                                       float* __restrict__ dinit,
                                                       float* __restrict__ dw_part) {
  const int d = blockIdx.x * NTHREADS + threadIdx.x, b = blockIdx.z;
  if (d >= a.D) return;
  const int T = a.T, t0 = blockIdx.y * CONV_TC;
  const float w0 = a.w[d * 4], w1 = a.w[d * 4 + 1], w2 = a.w[d * 4 + 2], w3 = a.w[d * 4 + 3];
  constexpr int NX = CONV_TC + 6, NA = CONV_TC + 3;
  float xv[NX];   // xs[t0-3 .. t0+CONV_TC+2]
  float gv[NA];   // dy[t0 .. t0+CONV_TC+2]
  conv_window(a, b, t0, d, xv);
#pragma unroll
  for (int j = 0; j < NA; ++j) {  // clamped token, then select
    const int t = t0 + j;
    gv[j] = keep_if(t < T, bf2f(dy[((long long)b * T + (t < T ? t : T - 1)) * a.D + d]));
  }
  float df[3] = {0.f, 0.f, 0.f};  // dfinal_m is the cotangent of xs[T-3+m]
  if (dfin)
#pragma unroll
    for (int m = 0; m < 3; ++m) df[m] = bf2f(dfin[((long long)b * a.D + d) * 3 + m]);
  float da[NA];
  float g0 = 0.f, g1 = 0.f, g2 = 0.f, g3 = 0.f;
#pragma unroll
  for (int j = 0; j < NA; ++j) {
    const float acc = w0 * xv[j] + w1 * xv[j + 1] + w2 * xv[j + 2] + w3 * xv[j + 3];
    const float sg = sigm(acc);
    da[j] = gv[j] * sg * (1.f + acc * (1.f - sg));   // gv = 0 beyond T
    if (j < CONV_TC) {
      g0 += da[j] * xv[j]; g1 += da[j] * xv[j + 1]; g2 += da[j] * xv[j + 2];
      g3 += da[j] * xv[j + 3];
    }
  }
#pragma unroll
  for (int j = 0; j < CONV_TC; ++j) {
    const int s = t0 + j;
    if (s < T) {
      float v = w3 * da[j] + w2 * da[j + 1] + w1 * da[j + 2] + w0 * da[j + 3];
      if (s >= T - 3) v += df[s - (T - 3)];
      dx[((long long)b * T + s) * a.D + d] = f2bf(v);
    }
  }
  if (t0 == 0 && dinit) {
    // xs[-3+j] feeds a_t for t = j - k >= 0 with weight w_k (k <= j)
    float v0 = w0 * da[0];
    float v1 = w1 * da[0] + w0 * da[1];
    float v2 = w2 * da[0] + w1 * da[1] + w0 * da[2];
#pragma unroll
    for (int m = 0; m < 3; ++m) {  // final-state cotangents that land on the initial state (T < 3)
      const int j = T + m;
      if (j < 3) (j == 0 ? v0 : j == 1 ? v1 : v2) += df[m];
    }
    float* di = dinit + ((long long)b * a.D + d) * 3;
    di[0] = v0; di[1] = v1; di[2] = v2;
  }
  float* p = dw_part + (((long long)b * gridDim.y + blockIdx.y) * a.D + d) * 4;
  p[0] = g0; p[1] = g1; p[2] = g2; p[3] = g3;
}

// out[i] = sum_p part[p][i]: COLS columns x 256 / COLS partial rows per workgroup,
// the row sums combined through LDS.  32 columns (whole lines) for wide sums; 8
// where the width alone would leave the chip idle and each thread a long chain
// of loads (1024 rows of 128: 11 us with 32 columns, 4 workgroups).  The row sums are
// added in chains of eight, the chains pairwise: one chain of 32 doubled the
// rounding error (125 rows of sums of 16 terms in [1, 2]: 8.9e-8 relative; 5.3e-8
// with the eight row sums of 32 columns, 4.3e-8 in chains).
template <int COLS>
__global__ __launch_bounds__(NTHREADS) void k_sum_parts(const float* __restrict__ part, int nparts,
                                                        int width, float* __restrict__ out) {
  constexpr int ROWS = NTHREADS / COLS;
  __shared__ float red[ROWS][COLS + 1];
  const int cx = threadIdx.x % COLS, ry = threadIdx.x / COLS;
  const int i = blockIdx.x * COLS + cx;
  float s = 0.f;
  if (i < width) {
#pragma unroll 8
    for (int p = ry; p < nparts; p += ROWS) s += part[(long long)p * width + i];
  }
  red[ry][cx] = s;
  __syncthreads();
  if (ry == 0 && i < width) {
    constexpr int NC = ROWS / 8;
    float t[NC] = {};
#pragma unroll
    for (int k = 0; k < ROWS; ++k) t[k % NC] += red[k][cx];
#pragma unroll
    for (int n = NC / 2; n > 0; n /= 2)
#pragma unroll
      for (int k = 0; k < n; ++k) t[k] += t[k + n];
    out[i] = t[0];
  }
}

static void launch_sum_parts(const float* part, int nparts, int width, float* out, hipStream_t st) {
  if (width <= 1024)
    SD_LAUNCH("k_sum_parts", k_sum_parts<8>, dim3((width + 7) / 8), dim3(NTHREADS), 0, st, part, nparts, width, out);
  else
    SD_LAUNCH("k_sum_parts", k_sum_parts<32>, dim3((width + 31) / 32), dim3(NTHREADS), 0, st, part, nparts, width,
              out);
}

// ---------------------------------------------------------------------------
// KDA decay gate.  raw [N][H*r] bf16 (row stride), bias [H*r], log_rate [H].
// ---------------------------------------------------------------------------
constexpr int GATE_TR = 16;  // rows per thread (and per partial row) in the backward
constexpr int GATE_FR = 8;   // rows per thread in the forward

// Thread (row group, VEC neighbouring columns): the columns' rate and bias are
// loaded once, the rows' loads are all in flight before the first use.  VEC = 4
// where rows start on 8-byte (raw) and 16-byte (FP32) boundaries; one column
// per element otherwise.  15 us forward (3.4 TB/s) and 22 us backward (3.0 TB/s) at
// 8192 rows of 1024, bound about equally by HBM and the transcendentals, where
// a thread per element (a 64-bit division each, log1pf) took 37 and 37 us.
struct GateArgs {
  int N, H, r, HR;
  const __bf16* __restrict__ raw;
  long long rs;
  const float* __restrict__ log_rate;
  const float* __restrict__ bias;
};
template <int VEC>
__device__ __forceinline__ void gate_cols(const GateArgs& a, int c, float (&rate)[VEC], float (&b)[VEC]) {
#pragma unroll
  for (int k = 0; k < VEC; ++k) {
    rate[k] = __expf(a.log_rate[(c + k) / a.r]);
    b[k] = a.bias[c + k];
  }
}
template <int VEC> struct FV { float v[VEC]; };

template <int VEC>
__global__ __launch_bounds__(NTHREADS) void k_gate_fwd(GateArgs a, float* __restrict__ out) {
  const unsigned Q = a.HR / VEC, idx = blockIdx.x * NTHREADS + threadIdx.x, rg = idx / Q;
  const unsigned N = a.N, n0 = rg * GATE_FR;
  const int c = (idx - rg * Q) * VEC;
  if (n0 >= N) return;
  BfV<VEC> x[GATE_FR];
#pragma unroll
  for (int j = 0; j < GATE_FR; ++j) x[j] = ldv<VEC>(a.raw + (long long)min(n0 + j, N - 1) * a.rs + c);
  float rate[VEC], b[VEC];
  gate_cols<VEC>(a, c, rate, b);
#pragma unroll
  for (int j = 0; j < GATE_FR; ++j) {
    float v[VEC];
    x[j].get(v);
    FV<VEC> o;
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
      const float t = v[k] + b[k];
      o.v[k] = -rate[k] * softplus_t(t, __expf(-fabsf(t)));
    }
    if (n0 + j < N) *reinterpret_cast<FV<VEC>*>(out + (long long)(n0 + j) * a.HR + c) = o;
  }
}

// draw = dout * (-exp(lr)) * sigmoid(raw + bias) (softplus' is 1 above the
// threshold); partials: dbias_c = sum draw, dlr_c = sum dout * out.
template <int VEC>
__global__ __launch_bounds__(NTHREADS) void k_gate_bwd(GateArgs a, const float* __restrict__ dout,
                                                       __bf16* __restrict__ draw,
                                                       float* __restrict__ part) {
  const unsigned Q = a.HR / VEC, idx = blockIdx.x * NTHREADS + threadIdx.x, rg = idx / Q;
  const unsigned N = a.N, n0 = rg * GATE_TR;
  const int c = (idx - rg * Q) * VEC;
  if (n0 >= N) return;
  BfV<VEC> x[GATE_TR];
  FV<VEC> g[GATE_TR];
#pragma unroll
  for (int j = 0; j < GATE_TR; ++j) {
    const long long n = min(n0 + j, N - 1);
    x[j] = ldv<VEC>(a.raw + n * a.rs + c);
    g[j] = *reinterpret_cast<const FV<VEC>*>(dout + n * a.HR + c);
  }
  float rate[VEC], b[VEC];
  gate_cols<VEC>(a, c, rate, b);
  FV<VEC> db = {}, dl = {};
#pragma unroll
  for (int j = 0; j < GATE_TR; ++j) {
    if (n0 + j >= N) break;
    float v[VEC], dx[VEC];
    x[j].get(v);
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
      const float t = v[k] + b[k];
      const float et = __expf(-fabsf(t));
      dx[k] = -rate[k] * g[j].v[k] * sigm_t(t, et);
      db.v[k] += dx[k];
      dl.v[k] += -rate[k] * softplus_t(t, et) * g[j].v[k];
    }
    stv<VEC>(draw + (long long)(n0 + j) * a.HR + c, dx);
  }
  float* p = part + (long long)rg * 2 * a.HR + c;
  *reinterpret_cast<FV<VEC>*>(p) = db;
  *reinterpret_cast<FV<VEC>*>(p + a.HR) = dl;
}

// One workgroup per head: dbias[c] for the head's columns, dlog_rate[h], from
// nparts partial rows (the backward passes the one row of column sums).
__global__ __launch_bounds__(NTHREADS) void k_gate_reduce(int H, int r, int nparts,
                                                          const float* part, float* dbias,
                                                          float* dlog_rate) {
  __shared__ float red[NTHREADS / 64];
  const int h = blockIdx.x, HR = H * r;
  float acc = 0.f;
  for (int cc = threadIdx.x; cc < r; cc += NTHREADS) {
    const int c = h * r + cc;
    float db = 0.f, dl = 0.f;
    for (int p = 0; p < nparts; ++p) {
      db += part[(long long)p * 2 * HR + c];
      dl += part[(long long)p * 2 * HR + HR + c];
    }
    dbias[c] = db;
    acc += dl;
  }
  acc = wave_sum(acc);
  if (lane_id() == 0) red[wave_id()] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = 0.f;
    for (int w = 0; w < NTHREADS / 64; ++w) s += red[w];
    dlog_rate[h] = s;
  }
}

// ---------------------------------------------------------------------------
// Sigmoid-gated RMSNorm: y = x rstd w sigmoid(g), rstd = 1/sqrt(mean(x^2) + eps).
// One wave per row of width D <= 256 (4 elements per lane).
// ---------------------------------------------------------------------------
constexpr int RMS_ROWS = 4;     // rows (waves) per workgroup
constexpr int RMS_PART = 64;    // rows per dweight partial

__device__ __forceinline__ void rms_row(const __bf16* x, const __bf16* g, const float* w, int D,
                                        float (&xv)[4], float (&gv)[4], float (&wv)[4]) {
  const int l = lane_id();
#pragma unroll
  for (int m = 0; m < 4; ++m) {  // clamped column, then select: no branch around the loads
    const int c = l + 64 * m, cc = c < D ? c : D - 1;
    const bool ok = c < D;
    xv[m] = keep_if(ok, bf2f(x[cc]));
    gv[m] = keep_if(ok, bf2f(g[cc]));
    wv[m] = keep_if(ok, w[cc]);
  }
}

__global__ __launch_bounds__(RMS_ROWS * 64) void k_rms_fwd(int N, int D, float eps,
                                                           const __bf16* x, const __bf16* g,
                                                           const float* w, __bf16* y,
                                                           float* rstd_out) {
  const int n = blockIdx.x * RMS_ROWS + wave_id();
  if (n >= N) return;
  float xv[4], gv[4], wv[4];
  rms_row(x + (long long)n * D, g + (long long)n * D, w, D, xv, gv, wv);
  const float ss = wave_sum(xv[0] * xv[0] + xv[1] * xv[1] + xv[2] * xv[2] + xv[3] * xv[3]);
  const float rs = rsqrtf(ss / D + eps);
  const int l = lane_id();
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int c = l + 64 * m;
    if (c < D) y[(long long)n * D + c] = f2bf(xv[m] * rs * wv[m] * sigm(gv[m]));
  }
  if (rstd_out && l == 0) rstd_out[n] = rs;
}

// dx = rstd (gy - xhat mean(gy xhat)), gy = dy w s;  dg = dy xhat w s (1 - s);
// dw_c = sum dy xhat s;  y (recomputed for the projection's weight gradient).
// Each wave takes RMS_U rows at a time, every row's loads issued before the
// first row's reductions (rows past N read row N - 1 and store nothing).
constexpr int RMS_U = 4;
static_assert(RMS_PART % (RMS_ROWS * RMS_U) == 0, "whole row groups per workgroup");

__global__ __launch_bounds__(RMS_ROWS * 64) void k_rms_bwd(int N, int D, float eps,
                                                           const __bf16* __restrict__ x,
                                                           const __bf16* __restrict__ g,
                                                           const float* __restrict__ w,
                                                           const __bf16* __restrict__ dy,
                                                           __bf16* __restrict__ dx,
                                                           __bf16* __restrict__ dg,
                                                           __bf16* __restrict__ y,
                                                           float* __restrict__ part) {
  __shared__ float pw[RMS_ROWS][256];
  const int l = lane_id(), wv_ = wave_id();
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  float wv[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int c = l + 64 * m;
    wv[m] = keep_if(c < D, w[c < D ? c : D - 1]);
  }
  // a workgroup covers RMS_PART rows: each wave walks RMS_PART / RMS_ROWS of them
  const int base = blockIdx.x * RMS_PART;
  for (int r0 = wv_; r0 < RMS_PART; r0 += RMS_ROWS * RMS_U) {
    if (base + r0 >= N) break;
    float xv[RMS_U][4], gv[RMS_U][4], dv[RMS_U][4];
#pragma unroll
    for (int u = 0; u < RMS_U; ++u) {
      const int n = base + r0 + u * RMS_ROWS, nc = n < N ? n : N - 1;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int c = l + 64 * m, cc = c < D ? c : D - 1;
        const long long o = (long long)nc * D + cc;
        xv[u][m] = keep_if(c < D, bf2f(x[o]));
        gv[u][m] = keep_if(c < D, bf2f(g[o]));
        dv[u][m] = keep_if(c < D && n < N, bf2f(dy[o]));
      }
    }
#pragma unroll
    for (int u = 0; u < RMS_U; ++u) {
      const int n = base + r0 + u * RMS_ROWS;
      const float ss = wave_sum(xv[u][0] * xv[u][0] + xv[u][1] * xv[u][1] + xv[u][2] * xv[u][2] +
                                xv[u][3] * xv[u][3]);
      const float rs = rsqrtf(ss / D + eps);
      float gy[4], xh[4], sg[4], dot = 0.f;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        sg[m] = sigm(gv[u][m]);
        xh[m] = xv[u][m] * rs;
        gy[m] = dv[u][m] * wv[m] * sg[m];
        dot += gy[m] * xh[m];
      }
      dot = wave_sum(dot) / D;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int c = l + 64 * m;
        acc[m] += dv[u][m] * xh[m] * sg[m];  // 0 on rows past N (dv = 0)
        if (c < D && n < N) {
          const long long o = (long long)n * D + c;
          dx[o] = f2bf(rs * (gy[m] - xh[m] * dot));
          dg[o] = f2bf(dv[u][m] * xh[m] * wv[m] * sg[m] * (1.f - sg[m]));
          if (y) y[o] = f2bf(xh[m] * wv[m] * sg[m]);
        }
      }
    }
  }
#pragma unroll
  for (int m = 0; m < 4; ++m) pw[wv_][l + 64 * m] = acc[m];
  __syncthreads();
  for (int c = threadIdx.x; c < D; c += RMS_ROWS * 64) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < RMS_ROWS; ++k) s += pw[k][c];
    part[(long long)blockIdx.x * D + c] = s;
  }
}

// The same with LPR (8, 16, 32) lanes per row, eight neighbouring columns each:
// D <= 8 LPR a multiple of 8 and 16-byte aligned rows, so a row is one 16-byte
// load per lane and a wave covers 64 / LPR rows.  HBM bound: 14 us forward,
// 17 us backward (3.6 and 4.9 TB/s) at 65536 rows of 128, where a wave per row with 2-byte loads
// (half its lanes idle at D = 128) took 19 and 30 us.
template <int LPR>
__device__ __forceinline__ float lanes_sum(float v) {
  v = dpp_add(v, 0);
  v = dpp_add(v, 1);
  v = dpp_add(v, 2);
  if constexpr (LPR >= 16) v = dpp_add(v, 3);
  if constexpr (LPR >= 32) v += __shfl_xor(v, 16);
  return v;
}
constexpr int RMSV_U = 4;  // rows per lane group and batch, all loads in flight

template <int LPR>
__global__ __launch_bounds__(NTHREADS) void k_rmsv_fwd(int N, int D, float eps, const __bf16* __restrict__ x,
                                                       const __bf16* __restrict__ g, const float* __restrict__ w,
                                                       __bf16* __restrict__ y, float* __restrict__ rstd_out) {
  constexpr int G = NTHREADS / LPR;
  const int c = (threadIdx.x % LPR) * 8, cc = c < D ? c : 0;
  const unsigned n0 = blockIdx.x * G * RMSV_U + threadIdx.x / LPR;  // (rows past N may pass 2^31)
  BfV<8> xr[RMSV_U], gr[RMSV_U];
#pragma unroll
  for (int u = 0; u < RMSV_U; ++u) {
    const long long o = (long long)min(n0 + u * G, (unsigned)N - 1) * D + cc;
    xr[u] = ldv<8>(x + o);
    gr[u] = ldv<8>(g + o);
  }
  float wv[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) wv[e] = w[cc + e];
#pragma unroll
  for (int u = 0; u < RMSV_U; ++u) {
    const unsigned n = n0 + u * G;
    float xv[8], gv[8], o[8], ss = 0.f;
    xr[u].get(xv);
    gr[u].get(gv);
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += xv[e] * xv[e];
    const float rs = rsqrtf(lanes_sum<LPR>(c < D ? ss : 0.f) / D + eps);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = xv[e] * rs * wv[e] * sigm(gv[e]);
    if (n < (unsigned)N && c < D) stv<8>(y + (long long)n * D + c, o);
    if (rstd_out && n < (unsigned)N && c == 0) rstd_out[n] = rs;
  }
}

// rows: per workgroup (rmsv_rows), a multiple of NTHREADS / LPR * RMSV_U
template <int LPR>
__global__ __launch_bounds__(NTHREADS) void k_rmsv_bwd(int N, int D, float eps, int rows,
                                                       const __bf16* __restrict__ x,
                                                       const __bf16* __restrict__ g,
                                                       const float* __restrict__ w,
                                                       const __bf16* __restrict__ dy,
                                                       __bf16* __restrict__ dx, __bf16* __restrict__ dg,
                                                       __bf16* __restrict__ y, float* __restrict__ part) {
  constexpr int G = NTHREADS / LPR;
  __shared__ float pw[G][LPR * 8 + 4];
  const int c = (threadIdx.x % LPR) * 8, cc = c < D ? c : 0, gr_ = threadIdx.x / LPR;
  const bool in = c < D;
  float wv[8], acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    wv[e] = w[cc + e];
    acc[e] = 0.f;
  }
  const unsigned base = blockIdx.x * rows;
  for (int r0 = gr_; r0 < rows; r0 += G * RMSV_U) {
    BfV<8> xr[RMSV_U], gr[RMSV_U], dr[RMSV_U];
#pragma unroll
    for (int u = 0; u < RMSV_U; ++u) {
      const long long o = (long long)min(base + r0 + u * G, (unsigned)N - 1) * D + cc;
      xr[u] = ldv<8>(x + o);
      gr[u] = ldv<8>(g + o);
      dr[u] = ldv<8>(dy + o);
    }
#pragma unroll
    for (int u = 0; u < RMSV_U; ++u) {
      const unsigned n = base + r0 + u * G;
      const bool ok = in && n < (unsigned)N;
      float xh[8], gv[8], dv[8], sg[8], gy[8], ss = 0.f, dot = 0.f;
      xr[u].get(xh);
      gr[u].get(gv);
      dr[u].get(dv);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += xh[e] * xh[e];
      const float rs = rsqrtf(lanes_sum<LPR>(in ? ss : 0.f) / D + eps);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        sg[e] = sigm(gv[e]);
        xh[e] *= rs;
        gy[e] = dv[e] * wv[e] * sg[e];
        dot += gy[e] * xh[e];
      }
      dot = lanes_sum<LPR>(in ? dot : 0.f) / D;
      float ox[8], og[8], oy[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        acc[e] += ok ? dv[e] * xh[e] * sg[e] : 0.f;
        ox[e] = rs * (gy[e] - xh[e] * dot);
        og[e] = dv[e] * xh[e] * wv[e] * sg[e] * (1.f - sg[e]);
        oy[e] = xh[e] * wv[e] * sg[e];
      }
      if (ok) {
        const long long o = (long long)n * D + c;
        stv<8>(dx + o, ox);
        stv<8>(dg + o, og);
        if (y) stv<8>(y + o, oy);
      }
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) pw[gr_][c + e] = acc[e];
  __syncthreads();
  for (int k = threadIdx.x; k < D; k += NTHREADS) {
    float t = 0.f;
#pragma unroll
    for (int q = 0; q < G; ++q) t += pw[q][k];
    part[(long long)blockIdx.x * D + k] = t;
  }
}

static inline int cdiv(long long a, int b) { return (int)((a + b - 1) / b); }


// ---------------------------------------------------------------------------
// conv4 + SiLU under valid / reset masks, the CPU loop's semantics
// (model.py:146-164): a reset on a valid token zeroes the 3-token state first;
// an invalid token emits 0 and leaves the state; a valid token emits
// silu(w . [state, x_t]) and shifts x_t into the state.
//
// A chunk's window depends on the row's history only through the last three
// valid tokens since the last reset, so each workgroup finds those by scanning
// the masks backwards from its chunk, 64 tokens per ballot (the result is wave
// uniform, held in scalar registers), and chunks run in parallel.  The scan ends
// within its first ballot unless the row holds long invalid stretches.  HBM
// bound: 33 us forward (3.1 TB/s of x and y) and 55 us backward (2.8 TB/s of x,
// dy and dx) at B4 T2048 D3072, where one thread walking a whole row serially
// (a load latency per 8 tokens, 48 workgroups in all) took 1374 and 1588 us.
// ---------------------------------------------------------------------------
struct ConvMask {
  const uint8_t* __restrict__ valid;  // [B,T] at b*sb + t*st, nullable (all valid)
  const uint8_t* __restrict__ reset;  // nullable (no reset)
  long long sb, st;
};
// Backward workgroups (and dw partial rows) per batch row: with more chunks than
// this a workgroup takes every MCONV_PARTS-th, which bounds the workspace
// whatever the row length.
constexpr int MCONV_PARTS = 64;
constexpr int MCONV_TC = 32;   // tokens per chunk (16 in the backward measured the same, 56 us)
constexpr int kNoSlot = -4;    // a window slot cleared by a reset

// Valid bits and reset-on-valid bits of tokens base .. base + 63 (0 outside [0, T)).
__device__ __forceinline__ void conv_mask_bits(const ConvMask& m, int b, int base, int T,
                                               unsigned long long& V, unsigned long long& R) {
  const int t = base + lane_id();
  const bool in = t >= 0 && t < T;
  const long long o = (long long)b * m.sb + (long long)(in ? t : 0) * m.st;
  const bool v = in && (m.valid ? m.valid[o] != 0 : true);
  const bool r = v && m.reset && m.reset[o] != 0;
  V = __ballot(v);
  R = __ballot(r);
}

// The window before token t0: p[0] the newest slot .. p[2] the oldest, each a
// token (>= 0), an initial-state slot (-1 newest .. -3) or kNoSlot.
__device__ __forceinline__ void conv_lookback(const ConvMask& m, int b, int t0, int T, int (&p)[3]) {
  int n = 0;
  bool closed = false;
  p[0] = p[1] = p[2] = kNoSlot;
  for (int base = t0 - 64; n < 3 && !closed && base > -64; base -= 64) {
    unsigned long long V, R;
    conv_mask_bits(m, b, base, T, V, R);
    while (V && n < 3 && !closed) {
      const int i = 63 - __clzll((long long)V);
      if (n == 0) p[0] = base + i;
      else if (n == 1) p[1] = base + i;
      else p[2] = base + i;
      ++n;
      closed = (R >> i) & 1;
      V &= ~(1ull << i);
    }
  }
  if (!closed) {  // the row's start: the initial state's newest slots follow
    if (n == 0) { p[0] = -1; p[1] = -2; p[2] = -3; }
    else if (n == 1) { p[1] = -1; p[2] = -2; }
    else if (n == 2) p[2] = -1;
  }
}

// Up to three valid tokens from t1 on, up to the first reset (which sees
// nothing earlier); returns their count.  closed: a reset ended the scan.
__device__ __forceinline__ int conv_lookahead(const ConvMask& m, int b, int t1, int T, int (&p)[3],
                                              bool& closed) {
  int n = 0;
  closed = false;
  p[0] = p[1] = p[2] = T - 1;
  for (int base = t1; n < 3 && !closed && base < T; base += 64) {
    unsigned long long V, R;
    conv_mask_bits(m, b, base, T, V, R);
    while (V && n < 3 && !closed) {
      const int i = __ffsll((unsigned long long)V) - 1;
      if ((R >> i) & 1) {
        closed = true;
      } else {
        if (n == 0) p[0] = base + i;
        else if (n == 1) p[1] = base + i;
        else p[2] = base + i;
        ++n;
        V &= ~(1ull << i);
      }
    }
  }
  return n;
}

// One window slot's values for this thread's channels.
template <int VEC>
__device__ __forceinline__ void conv_slot(const ConvArgs& a, int b, int p, unsigned d, float (&v)[VEC]) {
  ldv<VEC>(a.x + (long long)b * a.sb + (long long)(p >= 0 ? p : 0) * a.st + d).get(v);
#pragma unroll
  for (int c = 0; c < VEC; ++c) {
    if (p < 0) v[c] = 0.f;
    if (p < 0 && p > kNoSlot && a.init) v[c] = bf2f(a.init[((long long)b * a.D + d + c) * 3 + p + 3]);
  }
}

template <int VEC>
__global__ __launch_bounds__(NTHREADS) void k_conv_masked_fwd(ConvArgs a, ConvMask m,
                                                              __bf16* __restrict__ y,
                                                              __bf16* __restrict__ fin) {
  constexpr int TC = MCONV_TC;
  const int d0 = (blockIdx.x * NTHREADS + threadIdx.x) * VEC, b = blockIdx.z;
  const int T = a.T, D = a.D;
  const bool live = d0 < D;  // (whole waves take part in the ballots)
  const unsigned d = live ? d0 : 0;  // 32-bit lane offset from a wave-uniform row
  float w[VEC][4];
#pragma unroll
  for (int c = 0; c < VEC; ++c)
#pragma unroll
    for (int k = 0; k < 4; ++k) w[c][k] = a.w[(d + c) * 4 + k];
  for (int t0 = blockIdx.y * TC; t0 < T; t0 += gridDim.y * TC) {
    unsigned long long V, R;
    conv_mask_bits(m, b, t0, T, V, R);
    const bool last = t0 + TC >= T;
    __bf16* yr = y + ((long long)b * T + t0) * D;
    if ((unsigned)V == 0 && !(last && fin)) {  // no valid token in the chunk
      if (live)
#pragma unroll
        for (int j = 0; j < TC; ++j)
          if (t0 + j < T) stv<VEC>(yr + (long long)j * D + d, {});
      continue;
    }
    BfV<VEC> xv[TC];
#pragma unroll
    for (int j = 0; j < TC; ++j)
      xv[j] = ldv<VEC>(a.x + (long long)b * a.sb + (long long)min(t0 + j, T - 1) * a.st + d);
    int p[3];
    conv_lookback(m, b, t0, T, p);
    float s0[VEC], s1[VEC], s2[VEC];
    conv_slot<VEC>(a, b, p[2], d, s0);
    conv_slot<VEC>(a, b, p[1], d, s1);
    conv_slot<VEC>(a, b, p[0], d, s2);
    if (!live) continue;
#pragma unroll
    for (int j = 0; j < TC; ++j) {
      const bool v = (V >> j) & 1, r = (R >> j) & 1;
      float x[VEC], o[VEC];
      xv[j].get(x);
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        if (r) s0[c] = s1[c] = s2[c] = 0.f;
        const float acc = w[c][0] * s0[c] + w[c][1] * s1[c] + w[c][2] * s2[c] + w[c][3] * x[c];
        o[c] = v ? silu(acc) : 0.f;
        s0[c] = v ? s1[c] : s0[c];
        s1[c] = v ? s2[c] : s1[c];
        s2[c] = v ? x[c] : s2[c];
      }
      if (t0 + j < T) stv<VEC>(yr + (long long)j * D + d, o);
    }
    if (fin && last) {
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        __bf16* f = fin + ((long long)b * D + d + c) * 3;
        f[0] = f2bf(s0[c]);
        f[1] = f2bf(s1[c]);
        f[2] = f2bf(s2[c]);
      }
    }
  }
}

// Backward.  A forward sweep over the chunk's tokens and the next three valid
// ones forms da_t = dy_t silu'(a_t) and the dw partials; a reverse sweep then
// gathers dx_s = w3 da_s + w2 da_n1 + w1 da_n2 + w0 da_n3 over the next valid
// tokens n1, n2, n3 of s's segment, plus the final state's cotangent where s is
// one of the row's last three.  Chunk 0 holds (through its look-ahead) the
// row's first three valid tokens and forms dinit.
template <int VEC>
__global__ __launch_bounds__(NTHREADS) void k_conv_masked_bwd(ConvArgs a, ConvMask m,
                                                              const __bf16* __restrict__ dy,
                                                              const __bf16* __restrict__ dfin,
                                                              __bf16* __restrict__ dx,
                                                              float* __restrict__ dinit,
                                                              float* __restrict__ dw_part) {
  constexpr int TC = MCONV_TC;
  const int d0 = (blockIdx.x * NTHREADS + threadIdx.x) * VEC, b = blockIdx.z;
  const int T = a.T, D = a.D;
  const bool live = d0 < D;  // (whole waves take part in the ballots)
  const unsigned d = live ? d0 : 0;  // 32-bit lane offset from a wave-uniform row
  float w[VEC][4], gw[VEC][4];
#pragma unroll
  for (int c = 0; c < VEC; ++c)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      w[c][k] = a.w[(d + c) * 4 + k];
      gw[c][k] = 0.f;
    }
  for (int t0 = blockIdx.y * TC; t0 < T; t0 += gridDim.y * TC) {
    unsigned long long V, R;
    conv_mask_bits(m, b, t0, T, V, R);
    __bf16* dxr = dx + ((long long)b * T + t0) * D;
    if ((unsigned)V == 0 && !(t0 == 0 && dinit && a.init)) {
      if (live)
#pragma unroll
        for (int j = 0; j < TC; ++j)
          if (t0 + j < T) stv<VEC>(dxr + (long long)j * D + d, {});
      continue;
    }
    BfV<VEC> xv[TC], gv[TC], xh[3], gh[3];
#pragma unroll
    for (int j = 0; j < TC; ++j) {
      const int t = min(t0 + j, T - 1);
      xv[j] = ldv<VEC>(a.x + (long long)b * a.sb + (long long)t * a.st + d);
      gv[j] = ldv<VEC>(dy + ((long long)b * T + t) * D + d);
    }
    int p[3], q[3];
    bool closed;
    conv_lookback(m, b, t0, T, p);
    const int nh = conv_lookahead(m, b, t0 + TC, T, q, closed);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      xh[i] = ldv<VEC>(a.x + (long long)b * a.sb + (long long)q[i] * a.st + d);
      gh[i] = ldv<VEC>(dy + ((long long)b * T + q[i]) * D + d);
    }
    float s0[VEC], s1[VEC], s2[VEC];
    conv_slot<VEC>(a, b, p[2], d, s0);
    conv_slot<VEC>(a, b, p[1], d, s1);
    conv_slot<VEC>(a, b, p[0], d, s2);
    if (!live) continue;
    // (V and R are wave uniform: scalar branches, with no memory operation inside)
    float da[TC + 3][VEC];
#pragma unroll
    for (int j = 0; j < TC + 3; ++j) {
      const bool v = j < TC ? (V >> j) & 1 : j - TC < nh, r = j < TC ? (R >> j) & 1 : false;
#pragma unroll
      for (int c = 0; c < VEC; ++c) da[j][c] = 0.f;
      if (!v) continue;  // an invalid token's values may be anything
      float x[VEC], g[VEC];
      (j < TC ? xv[j < TC ? j : 0] : xh[j < TC ? 0 : j - TC]).get(x);
      (j < TC ? gv[j < TC ? j : 0] : gh[j < TC ? 0 : j - TC]).get(g);
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        if (r) s0[c] = s1[c] = s2[c] = 0.f;
        const float acc = w[c][0] * s0[c] + w[c][1] * s1[c] + w[c][2] * s2[c] + w[c][3] * x[c];
        const float sg = sigm(acc);
        da[j][c] = g[c] * sg * (1.f + acc * (1.f - sg));
        if (j < TC) {
          gw[c][0] += da[j][c] * s0[c];
          gw[c][1] += da[j][c] * s1[c];
          gw[c][2] += da[j][c] * s2[c];
          gw[c][3] += da[j][c] * x[c];
        }
        s0[c] = s1[c];
        s1[c] = s2[c];
        s2[c] = x[c];
      }
    }
    // the final state's cotangent: the token with `rank` valid ones after it, and
    // no reset in between, is slot 2 - rank of the final window
    float df[VEC][3], e1[VEC], e2[VEC], e3[VEC];
    int rank = nh;
    bool alive = dfin && !closed && nh < 3;
#pragma unroll
    for (int c = 0; c < VEC; ++c) {
#pragma unroll
      for (int k = 0; k < 3; ++k) df[c][k] = alive ? bf2f(dfin[((long long)b * D + d + c) * 3 + k]) : 0.f;
      e1[c] = da[TC][c];
      e2[c] = da[TC + 1][c];
      e3[c] = da[TC + 2][c];
    }
    auto dfin_at = [&](int c, int slot) {
      return !alive || slot < 0 ? 0.f : slot == 2 ? df[c][2] : slot == 1 ? df[c][1] : df[c][0];
    };
#pragma unroll
    for (int j = TC - 1; j >= 0; --j) {
      float o[VEC] = {};
      if ((V >> j) & 1) {
#pragma unroll
        for (int c = 0; c < VEC; ++c) {
          o[c] = w[c][3] * da[j][c] + w[c][2] * e1[c] + w[c][1] * e2[c] + w[c][0] * e3[c] +
                 dfin_at(c, 2 - rank);
          e3[c] = e2[c];
          e2[c] = e1[c];
          e1[c] = da[j][c];
        }
        ++rank;
        if ((R >> j) & 1) {
          alive = false;
#pragma unroll
          for (int c = 0; c < VEC; ++c) e1[c] = e2[c] = e3[c] = 0.f;
        }
      }
      if (t0 + j < T) stv<VEC>(dxr + (long long)j * D + d, o);
    }
    if (t0 == 0 && dinit && a.init) {  // e1, e2, e3: the row's first valid tokens, up to a reset
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        float* di = dinit + ((long long)b * D + d + c) * 3;
        di[0] = w[c][0] * e1[c] + dfin_at(c, 0 - rank);
        di[1] = w[c][1] * e1[c] + w[c][0] * e2[c] + dfin_at(c, 1 - rank);
        di[2] = w[c][2] * e1[c] + w[c][1] * e2[c] + w[c][0] * e3[c] + dfin_at(c, 2 - rank);
      }
    }
  }
  if (!live) return;
#pragma unroll
  for (int c = 0; c < VEC; ++c) {
    float* wp = dw_part + (((long long)b * gridDim.y + blockIdx.y) * D + d + c) * 4;
#pragma unroll
    for (int k = 0; k < 4; ++k) wp[k] = gw[c][k];
  }
}

}  // namespace sd

using namespace sd;

// Two channels per thread where every row of the three [.., D] operands starts
// on a 4-byte boundary (an even channel count and even strides).
static bool conv_pairs(const ConvArgs& a, const void* p, const void* q) {
  const uintptr_t bits = (uintptr_t)a.x | (uintptr_t)p | (uintptr_t)q;
  return a.D % 2 == 0 && a.sb % 2 == 0 && a.st % 2 == 0 && bits % 4 == 0;
}

// Backward workgroups per batch row (and dw partial rows) of a row of T tokens.
static int mconv_parts(int T) {
  const int nch = cdiv(T, MCONV_TC);
  return nch < MCONV_PARTS ? nch : MCONV_PARTS;
}

// Workgroups of a launch of one thread per (group of rows, column), whose index the
// kernels hold in 32 unsigned bits; 0 where it would not fit.
static int gate_blocks(int N, int rows, int cols) {
  const long long t = (long long)cdiv(N, rows) * cols;
  return t > 0xffffffffLL - NTHREADS ? 0 : cdiv(t, NTHREADS);
}

// Four columns per thread where every row of the bf16 operands starts on an
// 8-byte and of the FP32 operand on a 16-byte boundary.
static bool gate_quads(const GateArgs& a, const void* bf, const void* f32) {
  return a.HR % 4 == 0 && a.rs % 4 == 0 && (((uintptr_t)a.raw | (uintptr_t)bf) & 7) == 0 &&
         ((uintptr_t)f32 & 15) == 0;
}

// Rows per workgroup (and dweight partial) of the vector backward: one batch of its
// lanes (128 rows for D <= 64, 64 for D <= 128; two of 32 above, whose partials then
// fit the general path's workspace), and for D <= 128 two batches where that leaves
// two workgroups per CU and more.  Longer workgroups gain nothing and lose the CUs'
// balance; us with the sum of the partials, one / two / four batches, D = 128:
// 32768 rows 13.1 / 14.1 / 18.8, 65537 20.9 / 20.7 / 22.1, 98304 28.4 / 27.1 / 31.0,
// 262144 86.8 / 82.5 / 86.3.  D = 64: 32768 8.6 / 11.3 / 15.6, 262144 36.3 / 35.1 /
// 35.4.  D = 256: 131072 rows 82.5 in 64s, 84.8 in 128s.
static int rmsv_rows(int N, int D) {
  const int rows = D <= 64 ? 128 : RMS_PART;
  return D <= 128 && N > 2 * 512 * rows ? 2 * rows : rows;
}

// Eight columns per lane where rows are multiples of 8 wide and 16-byte aligned.
static bool rms_vec(int D, uintptr_t bits) { return D % 8 == 0 && (bits & 15) == 0; }

extern "C" {

size_t sd_conv4_workspace_bytes(int B, int T, int D) {
  if (B <= 0 || T <= 0 || D <= 0) return 0;
  return (size_t)B * cdiv(T, CONV_TC) * D * 4 * sizeof(float);
}

int sd_conv4_silu_fwd(int B, int T, int D, const void* x, int64_t x_sb, int64_t x_st,
                      const float* w, const void* init, void* y, void* final_state, void* stream) {
  if (B <= 0 || T <= 0 || D <= 0) return SD_ERR_SHAPE;
  if (!x || !w || !y) return SD_ERR_ARG;
  ConvArgs a{B, T, D, (const __bf16*)x, x_sb, x_st, w, (const __bf16*)init};
  dim3 grid(cdiv(D, NTHREADS), cdiv(T, CONV_TC), B);
  SD_LAUNCH("k_conv_fwd", k_conv_fwd, grid, dim3(NTHREADS), 0, (hipStream_t)stream, a,
            (__bf16*)y, (__bf16*)final_state);
  return hipGetLastError() == hipSuccess ? SD_OK : SD_ERR_LAUNCH;
}

int sd_conv4_silu_bwd(int B, int T, int D, const void* x, int64_t x_sb, int64_t x_st,
                      const float* w, const void* init, const void* dy, const void* dfinal,
                      void* dx, float* dw, float* dinit, void* workspace, size_t workspace_bytes,
                      void* stream) {
  if (B <= 0 || T <= 0 || D <= 0) return SD_ERR_SHAPE;
  if (!x || !w || !dy || !dx || !dw || !workspace) return SD_ERR_ARG;
  if (workspace_bytes < sd_conv4_workspace_bytes(B, T, D)) return SD_ERR_WORKSPACE;
  ConvArgs a{B, T, D, (const __bf16*)x, x_sb, x_st, w, (const __bf16*)init};
  const int nch = cdiv(T, CONV_TC);
  hipStream_t st = (hipStream_t)stream;
  SD_LAUNCH("k_conv_bwd", k_conv_bwd, dim3(cdiv(D, NTHREADS), nch, B), dim3(NTHREADS), 0, st, a,
            (const __bf16*)dy, (const __bf16*)dfinal, (__bf16*)dx, dinit, (float*)workspace);
  launch_sum_parts((const float*)workspace, B * nch, 4 * D, dw, st);
  return hipGetLastError() == hipSuccess ? SD_OK : SD_ERR_LAUNCH;
}

size_t sd_conv4_masked_workspace_bytes(int B, int D) {
  if (B <= 0 || D <= 0) return 0;
  return (size_t)B * MCONV_PARTS * D * 4 * sizeof(float);
}

size_t sd_conv4_masked_bwd_workspace_bytes(int B, int T, int D) {
  if (B <= 0 || T <= 0 || D <= 0) return 0;
  return (size_t)B * mconv_parts(T) * D * 4 * sizeof(float);
}

int sd_conv4_silu_masked_fwd(int B, int T, int D, const void* x, int64_t x_sb, int64_t x_st,
                             const float* w, const void* init, const uint8_t* valid,
                             const uint8_t* reset, int64_t m_sb, int64_t m_st, void* y,
                             void* final_state, void* stream) {
  if (B <= 0 || T <= 0 || D <= 0) return SD_ERR_SHAPE;
  if (!x || !w || !y) return SD_ERR_ARG;
  ConvArgs a{B, T, D, (const __bf16*)x, x_sb, x_st, w, (const __bf16*)init};
  ConvMask m{valid, reset, m_sb, m_st};
  const bool v2 = conv_pairs(a, y, y);
  const int nch = cdiv(T, MCONV_TC);
  const dim3 grid(cdiv(D, NTHREADS * (v2 ? 2 : 1)), nch < 32768 ? nch : 32768, B);
  if (v2)
    SD_LAUNCH("k_conv_masked_fwd", k_conv_masked_fwd<2>, grid, dim3(NTHREADS), 0,
              (hipStream_t)stream, a, m, (__bf16*)y, (__bf16*)final_state);
  else
    SD_LAUNCH("k_conv_masked_fwd", k_conv_masked_fwd<1>, grid, dim3(NTHREADS), 0,
              (hipStream_t)stream, a, m, (__bf16*)y, (__bf16*)final_state);
  return hipGetLastError() == hipSuccess ? SD_OK : SD_ERR_LAUNCH;
}

int sd_conv4_silu_masked_bwd(int B, int T, int D, const void* x, int64_t x_sb, int64_t x_st,
                             const float* w, const void* init, const uint8_t* valid,
                             const uint8_t* reset, int64_t m_sb, int64_t m_st, const void* dy,
                             const void* dfinal, void* dx, float* dw, float* dinit,
                             void* workspace, size_t workspace_bytes, void* stream) {
  if (B <= 0 || T <= 0 || D <= 0) return SD_ERR_SHAPE;
  if (!x || !w || !dy || !dx || !dw || !workspace) return SD_ERR_ARG;
  if (workspace_bytes < sd_conv4_masked_bwd_workspace_bytes(B, T, D)) return SD_ERR_WORKSPACE;
  ConvArgs a{B, T, D, (const __bf16*)x, x_sb, x_st, w, (const __bf16*)init};
  ConvMask m{valid, reset, m_sb, m_st};
  hipStream_t st = (hipStream_t)stream;
  const bool v2 = conv_pairs(a, dy, dx);
  const int parts = mconv_parts(T);
  const dim3 grid(cdiv(D, NTHREADS * (v2 ? 2 : 1)), parts, B);
  if (v2)
    SD_LAUNCH("k_conv_masked_bwd", k_conv_masked_bwd<2>, grid, dim3(NTHREADS), 0, st, a, m,
              (const __bf16*)dy, (const __bf16*)dfinal, (__bf16*)dx, dinit, (float*)workspace);
  else
    SD_LAUNCH("k_conv_masked_bwd", k_conv_masked_bwd<1>, grid, dim3(NTHREADS), 0, st, a, m,
              (const __bf16*)dy, (const __bf16*)dfinal, (__bf16*)dx, dinit, (float*)workspace);
  launch_sum_parts((const float*)workspace, B * parts, 4 * D, dw, st);
  return hipGetLastError() == hipSuccess ? SD_OK : SD_ERR_LAUNCH;
}

// Workspace: the [np][2][H*r] per-workgroup partials, then their [2][H*r] column sums.
size_t sd_kda_gate_workspace_bytes(int N, int H, int r) {
  if (N <= 0 || H <= 0 || r <= 0) return 0;
  return (size_t)(cdiv(N, GATE_TR) + 1) * 2 * H * r * sizeof(float);
}

int sd_kda_gate_fwd(int N, int H, int r, const void* raw, int64_t raw_row_stride,
                    const float* log_rate, const float* bias, float* out, void* stream) {
  if (N <= 0 || H <= 0 || r <= 0 || (long long)H * r > 0x7fffffff) return SD_ERR_SHAPE;
  if (!raw || !log_rate || !bias || !out) return SD_ERR_ARG;
  const GateArgs a{N, H, r, H * r, (const __bf16*)raw, raw_row_stride, log_rate, bias};
  const bool v4 = gate_quads(a, nullptr, out);
  const int blocks = gate_blocks(N, GATE_FR, v4 ? a.HR / 4 : a.HR);
  if (!blocks) return SD_ERR_SHAPE;
  if (v4)
    SD_LAUNCH("k_gate_fwd", k_gate_fwd<4>, dim3(blocks), dim3(NTHREADS), 0, (hipStream_t)stream, a, out);
  else
    SD_LAUNCH("k_gate_fwd", k_gate_fwd<1>, dim3(blocks), dim3(NTHREADS), 0, (hipStream_t)stream, a, out);
  return hipGetLastError() == hipSuccess ? SD_OK : SD_ERR_LAUNCH;
}

int sd_kda_gate_bwd(int N, int H, int r, const void* raw, int64_t raw_row_stride,
                    const float* log_rate, const float* bias, const float* dout, void* draw,
                    float* dlog_rate, float* dbias, void* workspace, size_t workspace_bytes,
                    void* stream) {
  if (N <= 0 || H <= 0 || r <= 0 || (long long)H * r > 0x3fffffff) return SD_ERR_SHAPE;  // (2 H r columns of sums)
  if (!raw || !log_rate || !bias || !dout || !draw || !dlog_rate || !dbias || !workspace)
    return SD_ERR_ARG;
  if (workspace_bytes < sd_kda_gate_workspace_bytes(N, H, r)) return SD_ERR_WORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  const int np = cdiv(N, GATE_TR);
  const GateArgs a{N, H, r, H * r, (const __bf16*)raw, raw_row_stride, log_rate, bias};
  const bool v4 = gate_quads(a, draw, dout) && ((uintptr_t)workspace & 15) == 0;
  const int blocks = gate_blocks(N, GATE_TR, v4 ? a.HR / 4 : a.HR);
  if (!blocks) return SD_ERR_SHAPE;
  if (v4)
    SD_LAUNCH("k_gate_bwd", k_gate_bwd<4>, dim3(blocks), dim3(NTHREADS), 0, st, a, dout, (__bf16*)draw,
              (float*)workspace);
  else
    SD_LAUNCH("k_gate_bwd", k_gate_bwd<1>, dim3(blocks), dim3(NTHREADS), 0, st, a, dout, (__bf16*)draw,
              (float*)workspace);
  // column sums over the partial rows spread over many workgroups (a per-head
  // walk over every partial row kept only H workgroups busy), then per head
  float* colsum = (float*)workspace + (size_t)np * 2 * H * r;
  launch_sum_parts((const float*)workspace, np, 2 * H * r, colsum, st);
  SD_LAUNCH("k_gate_reduce", k_gate_reduce, dim3(H), dim3(NTHREADS), 0, st, H, r, 1,
            (const float*)colsum, dbias, dlog_rate);
  return hipGetLastError() == hipSuccess ? SD_OK : SD_ERR_LAUNCH;
}

size_t sd_rmsnorm_gated_workspace_bytes(int N, int D) {
  if (N <= 0 || D <= 0) return 0;
  return (size_t)cdiv(N, RMS_PART) * D * sizeof(float);
}

int sd_rmsnorm_gated_fwd(int N, int D, float eps, const void* x, const void* gate,
                         const float* weight, void* y, float* rstd, void* stream) {
  if (N <= 0 || D <= 0 || D > 256) return SD_ERR_SHAPE;
  if (!x || !gate || !weight || !y) return SD_ERR_ARG;
  const __bf16 *xb = (const __bf16*)x, *gb = (const __bf16*)gate;
  __bf16* yb = (__bf16*)y;
  hipStream_t st = (hipStream_t)stream;
  if (!rms_vec(D, (uintptr_t)x | (uintptr_t)gate | (uintptr_t)y))
    SD_LAUNCH("k_rms_fwd", k_rms_fwd, dim3(cdiv(N, RMS_ROWS)), dim3(RMS_ROWS * 64), 0, st, N, D, eps, xb, gb,
              weight, yb, rstd);
  else if (D <= 64)
    SD_LAUNCH("k_rms_fwd", k_rmsv_fwd<8>, dim3(cdiv(N, NTHREADS / 8 * RMSV_U)), dim3(NTHREADS), 0, st, N, D, eps,
              xb, gb, weight, yb, rstd);
  else if (D <= 128)
    SD_LAUNCH("k_rms_fwd", k_rmsv_fwd<16>, dim3(cdiv(N, NTHREADS / 16 * RMSV_U)), dim3(NTHREADS), 0, st, N, D, eps,
              xb, gb, weight, yb, rstd);
  else
    SD_LAUNCH("k_rms_fwd", k_rmsv_fwd<32>, dim3(cdiv(N, NTHREADS / 32 * RMSV_U)), dim3(NTHREADS), 0, st, N, D, eps,
              xb, gb, weight, yb, rstd);
  return hipGetLastError() == hipSuccess ? SD_OK : SD_ERR_LAUNCH;
}

int sd_rmsnorm_gated_bwd(int N, int D, float eps, const void* x, const void* gate,
                         const float* weight, const void* dy, void* dx, void* dgate,
                         float* dweight, void* y, void* workspace, size_t workspace_bytes,
                         void* stream) {
  if (N <= 0 || D <= 0 || D > 256) return SD_ERR_SHAPE;
  if (!x || !gate || !weight || !dy || !dx || !dgate || !dweight || !workspace) return SD_ERR_ARG;
  if (workspace_bytes < sd_rmsnorm_gated_workspace_bytes(N, D)) return SD_ERR_WORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  const __bf16 *xb = (const __bf16*)x, *gb = (const __bf16*)gate, *db = (const __bf16*)dy;
  __bf16 *dxb = (__bf16*)dx, *dgb = (__bf16*)dgate, *yb = (__bf16*)y;
  float* part = (float*)workspace;
  int np = cdiv(N, RMS_PART);
  if (!rms_vec(D, (uintptr_t)x | (uintptr_t)gate | (uintptr_t)dy | (uintptr_t)dx | (uintptr_t)dgate | (uintptr_t)y)) {
    SD_LAUNCH("k_rms_bwd", k_rms_bwd, dim3(np), dim3(RMS_ROWS * 64), 0, st, N, D, eps, xb, gb, weight, db, dxb, dgb,
              yb, part);
  } else {
    const int rows = rmsv_rows(N, D);
    np = cdiv(N, rows);
    if (D <= 64)
      SD_LAUNCH("k_rms_bwd", k_rmsv_bwd<8>, dim3(np), dim3(NTHREADS), 0, st, N, D, eps, rows, xb, gb, weight, db,
                dxb, dgb, yb, part);
    else if (D <= 128)
      SD_LAUNCH("k_rms_bwd", k_rmsv_bwd<16>, dim3(np), dim3(NTHREADS), 0, st, N, D, eps, rows, xb, gb, weight, db,
                dxb, dgb, yb, part);
    else
      SD_LAUNCH("k_rms_bwd", k_rmsv_bwd<32>, dim3(np), dim3(NTHREADS), 0, st, N, D, eps, rows, xb, gb, weight, db,
                dxb, dgb, yb, part);
  }
  launch_sum_parts((const float*)workspace, np, D, dweight, st);
  return hipGetLastError() == hipSuccess ? SD_OK : SD_ERR_LAUNCH;
}

}  // extern "C"
