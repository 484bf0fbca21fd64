// Wide-width path of the SolveDelta recurrence: key widths 128 < r <= 256 and
// value widths up to 256 (gfx950).
//
// The reference runs its state pass for head widths up to 256
// (causallsso/ops/residual_frame/common_left_h.py:139-151).  The main kernels
// hold a 64-token chunk's 128-wide panels in LDS; at 256 they would not fit, so
// this path states the same chunked algebra (the generic pre-decay-read delta
// op restated in tests/chunk_model.py) with 32-token chunks, runtime padded
// widths KP, VP (multiples of 32, <= 256), u, k, q, h as packed bf16 rows with
// FP32 scalars per token, FP32 panels for what is computed, and a 16-bit
// matrix-core state pass (its panels and the chunk states in fp16 / bf16):
//
//   k_w_tokens  (chunk-parallel)  in-chunk log-decay prefix G, packed rows, L2
//               norms, gamma;
//   per op (predictor C: X = C^T, erase read before the token's decay, row
//   output; memory S: erase read after it, column output):
//     k_w_prep    decayed Gram L, (I+L)^-1, WY panels W, U (the memory's from
//                 z = sigmoid(write_raw) v, formed there), decayed keys, readout
//                 pair P (column output);
//     k_w_state   sequential chunk pass over one 32-column state tile;
//     k_w_out_c, k_w_out_s  chunk readouts (the predictor's forms d = k^ + C^T k^);
//   k_w_sources (per token)  dual sources e, chi;
// and backward, per op in reverse order:
//     k_w_bprep   dU = A^T (dW + pair^T dO), W' = -A^T K^, K' = -x~, injection;
//     k_w_state   reverse cotangent pass (lambda, dw);
//     k_w_grad    closed-form chunk gradients dk, dx, dq and the decay closure
//                 (the predictor's ends with the closures of u, k, h and gamma);
//   k_w_src_bwd (per token, between the ops)  source and q closures.
//
// Every decay factor is exp(a - b) with a <= b prefix sums inside one chunk (no
// reciprocal decays), formed per element; padding tokens and coordinates are
// zero and stay neutral.
#include <type_traits>

#include "sd_common.cuh"
#include "sd_internal.h"

namespace sd {
namespace wide {

constexpr int WBT = 32;    // chunk length
constexpr int WMAX = 256;  // widest padded width
constexpr int WT = 256;    // threads per workgroup

// Chunk-boundary state slots in a 2-byte type, as in the main kernels: the
// forward states X (C^T and S) in fp16, the reverse passes' cotangent states
// lambda in bf16.  The final states handed to the caller stay FP32.
using xs_t = xslot_t;
using ls_t = lslot_t;

// Workgroup ids are dealt round-robin over the 8 XCDs (each with its own L2).
// Maps a linear id over (inner, outer) = (L % inner, L / inner) so that, when the
// outer count is a multiple of 8, the inner indices of one outer index run on
// one XCD in consecutive order: the state pass's column tiles of a sequence
// share its L2 copy of the chunk panels, and the chunk gradients of neighbouring
// chunks share the state slot between them.
__device__ __forceinline__ void xcd_map(int L, int inner, int outer, int& in, int& out) {
  if (outer % 8 == 0) {
    const int x = L % 8, j = L / 8;
    in = j % inner;
    out = (j / inner) * 8 + x;
  } else {
    in = L % inner;
    out = L / inner;
  }
}

__device__ __forceinline__ const __bf16* wrow(const sd_view& v, int b, int t, int h) {
  return (const __bf16*)v.data + (long long)b * v.sb + (long long)t * v.st + (long long)h * v.sh;
}
__device__ __forceinline__ float wgamma(const sd_view& g, int b, int t, int h) {
  return ((const float*)g.data)[(long long)b * g.sb + (long long)t * g.st + (long long)h * g.sh];
}

// ---------------------------------------------------------------------------
// Token preparation: G prefix, packed rows, norms and gamma.
// ---------------------------------------------------------------------------
// Per-token scalars: the inverse norms 1/|u|, 1/|k|, 1/|q| (u^ = ru u and so on
// are formed from the packed bf16 rows where they are read: half the bytes of
// FP32 panels and the same values), gamma, the erase read's gamma (0 on fresh
// tokens), and 1/|k| again with 0 for a zero row, where it multiplies a
// cotangent of any scale.
struct Tok { float ru, rk, rq, gam, gx, rks, pad[2]; };

struct TokParams {
  sd_inputs in;
  int NT, Tp, KP;
  float *G;
  __bf16 *ub, *kb, *qb, *hb;  // packed raw rows [Tp][KP], zero past the widths and on invalid tokens (k, q)
  Tok* tok;
};

// Loads here are unconditional (indices clamped into the row, invalid values
// masked afterwards by a select): a load under a branch waits for every load
// issued before it, so guarded loads would run one round trip at a time.
__global__ __launch_bounds__(WT) void k_w_tokens(TokParams p) {
  const int ch = blockIdx.x, s = blockIdx.y;
  const int H = p.in.H, T = p.in.T, r = p.in.r, KP = p.KP;
  const int b = s / H, h = s % H, t0 = ch * WBT;
  const long long pb = (long long)s * p.Tp;
  // in-chunk inclusive log-decay prefix, one coordinate per thread: the chunk's
  // 32 values are loaded first, then summed
  const int c = threadIdx.x;
  // token flags (invalid: the log-decay reads 0; reset: the reset value): lane l
  // holds token t0 + l % 32's, read across lanes below (loaded by every lane)
  const int fl = tok_flag_row(p.in, b)[(long long)min(t0 + (int)(threadIdx.x & 31), T - 1) *
                                       tok_flag_st(p.in)];
  if (c < KP) {
    const float* g = (const float*)p.in.log_decay.data + (long long)b * p.in.log_decay.sb +
                     (long long)h * p.in.log_decay.sh + min(c, r - 1);
    float gv[WBT];
#pragma unroll
    for (int i = 0; i < WBT; ++i) gv[i] = g[(long long)min(t0 + i, T - 1) * p.in.log_decay.st];
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < WBT; ++i) {
      acc += (t0 + i < T && c < r) ? decay_eff(__builtin_amdgcn_readlane(fl, i), gv[i]) : 0.f;
      p.G[(pb + t0 + i) * KP + c] = acc;
    }
  }
  // per token: packed rows, norms and gamma, two tokens per wave at a time with
  // all their loads in flight together
  constexpr int NW = WT / 64, TU = 2;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  static_assert(WBT % (NW * TU) == 0, "tokens per wave");
  for (int i0 = w; i0 < WBT; i0 += NW * TU) {
    float uu[TU][4], kk[TU][4], qq[TU][4], hv[TU][4], gm[TU], ek[TU], om[TU];
#pragma unroll
    for (int u = 0; u < TU; ++u) {
      const int tc = min(t0 + i0 + u * NW, T - 1);
      const unsigned f = tok_flags(p.in, b, tc);
      gm[u] = wgamma(p.in.gamma, b, tc, h);
      ek[u] = erase_keep_f(f);
      om[u] = operand_keep(f);  // an invalid token's q, keys and gamma read 0
      const __bf16* ur = wrow(p.in.u, b, tc, h);
      const __bf16* kr = wrow(p.in.k, b, tc, h);
      const __bf16* qr = wrow(p.in.q, b, tc, h);
      const __bf16* hr = wrow(p.in.h, b, tc, h);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int cc = min(l + 64 * j, r - 1);
        uu[u][j] = bf2f(ur[cc]);
        kk[u][j] = bf2f(kr[cc]);
        qq[u][j] = bf2f(qr[cc]);
        hv[u][j] = bf2f(hr[cc]);
      }
    }
#pragma unroll
    for (int u = 0; u < TU; ++u) {
      const int t = t0 + i0 + u * NW;
      const bool tv = t < T;
      const float g1 = tv ? gm[u] * om[u] : 0.f;
      const float gx = tv ? g1 * ek[u] : 0.f;  // erase side: 0 on fresh tokens
      float su = 0.f, sk = 0.f, sq = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool ok = tv && l + 64 * j < r;
        uu[u][j] = ok ? uu[u][j] : 0.f;
        kk[u][j] = ok ? kk[u][j] * om[u] : 0.f;
        qq[u][j] = ok ? qq[u][j] * om[u] : 0.f;
        hv[u][j] = ok ? hv[u][j] : 0.f;
        su += uu[u][j] * uu[u][j];
        sk += kk[u][j] * kk[u][j];
        sq += qq[u][j] * qq[u][j];
      }
      const float ru = rsqrtf(wave_sum(su) + 1e-24f);
      sk = wave_sum(sk);
      const bool sk0 = sk == 0.f;
      const float rk = rsqrtf(sk + 1e-24f);
      const float rq = rsqrtf(wave_sum(sq) + 1e-24f);
      const long long row = (pb + t) * KP;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int cc = l + 64 * j;
        if (cc < KP) {  // (bf16 values and zeros: exact)
          p.ub[row + cc] = f2bf(uu[u][j]);
          p.kb[row + cc] = f2bf(kk[u][j]);
          p.qb[row + cc] = f2bf(qq[u][j]);
          p.hb[row + cc] = f2bf(hv[u][j]);
        }
      }
      if (l == 0) p.tok[pb + t] = {ru, rk, rq, g1, gx, sk0 ? 0.f : rk, {0.f, 0.f}};
    }
  }
}

// ---------------------------------------------------------------------------
// One op (state X [kw x vw]) of the chunked recurrence.
// ---------------------------------------------------------------------------
struct OpParams {
  int NT, Tp, kw, vw, colout;
  const float *k, *x, *q, *G;  // [Tp][kw] (k, x, q: column output)
  const __bf16 *ub, *hb;       // row output: k = u^, x = gx u^, v = gamma h
  const Tok* tok;
  sd_inputs in;                // column output: v = sigmoid(write_raw) v from the raw inputs
  float *A, *P;                    // [NT][32][32] (P: column output)
  _Float16 *Wneg, *Kt;             // state-pass panels: -W (w_off order), K^ transposed per chunk [NT][kw][32]
  float *U, *Qt, *Gam;             // Qt [Tp][kw] (column output); U [Tp][vw] (accumulator order); Gam [NT][kw]
};

// Decay factors of the matrix-core Grams and applies are factored per
// coordinate c as exp(Ga_i) * exp(-Gb_j), both prefixes inside the chunk.  That
// is exact up to rounding while the coordinate's decay over the chunk,
// -G_{31,c}, stays at most WILD (exp(WILD) is far inside FP32); "wild"
// coordinates beyond it are left out of the factored product and their terms
// added exactly.
// Accumulator order of a chunk's [32 tokens][C] FP32 panel (U, dU): the 16 x 16
// tile (token block tb, column block cb) is 64 lanes x 4 elements, lane (g, m)
// holding tokens 16 tb + 4 g .. + 3 of column 16 cb + m, as an MFMA writes it.
__device__ __forceinline__ unsigned acc_off(int tb, int cb, int lane, int C) {
  return (unsigned)(((tb * (C >> 4) + cb) * 64 + lane) * 4);
}

// Position of W's element (token t, state row) in its panel: the two token
// blocks' operands of a 16-row block side by side, 16 bytes per lane.
__device__ __forceinline__ unsigned w_off(int rb, int lane, int tb) {
  return (unsigned)(((rb * 64 + lane) * 2 + tb) * 4);
}

// A state slot [kw][vw] is kept in 32-column tiles, [vw / 32][kw][32]: a state
// workgroup writes whole lines of its own tile, and a 16-row operand fragment
// of 32 columns is 1 KiB contiguous.  Row-major slots held the state passes to
// the rate of their half-line stores (forward 187 us, in tiles 165).
constexpr int STILE = 32;  // state columns per workgroup
__device__ __forceinline__ unsigned slot_off(int row, int col, int kw) {
  return (unsigned)(((col / STILE) * kw + row) * STILE + col % STILE);
}

constexpr float WILD = 60.f;

// x * e^{g} for a factored decay operand, zero on a wild coordinate.  Both
// sides are evaluated (the operands are loaded unconditionally by the caller;
// a branch around them would serialise every operand behind its own memory
// wait), the exponent clamped so a wild coordinate's factor stays finite
// before the select drops it.
__device__ __forceinline__ float keep_exp(bool keep, float x, float g) {
  const float v = x * __expf(fminf(g, 80.f));
  return keep ? v : 0.f;
}

// v_mfma_f32_16x16x4f32: used with the sum index k = 4 g + e carried by MFMA e
// (e = 0..3) and lane group g = lane / 16, so an accumulator (lane (g, n)
// holding rows 4g..4g+3 of column n) is the B operand of a following product
// as it stands.
__device__ __forceinline__ f4 mfma4(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}


// The prep and backward-prep kernels: PW waves, wave w owning the 16-coordinate
// blocks w, w + 8 of the key axis.  Lane (g, m) holds coordinates 4 g .. 4 g + 3
// of tokens m and 16 + m: a 16-byte load per panel and token, and the operand
// layout of v_mfma_f32_16x16x4f32 with the sum index k = 4 g + e, so the decayed
// Grams run from registers, each operand element formed once.
constexpr int PW = 8;
constexpr int PT = PW * 64;
constexpr int PNB = WMAX / 16 / PW;  // 16-wide blocks per wave
constexpr int XTS = WMAX + 4;        // row stride (FP32) of a staged [32][kw] panel
constexpr int KHS = WMAX + 8;        // row stride (16-bit) of a staged [32][kw] panel
constexpr int AS = WBT + 4;          // row stride of the staged 32 x 32 matrices

struct Quad { float v[4]; };
__device__ __forceinline__ Quad ldq(const __bf16* p) {
  const bf16x4 h = *reinterpret_cast<const bf16x4*>(p);
  return {{bf2f(h[0]), bf2f(h[1]), bf2f(h[2]), bf2f(h[3])}};
}
__device__ __forceinline__ Quad scaled(const Quad& a, float f) {
  return {{a.v[0] * f, a.v[1] * f, a.v[2] * f, a.v[3] * f}};
}
__device__ __forceinline__ Quad ldq(const float* p) { return *reinterpret_cast<const Quad*>(p); }

// The three lower 16 x 16 blocks (0,0), (1,0), (1,1) of a 32 x 32 token Gram,
// summed over one 16-coordinate block from factored operands a (rows) and b
// (columns).
__device__ __forceinline__ void gram3(const Quad (&a)[2], const Quad (&b)[2], f4 (&acc)[3]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    acc[0] = mfma4(a[0].v[e], b[0].v[e], acc[0]);
    acc[1] = mfma4(a[1].v[e], b[0].v[e], acc[1]);
    acc[2] = mfma4(a[1].v[e], b[1].v[e], acc[2]);
  }
}

// Adds the exact terms of the block's wild coordinates (wild[e]: this lane
// group's coordinate 4 g + e is wild) to the lane's Gram entries.  left(i, c) /
// right(j, c) give a row's / column's {value, G} at coordinate c; strict keeps
// j < i, else j <= i.
template <class FL, class FR>
__device__ __forceinline__ void gram3_wild(const bool (&wild)[4], int c0, bool strict, FL left, FR right,
                                           f4 (&acc)[3]) {
  unsigned mask = 0;  // bit 4 g + e
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const unsigned long long b = __ballot(wild[e]);
#pragma unroll
    for (int gg = 0; gg < 4; ++gg) mask |= (unsigned)((b >> (gg * 16)) & 1) << (4 * gg + e);
  }
  while (mask) {
    const int c = c0 + __ffs(mask) - 1;
    mask &= mask - 1;
    // (opaque lane indices: hoisted out of this rare loop, its addresses would
    // stay in registers through the common path)
    int g = (threadIdx.x & 63) >> 4, m = threadIdx.x & 15;
    asm volatile("" : "+v"(g), "+v"(m));
    float2 lv[2][4], rv[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      rv[h] = right(h * 16 + m, c);
#pragma unroll
      for (int e = 0; e < 4; ++e) lv[h][e] = left(h * 16 + 4 * g + e, c);
    }
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int bi = q > 0, bj = q > 1, i = bi * 16 + 4 * g + e, j = bj * 16 + m;
        const float v = lv[bi][e].x * rv[bj].x * __expf(fminf(lv[bi][e].y - rv[bj].y, 0.f));
        acc[q][e] += (strict ? j < i : j <= i) ? v : 0.f;
      }
  }
}

// A wave's partial Gram blocks to LDS: [slot][3][64 lanes] x 4, and the sum of
// one block entry group over np slots from slot s0 on.
__device__ __forceinline__ void gram3_put(float* part, int slot, const f4 (&acc)[3]) {
  const int l = threadIdx.x & 63;
#pragma unroll
  for (int q = 0; q < 3; ++q) *reinterpret_cast<f4*>(part + ((slot * 3 + q) * 64 + l) * 4) = acc[q];
}
template <int NP>
__device__ __forceinline__ f4 gram3_sum(const float* part, int s0, int q, int l) {
  f4 a = zero4();
#pragma unroll
  for (int s = 0; s < NP; ++s) a += *reinterpret_cast<const f4*>(part + (((s0 + s) * 3 + q) * 64 + l) * 4);
  return a;
}

// (I + L)^-1 of a strictly lower 32 x 32 L in LDS (row stride AS), in place, by
// one wave: the two 16 x 16 diagonal blocks by forward substitution (one lane
// per column), then the off-diagonal block -D1 (L10 D0) on the matrix cores.
// Two 16-step chains side by side instead of one 32-step chain per column
// (32 lanes each walking a whole column took 10052 clocks of the kernel).
__device__ __forceinline__ void inverse32(float* L) {
  const int l = threadIdx.x & 63, g = l >> 4, m = l & 15;
  const int B0 = (g & 1) * 16;
  float col[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    float a = (i == m) ? 1.f : 0.f;
#pragma unroll
    for (int q = 0; q < i; ++q) a -= L[(B0 + i) * AS + B0 + q] * col[q];
    col[i] = (i < m) ? 0.f : a;
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  if (g < 2) {
#pragma unroll
    for (int i = 0; i < 16; ++i) L[(B0 + i) * AS + B0 + m] = col[i];
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  f4 t = zero4(), a = zero4();
#pragma unroll
  for (int e = 0; e < 4; ++e) t = mfma4(L[(16 + m) * AS + 4 * g + e], L[(4 * g + e) * AS + m], t);
#pragma unroll
  for (int e = 0; e < 4; ++e) a = mfma4(L[(16 + m) * AS + 16 + 4 * g + e], t[e], a);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int e = 0; e < 4; ++e) L[(16 + 4 * g + e) * AS + m] = -a[e];
}

// Chunk-transposed 16-bit panel dst[kw][32 tokens] from its staged rows
// src[32][KHS]: a thread's piece is 8 tokens of one coordinate (16 bytes), a
// wave's pieces contiguous.
template <class E>
__device__ __forceinline__ void store_transposed(E* dst, const E* src, int kw) {
  typedef E V8 __attribute__((ext_vector_type(8)));
#pragma unroll
  for (int q = 0; q < WMAX * 4 / PT; ++q) {
    const int pc = threadIdx.x + PT * q, c = pc >> 2, t8 = (pc & 3) * 8;
    if (c < kw) {
      V8 v;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = src[(t8 + e) * KHS + c];
      *reinterpret_cast<V8*>(dst + (long long)c * WBT + t8) = v;
    }
  }
}

// What bounds it: at r = V = 256 a chunk moves 133 KiB (C) / 265 KiB (S) through
// one or two workgroups per CU, so the phases between its loads and stores must
// be short: two workgroups fit a CU (79 KB of LDS, 128 VGPRs) and overlap.  76 us
// (C, 3.7 TB/s) and 132 us (S, 4.2 TB/s) at B4 T2048 H8 r = V = 256; 110 and 123
// when C read FP32 panels and S its z; one four-wave workgroup per CU with
// every operand panel staged in LDS (110-140 KB, each Gram element formed once per
// 16 x 16 block) took 226 us per op.
template <bool COL>
__global__ __launch_bounds__(PT, 4) void k_w_prep(OpParams p) {
  extern __shared__ __align__(16) float sm[];
  const int ch = blockIdx.x, s = blockIdx.y, kw = p.kw, vw = p.vw, nkb = kw / 16, nvb = vw / 16;
  float* xt = sm;                                               // x~ = x e^{Gx} [32][XTS]
  _Float16* kh = reinterpret_cast<_Float16*>(xt + WBT * XTS);   // K^ [32][KHS]
  float* part = reinterpret_cast<float*>(kh + WBT * KHS);       // partial Grams [8][3][64][4]
  float* Ls = part + PW * 3 * 256;                              // L, then A [32][AS]
  const long long tb = (long long)s * p.Tp + ch * WBT;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 4, m = l & 15;
  const long long cbase = (long long)s * p.NT + ch;
  // chunk-uniform bases, 32-bit lane offsets (64-bit lane addresses spill)
  const float* Gc = p.G + tb * kw;
  const float *kc = COL ? p.k + tb * kw : nullptr, *xc = COL ? p.x + tb * kw : nullptr,
              *qc = COL ? p.q + tb * kw : nullptr;
  const __bf16 *ubc = COL ? nullptr : p.ub + tb * kw, *hbc = COL ? nullptr : p.hb + tb * kw;
  const Tok* tokc = COL ? nullptr : p.tok + tb;
  // this lane's values for U = A v (the MFMA B operand: tokens kb * 16 + 4 g + e
  // of column block w + 8 j), loaded before any store of the kernel (a load
  // issued after a store waits for it: one counter retires both)
  __bf16 vr[PNB][2][4], wr[COL ? PNB : 1][2][4];
  [[maybe_unused]] const int b = s / (COL ? p.in.H : 1), hh = s - b * (COL ? p.in.H : 1);
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = kb * 16 + 4 * g + e;
      if constexpr (COL) {  // clamped, masked when used
        const int tc = min(ch * WBT + i, p.in.T - 1);
        const __bf16 *vp = wrow(p.in.v, b, tc, hh), *wp = wrow(p.in.write_raw, b, tc, hh);
#pragma unroll
        for (int j = 0; j < PNB; ++j) {
          const int cc = min(min(w + PW * j, nvb - 1) * 16 + m, p.in.V - 1);
          vr[j][kb][e] = vp[cc];
          wr[j][kb][e] = wp[cc];
        }
      } else {
#pragma unroll
        for (int j = 0; j < PNB; ++j) vr[j][kb][e] = hbc[(unsigned)(i * vw + min(w + PW * j, nvb - 1) * 16 + m)];
      }
    }
  // L_ij = sum_c x_ic k_jc e^{Gx_ic - G_jc} (j < i), and for the column output
  // P_ij = sum_c q_ic k_jc e^{G_ic - G_jc} (j <= i): the waves split the key
  // axis; with both Grams waves 0-3 form L's and waves 4-7 P's partials
  const bool second = COL && w >= PW / 2;
  constexpr int STEP = COL ? PW / 2 : PW;
  f4 acc[3] = {zero4(), zero4(), zero4()};
  [[maybe_unused]] float tru[2], tgx[2];
  if constexpr (!COL)
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      tru[t2] = tokc[t2 * 16 + m].ru;
      tgx[t2] = tokc[t2 * 16 + m].gx;
    }
#pragma unroll 1
  for (int kb = w % STEP; kb < nkb; kb += STEP) {
    const int c0 = kb * 16 + 4 * g;
    const float* lp = second ? qc : xc;
    const Quad gl = ldq(Gc + (unsigned)((WBT - 1) * kw + c0));
    Quad a[2], b[2], G[2], Gx[2];
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      const unsigned o = (t2 * 16 + m) * kw + c0;
      if constexpr (COL) {
        a[t2] = ldq(lp + o);
        b[t2] = ldq(kc + o);
      } else {
        b[t2] = scaled(ldq(ubc + o), tru[t2]);
        a[t2] = scaled(b[t2], tgx[t2]);
      }
      G[t2] = ldq(Gc + o);
      if constexpr (!COL) Gx[t2] = ldq(Gc + (t2 == 0 && m == 0 ? o : o - kw));  // prefix before the token
    }
    bool wild[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) wild[e] = -gl.v[e] > WILD;
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      f16x4 k4;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float gx = G[t2].v[e];
        if constexpr (!COL) gx = t2 == 0 && m == 0 ? 0.f : Gx[t2].v[e];
        a[t2].v[e] *= __expf(gx);
        k4[e] = (_Float16)(b[t2].v[e] * __expf(gl.v[e] - G[t2].v[e]));
        b[t2].v[e] = keep_exp(!wild[e], b[t2].v[e], -G[t2].v[e]);
      }
      const int i = t2 * 16 + m;
      if (second) {
        *reinterpret_cast<Quad*>(p.Qt + tb * kw + (unsigned)(i * kw + c0)) = a[t2];
      } else {
        *reinterpret_cast<Quad*>(xt + i * XTS + c0) = a[t2];
        *reinterpret_cast<f16x4*>(kh + i * KHS + c0) = k4;
      }
    }
    if (!second && m == 0) {
      Quad ge;
#pragma unroll
      for (int e = 0; e < 4; ++e) ge.v[e] = __expf(gl.v[e]);
      *reinterpret_cast<Quad*>(p.Gam + cbase * kw + c0) = ge;
    }
    gram3(a, b, acc);
    gram3_wild(wild, kb * 16, !second,
               [&](int i, int c) {
                 const float gx = COL ? Gc[i * kw + c] : i > 0 ? Gc[(i - 1) * kw + c] : 0.f;
                 if constexpr (COL) return make_float2(lp[i * kw + c], gx);
                 else return make_float2(tokc[i].gx * (bf2f(ubc[i * kw + c]) * tokc[i].ru), gx);
               },
               [&](int j, int c) {
                 if constexpr (COL) return make_float2(kc[j * kw + c], Gc[j * kw + c]);
                 else return make_float2(bf2f(ubc[j * kw + c]) * tokc[j].ru, Gc[j * kw + c]);
               }, acc);
  }
  gram3_put(part, w, acc);
  float vb[PNB][2][4];
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = kb * 16 + 4 * g + e;
      [[maybe_unused]] const float gm = COL ? 0.f : tokc[i].gam;
#pragma unroll
      for (int j = 0; j < PNB; ++j) {
        if constexpr (COL) {
          const bool ok = ch * WBT + i < p.in.T && (w + PW * j) * 16 + m < p.in.V;
          vb[j][kb][e] = ok ? bf2f(vr[j][kb][e]) / (1.f + __expf(-bf2f(wr[j][kb][e]))) : 0.f;
        } else {
          vb[j][kb][e] = gm * bf2f(vr[j][kb][e]);
        }
      }
    }
  __syncthreads();
  if (threadIdx.x < (COL ? 2 : 1) * 192) {
    const int half = threadIdx.x / 192, q = (threadIdx.x % 192) >> 6;
    const f4 v = gram3_sum<STEP>(part, half * STEP, q, l);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = (q > 0 ? 16 : 0) + 4 * g + e, j = (q > 1 ? 16 : 0) + m;
      if (half == 0) Ls[i * AS + j] = j < i ? v[e] : 0.f;
      else p.P[cbase * WBT * WBT + i * WBT + j] = j <= i ? v[e] : 0.f;
    }
  } else if (threadIdx.x >= 448) {  // the zero upper blocks
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      Ls[(4 * g + e) * AS + 16 + m] = 0.f;
      if constexpr (COL) p.P[cbase * WBT * WBT + (4 * g + e) * WBT + 16 + m] = 0.f;
    }
  }
  __syncthreads();
  if (w == 0) inverse32(Ls);  // A = (I + L)^-1
  __syncthreads();
  if (threadIdx.x < WBT * WBT / 4) {
    const int i = threadIdx.x >> 3, j = (threadIdx.x & 7) * 4;
    *reinterpret_cast<Quad*>(p.A + cbase * WBT * WBT + i * WBT + j) = *reinterpret_cast<const Quad*>(Ls + i * AS + j);
  }
  // W = A x~ and U = A v on FP32 matrix cores over A's lower blocks.  W is
  // formed transposed (a lane holds four neighbouring columns of a token, the
  // state pass's operand order), -W fp16; U in accumulator order.
#pragma unroll
  for (int j = 0; j < PNB; ++j) {
    const int nb = w + PW * j;
    f4 aw[2] = {zero4(), zero4()}, au[2] = {zero4(), zero4()};
    const int nk = min(nb, nkb - 1);
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = kb * 16 + 4 * g + e;
        const float xv = xt[k * XTS + nk * 16 + m];
#pragma unroll
        for (int t2 = kb; t2 < 2; ++t2) {
          const float av = Ls[(t2 * 16 + m) * AS + k];
          aw[t2] = mfma4(xv, av, aw[t2]);
          au[t2] = mfma4(av, vb[j][kb][e], au[t2]);
        }
      }
    if (nb < nkb) {
      f16x8 h;
#pragma unroll
      for (int e = 0; e < 8; ++e) h[e] = (_Float16)(-aw[e >> 2][e & 3]);
      *reinterpret_cast<f16x8*>(p.Wneg + tb * kw + w_off(nb, l, 0)) = h;
    }
    if (nb < nvb)
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) *reinterpret_cast<f4*>(p.U + tb * vw + acc_off(t2, nb, l, vw)) = au[t2];
  }
  store_transposed(p.Kt + cbase * kw * WBT, kh, kw);
}

constexpr size_t prep_smem() {
  return (size_t)(WBT * XTS + PW * 3 * 256 + WBT * AS) * sizeof(float) + (size_t)WBT * KHS * 2;
}

// ---------------------------------------------------------------------------
// Sequential chunk pass over a 32-column tile of X [kw x vw]:
//   slot[ch] = X;  w = U + Wneg X;  X = Gamma X + K^T w (+ At^T Ib)
// forward (chunks ascending; slot NT = final state) or reverse (descending).
// ---------------------------------------------------------------------------
struct WStateParams {
  int NT, Tp, kw, vw, rows, cols, rev;
  const void* Wneg;  // -W per chunk in w_off order (fp16 forward, bf16 reverse)
  const void* Kt;    // K^T per chunk [NT][kw][32] (fp16 forward, bf16 reverse)
  const __bf16* At;  // injection A^T per chunk [NT][kw][32] (reverse)
  const float *U, *Gam;  // U [Tp][vw] (accumulator order); Gam [NT][kw]
  const __bf16* Ib;      // [Tp][vw]
  void* slots;  // xs_t (forward) or ls_t (reverse)
  float* wout;
  const float* init; int init_t;
  float* fin; int fin_t;
};

// Matrix-core form on 16-bit MFMAs: a workgroup of 8 waves owns a 32-column
// tile of the state, wave w holding the 16-row blocks w and w + 8 of both
// 16-column halves in FP32 accumulators.  Per chunk step:
//   w = U + Wneg X0: an accumulator (lane (g, m): rows 4 g .. + 3 of column m)
//   is the B operand of v_mfma_f32_16x16x16 as it stands, so each wave
//   multiplies its own rows, split into high and low 16-bit halves, into a
//   partial w of all 32 tokens; the partials meet in LDS, where every thread
//   sums two elements over the eight waves, adds U and stores w, and w again
//   split and transposed ([column][token]) as the B operand of
//   X = Gamma X + K^T w (+ At^T Ib, reverse), which every wave forms for its
//   own rows.
// The state itself never passes through LDS (the form that staged it there for
// four waves to read moved 170 KB of LDS and 64 KB of Wneg per step against 90
// and 16): forward passes 159 us, reverse 190 at B4 T2048 H8 r = V = 256 (196 and
// 227 before), 59 us forward at 12 sequences of 1333 tokens, r = 192 (80 before).
// What is left is the slot store: a build without it runs the forward pass in 94 us.
// The panels Wneg, K^T and At are stored 16-bit by the prep kernels in the
// order the MFMA operands read them, so each lane's fragment is one 16-byte
// load; they, U, Gamma and Ib are fetched SPF - 1 chunks ahead into a ring of
// registers (Ib as two bf16 elements per thread, staged through LDS).
// Forward: panels fp16 (W and K are bounded by construction), X
// and w split into fp16 halves (~22 bits).  Reverse: bf16 throughout (its
// exponent range keeps any scale of the cotangent), lambda and dw split
// into bf16 halves (Ib, a bf16 input, enters as it is).  Two barriers per step:
// the partials are read between them and written again only before the next
// step's first; the split w is written between them and read before that.
constexpr int SW = 8;                // state-pass waves: two per SIMD
constexpr int ST = SW * 64;
constexpr int SRB = WMAX / 16 / SW;  // state-pass row blocks per wave
constexpr int NSUB = STILE / 16;
constexpr int SPF = 3;               // prefetch ring depth (chunks)
constexpr int WLD = WBT + 8;         // row stride (16-bit) of the staged w
constexpr int NTILE = WBT / 16 * NSUB;  // 16 x 16 tiles of w: tile = token block * NSUB + half
constexpr size_t state_smem() {
  return (size_t)SW * NTILE * 256 * 4 + (size_t)3 * STILE * WLD * 2;
}

template <bool REV> struct WStateT;
template <> struct WStateT<false> {
  using E = _Float16;
  using V8 = f16x8;
  using V4 = f16x4;
  static __device__ __forceinline__ f4 mma(V8 a, V8 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f4 mma16(V4 a, V4 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
  }
};
template <> struct WStateT<true> {
  using E = __bf16;
  using V8 = bf16x8;
  using V4 = bf16x4;
  static __device__ __forceinline__ f4 mma(V8 a, V8 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f4 mma16(V4 a, V4 b, f4 c) {
    typedef short s4 __attribute__((ext_vector_type(4)));
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s4, a), __builtin_bit_cast(s4, b), c,
                                                     0, 0, 0);
  }
};

template <bool REV>
struct WFrags {
  using V8 = typename WStateT<REV>::V8;
  V8 W[SRB];                      // Wneg's two token blocks against this wave's row blocks
  V8 K[SRB];                      // K^T rows of this wave's row blocks, the chunk's 32 tokens
  bf16x8 A[REV ? SRB : 1];        // At rows (reverse)
  unsigned ib;                    // reverse: this thread's two elements of the Ib tile
  float2 U;                       // this thread's two elements of the U tile
  float4 G[SRB];                  // Gamma of this wave's rows 16 rb + 4 g .. + 3
};

// Chunk-uniform bases with 32-bit lane offsets throughout: 64-bit per-lane
// addresses for a chunk's fragment loads would not fit in registers beside the
// prefetch ring.  Every load is unconditional (indices clamped into the
// panel): a memory operation under a branch gives the two paths different counts
// of operations in flight, and the compiler then waits for all of them (the
// ring's prefetches included) wherever the paths meet.
template <bool REV>
__device__ __forceinline__ void wstate_load(const WStateParams& p, int s, int ch, int c0,
                                            WFrags<REV>& f) {
  using E = typename WStateT<REV>::E;
  using V8 = typename WStateT<REV>::V8;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 4, m = l & 15, kq = g * 8;
  const int kw = p.kw, vw = p.vw, nrb = kw / 16;
  const long long tb = (long long)s * p.Tp + (long long)ch * WBT;
  const long long cb = ((long long)s * p.NT + ch) * kw;  // chunk base of [kw][32] and [kw] panels
  const E* Wc = static_cast<const E*>(p.Wneg) + tb * kw;
  {  // thread t: elements 2 t, 2 t + 1 of the tiles in accumulator order
    const int tile = threadIdx.x >> 7;
    f.U = *reinterpret_cast<const float2*>(
        p.U + tb * vw + acc_off(tile / NSUB, (c0 >> 4) + tile % NSUB, (threadIdx.x & 127) >> 1, vw) +
        (threadIdx.x & 1) * 2);
  }
  const E* Kc = static_cast<const E*>(p.Kt) + cb * WBT;
  const float* Gc = p.Gam + cb;
#pragma unroll
  for (int q = 0; q < SRB; ++q) {
    const int rb = min(w + SW * q, nrb - 1);
    const unsigned ko = (unsigned)((rb * 16 + m) * WBT + kq);
    f.W[q] = *reinterpret_cast<const V8*>(Wc + w_off(rb, l, 0));
    f.K[q] = *reinterpret_cast<const V8*>(Kc + ko);
    f.G[q] = *reinterpret_cast<const float4*>(Gc + (unsigned)(rb * 16 + 4 * g));
    if constexpr (REV) f.A[q] = *reinterpret_cast<const bf16x8*>(p.At + cb * WBT + ko);
  }
  if constexpr (REV) {
    static_assert(WBT * STILE == 2 * ST, "two Ib elements per thread");
    const int tok = threadIdx.x / (STILE / 2), col = (threadIdx.x % (STILE / 2)) * 2;
    f.ib = *reinterpret_cast<const unsigned*>(p.Ib + tb * vw + c0 + (unsigned)(tok * vw + col));
  }
}

// An accumulator fragment in 16 bits (lane (g, m): rows 4 g .. + 3 of column m)
// turned into four neighbouring columns of one row: a 4 x 4 transpose within
// each quad of lanes.  Lane m ends with row 4 g + quad_row(m), columns m & 12 .. + 3.
__device__ __forceinline__ int quad_row(int m) { return ((m & 1) << 1) | ((m >> 1) & 1); }
template <class V4>
__device__ __forceinline__ uint2 quad_transpose(V4 v) {
  const uint2 in = __builtin_bit_cast(uint2, v);  // rows 0, 1 and rows 2, 3 of this lane's column
  const bool odd = threadIdx.x & 1, up = threadIdx.x & 2;
  const unsigned got = __builtin_amdgcn_update_dpp(0, odd ? in.x : in.y, 0xB1, 0xF, 0xF, false);
  const unsigned own = odd ? in.y : in.x;
  const unsigned lo = odd ? got : own, hi = odd ? own : got;  // rows (0,1) or (2,3) of two columns
  const unsigned ra = (lo & 0xffffu) | (hi << 16), rb = (lo >> 16) | (hi & 0xffff0000u);
  const unsigned got2 = __builtin_amdgcn_update_dpp(0, up ? ra : rb, 0x4E, 0xF, 0xF, false);
  return up ? make_uint2(got2, rb) : make_uint2(ra, got2);
}

// FULL: kw = WMAX, every wave has all of its row blocks (a memory operation
// under a branch would make the compiler wait for more than it needs).
template <bool REV, bool FULL>
__device__ __forceinline__ void wstate_step(const WStateParams& p, int s, int ch, int c0,
                                            const WFrags<REV>& f, f4 (&X)[SRB][NSUB], unsigned char* sm) {
  using T = WStateT<REV>;
  using E = typename T::E;
  using V8 = typename T::V8;
  using V4 = typename T::V4;
  using S = typename std::conditional<REV, ls_t, xs_t>::type;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 4, m = l & 15, kq = g * 8;
  const int kw = p.kw, vw = p.vw, nrb = kw / 16;
  const long long tb = (long long)s * p.Tp + (long long)ch * WBT;
  float* part = reinterpret_cast<float*>(sm);  // partial w [wave][tile][lane][4]
  E* wh = reinterpret_cast<E*>(part + SW * NTILE * 256);  // w [32 columns][WLD], high and low halves
  E* wl = wh + STILE * WLD;
  E* ih = wl + STILE * WLD;          // reverse: the injection's Ib tile [32 columns][WLD]
  static_assert(std::is_same<S, E>::value, "the slot holds the high half");
  // this wave's partial w and its rows of slot[ch]
  f4 pw[NTILE];
#pragma unroll
  for (int t = 0; t < NTILE; ++t) pw[t] = zero4();
  S* slot = static_cast<S*>(p.slots) + ((long long)s * (p.NT + 1) + ch) * kw * vw + c0 * kw;
#pragma unroll
  for (int q = 0; q < SRB; ++q) {
    const int rb = w + SW * q;
    if (!FULL && rb >= nrb) continue;
    const V4 w0 = __builtin_shufflevector(f.W[q], f.W[q], 0, 1, 2, 3);
    const V4 w1 = __builtin_shufflevector(f.W[q], f.W[q], 4, 5, 6, 7);
#pragma unroll
    for (int h = 0; h < NSUB; ++h) {
      V4 xh, xl;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const E a = (E)X[q][h][e];
        xh[e] = a;
        xl[e] = (E)(X[q][h][e] - (float)a);
      }
      pw[h] = T::mma16(w0, xl, pw[h]);
      pw[NSUB + h] = T::mma16(w1, xl, pw[NSUB + h]);
      pw[h] = T::mma16(w0, xh, pw[h]);
      pw[NSUB + h] = T::mma16(w1, xh, pw[NSUB + h]);
      *reinterpret_cast<uint2*>(slot + (unsigned)((rb * 16 + 4 * g + quad_row(m)) * STILE + h * 16 + (m & 12))) =
          quad_transpose(xh);
    }
  }
#pragma unroll
  for (int t = 0; t < NTILE; ++t) *reinterpret_cast<f4*>(part + ((w * NTILE + t) * 64 + l) * 4) = pw[t];
  if constexpr (REV) {  // the Ib tile (exact in bf16) staged transposed ([column][token])
    const int tok = threadIdx.x / (STILE / 2), col = (threadIdx.x % (STILE / 2)) * 2;
    ih[col * WLD + tok] = __builtin_bit_cast(E, (unsigned short)f.ib);
    ih[(col + 1) * WLD + tok] = __builtin_bit_cast(E, (unsigned short)(f.ib >> 16));
  }
  __syncthreads();
  {  // w: two elements (neighbouring tokens of one column) per thread
    static_assert(NTILE * 256 == 2 * ST, "two w elements per thread");
    float2 v = f.U;
#pragma unroll
    for (int k = 0; k < SW; ++k) {
      const float2 a = *reinterpret_cast<const float2*>(part + k * NTILE * 256 + threadIdx.x * 2);
      v.x += a.x;
      v.y += a.y;
    }
    const int tile = threadIdx.x >> 7, wl_ = (threadIdx.x & 127) >> 1;
    const int col = (tile % NSUB) * 16 + (wl_ & 15);
    const int tok = (tile / NSUB) * 16 + (wl_ >> 4) * 4 + (threadIdx.x & 1) * 2;
    typedef E E2 __attribute__((ext_vector_type(2)));
    E2 hi, lo;
    hi[0] = (E)v.x;
    hi[1] = (E)v.y;
    lo[0] = (E)(v.x - (float)hi[0]);
    lo[1] = (E)(v.y - (float)hi[1]);
    *reinterpret_cast<E2*>(wh + col * WLD + tok) = hi;
    *reinterpret_cast<E2*>(wl + col * WLD + tok) = lo;
    float* wo = p.wout + tb * vw + c0;
    wo[(unsigned)(tok * vw + col)] = v.x;
    wo[(unsigned)((tok + 1) * vw + col)] = v.y;
  }
  // X = Gamma X (+ At^T Ib): independent of w
#pragma unroll
  for (int q = 0; q < SRB; ++q) {
    const int rb = w + SW * q;
    if (!FULL && rb >= nrb) continue;
    const float gv[4] = {f.G[q].x, f.G[q].y, f.G[q].z, f.G[q].w};
#pragma unroll
    for (int h = 0; h < NSUB; ++h) {
#pragma unroll
      for (int e = 0; e < 4; ++e) X[q][h][e] *= gv[e];
      if constexpr (REV) {
        const bf16x8 bh = *reinterpret_cast<const bf16x8*>(ih + (h * 16 + m) * WLD + kq);
        X[q][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.A[q], bh, X[q][h], 0, 0, 0);
      }
    }
  }
  __syncthreads();
  // X += K^T w
#pragma unroll
  for (int h = 0; h < NSUB; ++h) {
    const V8 whv = *reinterpret_cast<const V8*>(wh + (h * 16 + m) * WLD + kq);
    const V8 wlv = *reinterpret_cast<const V8*>(wl + (h * 16 + m) * WLD + kq);
#pragma unroll
    for (int q = 0; q < SRB; ++q) {
      const int rb = w + SW * q;
      if (!FULL && rb >= nrb) continue;
      X[q][h] = T::mma(f.K[q], wlv, X[q][h]);
      X[q][h] = T::mma(f.K[q], whv, X[q][h]);
    }
  }
}

template <bool REV, bool FULL>
__global__ __launch_bounds__(ST) void k_w_state(WStateParams p) {
  extern __shared__ __align__(16) unsigned char wsm[];
  int tile, s;
  xcd_map(blockIdx.x, p.vw / STILE, gridDim.x / (p.vw / STILE), tile, s);
  const int kw = p.kw, c0 = tile * STILE, NT = p.NT;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 4, m = l & 15;
  const int nrb = kw / 16;
  f4 X[SRB][NSUB];
#pragma unroll
  for (int q = 0; q < SRB; ++q) {
    const int rb = w + SW * q;
#pragma unroll
    for (int h = 0; h < NSUB; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = rb * 16 + 4 * g + e, col = c0 + h * 16 + m;
        float v = 0.f;
        if (rb < nrb && p.init && row < p.rows && col < p.cols)
          v = p.init_t ? p.init[((long long)s * p.cols + col) * p.rows + row]
                       : p.init[((long long)s * p.rows + row) * p.cols + col];
        X[q][h][e] = v;
      }
  }
  auto chunk_of = [&](int it) { return REV ? NT - 1 - it : it; };
  auto clampc = [&](int it) { return chunk_of(it < NT ? it : NT - 1); };
  // Straight-line ring (no breaks; clamped, unconditional prefetches) so the
  // compiler's wait counts only cover the buffer being consumed; the last
  // SPF - 1 or fewer chunks run after the loop.
  WFrags<REV> f[SPF];
#pragma unroll
  for (int j = 0; j < SPF - 1; ++j) wstate_load<REV>(p, s, clampc(j), c0, f[j]);
  int it = 0;
  for (; it + SPF - 1 < NT; it += SPF) {
#pragma unroll
    for (int j = 0; j < SPF; ++j) {
      wstate_load<REV>(p, s, clampc(it + j + SPF - 1), c0, f[(j + SPF - 1) % SPF]);
      __builtin_amdgcn_sched_barrier(0);
      wstate_step<REV, FULL>(p, s, chunk_of(it + j), c0, f[j], X, wsm);
    }
  }
#pragma unroll
  for (int j = 0; j < SPF - 1; ++j)
    if (it + j < NT) wstate_step<REV, FULL>(p, s, chunk_of(it + j), c0, f[j], X, wsm);
  // final state (forward: also slot NT for the backward)
  using S = typename std::conditional<REV, ls_t, xs_t>::type;
#pragma unroll
  for (int q = 0; q < SRB; ++q) {
    const int rb = w + SW * q;
    if (!FULL && rb >= nrb) continue;
#pragma unroll
    for (int h = 0; h < NSUB; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = rb * 16 + 4 * g + e, col = c0 + h * 16 + m;
        if (!REV)
          static_cast<S*>(p.slots)[((long long)s * (p.NT + 1) + p.NT) * kw * p.vw + slot_off(row, col, kw)] =
              (S)X[q][h][e];
        if (p.fin && row < p.rows && col < p.cols) {
          if (p.fin_t) p.fin[((long long)s * p.cols + col) * p.rows + row] = X[q][h][e];
          else p.fin[((long long)s * p.rows + row) * p.cols + col] = X[q][h][e];
        }
      }
  }
}

// Four elements of an output row at column c of r (a padded column is dropped).
__device__ __forceinline__ void store_row4(__bf16* row, int c, int r, int vec, bf16x4 h) {
  if (vec) {
    if (c < r) *reinterpret_cast<bf16x4*>(row + c) = h;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (c + e < r) row[c + e] = h[e];
  }
}
__device__ __forceinline__ void store_row4(__bf16* row, int c, int r, int vec, const Quad& q) {
  bf16x4 h;
#pragma unroll
  for (int e = 0; e < 4; ++e) h[e] = f2bf(q.v[e]);
  store_row4(row, c, r, vec, h);
}
__device__ __forceinline__ void store_row4(float* row, int c, int r, int vec, const Quad& q) {
  if (vec) {
    if (c < r) *reinterpret_cast<Quad*>(row + c) = q;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (c + e < r) row[c + e] = q.v[e];
  }
}

// ---------------------------------------------------------------------------
// Chunk readouts, transposed like the other chunk kernels' products (a lane
// holds four neighbouring coordinates of one token), two workgroups per CU.
// What bounds them: the state slot (128 KiB of a chunk's 208 (S) / 256 (C) KiB
// at r = V = 256).
// ---------------------------------------------------------------------------
struct OutParams {
  int NT, Tp, kw, vw;
  const xs_t* slots;
  const float *w, *G;           // w [Tp][vw]
  const float *Qt, *P;          // column output
  int H, T, V, vec;
  __bf16* out;
  const __bf16 *ub, *kb;        // row output: q = base = k^, k = u^
  const Tok* tok;
  float *o, *d;                 // o: null where no backward follows
};

constexpr int GS16 = 20;  // row stride (FP32) of a wave's staged [32 tokens][16 coordinates] panel

// Four values split into fp16 halves.
__device__ __forceinline__ void split4_h(_Float16* hi, _Float16* lo, const Quad& q) {
  f16x4 h, o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    h[e] = (_Float16)q.v[e];
    o[e] = (_Float16)(q.v[e] - (float)h[e]);
  }
  *reinterpret_cast<f16x4*>(hi) = h;
  *reinterpret_cast<f16x4*>(lo) = o;
}
__device__ __forceinline__ f4 mma_h(f16x8 a, f16x8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Column output o = Q~ X0 + P w.  Q~ X0 on fp16 matrix cores (Q~ split into high
// and low halves in LDS, X0 exact in its slot): the contraction runs along the
// slot's rows, so 32-row blocks pass through LDS (double buffered, one barrier
// each) and are read down their columns.  P w in FP32.  Wave w owns the
// 16-column blocks w, w + 8.  91 us (4.8 TB/s) at B4 T2048 H8
// r = V = 256, where four waves with one workgroup per CU took 155 us.
__global__ __launch_bounds__(PT, 4) void k_w_out_s(OutParams p) {
  extern __shared__ __align__(16) float sm[];
  const int ch = blockIdx.x, s = blockIdx.y, kw = p.kw, vw = p.vw, nvb = vw / 16;
  const long long tb = (long long)s * p.Tp + ch * WBT;
  const xs_t* X0 = p.slots + ((long long)s * (p.NT + 1) + ch) * kw * vw;
  const float *Qc = p.Qt + tb * kw, *wc = p.w + tb * vw;
  constexpr int RP = WBT * KHS;
  _Float16* Qh = reinterpret_cast<_Float16*>(sm);  // Q~ high / low [32][KHS]
  _Float16 *Ql = Qh + RP, *Xt = Ql + RP;           // X0 row blocks [2][32][KHS]
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 4, m = l & 15, kq = g * 8;
  constexpr int XQ = WBT * WMAX / 8 / PT, QQ = WBT * WMAX / 4 / PT;
  f16x8 xb[XQ];
  auto fetch = [&](int rb) {
#pragma unroll
    for (int q = 0; q < XQ; ++q) {
      // piece idx: column tile idx / 128, row (idx / 4) % 32, columns 8 (idx % 4) .. + 7
      const int idx = min((int)(threadIdx.x + PT * q), WBT * vw / 8 - 1);
      xb[q] = *reinterpret_cast<const f16x8*>(X0 + slot_off(rb + (idx >> 2) % 32, (idx >> 7) * STILE + (idx & 3) * 8, kw));
    }
  };
  auto put = [&](int f) {
#pragma unroll
    for (int q = 0; q < XQ; ++q) {
      const int idx = min((int)(threadIdx.x + PT * q), WBT * vw / 8 - 1);
      *reinterpret_cast<f16x8*>(Xt + f * RP + (idx >> 2) % 32 * KHS + (idx >> 7) * STILE + (idx & 3) * 8) = xb[q];
    }
  };
  fetch(0);
  {
    Quad qv[QQ];
#pragma unroll
    for (int q = 0; q < QQ; ++q) qv[q] = ldq(Qc + (unsigned)(min((int)(threadIdx.x + PT * q), WBT * kw / 4 - 1) * 4));
#pragma unroll
    for (int q = 0; q < QQ; ++q) {
      const int idx = min((int)(threadIdx.x + PT * q), WBT * kw / 4 - 1) * 4, o = idx / kw * KHS + idx % kw;
      split4_h(Qh + o, Ql + o, qv[q]);
    }
  }
  // P's rows and this lane's w values for P w, whose loads overlap the products
  float wv[PNB][2][4];
  int nb[PNB];
#pragma unroll
  for (int q = 0; q < PNB; ++q) {
    nb[q] = min(w + PW * q, nvb - 1) * 16;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 4; ++e) wv[q][kb][e] = wc[(unsigned)((kb * 16 + 4 * g + e) * vw + nb[q] + m)];
  }
  Quad pp[2][2];
#pragma unroll
  for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
    for (int kb = 0; kb <= t2; ++kb)
      pp[t2][kb] = ldq(p.P + ((long long)s * p.NT + ch) * WBT * WBT + (t2 * 16 + m) * WBT + kb * 16 + 4 * g);
  put(0);
  __syncthreads();
  f4 acc[PNB][2];
#pragma unroll
  for (int q = 0; q < PNB; ++q) acc[q][0] = acc[q][1] = zero4();
  for (int rb = 0; rb < kw; rb += 32) {
    const int f = (rb >> 5) & 1;
    if (rb + 32 < kw) fetch(rb + 32);
    f16x8 qh[2], ql[2];
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      qh[t2] = *reinterpret_cast<const f16x8*>(Qh + (t2 * 16 + m) * KHS + rb + kq);
      ql[t2] = *reinterpret_cast<const f16x8*>(Ql + (t2 * 16 + m) * KHS + rb + kq);
    }
#pragma unroll
    for (int q = 0; q < PNB; ++q) {
      f16x8 xc;
#pragma unroll
      for (int j = 0; j < 8; ++j) xc[j] = Xt[f * RP + (kq + j) * KHS + nb[q] + m];
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        acc[q][t2] = mma_h(xc, ql[t2], acc[q][t2]);
        acc[q][t2] = mma_h(xc, qh[t2], acc[q][t2]);
      }
    }
    if (rb + 32 < kw) put(f ^ 1);
    __syncthreads();
  }
  const int b = s / p.H, h = s % p.H;
#pragma unroll
  for (int q = 0; q < PNB; ++q)
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
#pragma unroll
      for (int kb = 0; kb <= t2; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[q][t2] = mfma4(wv[q][kb][e], pp[t2][kb].v[e], acc[q][t2]);
      const int t = ch * WBT + t2 * 16 + m;
      if (t < p.T && w + PW * q < nvb)
        store_row4(p.out + (((long long)b * p.T + t) * p.H + h) * p.V, nb[q] + 4 * g, p.V, p.vec,
                   Quad{{acc[q][t2][0], acc[q][t2][1], acc[q][t2][2], acc[q][t2][3]}});
    }
}

// Row output: M = q w^T (j <= i), then
//   o_ir = e^{G_ir} ((q X0^T)_ir + (M k~)_ir),  k~_jr = k_jr e^{-G_jr},  d = q + o
// with the decay factored per state row r (wild rows: exact per-term sum).  o is
// kept beside d for the backward's o dO: taken back from the rounded sum it would
// hold only the bits above k^'s last.  M as the prep's Grams, in FP32 over the
// waves; q X0^T on fp16 matrix cores (q, unit rows, split into high and low halves
// in LDS; X0 exact in its slot).  Wave w owns the 16-row blocks w, w + 8.  134 us
// (288 KiB a chunk, 4.5 TB/s) at B4 T2048 H8 r = V = 256, 117 without o; four waves
// with 4-byte panel accesses took 208 us.
__global__ __launch_bounds__(PT, 4) void k_w_out_c(OutParams p) {
  extern __shared__ __align__(16) float sm[];
  const int ch = blockIdx.x, s = blockIdx.y, kw = p.kw, nkb = kw / 16;
  const long long tb = (long long)s * p.Tp + ch * WBT;
  const xs_t* X0 = p.slots + ((long long)s * (p.NT + 1) + ch) * kw * kw;
  const __bf16 *ubc = p.ub + tb * kw, *kbc = p.kb + tb * kw;
  const float *Gc = p.G + tb * kw, *wc = p.w + tb * kw;
  const Tok* tokc = p.tok + tb;
  _Float16* Qh = reinterpret_cast<_Float16*>(sm);  // q high / low [32][KHS]
  _Float16* Ql = Qh + WBT * KHS;
  float* Ml = reinterpret_cast<float*>(Ql + WBT * KHS);  // M [32][AS]
  float* part = Ml + WBT * AS;  // partial Ms; then per wave k~ [32][GS16]
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 4, m = l & 15, kq = g * 8;
  float tru[2], trk[2];
#pragma unroll
  for (int t2 = 0; t2 < 2; ++t2) {
    tru[t2] = tokc[t2 * 16 + m].ru;
    trk[t2] = tokc[t2 * 16 + m].rk;
  }
  Quad kn[PNB][2], u[PNB][2], G[PNB][2], gl[PNB];
  int c0[PNB];
  f4 am[3] = {zero4(), zero4(), zero4()};
#pragma unroll
  for (int q = 0; q < PNB; ++q) {
    c0[q] = min(w + PW * q, nkb - 1) * 16 + 4 * g;
    Quad wv[2];
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      const unsigned o = (t2 * 16 + m) * kw + c0[q];
      kn[q][t2] = scaled(ldq(kbc + o), trk[t2]);
      wv[t2] = ldq(wc + o);
      u[q][t2] = scaled(ldq(ubc + o), tru[t2]);
      G[q][t2] = ldq(Gc + o);
    }
    gl[q] = ldq(Gc + (unsigned)((WBT - 1) * kw + c0[q]));
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      const int o = (t2 * 16 + m) * KHS + c0[q];
      split4_h(Qh + o, Ql + o, kn[q][t2]);
    }
    if (w + PW * q < nkb) gram3(kn[q], wv, am);
  }
  gram3_put(part, w, am);
  __syncthreads();
  if (threadIdx.x < 192) {
    const int q = threadIdx.x >> 6;
    const f4 v = gram3_sum<PW>(part, 0, q, l);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = (q > 0 ? 16 : 0) + 4 * g + e, j = (q > 1 ? 16 : 0) + m;
      Ml[i * AS + j] = j <= i ? v[e] : 0.f;
    }
  }
  f4 acc[PNB][2];
#pragma unroll
  for (int q = 0; q < PNB; ++q) acc[q][0] = acc[q][1] = zero4();
  unsigned ro[PNB];
#pragma unroll
  for (int q = 0; q < PNB; ++q) ro[q] = slot_off(min(w + PW * q, nkb - 1) * 16 + m, kq, kw);
#pragma unroll 4
  for (int cb = 0; cb < kw; cb += 32) {
    f16x8 x[PNB];
#pragma unroll
    for (int q = 0; q < PNB; ++q) x[q] = *reinterpret_cast<const f16x8*>(X0 + cb * kw + ro[q]);
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      const f16x8 qh = *reinterpret_cast<const f16x8*>(Qh + (t2 * 16 + m) * KHS + cb + kq);
      const f16x8 ql = *reinterpret_cast<const f16x8*>(Ql + (t2 * 16 + m) * KHS + cb + kq);
#pragma unroll
      for (int q = 0; q < PNB; ++q) {
        acc[q][t2] = mma_h(x[q], ql, acc[q][t2]);
        acc[q][t2] = mma_h(x[q], qh, acc[q][t2]);
      }
    }
  }
  __syncthreads();  // M complete, its partials dead
  float* kt = part + w * WBT * GS16;
#pragma unroll
  for (int q = 0; q < PNB; ++q) {
    if (w + PW * q >= nkb) continue;
    bool wild[4], any = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      wild[e] = -gl[q].v[e] > WILD;
      any |= wild[e];
    }
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      Quad a;
#pragma unroll
      for (int e = 0; e < 4; ++e) a.v[e] = keep_exp(!wild[e], u[q][t2].v[e], -G[q][t2].v[e]);
      *reinterpret_cast<Quad*>(kt + (t2 * 16 + m) * GS16 + 4 * g) = a;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wave's own panel
#pragma unroll
    for (int jb = 0; jb < 2; ++jb)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float kv = kt[(jb * 16 + 4 * g + e) * GS16 + m];
#pragma unroll
        for (int t2 = jb; t2 < 2; ++t2)
          acc[q][t2] = mfma4(kv, Ml[(t2 * 16 + m) * AS + jb * 16 + 4 * g + e], acc[q][t2]);
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the next block overwrites it
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      Quad o, d;
#pragma unroll
      for (int e = 0; e < 4; ++e) o.v[e] = __expf(G[q][t2].v[e]) * acc[q][t2][e];
      if (__any(any)) {  // exact sums of the wild rows' in-chunk terms
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (!wild[e]) continue;
          const int i = t2 * 16 + m, c = c0[q] + e;
          for (int j = 0; j <= i; ++j)
            o.v[e] += Ml[i * AS + j] * (bf2f(ubc[j * kw + c]) * tokc[j].ru) * __expf(G[q][t2].v[e] - Gc[j * kw + c]);
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) d.v[e] = kn[q][t2].v[e] + o.v[e];
      const unsigned off = (t2 * 16 + m) * kw + c0[q];
      if (p.o) *reinterpret_cast<Quad*>(p.o + tb * kw + off) = o;
      *reinterpret_cast<Quad*>(p.d + tb * kw + off) = d;
    }
  }
}

constexpr size_t out_s_smem() { return (size_t)4 * WBT * KHS * 2; }
constexpr size_t out_c_smem() {
  return (size_t)2 * WBT * KHS * 2 + (size_t)(WBT * AS + PW * 3 * 256) * sizeof(float);
}
static_assert(PW * 3 * 256 >= PW * WBT * GS16, "the waves' k~ panels fit the partial Ms' storage");

// ---------------------------------------------------------------------------
// Dual sources (per token): phi, den, e, chi.
// ---------------------------------------------------------------------------
struct SrcParams {
  sd_inputs in;
  int Tp, KP;
  const __bf16 *ub, *kb, *qb;
  const Tok* tok;
  const float* delta;
  float *e, *chi;
};

__global__ __launch_bounds__(WT) void k_w_sources(SrcParams p) {
  const int s = blockIdx.y, H = p.in.H, T = p.in.T, r = p.in.r;
  const int b = s / H, h = s % H;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int t = blockIdx.x * (WT / 64) + w;
  if (t >= p.Tp) return;
  const bool tv = t < T;
  const long long row = ((long long)s * p.Tp + t) * p.KP;
  // every load first, at clamped indices (masked below): no load under a branch
  const int tc = min(t, T - 1);
  const __bf16* err = wrow(p.in.erase_raw, b, tc, h);
  const Tok tk = p.tok[(long long)s * p.Tp + t];
  float u[4], dl[4], k[4], q[4], er[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = l + 64 * j, ck = min(c, p.KP - 1);
    u[j] = bf2f(p.ub[row + ck]);
    dl[j] = p.delta[row + ck];
    k[j] = bf2f(p.kb[row + ck]);
    q[j] = bf2f(p.qb[row + ck]);
    er[j] = bf2f(err[min(c, r - 1)]);
  }
  float usq = 0.f, dsq = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = l + 64 * j;
    const bool in = c < p.KP;
    u[j] = in ? u[j] * tk.ru : 0.f;
    dl[j] = in ? dl[j] : 0.f;
    k[j] = in ? k[j] * tk.rk : 0.f;
    q[j] = in ? q[j] * tk.rq : 0.f;
    er[j] = (tv && c < r) ? er[j] : 0.f;
    usq += u[j] * u[j];
    dsq += dl[j] * dl[j];
  }
  usq = wave_sum(usq);
  dsq = wave_sum(dsq);
  const float sc = RHO / sqrtf(RHO * RHO + usq * dsq);
  float phi[4], bb[4];
  float pu = 0.f, ub = 0.f, uq = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    phi[j] = sc * dl[j];
    bb[j] = k[j] / (1.f + __expf(-er[j]));
    pu += phi[j] * u[j];
    ub += u[j] * bb[j];
    uq += u[j] * q[j];
  }
  const float den = 1.f + wave_sum(pu);
  const float sb = wave_sum(ub) / den, sq = wave_sum(uq) / den;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = l + 64 * j;
    if (c < p.KP) {
      p.e[row + c] = bb[j] - phi[j] * sb;
      p.chi[row + c] = q[j] - phi[j] * sq;
    }
  }
}

// ---------------------------------------------------------------------------
// Backward preparation of one op's reverse pass.
//   column output: rhs = dW + P^T dO, injection Ia = q e^G, Ib = dO
//   row output:    Pp_ij = sum_r dO_ir k_jr e^{G_ir - G_jr} (j <= i), rhs = dW + Pp^T q,
//                  Ia = dO e^G / |k|, Ib = the raw k (q = k / |k|)
//   dU = A^T rhs,  Wn = -A^T Kh,  Kn = -x~  (Wn, Kn, Ia stored bf16 for the
//   reverse pass: -Wn token-major, Kn and Ia transposed per chunk)
// ---------------------------------------------------------------------------
struct BprepParams {
  int NT, Tp, kw, vw;
  const float *k, *x, *q, *G, *A, *P, *dO, *dW;  // k, x, q: column output; dO, dW: row output
  const __bf16 *dOb, *ub, *kb;  // column output: dO; row output: u, k (k = u^, x = gx u^, q = k^)
  const Tok* tok;
  float *dU, *Pp;  // dU [Tp][vw] in accumulator order (acc_off)
  __bf16 *Wneg, *Kt, *At;  // reverse-pass panels: -Wn (w_off order); Kn, Ia transposed per chunk [NT][kw][32]
};

// Same organisation as k_w_prep: a lane's four coordinates of a token are loaded
// once and give the Pp Gram's operands, K^, Kn and Ia; the value side runs
// straight from registers.  Two workgroups per CU (76 KB of LDS, 128 VGPRs):
// 92 us (S, 232 KiB a chunk, 5.3 TB/s with what the last-level cache still holds)
// and 104 us (C, 216 KiB, 4.4 TB/s) at B4 T2048 H8 r = V = 256, where one four-wave
// workgroup per CU (LDS copies of every operand, 4-byte loads of each panel's
// columns) took 174 us per op.
template <bool COL>
__global__ __launch_bounds__(PT, 4) void k_w_bprep(BprepParams p) {
  extern __shared__ __align__(16) float sm[];
  const int ch = blockIdx.x, s = blockIdx.y, kw = p.kw, vw = p.vw, nkb = kw / 16, nvb = vw / 16;
  const long long tb = (long long)s * p.Tp + ch * WBT;
  const long long cbase = (long long)s * p.NT + ch;
  // chunk-uniform bases, 32-bit lane offsets
  const __bf16* Y = (COL ? p.dOb : p.kb) + tb * vw;  // [32][vw] (row output: times 1/|k|)
  const float *Yk = (COL ? p.q : p.dO) + tb * kw, *Gc = p.G + tb * kw;  // [32][kw]
  const float *kc = COL ? p.k + tb * kw : nullptr, *xc = COL ? p.x + tb * kw : nullptr;
  const __bf16* ubc = COL ? nullptr : p.ub + tb * kw;
  const float* dWc = COL ? nullptr : p.dW + tb * vw;
  const Tok* tokc = COL ? nullptr : p.tok + tb;
  float* kh = sm;               // K^ [32][XTS]
  float* Al = kh + WBT * XTS;   // A [32][AS]
  float* Pl = Al + WBT * AS;    // P or Pp [32][AS]
  // Kn and Ia rows [32][KHS]; their storage first holds the partial Pp Grams
  __bf16* kn = reinterpret_cast<__bf16*>(Pl + WBT * AS);
  __bf16* ia = kn + WBT * KHS;
  float* part = reinterpret_cast<float*>(kn);
  static_assert(PW * 3 * 256 * sizeof(float) <= 2 * WBT * KHS * 2, "partial Grams fit");
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 4, m = l & 15;
  if (threadIdx.x < WBT * WBT / 4) {
    const int i = threadIdx.x >> 3, j = (threadIdx.x & 7) * 4;
    const long long o = cbase * WBT * WBT + i * WBT + j;
    const Quad av = ldq(p.A + o);
    if constexpr (COL) *reinterpret_cast<Quad*>(Pl + i * AS + j) = ldq(p.P + o);
    *reinterpret_cast<Quad*>(Al + i * AS + j) = av;
  }
  // key side: this lane's coordinates; row output: also the Gram
  // Pp_ij = sum_c dO_ic k_jc e^{G_ic - G_jc} (j <= i)
  f4 acc[3] = {zero4(), zero4(), zero4()};
  bf16x4 kn4[PNB][2], ia4[PNB][2];
  [[maybe_unused]] float tru[2], tgx[2], trk[2];
  if constexpr (!COL)
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      const Tok* tk = tokc + t2 * 16 + m;
      tru[t2] = tk->ru;
      tgx[t2] = tk->gx;
      trk[t2] = tk->rks;  // the injection's Ib is the raw bf16 k: its norm goes into Ia
    }
#pragma unroll
  for (int j = 0; j < PNB; ++j) {
    const int kb = w + PW * j;
    if (kb >= nkb) continue;
    const int c0 = kb * 16 + 4 * g;
    const Quad gl = ldq(Gc + (unsigned)((WBT - 1) * kw + c0));
    Quad x[2], k[2], y[2], G[2], Gx[2];
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      const unsigned o = (t2 * 16 + m) * kw + c0;
      if constexpr (COL) {
        x[t2] = ldq(xc + o);
        k[t2] = ldq(kc + o);
      } else {
        k[t2] = scaled(ldq(ubc + o), tru[t2]);
        x[t2] = scaled(k[t2], tgx[t2]);
      }
      y[t2] = ldq(Yk + o);
      G[t2] = ldq(Gc + o);
      if constexpr (!COL) Gx[t2] = ldq(Gc + (t2 == 0 && m == 0 ? o : o - kw));  // prefix before the token
    }
    bool wild[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) wild[e] = -gl.v[e] > WILD;
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      Quad kd;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float gx = G[t2].v[e];
        if constexpr (!COL) gx = t2 == 0 && m == 0 ? 0.f : Gx[t2].v[e];
        kd.v[e] = k[t2].v[e] * __expf(gl.v[e] - G[t2].v[e]);
        kn4[j][t2][e] = (__bf16)(-x[t2].v[e] * __expf(gx));
        y[t2].v[e] *= __expf(G[t2].v[e]);
        ia4[j][t2][e] = (__bf16)(COL ? y[t2].v[e] : y[t2].v[e] * trk[t2]);
        if constexpr (!COL) k[t2].v[e] = keep_exp(!wild[e], k[t2].v[e], -G[t2].v[e]);
      }
      *reinterpret_cast<Quad*>(kh + (t2 * 16 + m) * XTS + c0) = kd;
    }
    if constexpr (!COL) {
      gram3(y, k, acc);
      gram3_wild(wild, kb * 16, false,
                 [&](int i, int c) { return make_float2(Yk[i * kw + c], Gc[i * kw + c]); },
                 [&](int jj, int c) {
                   return make_float2(bf2f(ubc[jj * kw + c]) * tokc[jj].ru, Gc[jj * kw + c]);
                 }, acc);
    }
  }
  // the value side's rows, issued before any store of the kernel
  float yv[PNB][2][4];
  f4 rhs[PNB][2];
#pragma unroll
  for (int j = 0; j < PNB; ++j) {
    const int nb = min(w + PW * j, nvb - 1);
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned o = (t2 * 16 + 4 * g + e) * vw + nb * 16 + m;
        yv[j][t2][e] = bf2f(Y[o]);
        if constexpr (!COL) yv[j][t2][e] *= tokc[t2 * 16 + 4 * g + e].rk;
        rhs[j][t2][e] = COL ? 0.f : dWc[o];
      }
  }
  if constexpr (!COL) {
    gram3_put(part, w, acc);
    __syncthreads();
    if (threadIdx.x < 192) {
      const int q = threadIdx.x >> 6;
      const f4 v = gram3_sum<PW>(part, 0, q, l);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = (q > 0 ? 16 : 0) + 4 * g + e, j = (q > 1 ? 16 : 0) + m;
        Pl[i * AS + j] = j <= i ? v[e] : 0.f;
      }
    } else if (threadIdx.x < 256) {
#pragma unroll
      for (int e = 0; e < 4; ++e) Pl[(4 * g + e) * AS + 16 + m] = 0.f;
    }
    __syncthreads();
    if (threadIdx.x < WBT * WBT / 4) {
      const int i = threadIdx.x >> 3, j = (threadIdx.x & 7) * 4;
      *reinterpret_cast<Quad*>(p.Pp + cbase * WBT * WBT + i * WBT + j) =
          *reinterpret_cast<const Quad*>(Pl + i * AS + j);
    }
  }
#pragma unroll
  for (int j = 0; j < PNB; ++j) {
    const int kb = w + PW * j;
    if (kb >= nkb) continue;
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      const int o = (t2 * 16 + m) * KHS + kb * 16 + 4 * g;
      *reinterpret_cast<bf16x4*>(kn + o) = kn4[j][t2];
      *reinterpret_cast<bf16x4*>(ia + o) = ia4[j][t2];
    }
  }
  __syncthreads();
  // value side: rhs = dW + P^T Y and dU = A^T rhs on FP32 matrix cores over the
  // lower blocks of P and A (the rhs accumulators are the B operands of the dU
  // product as they stand)
#pragma unroll
  for (int j = 0; j < PNB; ++j) {
    const int nb = w + PW * j;
    f4 du[2] = {zero4(), zero4()};
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t2 = 0; t2 <= kb; ++t2)
          rhs[j][t2] = mfma4(Pl[(kb * 16 + 4 * g + e) * AS + t2 * 16 + m], yv[j][kb][e], rhs[j][t2]);
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t2 = 0; t2 <= kb; ++t2)
          du[t2] = mfma4(Al[(kb * 16 + 4 * g + e) * AS + t2 * 16 + m], rhs[j][kb][e], du[t2]);
    if (nb < nvb)
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) *reinterpret_cast<f4*>(p.dU + tb * vw + acc_off(t2, nb, l, vw)) = du[t2];
  }
  // key side: Wn = -A^T K^ (stored negated), transposed as k_w_prep's W
#pragma unroll
  for (int j = 0; j < PNB; ++j) {
    const int nb = w + PW * j, nk = min(nb, nkb - 1);
    f4 aw[2] = {zero4(), zero4()};
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = kb * 16 + 4 * g + e;
        const float kv = kh[k * XTS + nk * 16 + m];
#pragma unroll
        for (int t2 = 0; t2 <= kb; ++t2) aw[t2] = mfma4(kv, Al[k * AS + t2 * 16 + m], aw[t2]);
      }
    if (nb < nkb) {
      bf16x8 h;
#pragma unroll
      for (int e = 0; e < 8; ++e) h[e] = (__bf16)aw[e >> 2][e & 3];
      *reinterpret_cast<bf16x8*>(p.Wneg + tb * kw + w_off(nb, l, 0)) = h;
    }
  }
  store_transposed(p.Kt + cbase * kw * WBT, kn, kw);
  store_transposed(p.At + cbase * kw * WBT, ia, kw);
}

constexpr size_t bprep_smem() {
  return (size_t)(WBT * XTS + 2 * WBT * AS) * sizeof(float) + (size_t)2 * WBT * KHS * 2;
}

// ---------------------------------------------------------------------------
// Closed-form chunk gradients of one op (tests/chunk_model.py Op.backward):
//   M1_ij = dw_i.w_j (j < i);  M2_lj = Y_l.w_j (j <= l), Y = dO (column) / q (row)
//   dx = -(e^{Gx} (dw X0^T) + apply(M1, k, Gx, G))
//   dk = e^{G_C - G} (w lam^T) + apply_t(M2, Yk, G, G) - apply_t(M1, x, Gx, G)
//        with Yk = q (column) / dO (row)
//   dq = e^{G} (dO X0^T) + apply(M2, k, G, G)          (column)
//   dq = (dO e^G) X0 + Pp w                             (row)
//   dG = q dq - k dk (column) / o dO - k dk (row), + x dx (shifted one token
//   earlier when the erase reads before the decay), last row + rowsum(X_C lam);
//   dg = in-chunk reverse cumulative sum of dG.
// ---------------------------------------------------------------------------
struct GradParams {
  int NT, Tp, kw, vw;
  const float *k, *x, *q, *G, *dO, *o, *w, *dw, *Pp;  // k, x, q: column output; dO, o, Pp: row output
  const __bf16 *dOb, *ub, *kb;  // column output: dO; row output: u, k (k = u^, x = gx u^, q = k^)
  const Tok* tok;
  const xs_t* Xslots;
  const ls_t* Lslots;
  // column output (S): the panels dk, dx, dq, dg
  float *dk, *dx, *dq, *dg;
  // row output (C): the layer's closure of u, h, k, gamma and the log-decay
  sd_inputs in;
  const float *duh, *dkh, *dgS;
  __bf16 *du, *dh, *dkey;
  float *dlog_decay, *dgamma;
  int vec;  // the gradients' rows take 4-element stores
};


// Eight waves (two per SIMD, so one wave's loads overlap another's matrix
// work), each owning the 16-row blocks rb = wave + 8 q of the state.
constexpr int GW = 8;
constexpr int GT = GW * 64;
constexpr int GRB = WMAX / 16 / GW;
// Lane i of a 16-lane row takes lane i + N's value, 0 past the row's end.
template <int N>
__device__ __forceinline__ float row_next(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x100 + N, 0xF, 0xF, true));
}
// Lane i takes lane i - 1's value, 0 at the row's start.
__device__ __forceinline__ float row_prev(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x111, 0xF, 0xF, true));
}
// Sum over this and the following lanes of a 16-lane row.
__device__ __forceinline__ float row_suffix(float v) {
  v += row_next<1>(v);
  v += row_next<2>(v);
  v += row_next<4>(v);
  return v + row_next<8>(v);
}

__device__ __forceinline__ f4 mma_bf(bf16x8 a, bf16x8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
template <class V8>
__device__ __forceinline__ void split8(const V8& v, bf16x8& hi, bf16x8& lo) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float x = (float)v[j];
    const __bf16 h = (__bf16)x;
    hi[j] = h;
    lo[j] = (__bf16)(x - (float)h);
  }
}
__device__ __forceinline__ void split4_to(__bf16* hi, __bf16* lo, const Quad& q) {
  bf16x4 h, o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    h[e] = (__bf16)q.v[e];
    o[e] = (__bf16)(q.v[e] - (float)h[e]);
  }
  *reinterpret_cast<bf16x4*>(hi) = h;
  *reinterpret_cast<bf16x4*>(lo) = o;
}

// What bounds it: the state slots (X0 and lambda, 256 KiB of a chunk's 592 KiB
// (S) or 644 KiB (C) at r = V = 256) stream through phase 1; every product's output is formed
// transposed, so a lane holds four neighbouring coordinates of one token and
// reads and writes the token panels 16 bytes at a time, and the rows shared by
// all waves are split into bf16 halves once, in LDS.  290 us (S, 4.3 TB/s) and
// 460 us (C, with the layer's closure: 2.9 TB/s, one workgroup per CU whose tail
// reads more rows after its products) per launch at B4 T2048 H8 r = V = 256; with
// 4-byte panel accesses in the MFMA layout, the rows split by every wave and
// dO e^G X0 on FP32 MFMAs over 2-byte gathers of the slot, 360 us and, with the
// closure as a kernel of its own, 500 + 217 us.
template <bool COL>
__global__ __launch_bounds__(GT, 2) void k_w_grad(GradParams p) {
  extern __shared__ __align__(16) float sm[];
  int ch, s;
  xcd_map(blockIdx.x, p.NT, gridDim.x / p.NT, ch, s);
  const int kw = p.kw, vw = p.vw, nrb = kw / 16, nvb = vw / 16;
  const long long tb = (long long)s * p.Tp + ch * WBT;
  const long long slot = (long long)s * (p.NT + 1) + ch;
  const xs_t* X0 = p.Xslots + slot * kw * vw;
  const xs_t* XC = X0 + (long long)kw * vw;
  const ls_t* Lm = p.Lslots + slot * kw * vw;
  float* M1 = sm;              // token Grams [32][AS]
  float* M2 = M1 + WBT * AS;
  // phase 1: dw, w, Y rows split [32][KHS]; phase 2 (row output): dO e^G split
  // and two X0 row blocks; phase 3: per wave k~, Y~, x~ [32][GS16]
  __bf16* TR = reinterpret_cast<__bf16*>(M2 + WBT * AS);
  constexpr int RP = WBT * KHS;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, g = l >> 4, m = l & 15, kq = g * 8;
  // chunk-uniform bases, 32-bit lane offsets
  const __bf16* Y = (COL ? p.dOb : p.kb) + tb * vw;  // [32][vw]: exact in bf16 (row output: M2's rows take 1/|k| at the end)
  const float *Yk = (COL ? p.q : p.dO) + tb * kw, *Gc = p.G + tb * kw;  // [32][kw]
  const float *dwc = p.dw + tb * vw, *wc = p.w + tb * vw;
  const float *kpc = COL ? p.k + tb * kw : nullptr, *xpc = COL ? p.x + tb * kw : nullptr,
              *opc = COL ? nullptr : p.o + tb * kw;
  const __bf16 *ubc = COL ? nullptr : p.ub + tb * kw, *kbc = COL ? nullptr : p.kb + tb * kw;
  const Tok* tokc = COL ? nullptr : p.tok + tb;
  {
    constexpr int PQ = WBT * WMAX / 4 / GT;
    Quad v[PQ][2];
    bf16x4 y[PQ];
#pragma unroll
    for (int q = 0; q < PQ; ++q) {
      const int idx = min((int)(threadIdx.x + GT * q), WBT * vw / 4 - 1);
      const unsigned o = idx * 4;
      v[q][0] = ldq(dwc + o);
      v[q][1] = ldq(wc + o);
      y[q] = *reinterpret_cast<const bf16x4*>(Y + o);
    }
#pragma unroll
    for (int q = 0; q < PQ; ++q) {
      const int idx = min((int)(threadIdx.x + GT * q), WBT * vw / 4 - 1);
      const int i = (idx * 4) / vw, c = (idx * 4) % vw;
#pragma unroll
      for (int a = 0; a < 2; ++a)
        split4_to(TR + 2 * a * RP + i * KHS + c, TR + (2 * a + 1) * RP + i * KHS + c, v[q][a]);
      *reinterpret_cast<bf16x4*>(TR + 4 * RP + i * KHS + c) = y[q];
    }
  }
  __syncthreads();
  // phase 1 on bf16 matrix cores (the cotangents may take any scale), K = 32
  // value columns per step: this wave's rows of dwX = dw X0^T, wL = w lam^T and
  // (column output) dOX = dO X0^T, transposed (lane (g, m): rows 4 g .. + 3 of
  // token m), and one lower 16 x 16 block of M1 = dw w^T or M2 = Y w^T per wave
  // of the first six.  The rows and the fp16 state X0 enter split into bf16
  // high and low halves (three MFMAs per product); lambda is exact in its slot.
  f4 aX[GRB][2], aL[GRB][2], aO[GRB][2], am = zero4();
  float rs[GRB];  // partial rowsum(X_C (.) lam) of state row 16 rb + m over this lane's columns
#pragma unroll
  for (int q = 0; q < GRB; ++q) {
    rs[q] = 0.f;
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) aX[q][t2] = aL[q][t2] = aO[q][t2] = zero4();
  }
  const int gq = w % 3, bi = gq > 0, bj = gq > 1, gm = w < 3 ? 0 : 2;  // Gram block, left rows
  {
    unsigned ro[GRB];  // row offsets of this wave's blocks (clamped: loads stay unconditional)
#pragma unroll
    for (int q = 0; q < GRB; ++q) ro[q] = slot_off(min(w + GW * q, nrb - 1) * 16 + m, kq, kw);
    f16x8 x8[2][GRB], c8[2][GRB];
    bf16x8 l8[2][GRB];
    auto fetch = [&](int cb, int f) {
#pragma unroll
      for (int q = 0; q < GRB; ++q) {
        x8[f][q] = *reinterpret_cast<const f16x8*>(X0 + cb * kw + ro[q]);
        l8[f][q] = *reinterpret_cast<const bf16x8*>(Lm + cb * kw + ro[q]);
        c8[f][q] = *reinterpret_cast<const f16x8*>(XC + cb * kw + ro[q]);
      }
    };
    auto step = [&](int cb, int f) {
      auto row = [&](int a, int t2) { return *reinterpret_cast<const bf16x8*>(TR + a * RP + (t2 * 16 + m) * KHS + cb + kq); };
      bf16x8 xh[GRB], xl[GRB];
#pragma unroll
      for (int q = 0; q < GRB; ++q) {
        split8(x8[f][q], xh[q], xl[q]);
#pragma unroll
        for (int j = 0; j < 8; ++j) rs[q] += (float)c8[f][q][j] * (float)l8[f][q][j];
      }
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        const bf16x8 dh = row(0, t2), dl = row(1, t2), wh = row(2, t2), wl = row(3, t2);
#pragma unroll
        for (int q = 0; q < GRB; ++q) {
          aX[q][t2] = mma_bf(xh[q], dl, aX[q][t2]);
          aL[q][t2] = mma_bf(l8[f][q], wl, aL[q][t2]);
          aX[q][t2] = mma_bf(xl[q], dh, aX[q][t2]);
          aL[q][t2] = mma_bf(l8[f][q], wh, aL[q][t2]);
          aX[q][t2] = mma_bf(xh[q], dh, aX[q][t2]);
        }
        if constexpr (COL) {
          const bf16x8 yh = row(4, t2);
#pragma unroll
          for (int q = 0; q < GRB; ++q) {
            aO[q][t2] = mma_bf(xl[q], yh, aO[q][t2]);
            aO[q][t2] = mma_bf(xh[q], yh, aO[q][t2]);
          }
        }
      }
      if (w < 6) {
        const bf16x8 ah = row(gm * 2, bi), bh = row(2, bj), bl = row(3, bj);
        if (w < 3) am = mma_bf(row(1, bi), bh, am);
        am = mma_bf(ah, bl, am);
        am = mma_bf(ah, bh, am);
      }
    };
    fetch(0, 0);
    int cb = 0;
    for (; cb + 32 < vw; cb += 64) {  // (the last fetch past an odd count rereads the first columns)
      fetch(cb + 32, 1);
      step(cb, 0);
      fetch(cb + 64 < vw ? cb + 64 : 0, 0);
      step(cb + 32, 1);
    }
    if (cb < vw) step(cb, 0);
  }
  if (w < 6) {
    float* M = w < 3 ? M1 : M2;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = bi * 16 + 4 * g + e, j = bj * 16 + m;
      float v = am[e];
      if (!COL && w >= 3) {  // (a zero inverse norm: the raw row's products may have overflowed)
        const float rk = tokc[i].rk;
        v = rk != 0.f ? v * rk : 0.f;
      }
      M[i * AS + j] = (w < 3 ? j < i : j <= i) ? v : 0.f;
    }
  }
  // this lane's elements of the key-side panels (tokens m and 16 + m), loaded
  // before any store of the kernel
  Quad kr[GRB][2], yr[GRB][2], xr[GRB][2], G[GRB][2], orw[GRB][2], gl[GRB];
  int c0[GRB];
  Tok tk[2];
#pragma unroll
  for (int t2 = 0; t2 < 2; ++t2)
    if constexpr (!COL) tk[t2] = tokc[t2 * 16 + m];
#pragma unroll
  for (int q = 0; q < GRB; ++q) {
    c0[q] = min(w + GW * q, nrb - 1) * 16 + 4 * g;
    gl[q] = ldq(Gc + (unsigned)((WBT - 1) * kw + c0[q]));
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      const unsigned o = (t2 * 16 + m) * kw + c0[q];
      if constexpr (COL) {
        kr[q][t2] = ldq(kpc + o);
        xr[q][t2] = ldq(xpc + o);
      } else {
        kr[q][t2] = scaled(ldq(ubc + o), tk[t2].ru);
        xr[q][t2] = scaled(kr[q][t2], tk[t2].gx);
      }
      yr[q][t2] = ldq(Yk + o);
      G[q][t2] = ldq(Gc + o);
      if constexpr (!COL) orw[q][t2] = ldq(opc + o);
    }
  }
  // rowsum(X_C (.) lam): the four lane groups' partials of each state row
#pragma unroll
  for (int q = 0; q < GRB; ++q) {
    rs[q] += __shfl_xor(rs[q], 16);
    rs[q] += __shfl_xor(rs[q], 32);
  }
  __syncthreads();  // M1, M2 complete; the split rows are dead
  // phase 2 (row output): dq = (dO e^G) X0 + Pp w, this wave's 16-column blocks
  // of the value axis, transposed.  The contraction runs along the slot's rows,
  // so 32-row blocks pass through LDS (double buffered, one barrier each) and
  // are read down their columns; bf16 halves as in phase 1, Pp w in FP32.
  [[maybe_unused]] f4 dqc[GRB][2];
  if constexpr (!COL) {
    __bf16 *Dh = TR, *Dl = TR + RP;
    _Float16* Xt = reinterpret_cast<_Float16*>(TR + 2 * RP);  // [2][32][KHS]
    constexpr int XQ = WBT * WMAX / 8 / GT;
    f16x8 xb[XQ];
    auto fetch = [&](int rb) {
#pragma unroll
      for (int q = 0; q < XQ; ++q) {
        const int idx = min((int)(threadIdx.x + GT * q), WBT * vw / 8 - 1);
        // piece idx: column tile idx / 128, row (idx / 4) % 32, columns 8 (idx % 4) .. + 7
        xb[q] = *reinterpret_cast<const f16x8*>(X0 + slot_off(rb + (idx >> 2) % 32, (idx >> 7) * STILE + (idx & 3) * 8, kw));
      }
    };
    auto put = [&](int f) {
#pragma unroll
      for (int q = 0; q < XQ; ++q) {
        const int idx = min((int)(threadIdx.x + GT * q), WBT * vw / 8 - 1);
        *reinterpret_cast<f16x8*>(Xt + f * RP + (idx >> 2) % 32 * KHS + (idx >> 7) * STILE + (idx & 3) * 8) = xb[q];
      }
    };
    fetch(0);
    float wv[GRB][2][4];
    int nb[GRB];
#pragma unroll
    for (int q = 0; q < GRB; ++q) {
      nb[q] = min(w + GW * q, nvb - 1) * 16;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int e = 0; e < 4; ++e) wv[q][kb][e] = wc[(unsigned)((kb * 16 + 4 * g + e) * vw + nb[q] + m)];
    }
    Quad pp[2][2];
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
        pp[t2][kb] = ldq(p.Pp + ((long long)s * p.NT + ch) * WBT * WBT + (t2 * 16 + m) * WBT + kb * 16 + 4 * g);
#pragma unroll
    for (int q = 0; q < GRB; ++q)
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        Quad d;
#pragma unroll
        for (int e = 0; e < 4; ++e) d.v[e] = yr[q][t2].v[e] * __expf(G[q][t2].v[e]);
        const int o = (t2 * 16 + m) * KHS + c0[q];
        split4_to(Dh + o, Dl + o, d);
      }
    put(0);
    __syncthreads();
    f4 aq[GRB][2];
#pragma unroll
    for (int q = 0; q < GRB; ++q) aq[q][0] = aq[q][1] = zero4();
    for (int rb = 0; rb < kw; rb += 32) {
      const int f = (rb >> 5) & 1;
      if (rb + 32 < kw) fetch(rb + 32);
      bf16x8 dh[2], dl[2];
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        dh[t2] = *reinterpret_cast<const bf16x8*>(Dh + (t2 * 16 + m) * KHS + rb + kq);
        dl[t2] = *reinterpret_cast<const bf16x8*>(Dl + (t2 * 16 + m) * KHS + rb + kq);
      }
#pragma unroll
      for (int q = 0; q < GRB; ++q) {
        f16x8 xc;
#pragma unroll
        for (int j = 0; j < 8; ++j) xc[j] = Xt[f * RP + (kq + j) * KHS + nb[q] + m];
        bf16x8 xh, xl;
        split8(xc, xh, xl);
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2) {
          aq[q][t2] = mma_bf(xh, dl[t2], aq[q][t2]);
          aq[q][t2] = mma_bf(xl, dh[t2], aq[q][t2]);
          aq[q][t2] = mma_bf(xh, dh[t2], aq[q][t2]);
        }
      }
      if (rb + 32 < kw) put(f ^ 1);
      __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < GRB; ++q)
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
#pragma unroll
        for (int kb = 0; kb <= t2; ++kb)
#pragma unroll
          for (int e = 0; e < 4; ++e) aq[q][t2] = mfma4(wv[q][kb][e], pp[t2][kb].v[e], aq[q][t2]);
        dqc[q][t2] = aq[q][t2];  // vw = kw: the same coordinates as the key side's
      }
  }
  // phase 3: the in-chunk applies on FP32 matrix cores over the Grams' lower
  // blocks, decay factored per state row r as e^{Ga_i} e^{-Gb_j} (exact while r's
  // decay over the chunk is at most WILD; wild rows take the exact per-term sums):
  //   dx = -e^{Gx} (dwX + M1 k~),               k~_jr = k_jr e^{-G_jr}
  //   dk = e^{-G} (e^{G_C} wL + M2^T Y~ - M1^T x~),  Y~ = Yk e^{G}, x~ = x e^{Gx}
  //   dq = e^{G} (dOX + M2 k~)                   (column output)
  // k~, Y~, x~ of a wave's 16 coordinates pass through its own LDS panels.
  float* kt = reinterpret_cast<float*>(TR) + w * 3 * WBT * GS16;
  float *yt = kt + WBT * GS16, *xt = yt + WBT * GS16;
  // Row output: the closure of u, k, h, gamma follows from registers (the
  // workgroup holds its 32 tokens' whole rows): with du' = duh + dk + gamma dx,
  // dk' = dkh + dd + dq and the row sums su = du'.u, sk = dk'.k, sg = u.dx + h.dw
  // over all waves, du = (du' - su u) / |u|, dk = (dk' - sk k) / |k|, dh = gamma dw.
  // As a kernel of its own it read ten panels back (217 us at B4 T2048 H8 r = V = 256).
  [[maybe_unused]] Quad gu[GRB][2], gk[GRB][2], dgo[GRB][2];
  [[maybe_unused]] bf16x4 dh4[GRB][2];
  [[maybe_unused]] float su[2] = {0.f, 0.f}, sk[2] = {0.f, 0.f}, sg[2] = {0.f, 0.f}, gmv[2], xk[2];
  [[maybe_unused]] const int T = p.in.T, H = p.in.H, r = p.in.r, hb = s / H, hh = s % H;
  if constexpr (!COL) {
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      gmv[t2] = tk[t2].gam;
      xk[t2] = erase_keep(p.in, hb, min(ch * WBT + t2 * 16 + m, T - 1));  // fresh: dx reaches neither u nor gamma
    }
  }
#pragma unroll
  for (int q = 0; q < GRB; ++q) {
    if (w + GW * q >= nrb) continue;
    [[maybe_unused]] Quad hv[2], kn[2], dv[2];
    if constexpr (!COL) {
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        const unsigned o = (t2 * 16 + m) * kw + c0[q];
        gu[q][t2] = ldq(p.duh + tb * kw + o);
        gk[q][t2] = ldq(p.dkh + tb * kw + o);
        kn[t2] = scaled(ldq(kbc + o), tk[t2].rk);
        dv[t2] = ldq(dwc + o);
        dgo[q][t2] = ldq(p.dgS + tb * kw + o);
        const __bf16* hr = wrow(p.in.h, hb, min(ch * WBT + t2 * 16 + m, T - 1), hh);
#pragma unroll
        for (int e = 0; e < 4; ++e) hv[t2].v[e] = bf2f(hr[min(c0[q] + e, r - 1)]);
      }
    }
    bool wild[4];
    float gx[2][4];
    bool any = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      wild[e] = -gl[q].v[e] > WILD;
      any |= wild[e];
    }
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      Quad a, b, c;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (COL) {
          gx[t2][e] = G[q][t2].v[e];
        } else {  // the prefix before the token: the previous lane's, across the blocks lane 15's
          const float prev = row_prev(G[q][t2].v[e]), edge = __shfl(G[q][0].v[e], l | 15);
          gx[t2][e] = m > 0 ? prev : t2 ? edge : 0.f;
        }
        a.v[e] = keep_exp(!wild[e], kr[q][t2].v[e], -G[q][t2].v[e]);
        b.v[e] = keep_exp(!wild[e], yr[q][t2].v[e], G[q][t2].v[e]);
        c.v[e] = keep_exp(!wild[e], xr[q][t2].v[e], gx[t2][e]);
      }
      const int o = (t2 * 16 + m) * GS16 + 4 * g;
      *reinterpret_cast<Quad*>(kt + o) = a;
      *reinterpret_cast<Quad*>(yt + o) = b;
      *reinterpret_cast<Quad*>(xt + o) = c;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wave's own panels
    // M's blocks [i block][j block] and, for the transposed applies, -M1^T's and
    // M2^T's (read again per row block: held over both they spill)
    f4 m1[2][2], m2[2][2], m1t[2][2], m2t[2][2];
#pragma unroll
    for (int ib = 0; ib < 2; ++ib)
#pragma unroll
      for (int jb = 0; jb <= ib; ++jb) {
        m1[ib][jb] = *reinterpret_cast<const f4*>(M1 + (ib * 16 + m) * AS + jb * 16 + 4 * g);
        m2[ib][jb] = *reinterpret_cast<const f4*>(M2 + (ib * 16 + m) * AS + jb * 16 + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          m1t[ib][jb][e] = -M1[(ib * 16 + 4 * g + e) * AS + jb * 16 + m];
          m2t[ib][jb][e] = M2[(ib * 16 + 4 * g + e) * AS + jb * 16 + m];
        }
      }
    f4 ax[2], ak[2], aq[2];
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      ax[t2] = aX[q][t2];
      aq[t2] = aO[q][t2];
#pragma unroll
      for (int e = 0; e < 4; ++e) ak[t2][e] = __expf(gl[q].v[e]) * aL[q][t2][e];
    }
#pragma unroll
    for (int jb = 0; jb < 2; ++jb)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int o = (jb * 16 + 4 * g + e) * GS16 + m;
        const float kv = kt[o], yv = yt[o], xv = xt[o];
#pragma unroll
        for (int t2 = jb; t2 < 2; ++t2) {
          ax[t2] = mfma4(kv, m1[t2][jb][e], ax[t2]);
          if constexpr (COL) aq[t2] = mfma4(kv, m2[t2][jb][e], aq[t2]);
        }
#pragma unroll
        for (int t2 = 0; t2 <= jb; ++t2) {
          ak[t2] = mfma4(yv, m2t[jb][t2][e], ak[t2]);
          ak[t2] = mfma4(xv, m1t[jb][t2][e], ak[t2]);
        }
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the next block overwrites them
    Quad rdx[2], rdk[2], rdq[2];
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        rdx[t2].v[e] = -__expf(gx[t2][e]) * ax[t2][e];
        rdk[t2].v[e] = __expf(fminf(-G[q][t2].v[e], 80.f)) * ak[t2][e];
        rdq[t2].v[e] = __expf(G[q][t2].v[e]) * aq[t2][e];
      }
    if (__any(any)) {  // exact sums of the wild rows
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (!wild[e]) continue;
          const int i = t2 * 16 + m;
          const float* gc = Gc + c0[q] + e;
          const float* yc = Yk + c0[q] + e;
          auto kc = [&](int j) {
            const unsigned o = (j) * kw + c0[q] + e;
            return COL ? kpc[o] : bf2f(ubc[o]) * tokc[j].ru;
          };
          auto xc = [&](int j) { return COL ? xpc[j * kw + c0[q] + e] : kc(j) * tokc[j].gx; };
          const float gi = G[q][t2].v[e], gxi = gx[t2][e];
          auto gxa = [&](int j) { return COL ? gc[(long long)j * kw] : j > 0 ? gc[(long long)(j - 1) * kw] : 0.f; };
          float a = __expf(gxi) * aX[q][t2][e];
          for (int j = 0; j < i; ++j)
            a += M1[i * AS + j] * kc(j) * __expf(gxi - gc[(long long)j * kw]);
          rdx[t2].v[e] = -a;
          float b = __expf(gl[q].v[e] - gi) * aL[q][t2][e];
          for (int j = i; j < WBT; ++j)
            b += M2[j * AS + i] * yc[(long long)j * kw] * __expf(gc[(long long)j * kw] - gi);
          for (int j = i + 1; j < WBT; ++j)
            b -= M1[j * AS + i] * xc(j) * __expf(gxa(j) - gi);
          rdk[t2].v[e] = b;
          if constexpr (COL) {
            float c2 = __expf(gi) * aO[q][t2][e];
            for (int j = 0; j <= i; ++j)
              c2 += M2[i * AS + j] * kc(j) * __expf(gi - gc[(long long)j * kw]);
            rdq[t2].v[e] = c2;
          }
        }
    }
    // decay closure: dG = q dq - k dk (column) / o dO - k dk (row) + x dx (of the
    // next token when the erase reads before the decay), and
    // dg = rowsum(X_C lam) + the in-chunk reverse cumulative sum of dG: a
    // suffix scan over the row's 16 lanes (tokens), block 1's total added to block 0
    Quad rdg[2];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float dG[2], xd[2];
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        dG[t2] = -kr[q][t2].v[e] * rdk[t2].v[e] +
                 (COL ? yr[q][t2].v[e] * rdq[t2].v[e] : orw[q][t2].v[e] * yr[q][t2].v[e]);
        xd[t2] = xr[q][t2].v[e] * rdx[t2].v[e];
      }
      if constexpr (COL) {
        dG[0] += xd[0];
        dG[1] += xd[1];
      } else {
        // (every lane takes part: a lane read across lanes must not be switched off)
        const float n1 = __shfl(xd[1], l & 48), n0 = row_next<1>(xd[0]);
        dG[0] += m == 15 ? n1 : n0;
        dG[1] += row_next<1>(xd[1]);
      }
      const float rsum = __shfl(rs[q], 4 * g + e);
      const float s1 = row_suffix(dG[1]), s0 = row_suffix(dG[0]);
      rdg[1].v[e] = rsum + s1;
      rdg[0].v[e] = rsum + s0 + __shfl(s1, l & 48);
    }
    if constexpr (COL) {
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        const unsigned o = (t2 * 16 + m) * kw + c0[q];
        *reinterpret_cast<Quad*>(p.dx + tb * kw + o) = rdx[t2];
        *reinterpret_cast<Quad*>(p.dk + tb * kw + o) = rdk[t2];
        *reinterpret_cast<Quad*>(p.dq + tb * kw + o) = rdq[t2];
        *reinterpret_cast<Quad*>(p.dg + tb * kw + o) = rdg[t2];
      }
    } else {
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float u = kr[q][t2].v[e], dxc = xk[t2] * rdx[t2].v[e];
          gu[q][t2].v[e] += rdk[t2].v[e] + gmv[t2] * dxc;
          gk[q][t2].v[e] += yr[q][t2].v[e] + dqc[q][t2][e];
          su[t2] += gu[q][t2].v[e] * u;
          sk[t2] += gk[q][t2].v[e] * kn[t2].v[e];
          sg[t2] += u * dxc + (c0[q] + e < r ? hv[t2].v[e] : 0.f) * dv[t2].v[e];
          dh4[q][t2][e] = f2bf(gmv[t2] * dv[t2].v[e]);
          dgo[q][t2].v[e] += rdg[t2].v[e];
        }
    }
  }
  if constexpr (!COL) {
    // row sums over the lane groups, then over the waves: red[sum][token][wave]
    float* red = reinterpret_cast<float*>(TR) + GW * 3 * WBT * GS16;
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      float v[3] = {su[t2], sk[t2], sg[t2]};
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        v[a] += __shfl_xor(v[a], 16);
        v[a] += __shfl_xor(v[a], 32);
        if (g == 0) red[(a * WBT + t2 * 16 + m) * GW + w] = v[a];
      }
    }
    Quad kn[GRB][2];  // (read again: held through the loop above they spill)
#pragma unroll
    for (int q = 0; q < GRB; ++q)
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) kn[q][t2] = scaled(ldq(kbc + (unsigned)((t2 * 16 + m) * kw + c0[q])), tk[t2].rk);
    __syncthreads();
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      const int t = ch * WBT + t2 * 16 + m;
      float v[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const float* rr = red + (a * WBT + t2 * 16 + m) * GW;
        const Quad r0 = ldq(rr), r1 = ldq(rr + 4);
        v[a] = ((r0.v[0] + r0.v[1]) + (r0.v[2] + r0.v[3])) + ((r1.v[0] + r1.v[1]) + (r1.v[2] + r1.v[3]));
      }
      if (t >= T) continue;
      const float ru = tk[t2].ru, rk = tk[t2].rk;
      const long long ob = ((long long)hb * T + t) * H + hh, o = ob * r;
#pragma unroll
      for (int q = 0; q < GRB; ++q) {
        if (w + GW * q >= nrb) continue;
        Quad a, b;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          a.v[e] = (gu[q][t2].v[e] - v[0] * kr[q][t2].v[e]) * ru;
          b.v[e] = (gk[q][t2].v[e] - v[1] * kn[q][t2].v[e]) * rk;
        }
        store_row4(p.du + o, c0[q], r, p.vec, a);
        store_row4(p.dkey + o, c0[q], r, p.vec, b);
        store_row4(p.dh + o, c0[q], r, p.vec, dh4[q][t2]);
        store_row4(p.dlog_decay + o, c0[q], r, p.vec, dgo[q][t2]);
      }
      if (w == 0 && g == 0) p.dgamma[ob] = v[2];
    }
  }
}

constexpr size_t grad_smem() { return (size_t)2 * WBT * AS * sizeof(float) + (size_t)5 * WBT * KHS * 2; }
static_assert(5 * WBT * KHS * 2 >= (GW * 3 * WBT * GS16 + 3 * WBT * GW) * 4,
              "phase 3's panels and row sums fit the split rows' storage");

// ---------------------------------------------------------------------------
// Source closure (per token): cotangents of e, chi, z back to u^, delta, k^, q^,
// the raw gates and the values (tests/chunk_model.py sources_bwd).
// ---------------------------------------------------------------------------
struct SrcBwdParams {
  sd_inputs in;
  int Tp, KP, VP;
  const __bf16 *ub, *kb, *qb;
  const Tok* tok;
  const float *delta, *de, *dchi, *dz;
  float *duh, *ddelta, *dkh;
  __bf16 *dq, *derase, *dwrite, *dv;
};

__global__ __launch_bounds__(WT) void k_w_src_bwd(SrcBwdParams p) {
  const int s = blockIdx.y, H = p.in.H, T = p.in.T, r = p.in.r, V = p.in.V;
  const int b = s / H, h = s % H;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int t = blockIdx.x * (WT / 64) + w;
  if (t >= p.Tp) return;
  const bool tv = t < T;
  const long long row = ((long long)s * p.Tp + t) * p.KP, vr = ((long long)s * p.Tp + t) * p.VP;
  // every load first, at clamped indices (masked below): no load under a branch
  const int tc = min(t, T - 1);
  const __bf16 *err = wrow(p.in.erase_raw, b, tc, h), *vrow = wrow(p.in.v, b, tc, h),
               *wrr = wrow(p.in.write_raw, b, tc, h);
  const Tok tk = p.tok[(long long)s * p.Tp + t];
  float u[4], dl[4], k[4], q[4], er[4], de[4], dc[4], vv[4], wr[4], dzv[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = l + 64 * j, ck = min(c, p.KP - 1), cv = min(c, V - 1);
    u[j] = bf2f(p.ub[row + ck]);
    dl[j] = p.delta[row + ck];
    k[j] = bf2f(p.kb[row + ck]);
    q[j] = bf2f(p.qb[row + ck]);
    de[j] = p.de[row + ck];
    dc[j] = p.dchi[row + ck];
    er[j] = bf2f(err[min(c, r - 1)]);
    vv[j] = bf2f(vrow[cv]);
    wr[j] = bf2f(wrr[cv]);
    dzv[j] = p.dz[vr + cv];
  }
  float usq = 0.f, dsq = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = l + 64 * j;
    const bool in = c < p.KP;
    u[j] = in ? u[j] * tk.ru : 0.f;
    dl[j] = in ? dl[j] : 0.f;
    k[j] = in ? k[j] * tk.rk : 0.f;
    q[j] = in ? q[j] * tk.rq : 0.f;
    de[j] = in ? de[j] : 0.f;
    dc[j] = in ? dc[j] : 0.f;
    er[j] = (tv && c < r) ? er[j] : 0.f;
    usq += u[j] * u[j];
    dsq += dl[j] * dl[j];
  }
  usq = wave_sum(usq);
  dsq = wave_sum(dsq);
  const float N = sqrtf(RHO * RHO + usq * dsq), sc = RHO / N;
  float phi[4], se[4], bb[4];
  float pu = 0.f, ub = 0.f, uq = 0.f, pde = 0.f, pdc = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    phi[j] = sc * dl[j];
    se[j] = 1.f / (1.f + __expf(-er[j]));
    bb[j] = se[j] * k[j];
    pu += phi[j] * u[j];
    ub += u[j] * bb[j];
    uq += u[j] * q[j];
    pde += phi[j] * de[j];
    pdc += phi[j] * dc[j];
  }
  const float den = 1.f + wave_sum(pu);
  const float sb = wave_sum(ub) / den, sqv = wave_sum(uq) / den;
  const float dsb = -wave_sum(pde), dsqv = -wave_sum(pdc);
  const float dub = dsb / den, duq = dsqv / den;
  const float dden = -(dsb * sb + dsqv * sqv) / den;
  float dphi[4], duh[4], dqh[4], db[4];
  float ds = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    dphi[j] = -sb * de[j] - sqv * dc[j] + dden * u[j];
    duh[j] = dub * bb[j] + duq * q[j] + dden * phi[j];
    db[j] = de[j] + dub * u[j];
    dqh[j] = dc[j] + duq * u[j];
    ds += dphi[j] * dl[j];
  }
  ds = wave_sum(ds);
  float sqq = 0.f;  // the q norm's closure: dq = (dq^ - (dq^ . q^) q^) / |q|
#pragma unroll
  for (int j = 0; j < 4; ++j) sqq += dqh[j] * q[j];
  sqq = wave_sum(sqq);
  const float dN2 = (-RHO * ds / (N * N)) / (2.f * N);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = l + 64 * j;
    if (c < p.KP) {
      p.duh[row + c] = duh[j] + 2.f * dN2 * dsq * u[j];
      p.ddelta[row + c] = sc * dphi[j] + 2.f * dN2 * usq * dl[j];
      p.dkh[row + c] = db[j] * se[j];
    }
    const long long obase = ((long long)b * T + t) * H + h;
    if (tv && c < r) p.dq[obase * r + c] = f2bf((dqh[j] - sqq * q[j]) * tk.rq);
    if (tv && c < r) p.derase[obase * r + c] = f2bf(db[j] * k[j] * se[j] * (1.f - se[j]));
    if (tv && c < V) {
      const float sw = 1.f / (1.f + __expf(-wr[j]));
      p.dv[obase * V + c] = f2bf(sw * dzv[j]);
      p.dwrite[obase * V + c] = f2bf(dzv[j] * vv[j] * sw * (1.f - sw));
    }
  }
}

// Output cotangent as a padded bf16 panel (zero when absent and on padded entries).
struct DoutParams {
  int H, T, V, Tp, VP, vec;  // vec: rows take 4-element loads
  const __bf16* dout;
  __bf16* dO;
};
__global__ __launch_bounds__(WT) void k_w_dout(DoutParams p) {
  // four neighbouring elements per thread (64-bit divisions per element held
  // the copy to 2 TB/s: 34 us at B4 T2048 H8 V = 256, now 15)
  const int s = blockIdx.y, b = s / p.H, h = s % p.H, q4 = p.VP / 4;
  const long long ib = ((long long)b * p.T * p.H + h) * p.V;
  for (int idx = blockIdx.x * WT + threadIdx.x; idx < p.Tp * q4; idx += gridDim.x * WT) {
    const int t = idx / q4, c = (idx - t * q4) * 4;
    bf16x4 v = {};
    if (p.dout && t < p.T) {
      const __bf16* row = p.dout + ib + (long long)t * p.H * p.V;
      if (p.vec) {
        if (c < p.V) v = *reinterpret_cast<const bf16x4*>(row + c);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c + e < p.V) v[e] = row[c + e];
      }
    }
    *reinterpret_cast<bf16x4*>(p.dO + ((long long)s * p.Tp + t) * p.VP + c) = v;
  }
}

}  // namespace wide

// ---------------------------------------------------------------------------
// Host side: workspace layout and launch sequences.
// ---------------------------------------------------------------------------
namespace {

using namespace wide;

int pad32(int x) { return (x + 31) / 32 * 32; }

struct WideDims {
  int n, NT, Tp, KP, VP;
};
WideDims wide_dims(int B, int T, int H, int r, int V) {
  WideDims d;
  d.n = B * H;
  d.NT = (T + WBT - 1) / WBT;
  d.Tp = d.NT * WBT;
  d.KP = pad32(r);
  d.VP = pad32(V);
  return d;
}

struct WCarver {
  char* base;
  size_t off = 0;
  template <class T = float>
  T* take(size_t count) {
    off = (off + 255) & ~size_t(255);
    T* p = base ? reinterpret_cast<T*>(base + off) : nullptr;
    off += count * sizeof(T);
    return p;
  }
};

struct WideFwd {
  float* G;
  __bf16 *ub, *kb, *qb, *hb;
  Tok* tok;
  float *delta, *oC, *d, *e, *chi, *wS;
  float *AC, *AS, *PS;
  xs_t *XC, *XS;
  _Float16 *Wneg, *Kt;
  float *U, *Qt, *Gam;
};

// saved: what the backward reads; scratch: the forward-only panels (the packed h
// and both ops' W, U, K^, Q~).
WideFwd carve_wide_fwd(void* saved, void* scratch, const WideDims& d, size_t* saved_bytes,
                       size_t* scratch_bytes) {
  WCarver c{(char*)saved};
  const size_t tok = (size_t)d.n * d.Tp, pk = tok * d.KP, pv = tok * d.VP;
  const size_t mat = (size_t)d.n * d.NT * WBT * WBT;
  WideFwd w;
  w.G = c.take(pk);
  w.ub = c.take<__bf16>(pk); w.kb = c.take<__bf16>(pk); w.qb = c.take<__bf16>(pk);
  w.tok = c.take<Tok>(tok);
  w.delta = c.take(pk); w.oC = c.take(pk); w.d = c.take(pk); w.e = c.take(pk);
  w.chi = c.take(pk); w.wS = c.take(pv);
  w.AC = c.take(mat); w.AS = c.take(mat); w.PS = c.take(mat);
  w.XC = c.take<xs_t>((size_t)d.n * (d.NT + 1) * d.KP * d.KP);
  w.XS = c.take<xs_t>((size_t)d.n * (d.NT + 1) * d.KP * d.VP);
  w.Gam = c.take((size_t)d.n * d.NT * d.KP);
  if (saved_bytes) *saved_bytes = c.off + 256;
  WCarver t{(char*)scratch};
  const size_t pm = d.KP > d.VP ? pk : pv;
  w.hb = t.take<__bf16>(pk);
  w.Wneg = t.take<_Float16>(pk); w.U = t.take(pm); w.Kt = t.take<_Float16>(pk); w.Qt = t.take(pk);
  if (scratch_bytes) *scratch_bytes = t.off + 256;
  return w;
}

struct WideBwd {
  __bf16* dO;
  ls_t *LC, *LS;
  float *dU, *Pp;
  __bf16 *Wneg, *Kt, *At;
  float *dwS, *dwC, *dd, *de, *dchi, *dgS;
  float *duh, *ddelta, *dkh;
};

WideBwd carve_wide_bwd(void* base, const WideDims& d, size_t* total) {
  WCarver c{(char*)base};
  const size_t tok = (size_t)d.n * d.Tp, pk = tok * d.KP, pv = tok * d.VP;
  const size_t pm = d.KP > d.VP ? pk : pv;
  WideBwd w;
  w.dO = c.take<__bf16>(pv);
  w.LC = c.take<ls_t>((size_t)d.n * (d.NT + 1) * d.KP * d.KP);
  w.LS = c.take<ls_t>((size_t)d.n * (d.NT + 1) * d.KP * d.VP);
  w.dU = c.take(pm); w.Wneg = c.take<__bf16>(pk); w.Kt = c.take<__bf16>(pk); w.At = c.take<__bf16>(pk);
  w.Pp = c.take((size_t)d.n * d.NT * WBT * WBT);
  w.dwS = c.take(pv); w.dwC = c.take(pk);
  w.dd = c.take(pk); w.de = c.take(pk); w.dchi = c.take(pk); w.dgS = c.take(pk);
  w.duh = c.take(pk); w.ddelta = c.take(pk); w.dkh = c.take(pk);
  if (total) *total = c.off + 256;
  return w;
}

constexpr size_t kMaxLds = 160 * 1024;  // LDS of one gfx950 CU
static_assert(prep_smem() <= kMaxLds / 2 && state_smem() <= kMaxLds && out_s_smem() <= kMaxLds / 2 &&
                  out_c_smem() <= kMaxLds / 2 && bprep_smem() <= kMaxLds / 2 &&
                  grad_smem() <= kMaxLds,
              "a wide kernel's LDS exceeds the CU");

void launch_wprep(const OpParams& op, int n, hipStream_t st) {
  if (op.colout) {
    SD_SMEM_ONCE(k_w_prep<true>, (int)prep_smem());
    SD_LAUNCH("k_w_prep", k_w_prep<true>, dim3(op.NT, n), dim3(PT), prep_smem(), st, op);
  } else {
    SD_SMEM_ONCE(k_w_prep<false>, (int)prep_smem());
    SD_LAUNCH("k_w_prep", k_w_prep<false>, dim3(op.NT, n), dim3(PT), prep_smem(), st, op);
  }
}

void launch_wstate(const char* name, const WStateParams& sp, int n, hipStream_t st) {
  const dim3 grid(sp.vw / STILE * n), blk(ST);
  const bool full = sp.kw == WMAX;
  if (sp.rev && full)
    SD_LAUNCH(name, (k_w_state<true, true>), grid, blk, state_smem(), st, sp);
  else if (sp.rev)
    SD_LAUNCH(name, (k_w_state<true, false>), grid, blk, state_smem(), st, sp);
  else if (full)
    SD_LAUNCH(name, (k_w_state<false, true>), grid, blk, state_smem(), st, sp);
  else
    SD_LAUNCH(name, (k_w_state<false, false>), grid, blk, state_smem(), st, sp);
}

}  // namespace

void wide_fwd_sizes(int B, int T, int H, int r, int V, size_t* saved, size_t* scratch) {
  carve_wide_fwd(nullptr, nullptr, wide_dims(B, T, H, r, V), saved, scratch);
}

size_t wide_bwd_workspace_bytes(int B, int T, int H, int r, int V) {
  size_t total = 0;
  carve_wide_bwd(nullptr, wide_dims(B, T, H, r, V), &total);
  return total;
}

int launch_wide_fwd(const sd_inputs* in, void* out, float* C_T, float* S_T, void* saved,
                    void* scratch, bool keep, hipStream_t st) {
  const WideDims d = wide_dims(in->B, in->T, in->H, in->r, in->V);
  const WideFwd w = carve_wide_fwd(saved, scratch, d, nullptr, nullptr);

  TokParams tp{};
  tp.in = *in; tp.NT = d.NT; tp.Tp = d.Tp; tp.KP = d.KP;
  tp.G = w.G; tp.ub = w.ub; tp.kb = w.kb; tp.qb = w.qb; tp.hb = w.hb; tp.tok = w.tok;
  SD_LAUNCH("k_w_tokens", k_w_tokens, dim3(d.NT, d.n), dim3(WT), 0, st, tp);

  // predictor C: X = C^T, k = u^, x = gamma u^, v = gamma h, q = k^, row output
  OpParams oc{};
  oc.NT = d.NT; oc.Tp = d.Tp; oc.kw = d.KP; oc.vw = d.KP; oc.colout = 0;
  oc.ub = w.ub; oc.hb = w.hb; oc.tok = w.tok; oc.G = w.G;
  oc.A = w.AC; oc.Wneg = w.Wneg; oc.U = w.U; oc.Kt = w.Kt; oc.Gam = w.Gam;
  launch_wprep(oc, d.n, st);
  WStateParams sc{};
  sc.NT = d.NT; sc.Tp = d.Tp; sc.kw = d.KP; sc.vw = d.KP; sc.rows = in->r; sc.cols = in->r;
  sc.Wneg = w.Wneg; sc.U = w.U; sc.Kt = w.Kt; sc.Gam = w.Gam;
  sc.slots = w.XC; sc.wout = w.delta;
  sc.init = in->C0; sc.init_t = 1; sc.fin = C_T; sc.fin_t = 1;
  launch_wstate("w_state_c_fwd", sc, d.n, st);
  OutParams orow{};
  orow.NT = d.NT; orow.Tp = d.Tp; orow.kw = d.KP; orow.vw = d.KP;
  orow.slots = w.XC; orow.w = w.delta; orow.ub = w.ub; orow.kb = w.kb; orow.tok = w.tok;
  orow.G = w.G; orow.o = keep ? w.oC : nullptr; orow.d = w.d;
  SD_SMEM_ONCE(k_w_out_c, (int)out_c_smem());
  SD_LAUNCH("k_w_out_c", k_w_out_c, dim3(d.NT, d.n), dim3(PT), out_c_smem(), st, orow);

  SrcParams sp{};
  sp.in = *in; sp.Tp = d.Tp; sp.KP = d.KP;
  sp.ub = w.ub; sp.kb = w.kb; sp.qb = w.qb; sp.tok = w.tok; sp.delta = w.delta;
  sp.e = w.e; sp.chi = w.chi;
  SD_LAUNCH("k_w_sources", k_w_sources, dim3(d.Tp / (WT / 64), d.n), dim3(WT), 0, st, sp);

  // memory S: k = d, x = e, v = z, q = chi, column output
  OpParams os{};
  os.NT = d.NT; os.Tp = d.Tp; os.kw = d.KP; os.vw = d.VP; os.colout = 1;
  os.k = w.d; os.x = w.e; os.q = w.chi; os.G = w.G; os.in = *in;
  os.A = w.AS; os.P = w.PS; os.Wneg = w.Wneg; os.U = w.U; os.Kt = w.Kt; os.Qt = w.Qt; os.Gam = w.Gam;
  launch_wprep(os, d.n, st);
  WStateParams ss{};
  ss.NT = d.NT; ss.Tp = d.Tp; ss.kw = d.KP; ss.vw = d.VP; ss.rows = in->r; ss.cols = in->V;
  ss.Wneg = w.Wneg; ss.U = w.U; ss.Kt = w.Kt; ss.Gam = w.Gam;
  ss.slots = w.XS; ss.wout = w.wS;
  ss.init = in->S0; ss.init_t = 0; ss.fin = S_T; ss.fin_t = 0;
  launch_wstate("w_state_s_fwd", ss, d.n, st);
  OutParams ocol{};
  ocol.NT = d.NT; ocol.Tp = d.Tp; ocol.kw = d.KP; ocol.vw = d.VP;
  ocol.H = in->H; ocol.T = in->T; ocol.V = in->V;
  ocol.slots = w.XS; ocol.w = w.wS; ocol.Qt = w.Qt; ocol.P = w.PS; ocol.out = (__bf16*)out;
  ocol.vec = in->V % 4 == 0 && ((uintptr_t)out & 7) == 0;
  SD_SMEM_ONCE(k_w_out_s, (int)out_s_smem());
  SD_LAUNCH("k_w_out_s", k_w_out_s, dim3(d.NT, d.n), dim3(PT), out_s_smem(), st, ocol);
  return hipGetLastError() == hipSuccess ? SD_OK : SD_ERR_LAUNCH;
}

int launch_wide_bwd(const sd_inputs* in, const void* fws, void* bws, const void* dout,
                    const float* dC_T, const float* dS_T, void* du, void* dh, void* dq, void* dk,
                    void* dv, void* derase, void* dwrite, float* dlog_decay, float* dgamma,
                    float* dC0, float* dS0, hipStream_t st) {
  const WideDims d = wide_dims(in->B, in->T, in->H, in->r, in->V);
  const WideFwd f = carve_wide_fwd((void*)fws, nullptr, d, nullptr, nullptr);
  const WideBwd w = carve_wide_bwd(bws, d, nullptr);
  // The forward's Gam panel holds exp(G_C) of the last op it ran; both ops share
  // the log-decay, so it serves both reverse passes.

  DoutParams dp{};
  dp.H = in->H; dp.T = in->T; dp.V = in->V; dp.Tp = d.Tp; dp.VP = d.VP;
  dp.dout = (const __bf16*)dout; dp.dO = w.dO;
  dp.vec = in->V % 4 == 0 && ((uintptr_t)dout & 7) == 0;
  SD_LAUNCH("k_w_dout", k_w_dout, dim3(64, d.n), dim3(WT), 0, st, dp);

  // ---- memory S op ----
  BprepParams bs{};
  bs.NT = d.NT; bs.Tp = d.Tp; bs.kw = d.KP; bs.vw = d.VP;
  bs.k = f.d; bs.x = f.e; bs.q = f.chi; bs.G = f.G; bs.A = f.AS; bs.P = f.PS;
  bs.dOb = w.dO;
  bs.dU = w.dU; bs.Wneg = w.Wneg; bs.Kt = w.Kt; bs.At = w.At; bs.Pp = w.Pp;
  SD_SMEM_ONCE(k_w_bprep<true>, (int)bprep_smem());
  SD_LAUNCH("k_w_bprep_s", k_w_bprep<true>, dim3(d.NT, d.n), dim3(PT), bprep_smem(), st, bs);
  WStateParams rs{};
  rs.NT = d.NT; rs.Tp = d.Tp; rs.kw = d.KP; rs.vw = d.VP; rs.rows = in->r; rs.cols = in->V; rs.rev = 1;
  rs.Wneg = w.Wneg; rs.U = w.dU; rs.Kt = w.Kt; rs.Gam = f.Gam; rs.At = w.At; rs.Ib = w.dO;
  rs.slots = w.LS; rs.wout = w.dwS;
  rs.init = dS_T; rs.init_t = 0; rs.fin = dS0; rs.fin_t = 0;
  launch_wstate("w_state_s_bwd", rs, d.n, st);
  GradParams gs{};
  gs.NT = d.NT; gs.Tp = d.Tp; gs.kw = d.KP; gs.vw = d.VP;
  gs.k = f.d; gs.x = f.e; gs.q = f.chi; gs.G = f.G; gs.dOb = w.dO;
  gs.w = f.wS; gs.dw = w.dwS; gs.Xslots = f.XS; gs.Lslots = w.LS; gs.Pp = nullptr;
  gs.dk = w.dd; gs.dx = w.de; gs.dq = w.dchi; gs.dg = w.dgS;
  SD_SMEM_ONCE(k_w_grad<true>, (int)grad_smem());
  SD_LAUNCH("k_w_grad_s", k_w_grad<true>, dim3(d.NT * d.n), dim3(GT), grad_smem(), st, gs);

  SrcBwdParams sb{};
  sb.in = *in; sb.Tp = d.Tp; sb.KP = d.KP; sb.VP = d.VP;
  sb.ub = f.ub; sb.kb = f.kb; sb.qb = f.qb; sb.tok = f.tok; sb.delta = f.delta;
  sb.de = w.de; sb.dchi = w.dchi; sb.dz = w.dwS;
  sb.duh = w.duh; sb.ddelta = w.ddelta; sb.dkh = w.dkh; sb.dq = (__bf16*)dq;
  sb.derase = (__bf16*)derase; sb.dwrite = (__bf16*)dwrite; sb.dv = (__bf16*)dv;
  SD_LAUNCH("k_w_src_bwd", k_w_src_bwd, dim3(d.Tp / (WT / 64), d.n), dim3(WT), 0, st, sb);

  // ---- predictor C op: output cotangent dd (d = k^ + o_C), dW = ddelta ----
  BprepParams bc{};
  bc.NT = d.NT; bc.Tp = d.Tp; bc.kw = d.KP; bc.vw = d.KP;
  bc.ub = f.ub; bc.kb = f.kb; bc.tok = f.tok; bc.G = f.G; bc.A = f.AC;
  bc.dO = w.dd; bc.dW = w.ddelta;
  bc.dU = w.dU; bc.Wneg = w.Wneg; bc.Kt = w.Kt; bc.At = w.At; bc.Pp = w.Pp;
  SD_SMEM_ONCE(k_w_bprep<false>, (int)bprep_smem());
  SD_LAUNCH("k_w_bprep_c", k_w_bprep<false>, dim3(d.NT, d.n), dim3(PT), bprep_smem(), st, bc);
  WStateParams rc{};
  rc.NT = d.NT; rc.Tp = d.Tp; rc.kw = d.KP; rc.vw = d.KP; rc.rows = in->r; rc.cols = in->r; rc.rev = 1;
  rc.Wneg = w.Wneg; rc.U = w.dU; rc.Kt = w.Kt; rc.Gam = f.Gam; rc.At = w.At; rc.Ib = f.kb;
  rc.slots = w.LC; rc.wout = w.dwC;
  rc.init = dC_T; rc.init_t = 1; rc.fin = dC0; rc.fin_t = 1;
  launch_wstate("w_state_c_bwd", rc, d.n, st);
  GradParams gc{};
  gc.NT = d.NT; gc.Tp = d.Tp; gc.kw = d.KP; gc.vw = d.KP;
  gc.ub = f.ub; gc.kb = f.kb; gc.tok = f.tok; gc.G = f.G; gc.dO = w.dd; gc.o = f.oC;
  gc.w = f.delta; gc.dw = w.dwC; gc.Xslots = f.XC; gc.Lslots = w.LC; gc.Pp = w.Pp;
  gc.in = *in; gc.duh = w.duh; gc.dkh = w.dkh; gc.dgS = w.dgS;
  gc.du = (__bf16*)du; gc.dh = (__bf16*)dh; gc.dkey = (__bf16*)dk;
  gc.dlog_decay = dlog_decay; gc.dgamma = dgamma;
  gc.vec = in->r % 4 == 0 && (((uintptr_t)du | (uintptr_t)dh | (uintptr_t)dk) & 7) == 0 &&
           ((uintptr_t)dlog_decay & 15) == 0;
  SD_SMEM_ONCE(k_w_grad<false>, (int)grad_smem());
  SD_LAUNCH("k_w_grad_c", k_w_grad<false>, dim3(d.NT * d.n), dim3(GT), grad_smem(), st, gc);

  return hipGetLastError() == hipSuccess ? SD_OK : SD_ERR_LAUNCH;
}

}  // namespace sd
