// SequenceUnroller(GRU) training kernels (unroller.go:57-213, gru.go).
//
// Reference semantics kept (the quirks are the oracle's, see gru.go):
//  - gates (update u, reset r, candidate c); pre = b + Wx x, plus Wh_u h and
//    Wh_r h for u and r; the candidate adds Wh_r (r * h) with the *reset*
//    gate's recurrent block (gru.go:246-253); h' = h + u (c - h);
//  - backward per step (gru.go:347-510): dU = dh (c - h_prev) u (1 - u),
//    dC = dh (1 - u) (1 - c^2); the reset delta is never computed (0);
//    dh_prev = Wh_u^T dU + Wh_r^T (dC r) + dh u is added to the running dh
//    (unroller.go:189-206);
//  - input-weight gradients use the last step's input for every step.
//
// GPU formulation.  x W_x^T + b for every (sample, step) is one GEMM before
// the recurrence.  The recurrence runs one workgroup per sample: the forward
// reads W_h transposed ([H][2H], so that the threads of one row read
// consecutive floats), the backward reads W_h as stored (column i of W_h^T is
// row-contiguous across threads).  The forward saves the gates' activations
// (u, r, c), which are what the backward needs.  The backward stores dG =
// [dU | 0 | dC] per step; the weight gradients are then GEMMs over (sample,
// step): dW_h,u = dU^T h_prev, dW_h,r = dC^T (r * h_prev), dW_x = (sum_t
// dG)^T x_last, db = sum dG.
#include <algorithm>

#include "gn_common.h"

namespace gn {


// Both recurrences are chains of T steps, each a product with the 2H x H
// recurrent weights: 512 KB at H = 256, which one workgroup per sample would
// read from L2 every step (5 us of a step at one CU's 64 bytes per cycle; the
// first kernels here did, with one load in flight, at 20.8 us per forward and
// 17.8 us per backward step).  The weights therefore stay on the CU for the
// whole sequence: 512 threads with up to 192 of their 256 registers, and LDS,
// hold all of them up to H = 256; of wider layers the leading rows of every
// thread's share, the others streaming from L2 each step.
//
// Thread (c, q) owns columns 4c .. 4c+3 and the q-th share of `rows` input
// rows; the shares' partial sums meet in LDS.  What bounds a step then is the
// 3H^2 (forward) or 2H^2 (backward) fused multiply-adds on one CU's vector
// lanes (1.3 and 0.9 us at H = 256), the barriers between its phases and the
// float64 activations: 3.7 us per forward and 2.0 us per backward step at
// B = 64, H = 256 (the whole layer, T = 100: 3,957 -> 663 us; at T = 30 H = 64,
// B = 300: 374 -> 166, H = 320, B = 128: 1,600 -> 572, H = 1024: 10,390 ->
// 5,199).
// Rows past the matrix hold zero weights and meet zero inputs.
constexpr int GR_NT = 512;   // threads at most

struct GruPlan {
  int GB, NQ, rows, lrows, threads;  // column groups, shares, rows per share, of them in LDS
  size_t lds;
};

// the q-th share's rows e in [0, rows): RR rows in registers, lrows in LDS,
// the rest streamed
__device__ __forceinline__ void gru_fma4(float4 &s, const float4 &w, float x) {
  s.x = __builtin_fmaf(w.x, x, s.x);
  s.y = __builtin_fmaf(w.y, x, s.y);
  s.z = __builtin_fmaf(w.z, x, s.z);
  s.w = __builtin_fmaf(w.w, x, s.w);
}

// 16-byte load from any float's address (global_load_dwordx4 asks for 4 bytes)
typedef float gru_fx4 __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ float4 gru_ld4(const float *p) {
  const gru_fx4 v = *reinterpret_cast<const gru_fx4 *>(p);
  return make_float4(v.x, v.y, v.z, v.w);
}

// row k, columns 4c .. 4c+3 of W (K rows, pitch ld, columns below H, 4c < H);
// zero past the last row.  Columns past H come from what follows in memory
// (their sums are never read), but not past the last row's end.
__device__ __forceinline__ float4 gru_w4(const float *__restrict__ W, int ld, int k, int K, int c, int H) {
  float4 w = make_float4(0.f, 0.f, 0.f, 0.f);
  if (k >= K) return w;
  const float *p = W + (size_t)k * ld + 4 * c;
  if (4 * c + 3 < H || k + 1 < K) return gru_ld4(p);
  w.x = p[0];
  if (4 * c + 1 < H) w.y = p[1];
  if (4 * c + 2 < H) w.z = p[2];
  return w;
}

// s += the four rows w[0..3] of a share against inputs x
__device__ __forceinline__ void gru_rows4(float4 &s, const float4 *w, const float4 &x) {
  gru_fma4(s, w[0], x.x);
  gru_fma4(s, w[1], x.y);
  gru_fma4(s, w[2], x.z);
  gru_fma4(s, w[3], x.w);
}

// s += sum over rows e in [e0, rows) of the share, read from global memory,
// eight 16-byte loads in flight (W holds K rows).  A scalar form for widths
// that are no multiple of 4 had one row in flight: H 513, T 30, B 64 8085 us,
// with unaligned loads 1480 (H 512: 1158).
__device__ __forceinline__ void gru_stream(float4 &s, const float *__restrict__ W, int ld, int k0, int e0,
                                           int rows, int K, int c, int H, const float *v) {
  const int e1 = min(rows, K - k0);                                  // rows of the matrix
  const int ev = e1 - (4 * c + 3 >= H && k0 + e1 == K ? 1 : 0);      // of them those read whole
  int e = e0;
  const float *p = W + (size_t)(k0 + e0) * ld + 4 * c;
  for (; e + 8 <= ev; e += 8, p += 8 * (size_t)ld) {
    float4 w[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) w[u] = gru_ld4(p + u * (size_t)ld);
    gru_rows4(s, w, *reinterpret_cast<const float4 *>(v + k0 + e));
    gru_rows4(s, w + 4, *reinterpret_cast<const float4 *>(v + k0 + e + 4));
  }
  for (; e < e1; ++e) gru_fma4(s, gru_w4(W, ld, k0 + e, K, c, H), v[k0 + e]);
}

// xw [B*T][3H] = b + Wx x_t (from the GEMM); WhT [H][2H]; writes act [B*T][3H]
// (the activations u, r, c), hprev [B*T][H] (h before each step), rh [B*T][H]
// (r * h_prev) and out [B][H] (h_T; seq: every state, [B][T][H]).
// Of a thread's rows, RR (RU or 2 RU) of the reset block (used twice a step) and RU of the
// update block sit in registers, the next lrows of the update block in LDS;
// BIG: the rest streams (and a thread prefetches up to 6 projections, not 2).
template <int RR, int RU, bool BIG>
__global__ __launch_bounds__(GR_NT) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gru_fwd_kernel(const float *__restrict__ xw, const float *__restrict__ WhT, float *__restrict__ act,
                    float *__restrict__ hprev, float *__restrict__ rh, float *__restrict__ out, int T, int H,
                    int seq, GruPlan pl) {
  extern __shared__ __align__(16) float gsm[];
  const int GB = pl.GB, NQ = pl.NQ, rows = pl.rows, HC = 4 * GB, HP = NQ * rows;
  const int nt = blockDim.x, tid = threadIdx.x, b = blockIdx.x;
  float *hs = gsm, *srh = hs + HP, *us = srh + HP, *xs = us + HC;  // xs[2][3H], 16-byte aligned parts below
  float *part = xs + ((6 * H + 3) & ~3);                           // [NQ][2][HC]
  float4 *Wl = reinterpret_cast<float4 *>(part + NQ * 2 * HC);      // [lrows][GB * NQ]
  const int c = tid % GB, q = tid / GB, k0 = q * rows, np = GB * NQ;
  const bool mv = tid < np;
  float4 wr[RR], wu[RU];
#pragma unroll
  for (int e = 0; e < RR; ++e)
    wr[e] = mv && e < rows ? gru_w4(WhT + H, 2 * H, k0 + e, H, c, H) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int e = 0; e < RU; ++e)
    wu[e] = mv && e < rows ? gru_w4(WhT, 2 * H, k0 + e, H, c, H) : make_float4(0.f, 0.f, 0.f, 0.f);
  if (mv)
    for (int e = 0; e < pl.lrows; ++e)
      Wl[e * np + tid] = gru_w4(WhT, 2 * H, k0 + RU + e, H, c, H);
  for (int i = tid; i < HP; i += nt) hs[i] = srh[i] = 0.0f;  // GRU.Reset (gru.go:171-180); the pad stays 0
  const float *xb = xw + (size_t)b * T * 3 * H;
  for (int i = tid; i < 3 * H; i += nt) xs[i] = xb[i];
  __syncthreads();
  constexpr int NX = BIG ? 6 : 2;  // 3H <= NX * threads
  for (int t = 0; t < T; ++t) {
    const size_t row = (size_t)b * T + t;
    const float *xc = xs + (t & 1) * 3 * H;
    float *xn = xs + ((t & 1) ^ 1) * 3 * H;
    float nx[NX];  // the next step's projections, in flight during this one
    if (t + 1 < T) {
#pragma unroll
      for (int u = 0; u < NX; ++u)
        if (tid + u * nt < 3 * H) nx[u] = xb[(size_t)(t + 1) * 3 * H + tid + u * nt];
    }
    if (mv) {
      float4 su = make_float4(0.f, 0.f, 0.f, 0.f), sr = su;
      // the LDS rows of group g + RU/4 are in flight while the registers of
      // group g are worked
#pragma unroll
      for (int e = 0; e < RU; e += 4) {
        const bool ll = RU + e < RU + pl.lrows;
        float4 wl[4];
        if (ll) {
#pragma unroll
          for (int u = 0; u < 4; ++u) wl[u] = Wl[(e + u) * np + tid];
        }
        if (e < rows) {
          const float4 x = *reinterpret_cast<const float4 *>(hs + k0 + e);
          gru_rows4(sr, wr + e, x);
          gru_rows4(su, wu + e, x);
        }
        if (RU + e < rows && (RU < RR || ll)) {
          const float4 x = *reinterpret_cast<const float4 *>(hs + k0 + RU + e);
          if (RU < RR) gru_rows4(sr, wr + (RU < RR ? RU + e : 0), x);
          if (ll) gru_rows4(su, wl, x);
        }
      }
      if (BIG) {
        gru_stream(su, WhT, 2 * H, k0, RU + pl.lrows, rows, H, c, H, hs);
        gru_stream(sr, WhT + H, 2 * H, k0, RR, rows, H, c, H, hs);
      }
      *reinterpret_cast<float4 *>(part + q * 2 * HC + 4 * c) = su;
      *reinterpret_cast<float4 *>(part + q * 2 * HC + HC + 4 * c) = sr;
    }
    lds_barrier();
    for (int i = tid; i < 2 * H; i += nt) {
      const bool rg = i >= H;
      const int j = rg ? i - H : i;
      const float *p = part + (rg ? HC : 0) + j;
      float s = 0.f;
      for (int k = 0; k < NQ; ++k) s += p[k * 2 * HC];
      const float g = sigmoid_f64(xc[i] + s);
      act[row * 3 * H + i] = g;
      if (rg) {
        const float hi = hs[j], v = g * hi;
        srh[j] = v;
        rh[row * H + j] = v;
        hprev[row * H + j] = hi;
      } else {
        us[j] = g;
      }
    }
    lds_barrier();
    if (mv) {
      float4 sc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int e = 0; e < RR; e += 4)
        if (e < rows) gru_rows4(sc, wr + e, *reinterpret_cast<const float4 *>(srh + k0 + e));
      if (BIG) gru_stream(sc, WhT + H, 2 * H, k0, RR, rows, H, c, H, srh);
      *reinterpret_cast<float4 *>(part + q * 2 * HC + 4 * c) = sc;
    }
    lds_barrier();
    for (int j = tid; j < H; j += nt) {
      float s = 0.f;
      for (int k = 0; k < NQ; ++k) s += part[k * 2 * HC + j];
      const float cv = tanh_f64(xc[2 * H + j] + s);
      act[row * 3 * H + 2 * H + j] = cv;
      const float hi = hs[j], h = hi + us[j] * (cv - hi);
      hs[j] = h;
      if (seq) out[row * H + j] = h;  // returnSequences: every state, [B][T][H]
      else if (t == T - 1) out[(size_t)b * H + j] = h;
    }
    if (t + 1 < T) {
#pragma unroll
      for (int u = 0; u < NX; ++u)
        if (tid + u * nt < 3 * H) xn[tid + u * nt] = nx[u];
    }
    lds_barrier();
  }
}

// g [B][H] = dL/dh_T, or with seq dL/dh_t [B][T][H] added to the carried
// gradient at every step (unroller.go:192-198); act and hprev from the
// forward; Wh [2H][H] as stored; writes dG [B*T][3H].  Of a thread's rows, RW
// sit in registers and the next lrows in LDS; BIG: the rest streams (and a
// thread owns up to 4 hidden units, not 1).
template <int RW, bool BIG>
__global__ __launch_bounds__(GR_NT) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gru_bwd_kernel(const float *__restrict__ g, const float *__restrict__ act, const float *__restrict__ hprev,
                    const float *__restrict__ Wh, float *__restrict__ dG, int T, int H, int seq,
                    GruPlan pl) {
  extern __shared__ __align__(16) float gsm[];
  const int GB = pl.GB, NQ = pl.NQ, rows = pl.rows, HC = 4 * GB, VP = NQ * rows;
  const int nt = blockDim.x, tid = threadIdx.x, b = blockIdx.x;
  float *vs = gsm;                 // [dU | dC r], zero padded to the shares
  float *part = vs + VP;           // [NQ][HC]
  float4 *Wl = reinterpret_cast<float4 *>(part + NQ * HC);
  const int c = tid % GB, q = tid / GB, k0 = q * rows, np = GB * NQ;
  const bool mv = tid < np;
  float4 w[RW];
#pragma unroll
  for (int e = 0; e < RW; ++e)
    w[e] = mv && e < rows ? gru_w4(Wh, H, k0 + e, 2 * H, c, H) : make_float4(0.f, 0.f, 0.f, 0.f);
  if (mv)
    for (int e = 0; e < pl.lrows; ++e) Wl[e * np + tid] = gru_w4(Wh, H, k0 + RW + e, 2 * H, c, H);
  for (int i = tid; i < VP; i += nt) vs[i] = 0.f;
  constexpr int NE = BIG ? 4 : 1;  // hidden units per thread: H <= NE * threads
  float dh[NE], pu[NE], pr[NE], pc[NE], ph[NE], pg[NE];
  auto fetch = [&](int t) {  // step t's saved gates, state and (seq) gradient
#pragma unroll
    for (int n = 0; n < NE; ++n) {
      const int i = tid + n * nt;
      if (i < H) {
        const size_t row = (size_t)b * T + t;
        pu[n] = act[row * 3 * H + i];
        pr[n] = act[row * 3 * H + H + i];
        pc[n] = act[row * 3 * H + 2 * H + i];
        ph[n] = hprev[row * H + i];
        if (seq) pg[n] = g[row * H + i];
      }
    }
  };
#pragma unroll
  for (int n = 0; n < NE; ++n) dh[n] = !seq && tid + n * nt < H ? g[(size_t)b * H + tid + n * nt] : 0.f;
  fetch(T - 1);
  __syncthreads();
  for (int t = T - 1; t >= 0; --t) {
    const size_t row = (size_t)b * T + t;
    float uk[NE];
#pragma unroll
    for (int n = 0; n < NE; ++n) {
      const int i = tid + n * nt;
      if (i < H) {
        if (seq) dh[n] = t < T - 1 ? dh[n] + pg[n] : pg[n];
        const float u = pu[n], cv = pc[n], d = dh[n];
        const float du = d * (cv - ph[n]) * u * (1 - u);
        const float dc = d * (1 - u) * (1 - cv * cv);
        dG[row * 3 * H + i] = du;
        dG[row * 3 * H + H + i] = 0.0f;
        dG[row * 3 * H + 2 * H + i] = dc;
        vs[i] = du;
        vs[H + i] = dc * pr[n];
        uk[n] = u;
      }
    }
    lds_barrier();
    if (t > 0) fetch(t - 1);  // in flight during the product
    if (mv) {
      float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int e = 0; e < RW; e += 4) {
        // an LDS group in flight beside every third register group
        const int l = e / 12 * 4;
        const bool ll = e % 12 == 0 && l < pl.lrows;
        float4 wl[4];
        if (ll) {
#pragma unroll
          for (int u = 0; u < 4; ++u) wl[u] = Wl[(l + u) * np + tid];
        }
        if (e < rows) gru_rows4(s, w + e, *reinterpret_cast<const float4 *>(vs + k0 + e));
        if (ll) gru_rows4(s, wl, *reinterpret_cast<const float4 *>(vs + k0 + RW + l));
      }
      if (BIG) gru_stream(s, Wh, H, k0, RW + pl.lrows, rows, 2 * H, c, H, vs);
      *reinterpret_cast<float4 *>(part + q * HC + 4 * c) = s;
    }
    lds_barrier();
#pragma unroll
    for (int n = 0; n < NE; ++n) {
      const int i = tid + n * nt;
      if (i < H) {
        float s = 0.f;
        for (int k = 0; k < NQ; ++k) s += part[k * HC + i];
        s += dh[n] * uk[n];
        dh[n] += s;
      }
    }
  }
}

bool gru_supported(int H) { return H >= 1 && H <= 1024; }

// Shares: up to 16 of K input rows (fewer where a column group leaves fewer
// of the 512 threads), so small layers keep their partial sums short; rows per
// share a multiple of 4 (16-byte reads of the inputs).
static GruPlan gru_plan(int H, int K) {
  GruPlan p{};
  p.GB = (H + 3) / 4;
  p.NQ = std::max(1, std::min(16, GR_NT / p.GB));
  p.rows = ((K + p.NQ - 1) / p.NQ + 3) & ~3;
  p.NQ = (K + p.rows - 1) / p.rows;
  p.threads = std::max((p.GB * p.NQ + 63) / 64 * 64, std::min(GR_NT, (H + 63) / 64 * 64));
  return p;
}

// LDS for up to `most` of the rows that a thread's registers (`reg` rows) do
// not hold
static void gru_plan_lds(GruPlan &p, int reg, int most, size_t fixed) {
  const size_t row = (size_t)p.GB * p.NQ * sizeof(float4);
  p.lrows = std::min(std::max(p.rows - reg, 0), most);
  while (p.lrows > 0 && fixed + p.lrows * row > (160u << 10)) p.lrows -= 4;
  p.lds = fixed + p.lrows * row;
}

template <int RR, int RU, bool BIG = false>
static hipError_t gru_fwd_launch(GruPlan p, const float *xw, const float *WhT, float *act, float *hprev, float *rh,
                                 float *out, int B, int T, int H, hipStream_t s, int seq) {
  const int HC = 4 * p.GB, HP = p.NQ * p.rows;
  gru_plan_lds(p, RU, RU, (size_t)(2 * HP + HC + ((6 * H + 3) & ~3) + p.NQ * 2 * HC) * sizeof(float));
  static std::atomic<int> attr[kAttrDevices];
  const hipError_t e = ensure_lds_attr(reinterpret_cast<const void *>(gru_fwd_kernel<RR, RU, BIG>), (int)p.lds, attr);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((gru_fwd_kernel<RR, RU, BIG>), dim3(B), dim3(p.threads), p.lds, s, xw, WhT, act, hprev, rh, out, T,
                     H, seq, p);
  return hipGetLastError();
}

hipError_t launch_gru_fwd(const float *xw, const float *WhT, float *act, float *hprev, float *rh,
                          float *out, int B, int T, int H, hipStream_t s, int seq) {
  if (!gru_supported(H)) return hipErrorInvalidValue;
  const GruPlan p = gru_plan(H, H);
  if (p.rows <= 4) return gru_fwd_launch<4, 4>(p, xw, WhT, act, hprev, rh, out, B, T, H, s, seq);
  if (p.rows <= 8) return gru_fwd_launch<8, 8>(p, xw, WhT, act, hprev, rh, out, B, T, H, s, seq);
  if (p.rows <= 16) return gru_fwd_launch<16, 16>(p, xw, WhT, act, hprev, rh, out, B, T, H, s, seq);
  if (H <= 256) return gru_fwd_launch<32, 16>(p, xw, WhT, act, hprev, rh, out, B, T, H, s, seq);
  return gru_fwd_launch<16, 8, true>(p, xw, WhT, act, hprev, rh, out, B, T, H, s, seq);
}

template <int RW, bool BIG = false>
static hipError_t gru_bwd_launch(GruPlan p, const float *g, const float *act, const float *hprev, const float *Wh,
                                 float *dG, int B, int T, int H, hipStream_t s, int seq) {
  const int HC = 4 * p.GB, VP = p.NQ * p.rows;
  gru_plan_lds(p, RW, RW / 12 * 4, (size_t)(VP + p.NQ * HC) * sizeof(float));
  static std::atomic<int> attr[kAttrDevices];
  const hipError_t e = ensure_lds_attr(reinterpret_cast<const void *>(gru_bwd_kernel<RW, BIG>), (int)p.lds, attr);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((gru_bwd_kernel<RW, BIG>), dim3(B), dim3(p.threads), p.lds, s, g, act, hprev, Wh, dG, T, H, seq, p);
  return hipGetLastError();
}

hipError_t launch_gru_bwd(const float *g, const float *act, const float *hprev, const float *Wh,
                          float *dG, int B, int T, int H, hipStream_t s, int seq) {
  if (!gru_supported(H)) return hipErrorInvalidValue;
  const GruPlan p = gru_plan(H, 2 * H);
  if (p.rows <= 8) return gru_bwd_launch<8>(p, g, act, hprev, Wh, dG, B, T, H, s, seq);
  if (p.rows <= 16) return gru_bwd_launch<16>(p, g, act, hprev, Wh, dG, B, T, H, s, seq);
  if (p.rows <= 32) return gru_bwd_launch<32>(p, g, act, hprev, Wh, dG, B, T, H, s, seq);
  if (H <= 256) return gru_bwd_launch<48>(p, g, act, hprev, Wh, dG, B, T, H, s, seq);
  return gru_bwd_launch<24, true>(p, g, act, hprev, Wh, dG, B, T, H, s, seq);
}

}  // namespace gn
