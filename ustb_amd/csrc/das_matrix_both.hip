// das_matrix_both.hip — dimension both of the matrix contract outside das_c's
// summation order: out[f][p] = sum_w sum_n of das_c's terms, grouped by
// channel.
//
// A block is one tile of 64 consecutive pixels (lanes) x kWS wave64s. The
// tile's waves with a nonzero weight are listed first (ballots, ascending);
// each wave64 holds kWC of them, delay and weight in VGPRs, and runs over the
// channels, whose delay and weight are then read once for kWC waves instead
// of once per wave. Where the waves need fewer than kWS wave64s, the rest
// take shares of the channels. The partial sums are added in a fixed order.
//
// Phase. das_c rotates a term by exp(i p), p = fl32(wd * c), c = fl32(td +
// rd) (das_c.cpp:372, 383-387). With exact FP32 error terms, c = td + rd - e
// (two-sum) and p = wd c - r (one FMA), so p = wd td + wd rd - (r + wd e): the
// rotation is exp(i wd td) exp(i wd rd) exp(i D), D = -(r + wd e), |D| below
// 2^-23 |p|. The first two are formed once per (pixel, wave) and (pixel,
// channel) with the FP64 argument of sincos_wd, the last to second order: up to
// |p| = 32768, |D| < 2^-8, what that leaves out is below 1e-8, a sixth of the
// rounding of the rotation itself. So a term keeps das_c's rounded phase (the
// result is das_c's within FP32 rounding) at 11 instructions instead of a sine
// and cosine of an unreduced argument (about 45). A tile with larger phases is
// summed from das_c's own terms (dasc_sum).
//
// Bound by latency (the waves wait 46 % of their cycles; about 35 VALU instructions
// per 64 terms take 32-64 % of the issue slots, 25 waves 25 of 32 wave slots). Against
// das_matrix_kernel, whose lanes take a sine, a cosine and two branches per
// term and read the receive rows once per wave (128 channels, 256 x 256 pixels,
// IQ): 25 waves 0.401 -> 0.180 ms, 16 0.264 -> 0.099, 8 0.135 -> 0.057, 4 0.071
// -> 0.035, 2 0.039 -> 0.033; 25 waves cubic 0.418 -> 0.223; 9 waves x 5 frames
// 0.734 -> 0.292. One wave stays there (0.022 against 0.033 ms: nothing to
// share, and its deeper row loads count).
#include "das_launch.h"
#include "das_rxtab.h"

namespace ustbx {

namespace {

constexpr int kWS = 4;        // wave64s per block
constexpr int kWC = 8;        // waves held by a wave64 per round
constexpr int kMaxList = 2048;  // waves of a call (the tile's list in LDS)

struct MatBoth {
  const void* ch;
  const float* tx_apo;
  const float* rx_apo;
  const float* tx_delay;
  const float* rx_delay;
  float2* out;
  int L, N, W, F, P;
  float fs, t0, wd, lo;
  int frame_bytes, edge;
};

// exp(i D) T for das_c's phase of the term (see above); d0 receives c.
__device__ __forceinline__ float2 dasc_rotation(float2 T, float td, float rd, float wd, float c) {
#pragma clang fp contract(off)
  const float t = c - td;
  const float e = (td - (c - t)) + (rd - t);      // td + rd = c + e
  const float p = wd * c;
  const float r = __builtin_fmaf(wd, c, -p);      // wd c = p + r
  const float D = -__builtin_fmaf(wd, e, r);
  const float h = __builtin_fmaf(-0.5f * D, D, 1.0f);
  return make_float2(__builtin_fmaf(-D, T.y, h * T.x), __builtin_fmaf(D, T.x, h * T.y));
}

constexpr float kNearPhase = 32768.0f;  // rad: |D| < 2^-8

// The channels n = s, s + kWS, ... of pixel p summed from das_c's terms
// (das_c.cpp:366-399), for tiles outside the range of the split rotation or
// with sums that are not finite.
template <int SM, bool IQ, int FC>
__device__ __forceinline__ void dasc_sum(const MatBoth& A, const int* list, int nw, int s, unsigned p, int f0, int nfr,
                                         float2 (&acc)[FC]) {
  constexpr int INTERP = SM == SM_CUBIC ? INTERP_CUBIC : INTERP_LINEAR;
  const size_t PS = (size_t)A.P, LN = (size_t)A.L * A.N;
#pragma unroll
  for (int f = 0; f < FC; ++f) acc[f] = make_float2(0.0f, 0.0f);
#pragma unroll 1
  for (int n = s; n < A.N; n += kWS) {
    const float ra = (A.rx_apo + (size_t)n * PS)[p], rd = (A.rx_delay + (size_t)n * PS)[p];
    if (!__any(ra != 0.0f)) continue;
#pragma unroll 1
    for (int k = 0; k < nw; ++k) {
      const int w = __builtin_amdgcn_readfirstlane(list[k]);
      const float ta = (A.tx_apo + (size_t)w * PS)[p], td = (A.tx_delay + (size_t)w * PS)[p];
      if (ta != 0.0f && ra != 0.0f) {
        const Term t = dasc_term<INTERP, IQ>(td, rd, ta, ra, A.t0, A.fs, A.wd, A.L, A.edge);
        if (t.valid) {
          const float2* trace = reinterpret_cast<const float2*>(A.ch) + (size_t)f0 * LN * A.W + (size_t)w * LN + (size_t)n * A.L;
#pragma unroll
          for (int f = 0; f < FC; ++f)
            if (f < nfr) cadd(acc[f], mat_contrib<INTERP>(t, trace + (size_t)f * LN * A.W));
        }
      }
    }
  }
}

template <int SM, bool IQ, int FC>
__global__ __launch_bounds__(64 * kWS) void das_matrix_both_kernel(MatBoth A) {
  constexpr int NL = SM == SM_CUBIC ? 2 : 1;
  __shared__ float2 red[kWS][64];
  __shared__ int list[kMaxList];
  __shared__ int count;
  __shared__ int far_tile, redo;
  const int lane = threadIdx.x & 63;
  const int s = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int tile = xcd_tile((int)blockIdx.x, (int)gridDim.x);
  const int pp = tile * 64 + lane;
  const bool active = pp < A.P;
  const unsigned p = (unsigned)min(pp, A.P - 1);  // lanes past the end repeat the last pixel
  const size_t PS = (size_t)A.P;
  const int f0 = (int)blockIdx.y * FC;
  const int nfr = min(FC, A.F - f0);

  // the waves with a nonzero weight on some pixel of the tile, ascending
  for (int w = s; w < A.W; w += kWS) {
    const bool any = __any((A.tx_apo + (size_t)w * PS)[p] != 0.0f);
    if (lane == 0) list[w] = any ? 1 : 0;
  }
  __syncthreads();
  if (s == 0) {
    int n = 0;
    for (int b = 0; b < A.W; b += 64) {
      const bool on = b + lane < A.W && list[b + lane] != 0;
      const unsigned long long m = __ballot(on);
      // entry n + k <= b + lane: written after every lane of this step has read
      __builtin_amdgcn_wave_barrier();
      if (on) list[n + __popcll(m & ((1ull << lane) - 1ull))] = b + lane;
      n += __popcll(m);
    }
    if (lane == 0) {
      count = n;
      far_tile = redo = 0;
    }
  }
  __syncthreads();
  const int nw = __builtin_amdgcn_readfirstlane(count);

  __amdgpu_buffer_rsrc_t rs[FC];
#pragma unroll
  for (int f = 0; f < FC; ++f)
    rs[f] = make_rsrc((const char*)A.ch + (size_t)(f0 + min(f, nfr - 1)) * (size_t)A.frame_bytes, A.frame_bytes);
  const int lst = A.L * 8, wst = lst * A.N;
  const float lim = (float)(SM == SM_LINEAR ? A.L - 1 : A.L - 2);
  const float t0 = A.t0, fs = A.fs, wd = A.wd, lo = A.lo;

  // wave64s per channel group, channel groups (as rxtab_tile)
  const int wneed = (nw + kWC - 1) / kWC;
  const int cg = (wneed > 0 && wneed < kWS) ? kWS / wneed : 1;
  const int wsp = cg > 1 ? wneed : kWS;
  const int g = s / wsp, sw = s - g * wsp;

  float2 acc[FC];
#pragma unroll
  for (int f = 0; f < FC; ++f) acc[f] = make_float2(0.0f, 0.0f);
  bool far = false;  // wave-uniform: a phase beyond the split rotation's range
  for (int k0 = 0; g < cg && k0 < nw && !far; k0 += wsp * kWC) {
    const int nj = __builtin_amdgcn_readfirstlane(min(kWC, max(0, (nw - k0 - sw + wsp - 1) / wsp)));
    if (nj == 0) break;
    float td[kWC];
    float2 T[kWC];
    int wb[kWC];
    float tmax = 0.0f;  // largest |delay| of the round's waves
#pragma unroll
    for (int j = 0; j < kWC; ++j) {
      td[j] = kFar;
      T[j] = make_float2(0.0f, 0.0f);
      wb[j] = 0;
      if (j < nj) {
        const int w = __builtin_amdgcn_readfirstlane(list[k0 + sw + wsp * j]);
        wb[j] = w * wst;
        const float ta = (A.tx_apo + (size_t)w * PS)[p], d = (A.tx_delay + (size_t)w * PS)[p];
        if (ta != 0.0f) {
          td[j] = d;
          if (IQ) tmax = fmaxf(tmax, fabsf(d));
          float sv = 0.0f, cv = 1.0f;
          if (IQ) sincos_wd(wd, d, sv, cv);
          T[j] = make_float2(ta * cv, IQ ? ta * sv : 0.0f);
        }
      }
    }
    // the next channel's receive rows are in flight during this one's terms
    float ran = (A.rx_apo + (size_t)min(g, A.N - 1) * PS)[p], rdn = (A.rx_delay + (size_t)min(g, A.N - 1) * PS)[p];
    // a test here spares most far tiles the round; one per channel costs 3 %
    float rmax = ran != 0.0f ? fabsf(rdn) : 0.0f;
    if (IQ) {
      far = __any(fabsf(wd) * (tmax + rmax) > kNearPhase);
      if (far) break;
    }
    for (int n = g; n < A.N; n += cg) {
      const float ra = ran, rdv = rdn;
      const size_t nx = (size_t)min(n + cg, A.N - 1) * PS;
      ran = (A.rx_apo + nx)[p];
      rdn = (A.rx_delay + nx)[p];
      const bool ron = ra != 0.0f;
      if (!__any(ron)) continue;  // wave-uniform
      if (IQ) rmax = ron ? fmaxf(rmax, fabsf(rdv)) : rmax;
      const float rd = ron ? rdv : kFar;
      const int nb = n * lst;
      float2 part[FC];
#pragma unroll
      for (int f = 0; f < FC; ++f) part[f] = make_float2(0.0f, 0.0f);
      bool any = false;
      constexpr int RB = FC == 1 ? 4 : 1;  // terms whose gathers are issued together
#pragma unroll
      for (int j0 = 0; j0 < kWC; j0 += RB) {
        if (j0 < nj) {
          float4 x[RB][FC][NL];
          float b[RB], c[RB];
          bool ok[RB];
#pragma unroll
          for (int i = 0; i < RB; ++i) {
            const int j = j0 + i;
            float d;
            {
#pragma clang fp contract(off)
              c[i] = td[j] + rd;      // das_c.cpp:372
              d = (c[i] - t0) * fs;   // das_c.cpp:375
            }
            ok[i] = d >= lo && d < lim;
            b[i] = __builtin_amdgcn_fractf(d);
            const int off = ok[i] ? (int)d * 8 + (nb + wb[j] - (SM == SM_CUBIC ? 8 : 0)) : kOOB;
#pragma unroll
            for (int f = 0; f < FC; ++f) {
              x[i][f][0] = buf_load16(rs[f], off);
              if (NL == 2) x[i][f][NL - 1] = buf_load16(rs[f], off + 16);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < RB; ++i) {
            const int j = j0 + i;
            const float2 w = IQ ? dasc_rotation(T[j], ok[i] ? td[j] : 0.0f, ok[i] ? rd : 0.0f, wd, ok[i] ? c[i] : 0.0f)
                                : T[j];
            float k0w = 0.f, k1w = 0.f, k2w = 0.f, k3w = 0.f;
            if (SM == SM_CUBIC) keys_weights_horner(b[i], k0w, k1w, k2w, k3w);
#pragma unroll
            for (int f = 0; f < FC; ++f) {
              float2 sm;
              const float4 q = x[i][f][0];
              if (SM == SM_LINEAR) {
                sm = make_float2(fmaf(b[i], q.z - q.x, q.x), fmaf(b[i], q.w - q.y, q.y));
              } else {
                const float4 h = x[i][f][NL - 1];
                sm = make_float2(fmaf(k3w, h.z, fmaf(k2w, h.x, fmaf(k1w, q.z, k0w * q.x))),
                                 fmaf(k3w, h.w, fmaf(k2w, h.y, fmaf(k1w, q.w, k0w * q.y))));
              }
              float2 v = part[f];
              cfma(v, w, sm);
              part[f] = ok[i] ? v : part[f];  // das_c skips the others before it multiplies
            }
            any = any || ok[i];
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      float sv = 0.0f, cv = 1.0f;
      if (IQ) sincos_wd_hw(wd, any ? rdv : 0.0f, sv, cv);
      const float2 R = make_float2(ra * cv, IQ ? ra * sv : 0.0f);
#pragma unroll
      for (int f = 0; f < FC; ++f) {
        float2 v = acc[f];
        cfma(v, R, part[f]);
        acc[f] = any ? v : acc[f];
      }
    }
    if (IQ) far = __any(fabsf(wd) * (tmax + rmax) > kNearPhase);
  }
  if (IQ) {
    if (far && lane == 0) far_tile = 1;
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(far_tile)) dasc_sum<SM, IQ, FC>(A, list, nw, s, p, f0, nfr, acc);
  }
#pragma unroll
  for (int f = 0; f < FC; ++f) {
    red[s][lane] = acc[f];
    __syncthreads();
    if (s == 0 && active && f < nfr) {
      float2 v = red[0][lane];
#pragma unroll
      for (int k = 1; k < kWS; ++k) cadd(v, red[k][lane]);
      A.out[(size_t)(f0 + f) * PS + p] = v;
      if (!(isfinite(v.x) && isfinite(v.y))) redo = 1;
    }
    __syncthreads();
  }
  // Infinities: the split weights and x0 + b (x1 - x0) turn some into NaN that
  // das_c's products keep, and weights far from 1 can overflow in between.
  // Sums that are not finite are das_c's.
  if (__builtin_amdgcn_readfirstlane(redo)) {
    dasc_sum<SM, IQ, FC>(A, list, nw, s, p, f0, nfr, acc);
#pragma unroll
    for (int f = 0; f < FC; ++f) {
      red[s][lane] = acc[f];
      __syncthreads();
      if (s == 0 && active && f < nfr) {
        float2* o = A.out + (size_t)(f0 + f) * PS + p;
        if (!(isfinite(o->x) && isfinite(o->y))) {
          float2 v = red[0][lane];
#pragma unroll
          for (int k = 1; k < kWS; ++k) cadd(v, red[k][lane]);
          *o = v;
        }
      }
      __syncthreads();
    }
  }
}

template <int SM, bool IQ>
hipError_t matrix_both_t(const MatBoth& A, hipStream_t s) {
  const unsigned tiles = (unsigned)((A.P + 63) / 64);
  if (A.F == 1)
    hipLaunchKernelGGL((das_matrix_both_kernel<SM, IQ, 1>), dim3(tiles, 1u), dim3(64 * kWS), 0, s, A);
  else
    hipLaunchKernelGGL((das_matrix_both_kernel<SM, IQ, 4>), dim3(tiles, (unsigned)((A.F + 3) / 4)), dim3(64 * kWS), 0, s,
                       A);
  return hipGetLastError();
}

}  // namespace

bool matrix_both_applies(const MatLaunch& m) {
  return m.dim == 3 && !m.py && m.W >= 2 && m.W <= kMaxList && m.L >= 4 && (int64_t)m.L * m.N * m.W * 8 <= 0x7FFFFE00;
}

hipError_t launch_das_matrix_both(const MatLaunch& m, hipStream_t s) {
  MatBoth A;
  A.ch = m.ch;
  A.tx_apo = m.tx_apo;
  A.rx_apo = m.rx_apo;
  A.tx_delay = m.tx_delay;
  A.rx_delay = m.rx_delay;
  A.out = reinterpret_cast<float2*>(m.out);
  A.L = m.L;
  A.N = m.N;
  A.W = m.W;
  A.F = m.F;
  A.P = m.P;
  A.fs = m.fs;
  A.t0 = m.t0;
  A.wd = m.wd;
  A.lo = m.edge == EDGE_PYTHON && m.interp == INTERP_LINEAR ? 0.0f : 1.0f;
  A.frame_bytes = m.L * m.N * m.W * 8;
  A.edge = m.edge;
  if (m.interp == INTERP_CUBIC)
    return m.wd != 0.0f ? matrix_both_t<SM_CUBIC, true>(A, s) : matrix_both_t<SM_CUBIC, false>(A, s);
  return m.wd != 0.0f ? matrix_both_t<SM_LINEAR, true>(A, s) : matrix_both_t<SM_LINEAR, false>(A, s);
}

}  // namespace ustbx
