// demodulate.hip — RF -> IQ on the device: preprocess.fast_demodulation
// (+preprocess/fast_demodulation.m:58-183) and the Python reference's
// FastDemodulation (python/src/ustb/preprocess/fast_demodulation.py:24-85).
//
// Both are: mix each trace by exp(-1j 2 pi fmod t), t = t0 + n / fs (the
// phase in FP64, the factor rounded to FP32 and multiplied in FP32 as MATLAB
// does with single data); low-pass FIR; keep every down-th sample from the
// first. The two filters differ:
//  - causal (MATLAB filter(b, 1, x) with zero initial state): taps at offsets
//    -(K-1) .. 0, samples before the trace are zero;
//  - zero-phase (scipy filtfilt(b, 1, x) with its odd extension of 3K
//    samples): on the cropped output the forward and backward passes never
//    reach the extension's ends, so the result is one FIR with the taps'
//    autocorrelation c[d] = sum_k b[k] b[k+d], d = -(K-1) .. K-1, over the
//    odd-extended signal (2 e[0] - e[-m] before the start, 2 e[L-1] -
//    e[2L-2-m] after the end).
//
// The mixing factors depend on the sample index only: they are computed once
// per (device, L, fs, t0, fmod) into a small device table that later calls
// reuse. One block per (trace, run of up to R * kDB outputs) stages the
// mixed samples of its input window in LDS, split by decimation phase
// (phase r holds window samples r, r + down, ...; one pad slot every R
// entries, so the lanes' reads, R entries apart, hit distinct banks). Each
// lane forms R consecutive outputs (R = 8 without decimation, 4 with): per
// phase, a window of R samples slides along the phase's taps in registers, so
// every staged sample a lane needs is read once. The sum runs phase by phase
// (within a phase in tap order), whatever R is.
//
// The kernel's time is VALU issue next to HBM, so what is not a multiply-add
// is kept off it: the decimation is a template argument at 1 and 2 (else a
// multiplication by its inverse), samples outside a causal filter's trace come
// as zeros from a buffer load's bounds check, taps lie phase by phase in the
// kernel's arguments and come as scalars. 16384 traces of 2048 samples: 86 ->
// 68 us at decimation 2 with the standard low-pass (53 us is a copy of the
// bytes); with 21 taps at decimation 1, 2, 3 and 4 causal 200 -> 128, 74 -> 55,
// 76 -> 59 and 98 -> 72 us, zero-phase 201 -> 130, 84 -> 70, 92 -> 78 and 122 ->
// 102 us. A scalar load's wait is a wait for every LDS read before it, so long
// filters at decimation 1, whose time is the tap loop, read their taps from LDS,
// eight at a time: zero-phase 65 taps 175 -> 161 us, 129 247 -> 210, 257 470 -> 375;
// causal 65 taps 138 -> 136, 129 240 -> 203; 57 and fewer 0-20 % slower, mostly on
// few traces. The sums are the same bits.
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>

#include "das_common.h"
#include "das_status.h"

namespace ustbx {

namespace {

constexpr int kDB = 256;         // threads per block
// window samples a lane loads per staging round: 9 x 256 covers the window of
// 1024 outputs at decimation 2, or 2048 at decimation 1, with up to 241 taps
// in one round, so a block waits for memory once (8: two rounds, 12 % slower
// on 128 x 128 traces of 2048 samples, 31 taps, decimation 2)
constexpr int kSB = 9;
constexpr int kMaxTaps = 767;    // passed by value (kernel arguments stay under 4 KB); zero-phase: K <= 384
constexpr size_t kLdsMax = 64 * 1024;
constexpr int kLdsTaps = 64;     // decimation 1: from here on the taps lie in LDS

struct DemodArgs {
  const float* rf;
  const float2* mix;   // [L] mixing factors
  float2* out;
  int L, Lout, down, ntaps, off0, OB;
  int PS;              // LDS entries per phase (padded)
  unsigned inv;        // ceil(2^32 / down)
  float taps[kMaxTaps];  // phase by phase: taps r, r + down, ... of phase r
};

// entries of one phase for m window samples (one pad slot per R) and the LDS
// that a block of OB outputs may take (samples, and room for the taps)
inline int phase_slots(int mr, int R) { return mr + mr / R + 1; }
inline int phase_len(int OB, int down, int T, int R) {
  const int count = (OB - 1) * down + T;
  return (count + down - 1) / down + 2 * R;
}
inline size_t demod_lds(int OB, int down, int T, int R) {
  return sizeof(float2) * (size_t)down * phase_slots(phase_len(OB, down, T, R), R) +
         sizeof(float) * (size_t)(T + (R + 1) * down);
}

__global__ __launch_bounds__(kDB) void mix_table_kernel(float2* __restrict__ tab, int L, double fs, double t0,
                                                        double fmod) {
#pragma clang fp contract(off)
  const int m = blockIdx.x * kDB + threadIdx.x;
  if (m >= L) return;
  const double t = t0 + (double)m / fs;
  const double ph = ((-2.0 * M_PI) * fmod) * t;
  double s, c;
  sincos(ph, &s, &c);
  tab[m] = make_float2((float)c, (float)s);
}

// mixed sample e[m] of the trace, m in [0, L)
__device__ __forceinline__ float2 mixed(const float* __restrict__ x, int m, const DemodArgs& A) {
  const float v = x[m];
  const float2 e = A.mix[m];
  return make_float2(v * e.x, v * e.y);
}

// two complex outputs in one store, at the alignment of one
typedef float out4 __attribute__((ext_vector_type(4), aligned(8)));

template <int kR, int DOWN, bool ZP, bool LT = false>
__global__ __launch_bounds__(kDB) void demodulate_kernel(DemodArgs A) {
  extern __shared__ float2 lds[];
  const int down = DOWN ? DOWN : A.down, T = A.ntaps, PS = A.PS;
  const int tid = (int)threadIdx.x;
  const size_t trace = blockIdx.x;
  const float* __restrict__ x = A.rf + trace * (size_t)A.L;
  const int j0 = (int)blockIdx.y * A.OB;
  const int jn = min(A.OB, A.Lout - j0);
  const int lo = j0 * down + A.off0;            // extended index of window sample 0
  const int count = (jn - 1) * down + T;        // window samples the outputs read
  // Window sample i (extended index lo + i) goes to phase i mod down, entry
  // i / down. Each lane issues kSB loads per round, all in bounds (zero phase:
  // an index outside the trace reads its odd-extension reflection) or answered
  // with zero (causal), then forms and stores the samples. What the window
  // does not hold stays unwritten: only outputs that are not stored read it.
  float2 e0 = make_float2(0.0f, 0.0f), e1 = e0;
  if (ZP) {
    e0 = mixed(x, 0, A);
    e1 = mixed(x, A.L - 1, A);
  }
  const int bs = max(lo, 0), n = min(A.L, lo + count) - bs;  // the trace's samples in the window: n >= 1
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(x + bs, n * 4), rm = make_rsrc(A.mix + bs, n * 8);
  for (int base = 0; base < count; base += kSB * kDB) {
    float xv[kSB];
    float2 mv[kSB];
#pragma unroll
    for (int k = 0; k < kSB; ++k) {
      const int i = base + k * kDB + tid;
      const int m = lo + i;
      if (ZP) {
        int src = m;
        const int c0 = lo + base + k * kDB;
        if (c0 < 0 || c0 + kDB > A.L) {
          src = m < 0 ? -m : (m >= A.L ? 2 * A.L - 2 - m : m);
          // lanes past the window read the window's first sample (unused)
          src = i < count ? min(max(src, 0), A.L - 1) : min(bs, A.L - 1);
        }
        xv[k] = x[src];
        mv[k] = A.mix[src];
      } else {
        const int q = m < 0 ? 0x0FFFFFF0 : m - bs;  // past the end, also times 8
        xv[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, q * 4, 0, 0));
        mv[k] = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(rm, q * 8, 0, 0));
      }
    }
#pragma unroll
    for (int k = 0; k < kSB; ++k) {
      const int i = base + k * kDB + tid;
      if (i < count) {
#pragma clang fp contract(off)
        const int m = lo + i;
        float2 v = make_float2(xv[k] * mv[k].x, xv[k] * mv[k].y);
        if (ZP && (m < 0 || m >= A.L)) {
          const float2 edge = m < 0 ? e0 : e1;
          v = make_float2(2.0f * edge.x - v.x, 2.0f * edge.y - v.y);
        }
        const unsigned q = DOWN ? (unsigned)i / (unsigned)(DOWN ? DOWN : 1) : __umulhi((unsigned)i, A.inv);
        lds[(size_t)((unsigned)i - q * (unsigned)down) * PS + q + q / kR] = v;
      }
    }
  }
  // LT: the taps beside the samples, for lanes to read together
  const float* tl = reinterpret_cast<const float*>(lds + ((down * PS + 1) & ~1));
  if (LT)
    for (int i = tid; i < T; i += kDB) const_cast<float*>(tl)[i] = A.taps[i];
  __syncthreads();
  const int jt = kR * tid;                      // first output of this lane (block-local)
  if (jt >= jn) return;
  float2 acc[kR];
#pragma unroll
  for (int k = 0; k < kR; ++k) acc[k] = make_float2(0.0f, 0.0f);
  int tq = 0;                                   // the phase's first tap
  for (int r = 0; r < down; ++r) {
    const float2* __restrict__ p = lds + (size_t)r * PS + (kR + 1) * tid;
    const int Q = (T - r + down - 1) / down;    // taps r, r + down, ... of this phase
    // w[s] holds phase sample jt + q0 + s at the start of each block of kR taps
    float2 w[kR];
#pragma unroll
    for (int k = 0; k < kR; ++k) w[k] = p[k];
    auto tap = [&](int q, int u) {
      const float t = LT ? tl[tq + q + u] : A.taps[tq + q + u];
#pragma unroll
      for (int k = 0; k < kR; ++k) {
        const float2 s = w[(u + k) % kR];
        acc[k].x = fmaf(t, s.x, acc[k].x);
        acc[k].y = fmaf(t, s.y, acc[k].y);
      }
      w[u] = p[u];
    };
    int q0 = 0;
    for (; q0 + kR <= Q; q0 += kR) {
      p += kR + 1;
#pragma unroll
      for (int u = 0; u < kR; ++u) tap(q0, u);
    }
    p += kR + 1;
#pragma unroll
    for (int u = 0; u < kR - 1; ++u)
      if (q0 + u < Q) tap(q0, u);               // uniform
    tq += Q;
  }
  float2* __restrict__ o = A.out + trace * (size_t)A.Lout + j0 + jt;
  if (jt + kR <= jn) {
#pragma unroll
    for (int k = 0; k < kR; k += 2) *(out4*)(o + k) = out4{acc[k].x, acc[k].y, acc[k + 1].x, acc[k + 1].y};
  } else {
#pragma unroll
    for (int k = 0; k < kR; ++k)
      if (jt + k < jn) o[k] = acc[k];
  }
}

struct MixTable {
  float2* tab = nullptr;
  unsigned long long last_use = 0;
};

std::mutex g_mu;
std::map<std::tuple<int, int, double, double, double>, MixTable> g_mix;
unsigned long long g_mix_clock = 0;
// tables kept per device; the least recently used one is released (after the
// device has finished its queued work) to make room for a new one
constexpr int kMaxMixTables = 64;

hipError_t evict_mix(int dev) {
  for (;;) {
    int n = 0;
    auto lru = g_mix.end();
    for (auto it = g_mix.begin(); it != g_mix.end(); ++it) {
      if (std::get<0>(it->first) != dev) continue;
      ++n;
      if (lru == g_mix.end() || it->second.last_use < lru->second.last_use) lru = it;
    }
    if (n < kMaxMixTables) return hipSuccess;
    const hipError_t e = hipDeviceSynchronize();  // no queued work still reads it
    if (e != hipSuccess) return e;
    (void)hipFree(lru->second.tab);
    g_mix.erase(lru);
  }
}

// The mixing-factor table of (device, L, fs, t0, fmod), built on first use on
// the caller's stream (and waited for, so that other streams may read it).
// The caller holds g_mu until it has launched the kernel that reads the
// table, so that no other call releases the table before that launch.
int mix_table(int L, double fs, double t0, double fmod, hipStream_t s, const float2** out, ustbx_status* st) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(st, e, "hipGetDevice");
  const auto key = std::make_tuple(dev, L, fs, t0, fmod);
  auto it = g_mix.find(key);
  if (it != g_mix.end()) {
    it->second.last_use = ++g_mix_clock;
    *out = it->second.tab;
    return ok(st);
  }
  e = evict_mix(dev);
  if (e != hipSuccess) return hip_fail(st, e, "releasing a mixing-factor table");
  float2* tab = nullptr;
  e = hipMalloc(&tab, sizeof(float2) * (size_t)L);
  if (e != hipSuccess) return hip_fail(st, e, "hipMalloc (mixing factors)");
  hipLaunchKernelGGL(mix_table_kernel, dim3((unsigned)((L + kDB - 1) / kDB)), dim3(kDB), 0, s, tab, L, fs, t0, fmod);
  e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    (void)hipFree(tab);
    return hip_fail(st, e, "mixing factors");
  }
  g_mix.emplace(key, MixTable{tab, ++g_mix_clock});
  *out = tab;
  return ok(st);
}

}  // namespace
}  // namespace ustbx

using namespace ustbx;

extern "C" {

int ustbx_demodulate(const float* rf, void* iq, int32_t L, int64_t traces, double fs, double t0, double fmod,
                     const double* b, int32_t ntaps, int32_t down, int32_t mode, void* stream, ustbx_status* st) {
  if (mode != USTBX_FIR_CAUSAL && mode != USTBX_FIR_ZERO_PHASE)
    return set_status(st, USTBX_E_ARG, "mode must be USTBX_FIR_CAUSAL or USTBX_FIR_ZERO_PHASE");
  if (L < 0 || traces < 0) return set_status(st, USTBX_E_ARG, "negative size");
  if (!b || ntaps < 1) return set_status(st, USTBX_E_ARG, "the filter needs at least one tap");
  if (down < 1) return set_status(st, USTBX_E_ARG, "the decimation factor must be at least 1");
  if (!(fs > 0.0)) return set_status(st, USTBX_E_ARG, "the sampling frequency must be positive");
  const int K = ntaps;
  const int T = mode == USTBX_FIR_CAUSAL ? K : 2 * K - 1;
  if (T > kMaxTaps)
    return set_status(st, USTBX_E_ARG, "at most %d taps", mode == USTBX_FIR_CAUSAL ? kMaxTaps : (kMaxTaps + 1) / 2);
  if (mode == USTBX_FIR_ZERO_PHASE && L <= 3 * K)
    return set_status(st, USTBX_E_ARG, "The length of the input vector x must be greater than padlen, which is %d.",
                      3 * K);
  if (L == 0 || traces == 0) return ok(st);
  if (traces > 0x7FFFFFFF) return set_status(st, USTBX_E_ARG, "too many traces");
  if (!rf || !iq) return set_status(st, USTBX_E_ARG, "NULL buffer");
  // outputs per lane: 8 halves the LDS reads per FMA (the zero-phase form,
  // decimation 1, is VALU-bound: 14 % faster than 4); with decimation the
  // traces have fewer outputs (1024 of 2048 samples at 2), which 4 per lane
  // spreads over every lane of a block
  const int R = down == 1 ? 8 : 4;
  // outputs per block: R per lane, fewer where the window would not fit in LDS
  int OB = R * kDB;
  while (OB > R && demod_lds(OB, down, T, R) > kLdsMax) OB /= 2;
  if (demod_lds(OB, down, T, R) > kLdsMax)
    return set_status(st, USTBX_E_ARG, "decimation factor too large for the filter");
  // taps in FP32 (MATLAB filter runs in the data's single precision); the
  // zero-phase form's autocorrelation is formed in FP64 first
  DemodArgs A;
  float taps[kMaxTaps];
  if (mode == USTBX_FIR_CAUSAL) {
    for (int i = 0; i < K; ++i) taps[i] = (float)b[K - 1 - i];  // offsets -(K-1) .. 0
  } else {
    for (int d = -(K - 1); d <= K - 1; ++d) {
      double c = 0.0;
      for (int k = 0; k < K; ++k)
        if (k + d >= 0 && k + d < K) c += b[k] * b[k + d];
      taps[d + K - 1] = (float)c;
    }
  }
  for (int r = 0, n = 0; r < down; ++r)
    for (int i = r; i < T; i += down) A.taps[n++] = taps[i];
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const float2* mix = nullptr;
  std::lock_guard<std::mutex> lock(g_mu);  // held through the launch that reads the table
  const int rc = mix_table(L, fs, t0, fmod, s, &mix, st);
  if (rc != USTBX_OK) return rc;
  A.rf = rf;
  A.mix = mix;
  A.out = reinterpret_cast<float2*>(iq);
  A.L = L;
  A.Lout = (L + down - 1) / down;
  A.down = down;
  A.ntaps = T;
  A.off0 = -(K - 1);
  A.OB = OB;
  A.PS = phase_slots(phase_len(OB, down, T, R), R);
  A.inv = down == 1 ? 0u : (unsigned)((0x100000000ull + (unsigned)down - 1) / (unsigned)down);
  const int64_t gy = (A.Lout + A.OB - 1) / A.OB;
  if (gy > 65535) return set_status(st, USTBX_E_ARG, "trace too long for the decimation factor");
  const dim3 grid((unsigned)traces, (unsigned)gy);
  const bool zp = mode == USTBX_FIR_ZERO_PHASE, lt = down == 1 && T >= kLdsTaps;
  const size_t bytes = sizeof(float2) * (((size_t)down * A.PS + 1) & ~size_t(1)) + (lt ? sizeof(float) * (size_t)T : 0);
  if (lt)
    hipLaunchKernelGGL((zp ? demodulate_kernel<8, 1, true, true> : demodulate_kernel<8, 1, false, true>), grid,
                       dim3(kDB), bytes, s, A);
  else if (down == 1)
    hipLaunchKernelGGL((zp ? demodulate_kernel<8, 1, true> : demodulate_kernel<8, 1, false>), grid, dim3(kDB), bytes, s, A);
  else if (down == 2)
    hipLaunchKernelGGL((zp ? demodulate_kernel<4, 2, true> : demodulate_kernel<4, 2, false>), grid, dim3(kDB), bytes, s, A);
  else
    hipLaunchKernelGGL((zp ? demodulate_kernel<4, 0, true> : demodulate_kernel<4, 0, false>), grid, dim3(kDB), bytes, s, A);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(st, e, "demodulate_kernel launch");
  return ok(st);
}

}  // extern "C"
