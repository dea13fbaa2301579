// das_window.h — delay-and-sum on patches of 256 pixels whose sample windows
// are staged in LDS (dimension both with the separable or RF phase, receive
// and none with any phase, on linear and sector scans).
//
// A tile is a patch of DZ consecutive depths by 256 / DZ neighbouring scan
// lines (WinTiles), one lane per pixel. For a (channel, wave, frame) all of
// the tile's terms read one short run of the trace, the tile's window: the
// block loads it once, coalesced, into an LDS row, and every lane reads its
// samples from there. That replaces one or two 16-byte gathers per term
// through the texture path (20 cycles per 64 lanes, the roof of the gathering
// kernels) by 8 cycles of LDS reads, and the windows that 256 pixels share by
// one read of L2 or HBM instead of four.
//
// Window position. With per-tile integer bounds of a wave's transmit delay and
// of a channel's receive delay in samples (floor of the tile's minimum and
// maximum, tables of the plan), every term's index n0 lies in [lo_w + lo_n -
// 1, hi_w + hi_n + 2]: the -1 and +2 cover both floors and the FP32 rounding
// of das_c's index (below a quarter sample; the plan checks the magnitude). So a
// window's place is one scalar addition, and whether all of a channel's terms
// are inside the sample window (no lane tests anything) one comparison.
//
// Loop: rounds of up to WC waves (transmit state in VGPRs) x the tile's
// channel list; a step stages NCH channels' WC x FT windows (FT frames) while
// the previous step's are used (two LDS buffers, one barrier per step). The
// index, the fraction and the weights of a term are formed once for its FT
// frames. A block is one group of 256 threads, or CG x WG groups that share
// out the channels (CG) and the waves (WG) of one tile.
//
// Rows hold 64 samples, or 128 on coarse scans. Linear interpolation with the
// separable phase keeps {x, x[+1] - x} per sample in rows of 64, so a term
// costs two FMAs and no subtraction; the other forms keep the samples.
#pragma once
#include <algorithm>
#include <type_traits>
#include <utility>

#include "das_rxtab.h"

namespace ustbx {

// The sample positions a row must hold beyond hi - lo of the bounds: n0 from
// lo - 1 to hi + 2, and the samples a term reads around n0.
template <int SM>
struct WinSpan {
  static constexpr int kBack = SM == SM_CUBIC ? 1 : 0;
  static constexpr int kSlack = 3 + (SM == SM_CUBIC ? 4 : 2);  // samples = (hi - lo) + kSlack
};

struct WinArgs {
  const void* ch;      // [F][W][N][L] complex64
  float2* out;
  const float4* tx;    // [W][P]
  const float4* rx;    // [N][P] float4, or float2 (RF plans)
  const float2* ref;   // [P] or null
  WinTiles T;
  int P, N, W, L, F;
  float t0, fs, wd;
  int frame_bytes;
};

typedef const __attribute__((address_space(3))) f4v lds_f4;
typedef __attribute__((address_space(3))) f4v lds_f4w;

__device__ __forceinline__ int4 scalar_int4(const int4* p) {
  const __attribute__((address_space(4))) int* q = (const __attribute__((address_space(4))) int*)p;
  return make_int4(q[0], q[1], q[2], q[3]);
}

// v of the next lane (lane 63: zero)
__device__ __forceinline__ float next_lane(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));  // wave_shl:1
}

// f(integral_constant 0), .., f(integral_constant N - 1): the indices of
// register arrays are constants before any pass runs.
template <typename F, int... I>
__device__ __forceinline__ void static_for_seq(const F& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>()), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(const F& f) {
  static_for_seq(f, std::make_integer_sequence<int, N>());
}

template <int SM, int MODE, int PH, int ROW, int WC, int FT, int NCH, int CG, int WG>
struct WinKernel {
  static_assert(MODE == MODE_BOTH || MODE == MODE_RX || MODE == MODE_NONE, "dimension transmit has its own kernel");
  static_assert(WG == 1 || MODE == MODE_BOTH, "wave groups add into one image");
  static constexpr bool kSep = MODE == MODE_BOTH || PH == PH_SEP;  // T and R from the tables
  static_assert(ROW == 64 || ROW == 128, "samples of an LDS row");
  static constexpr bool kDelta = SM == SM_LINEAR && kSep && ROW == 64;
  static constexpr int kLd = ROW / 64;  // loads per row
  static constexpr bool kCompact = PH == PH_RF;
  static constexpr int kShift = kDelta ? 4 : 3;  // log2 bytes per staged sample
  static constexpr int kRows = NCH * WC * FT;    // row (channel, wave, frame), frame fastest
  static constexpr int kRowBytes = ROW << kShift;
  static constexpr int kBufBytes = kRows * kRowBytes;
  static constexpr int kPer = (kRows + 3) / 4;  // rows a wave stages per step: wave + 4 i
  static constexpr int kAcc = MODE == MODE_RX ? WC : 1;
  static constexpr int kGroups = CG * WG;
  // dimension both: the sums are closed every 32 steps (and at the end of a
  // round), so that their rounding grows with 32 + steps / 32 additions, not
  // with the channels (1024 of the volume: 4.7e-7 by the gathering kernel's
  // splits, 6.2e-7 in one running sum). One frame keeps its closed sum in
  // registers; several keep one per pixel in LDS, which the groups add to in
  // turn: two more register pairs leave a block less per CU (cine 0.56 -> 0.72
  // ms).
  static constexpr bool kClose = MODE == MODE_BOTH;
  static constexpr bool kCloseLds = kClose && FT > 1;
  static constexpr int kTot = kCloseLds ? FT * 256 * 8 : 0;
  static constexpr int kSmem = kGroups * 2 * kBufBytes + kTot;

  // One staged term: its fraction, the LDS address of its samples and whether it counts.
  struct Term1 {
    float b;
    unsigned la;
    bool ok;
  };

  template <bool CHK>
  static __device__ __forceinline__ Term1 term(float td, float rd, float t0, float fs, float lim, unsigned soff,
                                               unsigned zero) {
    const float d = term_index(td, rd, t0, fs);
    Term1 t;
    t.b = __builtin_amdgcn_fractf(d);
    const int n0 = (int)d;
    t.la = ((unsigned)n0 << kShift) + soff;
    t.ok = true;
    if (CHK) {
      t.ok = d >= 1.0f && d < lim;
      t.la = t.ok ? t.la : zero;  // in the buffer, whatever is there
    }
    return t;
  }

  struct Samples {
    f4v lo, hi;
  };
  static __device__ __forceinline__ Samples fetch(unsigned la, int row) {
    Samples s;
    const unsigned a = la + (unsigned)(row * kRowBytes);
    if (kDelta) {
      s.lo = *reinterpret_cast<lds_f4*>((size_t)a);
      s.hi = s.lo;
    } else {
      const f4a8 v = *reinterpret_cast<lds_f4a8*>((size_t)a);
      s.lo = f4v{v.x, v.y, v.z, v.w};
      if (SM == SM_CUBIC) {
        const f4a8 u = *reinterpret_cast<lds_f4a8*>((size_t)a + 16);
        s.hi = f4v{u.x, u.y, u.z, u.w};
      } else {
        s.hi = s.lo;
      }
    }
    return s;
  }
  static __device__ __forceinline__ float2 interp(const Samples& s, float b, const float (&k)[4]) {
    if (kDelta) return make_float2(fmaf(b, s.lo.z, s.lo.x), fmaf(b, s.lo.w, s.lo.y));
    if (SM == SM_LINEAR) return make_float2(fmaf(b, s.lo.z - s.lo.x, s.lo.x), fmaf(b, s.lo.w - s.lo.y, s.lo.y));
    return make_float2(fmaf(k[3], s.hi.z, fmaf(k[2], s.hi.x, fmaf(k[1], s.lo.z, k[0] * s.lo.x))),
                       fmaf(k[3], s.hi.w, fmaf(k[2], s.hi.y, fmaf(k[1], s.lo.w, k[0] * s.lo.y))));
  }

  // das_c's weight of a term (das_c.cpp:372-387)
  static __device__ __forceinline__ void exact_weight(float td, float rd, float ta, float ra, float wd, float& wr,
                                                      float& wi) {
#pragma clang fp contract(off)
    const float c_apo = ta * ra;
    wr = c_apo;
    wi = 0.0f;
    if (PH == PH_DASC) {
      float sv, cv;
      sincosf(wd * (td + rd), &sv, &cv);
      wr = cv * c_apo;
      wi = sv * c_apo;
    }
  }
  static __device__ __forceinline__ float2 exact_value(const Samples& s, float b, const float (&k)[4], float wr,
                                                       float wi) {
#pragma clang fp contract(off)
    if (SM == SM_LINEAR) {
      ustbx::Term t;
      t.a = 1.0f - b;
      t.b = b;
      t.wr = wr;
      t.wi = wi;
      return dasc_contrib(t, make_float4(s.lo.x, s.lo.y, s.lo.z, s.lo.w));  // das_c.cpp:389-399
    }
    const float2 sm = interp(s, b, k);
    return make_float2(wr * sm.x - wi * sm.y, wr * sm.y + wi * sm.x);
  }

  static __device__ __forceinline__ void run(const WinArgs& A, char* smem) {
    const int lane = threadIdx.x & 63;
    const int lid = threadIdx.x & 255;
    const int wave = __builtin_amdgcn_readfirstlane(lid >> 6);
    const int g = kGroups > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8) : 0;
    const int wgi = g / CG;  // this group's share of the waves
    const WinTiles& T = A.T;
    // a tile's frame chunks next to each other on one XCD: they read the same
    // receive rows at about the same time
    const int fcs = (A.F + FT - 1) / FT;
    const int item = xcd_tile((int)blockIdx.x, (int)gridDim.x);
    const int tile = __builtin_amdgcn_readfirstlane(T.order[item / fcs]);
    const int f0 = (item % fcs) * FT;
    const int nfr = min(FT, A.F - f0);
    const size_t PS = (size_t)A.P;

    // this lane's pixel; lanes past the scan's edge take the nearest pixel
    // (their terms are computed like the others', their results dropped)
    const int tz = tile % T.ntz, tg = tile / T.ntz;
    const int gx = tg % T.nlx, gy = tg / T.nlx;
    const int zl = T.zl, lb = T.lxb + T.lyb;
    const int dz = (lid & ((1 << zl) - 1)) | ((lid >> (zl + lb)) << zl);
    const int line = (lid >> zl) & ((1 << lb) - 1);
    const int iz = (tz << T.dzb) + dz, ix = (gx << T.lxb) + (line & ((1 << T.lxb) - 1)),
              iy = (gy << T.lyb) + (line >> T.lxb);
    const bool act = iz < T.n0 && ix < T.n1 && iy < T.n2;
    const unsigned p = (unsigned)(min(iz, T.n0 - 1) + T.n0 * (min(ix, T.n1 - 1) + T.n1 * min(iy, T.n2 - 1)));

    const int nw = __builtin_amdgcn_readfirstlane(T.nw[tile]);
    const int nc = __builtin_amdgcn_readfirstlane(T.nc[tile]);
    const int4* __restrict__ wl = T.wl + (size_t)tile * A.W;
    const int4* __restrict__ cl = T.cl + (size_t)tile * A.N;
    const float t0 = A.t0, fs = A.fs, wd = A.wd;
    const int ilim = A.L - (SM == SM_LINEAR ? 1 : 2);
    const float lim = (float)ilim;
    const float2 refp = A.ref ? A.ref[p] : make_float2(1.0f, 0.0f);
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char*)smem + (unsigned)(g * 2 * kBufBytes);
    const unsigned lane8 = (unsigned)lane * 8u;

    // channel steps of this group: s = q, q + Q, ...
    const int Q = CG * (int)gridDim.z, q = (int)blockIdx.z * CG + g % CG;
    const int steps = (nc + NCH - 1) / NCH;
    const int nit = (steps + Q - 1) / Q;  // the same for every group (they share the barriers)

    constexpr int kAF = MODE == MODE_NONE ? 1 : FT;
    constexpr bool kT = !(MODE == MODE_RX && kSep);  // the transmit weight is held per wave
    float2 acc[kAF][kAcc];
    static_for<kAF>([&](auto f) { static_for<kAcc>([&](auto j) { acc[f][j] = make_float2(0.0f, 0.0f); }); });
    float2 tot = make_float2(0.0f, 0.0f);
    // this lane's closed sum of frame f, its address formed where it is used (a
    // register held through the loop would cost a block per CU)
    auto closed = [&](int f) {
      unsigned t = threadIdx.x;
      asm volatile("" : "+v"(t));
      return reinterpret_cast<lds_f2*>((size_t)((unsigned)(size_t)(__attribute__((address_space(3))) char*)smem +
                                                (unsigned)(kSmem - kTot + f * 2048) + (t & 255u) * 8u));
    };
    auto close = [&]() {
      if constexpr (kCloseLds) {
        static_for<kGroups>([&](auto turn) {
          if (g == turn)
            static_for<FT>([&](auto f) {
              lds_f2* t = closed(f);
              const f2v v = *t;
              *t = f2v{v.x + acc[f][0].x, v.y + acc[f][0].y};
            });
          __syncthreads();
        });
      } else {
        cadd(tot, acc[0][0]);
      }
      static_for<kAF>([&](auto f) { acc[f][0] = make_float2(0.0f, 0.0f); });
    };
    if constexpr (kCloseLds) {
      if (g == 0) static_for<FT>([&](auto f) { *closed(f) = f2v{0.0f, 0.0f}; });
    }

    for (int kr = 0; kr < nw; kr += WG * WC) {
      const int k0 = __builtin_amdgcn_readfirstlane(kr + wgi * WC);
      const int nj = __builtin_amdgcn_readfirstlane(min(WC, max(0, nw - k0)));  // this group's waves of the round
      float td[WC];
      float2 Tw[kT ? WC : 1];  // T, or {ta, -} in the exact phases
      // scalars: of term J, the part of its LDS address that the wave fixes
      unsigned woff[WC];
      int amin = 0x3fffffff, amax = -0x3fffffff, all_t = 1;
      static_for<WC>([&](auto j) {
        td[j] = kFar;
        if constexpr (kT) Tw[j] = make_float2(0.0f, 0.0f);
        // slots past the list repeat its last wave with weight zero (their rows
        // are staged as zeros; a group with no waves computes no terms): no
        // entry past the list is read
        const int4 e = scalar_int4(wl + min(k0 + (int)j, nw - 1));
        woff[j] = lds0 + (unsigned)(j * FT * kRowBytes) - (unsigned)((e.y - 1) << kShift);
        all_t &= e.w;
        if (e.w & 2) {
          amin = min(amin, e.y);
          amax = max(amax, e.z);
        }
        const float4 v = (A.tx + (size_t)e.x * PS)[p];
        if (v.y != 0.0f) {
          td[j] = v.x;
          if constexpr (kT) {
            if (j < nj) Tw[j] = kSep ? make_float2(v.z, v.w) : make_float2(v.y, 0.0f);
          }
        }
      });
      if constexpr (MODE == MODE_RX)
        static_for<kAF>([&](auto f) { static_for<kAcc>([&](auto j) { acc[f][j] = make_float2(0.0f, 0.0f); }); });

      // The rows this wave stages, r = wave + 4 i: the byte offset that the
      // wave (and the frame) fixes, the samples its delay's spread takes (0:
      // no row), the channel of the step.
      int roff[kPer], rcnt[kPer];
      __amdgpu_buffer_rsrc_t rs[FT];
      static_for<FT>([&](auto f) {
        rs[f] = make_rsrc((const char*)A.ch + (size_t)(f0 + min((int)f, nfr - 1)) * (size_t)A.frame_bytes, A.frame_bytes);
      });
      static_for<kPer>([&](auto i) {
        const int r = wave + 4 * i;
        const int rem = r % (WC * FT);
        const int j = rem / FT, f = rem % FT;
        roff[i] = rcnt[i] = 0;
        if ((kRows % 4 == 0 || r < kRows) && j < nj && f < nfr) {
          const int4 we = scalar_int4(wl + k0 + j);
          roff[i] = (we.x * A.N * A.L + we.y - 1 - WinSpan<SM>::kBack) * 8;
          rcnt[i] = we.z - we.y + WinSpan<SM>::kSlack;
        }
        roff[i] = __builtin_amdgcn_readfirstlane(roff[i]);
        rcnt[i] = __builtin_amdgcn_readfirstlane(rcnt[i]);
      });
      float2 st[kPer][kLd];
      auto stage_load = [&](int s) {
        int4 ce[NCH];
        static_for<NCH>([&](auto c) { ce[c] = scalar_int4(cl + min(s * NCH + c, nc - 1)); });
        static_for<kPer>([&](auto i) {
          const int r = wave + 4 * i;
          int4 e = ce[0];
          static_for<NCH>([&](auto c) {
            if (c > 0 && r >= c * WC * FT) e = ce[c];
          });
          const int cnt = rcnt[i] > 0 ? rcnt[i] + (e.z - e.y) : 0;
          const unsigned off = (unsigned)(roff[i] + (e.x * A.L + e.y) * 8) + lane8;
          // FT 1, 2 or 4: the row's frame is r % FT
          __amdgpu_buffer_rsrc_t rsf = rs[0];
          if constexpr (FT > 1) {
            static_for<FT>([&](auto f) {
              if ((r % FT) == f) rsf = rs[f];
            });
          }
          static_for<kLd>([&](auto h) {
            st[i][h] = make_float2(0.0f, 0.0f);
            if (h == 0 || cnt > 64 * h)  // uniform
              st[i][h] = buf_load8(rsf, lane + 64 * h < cnt ? (int)(off + 512u * h) : kOOB);
          });
        });
      };
      auto stage_store = [&](int buf) {
        static_for<kPer>([&](auto i) {
          const int r = wave + 4 * i;
          if (kRows % 4 == 0 || r < kRows) {
            const unsigned a = lds0 + (unsigned)(buf * kBufBytes + r * kRowBytes) + ((unsigned)lane << kShift);
            if constexpr (kDelta) {
              const float2 x = st[i][0];
              const float nx = next_lane(x.x), ny = next_lane(x.y);
              *reinterpret_cast<lds_f4w*>((size_t)a) = f4v{x.x, x.y, nx - x.x, ny - x.y};
            } else {
              static_for<kLd>([&](auto h) {
                *reinterpret_cast<lds_f2*>((size_t)a + 512 * h) = f2v{st[i][h].x, st[i][h].y};
              });
            }
          }
        });
      };
      // receive entries of the step's channels
      float4 rv[NCH];
      static_for<NCH>([&](auto c) { rv[c] = make_float4(0.f, 0.f, 0.f, 0.f); });
      auto rx_load = [&](int s) {
        static_for<NCH>([&](auto c) {
          rv[c] = make_float4(0.f, 0.f, 0.f, 0.f);
          if (s * NCH + c < nc) {
            const size_t row = (size_t)scalar_int4(cl + s * NCH + c).x * PS;
            if constexpr (kCompact) {
              const float2 v = (reinterpret_cast<const float2*>(A.rx) + row)[p];
              rv[c] = make_float4(v.x, v.y, v.y, v.y * 0.0f);
            } else {
              rv[c] = (A.rx + row)[p];
            }
          }
        });
      };

      // the terms of channel C of the step (channel n, receive bound blo)
      auto compute = [&](auto chk, auto c, int n, int blo, int buf, float rd, float2 R, float ra, float2(&part)[FT]) {
        constexpr bool CHK = decltype(chk)::value;
        constexpr int C = decltype(c)::value;
        const unsigned zero = lds0 + (unsigned)(buf * kBufBytes);
        const unsigned coff = (unsigned)(buf * kBufBytes + C * WC * FT * kRowBytes) - (unsigned)(blo << kShift);
        // batches of kB waves: their samples are all asked for before the first
        // is used
        constexpr int kBmax = WC * FT <= 4 ? WC : 4 / FT;  // FT 1 or 2
        static_for<(WC + kBmax - 1) / kBmax>([&](auto gr) {
          constexpr int J0 = kBmax * decltype(gr)::value;
          constexpr int kB = WC - J0 < kBmax ? WC - J0 : kBmax;
          Term1 t[kB];
          Samples sm[kB][FT];
          static_for<kB>([&](auto u) {
            constexpr int J = J0 + decltype(u)::value;
            unsigned soff = woff[J] + coff;
            asm("" : "+s"(soff));  // one scalar operand of the address
            t[u] = term<CHK>(td[J], rd, t0, fs, lim, soff, zero);
            static_for<FT>([&](auto f) { sm[u][f] = fetch(t[u].la, f); });
          });
          __builtin_amdgcn_sched_barrier(0);
          static_for<kB>([&](auto u) {
            constexpr int J = J0 + decltype(u)::value;
            float kw[4] = {0.f, 0.f, 0.f, 0.f};
            if constexpr (SM == SM_CUBIC) keys_weights_horner(t[u].b, kw[0], kw[1], kw[2], kw[3]);
            float wr = 0.0f, wi = 0.0f;
            if constexpr (!kSep) exact_weight(t[u].ok ? td[J] : 0.0f, t[u].ok ? rd : 0.0f, Tw[J].x, ra, wd, wr, wi);
            static_for<FT>([&](auto f) {
              if constexpr (MODE == MODE_BOTH) {
                float2 v = part[f];
                cfma(v, Tw[J], interp(sm[u][f], t[u].b, kw));
                part[f] = !CHK || t[u].ok ? v : part[f];
              } else if constexpr (MODE == MODE_RX) {
                float2 v = acc[f][J];
                if constexpr (kSep) cfma(v, R, interp(sm[u][f], t[u].b, kw));
                else cadd(v, exact_value(sm[u][f], t[u].b, kw, wr, wi));
                acc[f][J] = !CHK || t[u].ok ? v : acc[f][J];
              } else {
                float2 v;
                if constexpr (kSep) v = cmul(cmul(R, Tw[J]), interp(sm[u][f], t[u].b, kw));
                else v = exact_value(sm[u][f], t[u].b, kw, wr, wi);
                if (CHK && !t[u].ok) v = make_float2(0.0f, 0.0f);
                if (A.ref) v = cmul(v, refp);
                if (act && J < nj && f < nfr) {
                  const int w = scalar_int4(wl + k0 + J).x;
                  (A.out + (((size_t)(f0 + f) * A.W + w) * A.N + n) * PS)[p] = v;
                }
              }
            });
          });
          __builtin_amdgcn_sched_barrier(0);
        });
      };

      int buf = 0;
      if (q < steps) {
        stage_load(q);
        stage_store(0);
        rx_load(q);
      }
      __syncthreads();
      for (int i0 = 0, i1; i0 < nit; i0 = i1) {
        i1 = kClose ? min(i0 + 32, nit) : nit;
        for (int it = i0; it < i1; ++it) {
          const int s = q + it * Q;
          const bool more = s + Q < steps;           // wave-uniform
          if (more) stage_load(s + Q);
          if (s < steps && nj > 0) {
            static_for<NCH>([&](auto c) {
              const int ci = s * NCH + c;
              if (ci < nc) {
                const int4 ce = scalar_int4(cl + ci);
                const bool ron = rv[c].y != 0.0f;
                const float2 R = ron ? make_float2(rv[c].z, rv[c].w) : make_float2(0.0f, 0.0f);
                float2 part[FT];
                static_for<FT>([&](auto f) { part[f] = make_float2(0.0f, 0.0f); });
                // every term of the channel in the sample window, every weight
                // nonzero (dimension both drops the sums of the lanes with no
                // receive weight below)
                const bool dense = (all_t & 1) && (MODE == MODE_BOTH || (ce.w & 1)) && amin + ce.y - 1 >= 1 &&
                                   amax + ce.z + 2 < ilim;
                if (dense)
                  compute(std::false_type(), c, ce.x, ce.y, buf, rv[c].x, R, rv[c].y, part);
                else
                  compute(std::true_type(), c, ce.x, ce.y, buf, ron ? rv[c].x : kFar, R, rv[c].y, part);
                if constexpr (MODE == MODE_BOTH)
                  static_for<FT>([&](auto f) {
                    float2 v = acc[f][0];
                    cfma(v, make_float2(rv[c].z, rv[c].w), part[f]);
                    acc[f][0] = ron ? v : acc[f][0];
                  });
              }
            });
          }
          // the next entries into the same registers: a second set, in flight
          // during the terms, costs a block per CU and time (cine 0.60 -> 0.77 ms)
          if (more) {
            rx_load(s + Q);
            stage_store(buf ^ 1);
          }
          __syncthreads();
          buf ^= 1;
        }
        if constexpr (kClose) close();
      }

      if constexpr (MODE == MODE_RX) {
        // out[f][w][p] = T * sum (the exact phases: the sum)
        static_for<kAcc>([&](auto j) {
          if (j < nj) {
            const int w = scalar_int4(wl + k0 + j).x;
            float2 Tj = make_float2(0.0f, 0.0f);
            if constexpr (kSep) {
              const float4 v = (A.tx + (size_t)w * PS)[p];
              if (v.y != 0.0f) Tj = make_float2(v.z, v.w);
            }
            static_for<FT>([&](auto f) {
              if (f < nfr) {
                float2 v = group_sum(acc[f][j], smem, g, lid);
                if constexpr (kSep) v = cmul(Tj, v);
                if (A.ref) v = cmul(v, refp);
                if (act && g == 0) (A.out + ((size_t)(f0 + f) * A.W + w) * PS)[p] = v;
              }
            });
          }
        });
      }
    }  // round

    if constexpr (MODE == MODE_BOTH)
      static_for<FT>([&](auto f) {
        if (f < nfr) {
          float2 v;
          if constexpr (kCloseLds) {
            const f2v t = *closed(f);
            v = make_float2(t.x, t.y);
          } else {
            v = group_sum(tot, smem, g, lid);
          }
          if (A.ref) v = cmul(v, refp);
          if (act && g == 0) (A.out + (size_t)(f0 + f) * PS)[p] = v;
        }
      });
  }

  // The groups' sums in group order (group 0 gets them).
  static __device__ __forceinline__ float2 group_sum(float2 v, char* smem, int g, int lid) {
    if constexpr (kGroups > 1) {
      float2* red = reinterpret_cast<float2*>(smem);
      red[threadIdx.x] = v;
      __syncthreads();
      if (g == 0)
        static_for<kGroups - 1>([&](auto k) { cadd(v, red[(k + 1) * 256 + lid]); });
      __syncthreads();
    }
    return v;
  }
};

template <int SM, int MODE, int PH, int ROW, int WC, int FT, int NCH, int CG, int WG>
__global__ __launch_bounds__(256 * CG * WG, 4) void das_window_kernel(WinArgs A) {
  using K = WinKernel<SM, MODE, PH, ROW, WC, FT, NCH, CG, WG>;
  __shared__ __align__(16) char smem[K::kSmem];
  K::run(A, smem);
}

// Channel groups per tile: blocks of 1024 threads (or, in dimension none,
// more blocks per tile) where the tiles alone leave the chip idle.
template <int SM, int MODE, int PH, int ROW, int WC, int FT, int NCH, int CG, int WG>
static hipError_t launch_window_t(const GeomLaunch& G, int zsplit, hipStream_t stream) {
  WinArgs A;
  A.ch = G.ch;
  A.out = reinterpret_cast<float2*>(G.out);
  A.tx = G.tx_table;
  A.rx = G.dim == MODE_BOTH ? G.rx_table : G.win_rx;
  A.ref = G.ref_phase ? (G.dim == MODE_BOTH ? G.ref_table : G.win_ref) : nullptr;
  A.T = G.win;
  A.P = G.P;
  A.N = G.N;
  A.W = G.W;
  A.L = G.L;
  A.F = G.F;
  A.t0 = G.t0;
  A.fs = G.fs;
  A.wd = G.wd;
  A.frame_bytes = G.L * G.N * G.W * 8;
  // a grid holds fewer than 2^32 threads: as many frames per launch as fit
  constexpr int kThreads = 256 * CG * WG;
  const size_t chunks = (size_t)(0xFFFFFFFFu / kThreads) / (size_t)G.win.tiles;
  const int most = (int)std::min<size_t>((size_t)G.F, std::max<size_t>(chunks, 1) * FT);
  const size_t frame_out = (size_t)G.P * (size_t)(MODE == MODE_BOTH ? 1 : G.W) * (size_t)(MODE == MODE_NONE ? G.N : 1);
  hipError_t e = hipSuccess;
  for (int64_t f = 0; e == hipSuccess && f < G.F; f += most) {
    A.F = (int)std::min<int64_t>(most, G.F - f);
    A.ch = (const char*)G.ch + (size_t)f * (size_t)A.frame_bytes;
    A.out = reinterpret_cast<float2*>(G.out) + (size_t)f * frame_out;
    hipLaunchKernelGGL((das_window_kernel<SM, MODE, PH, ROW, WC, FT, NCH, CG, WG>),
                       dim3((unsigned)G.win.tiles * (unsigned)((A.F + FT - 1) / FT), 1u, (unsigned)zsplit),
                       dim3(kThreads), 0, stream, A);
    e = hipGetLastError();
  }
  return e;
}

hipError_t launch_window_rx(const GeomLaunch& G, int ph, hipStream_t stream);
hipError_t launch_window_none(const GeomLaunch& G, int ph, hipStream_t stream);
hipError_t launch_window_both_iq(const GeomLaunch& G, hipStream_t stream);
hipError_t launch_window_both_rf(const GeomLaunch& G, hipStream_t stream);
hipError_t launch_window_both_cubic(const GeomLaunch& G, hipStream_t stream);
inline hipError_t launch_window_both(const GeomLaunch& G, hipStream_t stream) {
  if (G.interp == INTERP_CUBIC) return launch_window_both_cubic(G, stream);
  return G.wd == 0.0f ? launch_window_both_rf(G, stream) : launch_window_both_iq(G, stream);
}

}  // namespace ustbx
