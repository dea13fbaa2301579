// das_window_rxnone.hip — the window-staged kernels of dimension receive (sum
// over channels per wave) and none, and the tile lists they all read.
//
// Bound: dimension receive by the wait for a step's receive entries (53 % of the
// wave cycles; VALU 32-64 %, LDS 27 %), none by its stores. Measured against the per-lane kernel, which
// forms delay, weight and phase of every (pixel, channel) in FP64 for every 8
// waves and every frame: 64 channels x 31 waves x 4 frames on 193 x 512 pixels
// of a sector (receive, then the coherence factor) 4.69 -> 0.48 ms; 128
// channels x 5 waves on 150 x 201 pixels (none, 154 MB of output) 0.42 -> 0.087
// ms.
//
// Shapes: 8 waves held per round and 2 channels per step (16 rows); up to 4
// waves: 4 channels per step; several frames: 2 at a time (receive holds 8
// waves x 2 frames of sums; 8 x 4, and 16 waves of one frame, spilled
// registers: 2.8 ms instead of 0.6).
#include <algorithm>

#include "das_window.h"

namespace ustbx {

// A launch should hold several thousand wave64s (256 CUs x 4 SIMDs x a few);
// with fewer tiles the channels of a tile are shared out.
static int tiles_short(const GeomLaunch& G, int ft) {
  return (int64_t)G.win.tiles * ((G.F + ft - 1) / ft) < 1024;
}

template <int SM, int PH, int ROW, int WC, int FT, int NCH>
static hipError_t rx_cg(const GeomLaunch& G, hipStream_t s) {
  // the exact phases add a wave's channels in das_c's ascending order
  constexpr int kCG = PH == PH_SEP && FT == 1 ? 4 : 1;
  if (kCG > 1 && tiles_short(G, FT))
    return launch_window_t<SM, MODE_RX, PH, ROW, WC, FT, NCH, kCG, 1>(G, 1, s);
  return launch_window_t<SM, MODE_RX, PH, ROW, WC, FT, NCH, 1, 1>(G, 1, s);
}

template <int SM, int PH, int ROW>
static hipError_t rx_shape(const GeomLaunch& G, hipStream_t s) {
  if (G.F > 1) {
    if constexpr (PH == PH_SEP) return rx_cg<SM, PH, ROW, 8, 2, 1>(G, s);
    else return rx_cg<SM, PH, ROW, 4, 2, 2>(G, s);
  }
  if (G.W <= 4) return rx_cg<SM, PH, ROW, 4, 1, 4>(G, s);
  return rx_cg<SM, PH, ROW, 8, 1, 2>(G, s);
}

template <int SM, int ROW>
static hipError_t rx_ph(const GeomLaunch& G, int ph, hipStream_t s) {
  if (ph == PH_RF) return rx_shape<SM, PH_RF, ROW>(G, s);
  if (ph == PH_DASC) return rx_shape<SM, PH_DASC, ROW>(G, s);
  return rx_shape<SM, PH_SEP, ROW>(G, s);
}

hipError_t launch_window_rx(const GeomLaunch& G, int ph, hipStream_t s) {
  if (G.win.row == 64)
    return G.interp == INTERP_CUBIC ? rx_ph<SM_CUBIC, 64>(G, ph, s) : rx_ph<SM_LINEAR, 64>(G, ph, s);
  return G.interp == INTERP_CUBIC ? rx_ph<SM_CUBIC, 128>(G, ph, s) : rx_ph<SM_LINEAR, 128>(G, ph, s);
}

template <int SM, int PH, int ROW, int WC, int FT, int NCH>
static hipError_t none_z(const GeomLaunch& G, hipStream_t s) {
  const int64_t blocks = (int64_t)G.win.tiles * ((G.F + FT - 1) / FT);
  const int steps = (G.N + NCH - 1) / NCH;
  int z = (int)std::min<int64_t>((2048 + blocks - 1) / blocks, std::max(1, steps / 4));
  return launch_window_t<SM, MODE_NONE, PH, ROW, WC, FT, NCH, 1, 1>(G, std::max(1, std::min(z, 64)), s);
}

template <int SM, int PH, int ROW>
static hipError_t none_shape(const GeomLaunch& G, hipStream_t s) {
  if (G.F > 1) return none_z<SM, PH, ROW, 4, 2, 2>(G, s);
  if (G.W <= 4) return none_z<SM, PH, ROW, 4, 1, 4>(G, s);
  return none_z<SM, PH, ROW, 8, 1, 2>(G, s);
}

template <int SM, int ROW>
static hipError_t none_ph(const GeomLaunch& G, int ph, hipStream_t s) {
  if (ph == PH_RF) return none_shape<SM, PH_RF, ROW>(G, s);
  if (ph == PH_DASC) return none_shape<SM, PH_DASC, ROW>(G, s);
  return none_shape<SM, PH_SEP, ROW>(G, s);
}

hipError_t launch_window_none(const GeomLaunch& G, int ph, hipStream_t s) {
  if (G.win.row == 64)
    return G.interp == INTERP_CUBIC ? none_ph<SM_CUBIC, 64>(G, ph, s) : none_ph<SM_LINEAR, 64>(G, ph, s);
  return G.interp == INTERP_CUBIC ? none_ph<SM_CUBIC, 128>(G, ph, s) : none_ph<SM_LINEAR, 128>(G, ph, s);
}

// ---------------------------------------------------------------------------
// Tile lists, once per plan. One block of 16 wave64s per tile; wave s takes
// every 16th wave and channel, its lanes the tile's 256 pixels in four passes.
// A slot of cl / wl is first filled in index order, then wave 0 closes the gaps
// (ballots keep the order).
// ---------------------------------------------------------------------------
__device__ __forceinline__ int win_pixel(const WinTiles& T, int tile, int lid) {
  const int tz = tile % T.ntz, tg = tile / T.ntz;
  const int gx = tg % T.nlx, gy = tg / T.nlx;
  const int lb = T.lxb + T.lyb;
  const int dz = (lid & ((1 << T.zl) - 1)) | ((lid >> (T.zl + lb)) << T.zl);
  const int line = (lid >> T.zl) & ((1 << lb) - 1);
  const int iz = min((tz << T.dzb) + dz, T.n0 - 1), ix = min((gx << T.lxb) + (line & ((1 << T.lxb) - 1)), T.n1 - 1),
            iy = min((gy << T.lyb) + (line >> T.lxb), T.n2 - 1);
  return iz + T.n0 * (ix + T.n1 * iy);
}

__device__ __forceinline__ float wave_fmin(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o));
  return v;
}
__device__ __forceinline__ float wave_fmax(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  return v;
}

// floor of a delay in samples; bad where it is beyond what the bounds' slack
// covers (FP32 index rounding below a quarter sample)
__device__ __forceinline__ int sample_floor(float d, double t0, double fs, bool& bad) {
  const double v = ((double)d - t0) * fs;
  if (!(fabs((double)d * fs) < 524288.0) || !(fabs(t0 * fs) < 524288.0)) bad = true;
  return bad ? 0 : (int)floor(v);
}

constexpr int kListWaves = 16;

struct WinLists {
  WinTiles t[kWinShapes];
  int count;
};

// Place of tile t in the visiting order: each of 8 contiguous shares of the
// tiles (one per XCD) depth band by depth band, tpl tiles down a line group.
__device__ __forceinline__ int band_place(int t, int tpl, int tiles) {
  const int q = tiles / 8, r = tiles % 8;
  const int k = t < r * (q + 1) ? t / (q + 1) : r + (t - r * (q + 1)) / q;
  const int s0 = k * q + min(k, r), cnt = q + (k < r ? 1 : 0);
  const int b = t % tpl, r0 = s0 % tpl, rem = cnt % tpl;
  // tiles of the share in a band: cnt / tpl, and one more in the rem bands from r0 on (cyclic)
  const int wrap = r0 + rem - tpl;
  const int more = wrap <= 0 ? max(0, min(b, r0 + rem) - r0) : min(b, wrap) + max(0, b - r0);
  const int first = s0 + (b - r0 + tpl) % tpl;
  return s0 + b * (cnt / tpl) + more + (t - first) / tpl;
}

__global__ __launch_bounds__(64 * kListWaves) void window_lists_kernel(GeomLaunch G, WinLists C,
                                                                       WinInfo* __restrict__ infos, int full_w,
                                                                       int full_n) {
  __shared__ int spans[2];   // largest hi - lo of the tile's waves, channels
  __shared__ int counts[2];  // entries
  int k = 0, tile = blockIdx.x;
  while (tile >= C.t[k].tiles) tile -= C.t[k++].tiles;
  const WinTiles T = C.t[k];
  WinInfo* info = infos + k;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t PS = (size_t)G.P;
  int px[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) px[i] = win_pixel(T, tile, i * 64 + lane);
  int4* tw = T.wl + (size_t)tile * G.W;
  int4* tc = T.cl + (size_t)tile * G.N;
  bool bad = false;
  for (int e = wave; e < G.W + G.N; e += kListWaves) {
    const bool rx = e >= G.W;
    const int k = rx ? e - G.W : e;
    float lo = INFINITY, hi = -INFINITY;
    bool any = false, all = true;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float4 v = rx ? rx_entry(G.win_rx, G.rx_compact, (size_t)k * PS + px[i]) : G.tx_table[(size_t)k * PS + px[i]];
      const bool on = v.y != 0.0f;
      if (on && !(isfinite(v.x) && isfinite(v.z) && isfinite(v.w))) bad = true;
      if (rx && !isfinite(v.x)) bad = true;
      // receive: the range of every pixel (a lane with no weight is computed
      // and dropped); transmit: of the weighted ones
      if (rx || on) {
        lo = fminf(lo, v.x);
        hi = fmaxf(hi, v.x);
      }
      any = any || on;
      all = all && on;
    }
    lo = wave_fmin(lo);
    hi = wave_fmax(hi);
    const bool wany = __any(any), wall = __all(all);
    int4 out = make_int4(k, 0, 0, (wall ? 1 : 0) | (wany ? 2 : 0));
    if (wany) {
      out.y = sample_floor(lo, rx ? (double)G.t0 : 0.0, (double)G.fs, bad);
      out.z = sample_floor(hi, rx ? (double)G.t0 : 0.0, (double)G.fs, bad);
    }
    if (lane == 0) (rx ? tc : tw)[k] = out;
  }
  if (__any(bad) && lane == 0) atomicOr(&info->bad, 1);
  __syncthreads();
  if (wave < 2) {  // wave 0: the transmit list, wave 1: the channels
    int4* t = wave == 0 ? tw : tc;
    const int n = wave == 0 ? G.W : G.N, full = wave == 0 ? full_w : full_n;
    int cnt = 0, span = 0;
    for (int b = 0; b < n; b += 64) {
      const bool in = b + lane < n;
      const int4 v = in ? t[b + lane] : make_int4(0, 0, 0, 0);
      const bool keep = in && (full || (v.w & 2));
      const unsigned long long m = __ballot(keep);
      if (keep) t[cnt + __popcll(m & ((1ull << lane) - 1ull))] = v;
      if (in && (v.w & 2)) span = max(span, v.z - v.y);
      cnt += __popcll(m);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) span = max(span, __shfl_xor(span, o));
    if (lane == 0) {
      (wave == 0 ? T.nw : T.nc)[tile] = cnt;
      counts[wave] = cnt;
      spans[wave] = span;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned long long terms = (unsigned long long)counts[0] * (unsigned long long)counts[1];
    atomicMax(&info->span, spans[0] + spans[1]);
    atomicMax(&info->max_nw, counts[0]);
    atomicAdd(&info->terms, terms);
    atomicMax(&info->most, terms);
    T.order[band_place(tile, T.ntz, T.tiles)] = tile;
  }
}

hipError_t launch_window_lists(const GeomLaunch& G, const WinTiles* T, int count, WinInfo* info, int full_w, int full_n,
                               hipStream_t stream) {
  WinLists C;
  unsigned tiles = 0;
  for (int k = 0; k < count; ++k) {
    C.t[k] = T[k];
    tiles += (unsigned)T[k].tiles;
  }
  C.count = count;
  hipLaunchKernelGGL(window_lists_kernel, dim3(tiles), dim3(64 * kListWaves), 0, stream, G, C, info, full_w, full_n);
  return hipGetLastError();
}

}  // namespace ustbx
