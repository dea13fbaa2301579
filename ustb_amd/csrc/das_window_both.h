// das_window_both.h — shapes of the window-staged kernel of dimension both
// (instantiated per data type, one translation unit each).
//
// A block is two groups of 256 threads that share out the tile's waves: the
// receive entries are read once from memory for both (the second read hits
// the CU's cache), and the 6-13 waves a group holds leave registers for 4-6
// waves per SIMD. Bound: the latency between a step's barrier and its receive
// entries (the waves wait 51 and 52 % of their cycles on the two below); 12 VALU
// instructions per 64 terms take 26-66 % of the issue slots.
// Against the gathering kernel:
//   volume, 1024 channels x 25 waves on 96 x 96 x 128 voxels: 29.9 -> 10.1 ms
//     (two groups of 13; one group of 16 in two rounds 11.5, of 25 at 3 waves
//     per SIMD 9.8; four groups of 7: 14.1)
//   cine, 128 channels x 11 waves x 16 frames on 301 x 387 pixels: 1.08 -> 0.58
//     ms (two groups of 6, 2 frames; one group of 12: 0.69; 4 frames: 1.0)
#pragma once
#include "das_window.h"

namespace ustbx {

template <int SM, int PH, int ROW, int WC, int FT>
static hipError_t both_launch(const GeomLaunch& G, hipStream_t s) {
  return launch_window_t<SM, MODE_BOTH, PH, ROW, WC, FT, 1, 1, 2>(G, 1, s);
}

// Waves per group of a block's two groups: the shape whose rounds leave the
// fewest slots empty, the fewer rounds where they tie.
template <int N>
static int fewest_slots(int W, const int (&wc)[N]) {
  int best = 0, slots = 0x7fffffff;
  for (int k = 0; k < N; ++k) {
    const int per = 2 * wc[k], n = (W + per - 1) / per * per;
    if (n < slots || (n == slots && wc[k] > wc[best])) {
      best = k;
      slots = n;
    }
  }
  return wc[best];
}

template <int SM, int PH, int ROW>
static hipError_t both_shape(const GeomLaunch& G, hipStream_t s) {
  if (G.F > 1) {
    const int wc[2] = {6, 8};
    return fewest_slots(G.win_max_nw, wc) == 6 ? both_launch<SM, PH, ROW, 6, 2>(G, s)
                                               : both_launch<SM, PH, ROW, 8, 2>(G, s);
  }
  if constexpr (SM == SM_LINEAR) {
    const int wc[4] = {6, 8, 13, 16};
    switch (fewest_slots(G.win_max_nw, wc)) {
      case 6: return both_launch<SM, PH, ROW, 6, 1>(G, s);
      case 8: return both_launch<SM, PH, ROW, 8, 1>(G, s);
      case 13: return both_launch<SM, PH, ROW, 13, 1>(G, s);
      default: return both_launch<SM, PH, ROW, 16, 1>(G, s);
    }
  } else {
    return hipErrorInvalidValue;  // one cubic frame runs the gathering kernel
  }
}

}  // namespace ustbx
