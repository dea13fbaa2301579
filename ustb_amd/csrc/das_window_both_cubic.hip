// das_window_both_cubic.hip — the window-staged kernel of dimension both, cubic data of several frames.
#include "das_window_both.h"

namespace ustbx {

hipError_t launch_window_both_cubic(const GeomLaunch& G, hipStream_t s) {
  if (G.wd == 0.0f)
    return G.win.row == 64 ? both_shape<SM_CUBIC, PH_RF, 64>(G, s) : both_shape<SM_CUBIC, PH_RF, 128>(G, s);
  return G.win.row == 64 ? both_shape<SM_CUBIC, PH_SEP, 64>(G, s) : both_shape<SM_CUBIC, PH_SEP, 128>(G, s);
}

}  // namespace ustbx
