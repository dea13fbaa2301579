// das_window_both_iq.hip — the window-staged kernel of dimension both, linear IQ data.
#include "das_window_both.h"

namespace ustbx {

hipError_t launch_window_both_iq(const GeomLaunch& G, hipStream_t s) {
  return G.win.row == 64 ? both_shape<SM_LINEAR, PH_SEP, 64>(G, s) : both_shape<SM_LINEAR, PH_SEP, 128>(G, s);
}

}  // namespace ustbx
