// The deep convolution kernel's MXFP8 tiles.
#include "deep_launch.h"

namespace fim {

template <int OUT>
static int launch_out(const ConvArgs& a, DeepPlan p, hipStream_t stream) {
  if (p.wn == 4) {
    switch (p.mbw) {
      case 4: return launch_deep_tile<KIND_MX, OUT, 4, 4, false>(a, stream);
      case 5: return launch_deep_tile<KIND_MX, OUT, 4, 5, false>(a, stream);
      case 6: return launch_deep_tile<KIND_MX, OUT, 4, 6, false>(a, stream);
      case 7: return launch_deep_tile<KIND_MX, OUT, 4, 7, false>(a, stream);
      case 8: return launch_deep_tile<KIND_MX, OUT, 4, 8, false>(a, stream);
    }
  } else if (p.wn == 2) {
    switch (p.mbw) {
      case 2:
        return p.two ? launch_deep_tile<KIND_MX, OUT, 2, 2, false, true>(a, stream)
                     : launch_deep_tile<KIND_MX, OUT, 2, 2, false>(a, stream);
      case 3: return launch_deep_tile<KIND_MX, OUT, 2, 3, false>(a, stream);
      case 4: return launch_deep_tile<KIND_MX, OUT, 2, 4, false>(a, stream);
      case 5: return launch_deep_tile<KIND_MX, OUT, 2, 5, false>(a, stream);
    }
  }
  return FIM_ERR_UNSUPPORTED;
}

int launch_deep_mx(const ConvArgs& a, DeepPlan p, hipStream_t stream) {
  return a.out_mode == OUT_BF16 ? launch_out<OUT_BF16>(a, p, stream) : launch_out<OUT_E4M3>(a, p, stream);
}

}  // namespace fim
