// The deep convolution kernel's INT8 tiles.
#include "deep_launch.h"

namespace fim {

template <int OUT, bool RAG>
static int launch_out(const ConvArgs& a, DeepPlan p, hipStream_t stream) {
  if (p.wn == 4) {
    switch (p.mbw) {
      case 4: return launch_deep_tile<KIND_INT8, OUT, 4, 4, RAG>(a, stream);
      case 5: return launch_deep_tile<KIND_INT8, OUT, 4, 5, RAG>(a, stream);
      case 6: return launch_deep_tile<KIND_INT8, OUT, 4, 6, RAG>(a, stream);
      case 7: return launch_deep_tile<KIND_INT8, OUT, 4, 7, RAG>(a, stream);
      case 8: return launch_deep_tile<KIND_INT8, OUT, 4, 8, RAG>(a, stream);
    }
  } else if (p.wn == 2) {
    switch (p.mbw) {
      case 2:
        return p.two ? launch_deep_tile<KIND_INT8, OUT, 2, 2, RAG, true>(a, stream)
                     : launch_deep_tile<KIND_INT8, OUT, 2, 2, RAG>(a, stream);
      case 3: return launch_deep_tile<KIND_INT8, OUT, 2, 3, RAG>(a, stream);
      case 4: return launch_deep_tile<KIND_INT8, OUT, 2, 4, RAG>(a, stream);
      case 5: return launch_deep_tile<KIND_INT8, OUT, 2, 5, RAG>(a, stream);
    }
  }
  return FIM_ERR_UNSUPPORTED;
}

int launch_deep_int8(const ConvArgs& a, DeepPlan p, hipStream_t stream) {
  if (a.out_mode == OUT_BF16)
    return p.rag ? launch_out<OUT_BF16, true>(a, p, stream) : launch_out<OUT_BF16, false>(a, p, stream);
  return p.rag ? launch_out<OUT_INT8, true>(a, p, stream) : launch_out<OUT_INT8, false>(a, p, stream);
}

}  // namespace fim
