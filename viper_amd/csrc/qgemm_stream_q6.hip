// Streaming skinny-GEMM kernels of format 6 (the template is in qgemm_stream.h).
#include "qgemm_stream.h"

namespace vq {

sg_fn sg_pick_q6(int gw, int am, bool pack, bool part, int senc, size_t* lds) {
    return sg_pick<6>(gw, am, pack, part, senc, lds);
}

}  // namespace vq
