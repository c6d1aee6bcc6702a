// Streaming skinny-GEMM kernels of format 5 (the template is in qgemm_stream.h).
#include "qgemm_stream.h"

namespace vq {

sg_fn sg_pick_q5(int gw, int am, bool pack, bool part, int senc, size_t* lds) {
    return sg_pick<5>(gw, am, pack, part, senc, lds);
}

}  // namespace vq
