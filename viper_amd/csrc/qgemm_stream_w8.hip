// Streaming skinny-GEMM kernels of format 8 (the template is in qgemm_stream.h).
#include "qgemm_stream.h"

namespace vq {

sg_fn sg_pick_w8(int gw, int am, bool pack, bool part, int senc, size_t* lds) {
    return sg_pick<8>(gw, am, pack, part, senc, lds);
}
sg_fn sg_pick_tl8(int gw, bool pack) { return sg_pick_tl<8>(gw, pack); }

}  // namespace vq
