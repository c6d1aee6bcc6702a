// Streaming M = 1 GEMV kernels of format 6 (the template is in qgemv_stream.h).
#include "qgemv_stream.h"

namespace vq {

VQ_ST_PICK(6)

}  // namespace vq
