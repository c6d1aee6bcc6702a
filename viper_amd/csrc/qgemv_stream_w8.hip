// Streaming M = 1 GEMV kernels of format 8 (the template is in qgemv_stream.h).
#include "qgemv_stream.h"

namespace vq {

VQ_ST_PICK(8)

}  // namespace vq
