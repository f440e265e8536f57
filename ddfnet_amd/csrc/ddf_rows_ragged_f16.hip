// Row-register kernels for ragged rows, fp16 storage (fp32 accumulation).
#include "ddf_rows_ragged.h"

namespace ddf {
DDF_INSTANTIATE_RAGGED(__half)
}  // namespace ddf
