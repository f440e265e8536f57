// Row-register kernels for ragged rows, fp32.
#include "ddf_rows_ragged.h"

namespace ddf {
DDF_INSTANTIATE_RAGGED(float)
}  // namespace ddf
