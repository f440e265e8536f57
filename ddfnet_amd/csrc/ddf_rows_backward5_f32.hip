// All gradients of 5 x 5 filters in one launch, fp32 storage.
#include "ddf_rows_backward5.h"

namespace ddf {
DDF_INSTANTIATE_BACKWARD5(float)
}  // namespace ddf
