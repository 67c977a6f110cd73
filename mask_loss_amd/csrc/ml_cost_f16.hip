// The contraction's kernels for float16 logits.
#include "ml_cost.h"

namespace ml {
ML_COST_TYPE(ML_F16)
}  // namespace ml
