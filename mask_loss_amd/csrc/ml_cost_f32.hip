// The contraction's kernels for float32 logits.
#include "ml_cost.h"

namespace ml {
ML_COST_TYPE(ML_F32)
}  // namespace ml
