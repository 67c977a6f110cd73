// The contraction's kernels for bfloat16 logits.
#include "ml_cost.h"

namespace ml {
ML_COST_TYPE(ML_BF16)
}  // namespace ml
