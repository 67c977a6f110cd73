// The contraction's host side: operand form, launch plan and dispatch on the logit
// type (kernels: ml_cost.h).
#include "ml_cost.h"

namespace ml {

// instantiated in the types' own files
#define ML_COST_EXTERN(DT)                                                           \
  extern template void plan_slots<DT>(CostPlan&, int, bool, bool, int64_t);          \
  extern template int launch_classes<DT>(const CostArgs&, const Dims&, unsigned, hipStream_t);
ML_COST_EXTERN(ML_F32)
ML_COST_EXTERN(ML_BF16)
ML_COST_EXTERN(ML_F16)

// Operands of the contraction for the call's per-logit terms (see ml_cost.h).
CostForm cost_form(const Dims& d, int dtype, const ElemParams& ep, bool force_masks) {
  CostForm f;
  // focal powers, and weights below 2^-6, leave planes of any size
  f.wide = ep.gamma_mode != 0 || (ep.ug_mode != 0 && ep.ug_min < 0.015625f);
  // bf16 table: a wide one holds label maps only, float16 counts being its right operand
  f.tab = dtype == ML_BF16 && g_use_lut && !force_masks && !(f.wide && d.counts_mode);
  // the largest power of two that keeps the planes of |z| <= zmax below 65504:
  // w softplus(|z|) <= zmax without weights, and H softplus(|z|) < 1.2 where the
  // weight is H^ug, ug >= 1, above its floor
  const float zmax = f.tab ? 63.75f : kNarrowMax;
  float most = zmax * 1.0001f;
  if (ep.ug_mode != 0 && ep.ug >= 1.f) most = std::max(1.2f, ep.ug_min * (zmax + 1.f));
  f.lg = 0;
  while (f.lg < 14 && std::max(most, 1.f) * (float)(2 << f.lg) <= 65504.f) ++f.lg;
  return f;
}

CostPlan make_cost_plan(const Dims& d, int dtype, const CostForm& f) {
  CostPlan p = bound_cost_plan(d);
  const int cnt = d.counts_mode ? d.cw : 0;
  p.pair0 = f.tab && d.pair_ok ? 1 : 0;
  const int64_t side = std::min<int64_t>(d.LB, kSideCUs);
  switch (dtype) {
    case ML_F32: plan_slots<ML_F32>(p, cnt, false, f.wide, side); break;
    case ML_BF16: plan_slots<ML_BF16>(p, cnt, f.tab, f.wide, side); break;
    case ML_F16: plan_slots<ML_F16>(p, cnt, false, f.wide, side); break;
  }
  return p;
}

int launch_cost(const CostArgs& a, const Dims& d, int dtype, hipStream_t st, unsigned classes, bool prof) {
  ProfScope ps_(prof ? "pair_cost" : nullptr, st);
  switch (dtype) {
    case ML_F32: return launch_classes<ML_F32>(a, d, classes, st);
    case ML_BF16: return launch_classes<ML_BF16>(a, d, classes, st);
    case ML_F16: return launch_classes<ML_F16>(a, d, classes, st);
  }
  return fail(ML_EINVAL, "unsupported mask logits dtype");
}

}  // namespace ml
