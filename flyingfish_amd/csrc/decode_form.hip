// Decode expert FFN in the reference's Lane16 / Lane8 reduction orders (form_kernel.cuh) for the BF16 and per-channel
// FP8 expert formats.
#include "form_kernel.cuh"

namespace ffmoe {
int decode_form_launch(int fmt, int form, const DecodeParams& p, int stage_mask, hipStream_t st) {
  if (fmt == FFMOE_FMT_BF16)
    return form == FFMOE_FORM_LANE16 ? launch_form<FmtBf16, FFMOE_FORM_LANE16_>(p, stage_mask, st) : launch_form<FmtBf16, FFMOE_FORM_LANE8_>(p, stage_mask, st);
  return form == FFMOE_FORM_LANE16 ? launch_form<FmtFp8Channel, FFMOE_FORM_LANE16_>(p, stage_mask, st)
                                   : launch_form<FmtFp8Channel, FFMOE_FORM_LANE8_>(p, stage_mask, st);
}

template <class F>
static int form_grouped_fmt(int form, int rg, const DecodeParams& p, unsigned max_groups, int stage_mask, hipStream_t st) {
  const bool l16 = form == FFMOE_FORM_LANE16;
  switch (rg) {
    case 8: return l16 ? launch_form_grouped<F, FFMOE_FORM_LANE16_, 8>(p, max_groups, stage_mask, st) : launch_form_grouped<F, FFMOE_FORM_LANE8_, 8>(p, max_groups, stage_mask, st);
    case 4: return l16 ? launch_form_grouped<F, FFMOE_FORM_LANE16_, 4>(p, max_groups, stage_mask, st) : launch_form_grouped<F, FFMOE_FORM_LANE8_, 4>(p, max_groups, stage_mask, st);
    default: return l16 ? launch_form_grouped<F, FFMOE_FORM_LANE16_, 2>(p, max_groups, stage_mask, st) : launch_form_grouped<F, FFMOE_FORM_LANE8_, 2>(p, max_groups, stage_mask, st);
  }
}
// groups of rg = 2, 4 or 8 assignments per expert (p.groups / p.counters filled by k_group_assignments)
int decode_form_grouped_launch(int fmt, int form, int rg, const DecodeParams& p, unsigned max_groups, int stage_mask, hipStream_t st) {
  if (fmt == FFMOE_FMT_BF16) return form_grouped_fmt<FmtBf16>(form, rg, p, max_groups, stage_mask, st);
  return form_grouped_fmt<FmtFp8Channel>(form, rg, p, max_groups, stage_mask, st);
}

template <class F>
static int form_rows_fmt(int form, int rg, const DecodeParams& p, long long routed, long long shared, int stage_mask, hipStream_t st) {
  const bool l16 = form == FFMOE_FORM_LANE16;
#define FF_FORM_ROWS(T) \
  (l16 ? launch_form_rows<F, FFMOE_FORM_LANE16_, T>(p, routed, shared, stage_mask, st) : launch_form_rows<F, FFMOE_FORM_LANE8_, T>(p, routed, shared, stage_mask, st))
  switch (rg) {
    case 8: return FF_FORM_ROWS(8);
    case 4: return FF_FORM_ROWS(4);
    case 2: return FF_FORM_ROWS(2);
    default: return FF_FORM_ROWS(1);
  }
#undef FF_FORM_ROWS
}
bool decode_form_rows_fit(int fmt, const DecodeParams& p) { return fmt == FFMOE_FMT_BF16 ? form_rows_fit<FmtBf16>(p) : form_rows_fit<FmtFp8Channel>(p); }
// rg: assignments of one expert per group (1: every assignment its own, no descriptors); routed, shared: upper bounds of the groups
int decode_form_rows_launch(int fmt, int form, int rg, const DecodeParams& p, long long routed, long long shared, int stage_mask, hipStream_t st) {
  if (fmt == FFMOE_FMT_BF16) return form_rows_fmt<FmtBf16>(form, rg, p, routed, shared, stage_mask, st);
  return form_rows_fmt<FmtFp8Channel>(form, rg, p, routed, shared, stage_mask, st);
}
}  // namespace ffmoe
