// The launches of a small decode batch that take the routed experts and a block-FP8 shared expert together.
#define DGPP_GEMV_IMPL
#include "gemv_shared.hpp"

namespace dgpp_amd {
bool launch_gate_up_shared(int fmt, const SlotArgs& a, const SlotArgs& sh, const SelectArgs* sel, bool ask, hipStream_t s, hipError_t& err) {
  switch (fmt) {
    case kFmtFp8F32: return launch_gate_up_shared_fmt<kFmtFp8F32>(a, sh, sel, ask, s, err);
    case kFmtNvfp4: return launch_gate_up_shared_fmt<kFmtNvfp4>(a, sh, sel, ask, s, err);
    default: return launch_gate_up_shared_fmt<kFmtMxfp4>(a, sh, sel, ask, s, err);
  }
}
bool launch_token_down_shared(int fmt, const TokenDownArgs& a, const MatRef& shared, int k_shared, bool ask, hipStream_t s, hipError_t& err) {
  switch (fmt) {
    case kFmtFp8F32: return launch_token_down_shared_fmt<kFmtFp8F32>(a, shared, k_shared, ask, s, err);
    case kFmtNvfp4: return launch_token_down_shared_fmt<kFmtNvfp4>(a, shared, k_shared, ask, s, err);
    default: return launch_token_down_shared_fmt<kFmtMxfp4>(a, shared, k_shared, ask, s, err);
  }
}
}  // namespace dgpp_amd
