// Paged attention kernels instantiated for bf16 inputs (see attn_impl.h).
#include "attn_impl.h"

namespace fxpr {
namespace attn {

int run_attn_bf16(const AttnArgs& a, const LongPlan& lp, int bits, int num_requests, int max_qtiles,
                  int64_t num_tokens, hipStream_t st) {
  switch (bits) {
    case 16: return dispatch_dmax<FXPR_DTYPE_BF16, 16>(a, lp, num_requests, max_qtiles, num_tokens, st);
    case 32: return dispatch_dmax<FXPR_DTYPE_BF16, 32>(a, lp, num_requests, max_qtiles, num_tokens, st);
    default: return dispatch_dmax<FXPR_DTYPE_BF16, 64>(a, lp, num_requests, max_qtiles, num_tokens, st);
  }
}

}  // namespace attn
}  // namespace fxpr
