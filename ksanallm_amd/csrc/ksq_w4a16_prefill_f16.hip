// The forms of the W4A16 prefill kernel for f16 (ksq_w4a16_prefill_kernel.h).
#include "ksq_w4a16_prefill_kernel.h"

namespace ksq {

bool w4a16_prefill_launch_f16(const PrefillArgs& a, int gpt, const PrefillPlan& plan, dim3 grid, dim3 block, hipStream_t s) {
  return launch_typed<_Float16>(a, gpt, plan, grid, block, s);
}

}  // namespace ksq
