// Instantiates the head_dim 128 prefill kernels whose tile loop is scheduled assembly (bf16 / fp16, without and with
// lower bounds; without, for one and for several groups a workgroup).
#include "prefill_asm.h"

namespace pa_decode_detail {

prefill_mfma_fn pa_prefill_asm_kernel_d128(int dtype, bool lower_bounds, bool one) {
    if (dtype == PA_BF16) return lower_bounds ? prefill_asm_kernel<pa_bf16, true, 128> : one ? prefill_asm_kernel<pa_bf16, false, 128, false, true> : prefill_asm_kernel<pa_bf16, false, 128>;
    if (dtype == PA_F16) return lower_bounds ? prefill_asm_kernel<pa_f16, true, 128> : one ? prefill_asm_kernel<pa_f16, false, 128, false, true> : prefill_asm_kernel<pa_f16, false, 128>;
    return nullptr;
}

}  // namespace pa_decode_detail
