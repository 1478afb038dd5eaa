// Instantiates the single-query-row attention kernels for a f16 KV pool.
#include "decode_short.h"

namespace pa_decode_detail {
KernelSet pa_kernels_f16(int d, int nrep_t) { return with_short<pa_f16, pa_f16>(kernels_for<pa_f16, pa_f16>(d, nrep_t), d); }
}  // namespace pa_decode_detail
