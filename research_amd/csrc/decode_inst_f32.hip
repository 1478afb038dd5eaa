// Instantiates the single-query-row attention kernels for a f32 KV pool.
#include "decode_short.h"

namespace pa_decode_detail {
KernelSet pa_kernels_f32(int d, int nrep_t) { return with_short<float, float>(kernels_for<float, float>(d, nrep_t), d); }
}  // namespace pa_decode_detail
