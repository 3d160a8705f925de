// head_dim 96 instantiations of the decode kernels of tq_decode_mfma.h.

#include "tq_decode_mfma.h"

namespace tq {

int launch_mfma_d96(const MfmaArgs& a, int kk, hipStream_t s) { return mk::launch_mfma<96, false>(a, kk, s); }

}  // namespace tq
