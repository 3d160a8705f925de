// head_dim 128 instantiations of the decode kernels of tq_decode_mfma.h with a
// 32-projection QJL sketch.

#include "tq_decode_mfma.h"

namespace tq {

int launch_mfma_d128_qjl(const MfmaArgs& a, int kk, hipStream_t s) { return mk::launch_mfma<128, true>(a, kk, s); }

}  // namespace tq
