// The generic attention kernels for f32 tensors (attention_g_impl.h).
#include "attention_g_impl.h"

namespace reels {
template int attng_fwd<REELS_HIP_F32>(const AttgArgs&, int64_t, hipStream_t);
template int attng_bwd<REELS_HIP_F32>(const AttgArgs&, int64_t, hipStream_t);
}  // namespace reels
