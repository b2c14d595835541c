// Launchers of the generic attention kernels (attention_g_impl.h) by element type, called by the entry
// points of attention.hip after their argument checks.
#include "attention_g.h"

namespace reels {

int attn_generic_fwd(const AttgArgs& a, int dtype, int64_t B, hipStream_t st) {
  if (dtype == REELS_HIP_F32) return attng_fwd<REELS_HIP_F32>(a, B, st);
  if (dtype == REELS_HIP_F16) return attng_fwd<REELS_HIP_F16>(a, B, st);
  return attng_fwd<REELS_HIP_BF16>(a, B, st);
}

int attn_generic_bwd(const AttgArgs& a, int dtype, int64_t B, hipStream_t st) {
  if (dtype == REELS_HIP_F32) return attng_bwd<REELS_HIP_F32>(a, B, st);
  if (dtype == REELS_HIP_F16) return attng_bwd<REELS_HIP_F16>(a, B, st);
  return attng_bwd<REELS_HIP_BF16>(a, B, st);
}

}  // namespace reels
