// Attention for element types and head dims outside the tuned kernels (attention_g_impl.h):
// arguments and launchers, called by the entry points of attention.hip.
#pragma once
#include "common.h"

namespace reels {

struct AttgArgs {
  const void* q;
  const void* k;
  const void* v;
  const void* out;   // backward: the forward's output
  const void* dy;
  const float* lse;  // backward: [B][H][Sq]
  float* corr;       // backward: sum(dy .* out) per query, [B][H][Sq] (workspace)
  const uint8_t* mask;
  void* o;           // forward output / dq
  void* dk;
  void* dv;
  float* lse_out;
  int64_t Sq, Sk, H, D;
  int causal;
  float scale;       // 1 / sqrt(Float32(D)) (attention.jl:129)
  float ch, cl;      // scale log2(e) = ch + cl, ch rounded down so that cl > 0 (set by the launchers)
  // dK / dV with the queries split over qsplits workgroups per key block (qper query tiles each): the
  // f32 sums of split sp go to part[sp][dV, then dK][B][Sk][H][D] (dK unscaled)
  float* part;
  int qsplits, qper;
};

// Bytes of dQ's buffer (a.o, elements of esz bytes) that partials of dK and dV may use before the dQ
// kernel fills it: none if it overlaps another operand. Args: AttArgs or AttgArgs.
template <typename Args>
inline int64_t dq_scratch_bytes(const Args& a, int64_t B, int64_t D, int esz) {
  const int64_t nq = B * a.Sq * a.H * D * esz, nk = B * a.Sk * a.H * D * esz, nl = B * a.Sq * a.H * 4;
  const uintptr_t lo = reinterpret_cast<uintptr_t>(a.o), hi = lo + (uintptr_t)nq;
  auto apart = [&](const void* p, int64_t bytes) {
    const uintptr_t b = reinterpret_cast<uintptr_t>(p);
    return p == nullptr || b >= hi || b + (uintptr_t)bytes <= lo;
  };
  const bool ok = apart(a.q, nq) && apart(a.out, nq) && apart(a.dy, nq) && apart(a.k, nk) && apart(a.v, nk) &&
                  apart(a.dk, nk) && apart(a.dv, nk) && apart(a.lse, nl) && apart(a.corr, nl) &&
                  apart(a.mask, a.Sq * a.Sk);
  return ok ? nq : 0;
}

// forward (out, lse) and backward (dq, dk, dv; corr is the [B][H][Sq] f32 workspace) for dtype
// REELS_HIP_F32, _BF16 or _F16 and 1 <= D <= 128; the caller has checked the arguments
int attn_generic_fwd(const AttgArgs& a, int dtype, int64_t B, hipStream_t st);
int attn_generic_bwd(const AttgArgs& a, int dtype, int64_t B, hipStream_t st);
// the same of one element type, instantiated in attention_g_<type>.hip
template <int ELT> int attng_fwd(const AttgArgs& a, int64_t B, hipStream_t st);
template <int ELT> int attng_bwd(const AttgArgs& a, int64_t B, hipStream_t st);

}  // namespace reels
