// Attention for the element types and head dims the tuned kernels of attention.hip do not take:
// f32 tensors (the reference's Float32 path, the partner of the f32 int8 LoRA linear), and bf16 /
// f16 tensors whose head dim is not 64 or 128 (any D up to 128). memory_efficient_attention and
// its backward (src/layers/attention.jl:106-221) are generic in both.
//
// Everything is f32 in value; unlike the tuned kernels the probabilities and dS are not rounded to
// the element type (the reference's own order: scores, softmax and P V in Float32), and only the
// results are. The products run on bf16 MFMA with f32 sums: every f32 operand is taken apart into
// three bf16 values that sum to it exactly (an f16 one into two, a bf16 one is itself), and a
// product keeps the pairs of parts i, j with i + j <= 2; the pairs left out are below 2^-25 of the
// product, with random sign (parts are the nearest bf16 values: a second part is at most 2^-9, a third
// 2^-18 of the element; with truncated first parts the pairs reached 2^-23). Six (f32) or three (P times
// a bf16 tensor) products at 16 times the rate of fp32 MFMA, and from sums of two terms on they come out
// closer to 64 bits than a chain of v_mfma_f32_16x16x4_f32 (fewer roundings; small pairs are added before
// large ones or in accumulators of their own): dP of normal f32 data, rms error over the norms at head
// dim 1, 2, 3: 2.60e-8, 1.84e-8, 1.54e-8 against 2.53e-8, 2.62e-8, 2.43e-8; at 128 (emulated) 3.2e-9
// against 1.8e-8.
// Deterministic: no atomics, fixed summation order.
//
// MFMA layouts (v_mfma_f32_16x16x32_bf16): lane l holds row l % 16 of A and of B with k = 8 (l / 16)
// + (0..7), and D[4 g + v][l % 16], v = 0..3, g = l / 16. A score product S^T = K Q^T leaves lane
// (query l % 16, g) holding keys 4 g + v of a 16-key tile; the product that consumes those
// probabilities takes the lane's 8 k slots as keys {4 g ..} and {16 + 4 g ..} of a 32-key block,
// which are its own scores: no lane exchange. The transposed operand of that product is read from
// the row-major LDS tile with ds_read_b64_tr_b16 in the same key order.
//
// Measured, forward / backward: 1560 tokens, 12 heads x 128, f32: 148 / 425 us (fp32 MFMA
// with single-element LDS reads: 610 / 1556); 2 x 1024 tokens, 16 heads x 80, bf16: 46 /
// 115 us (460 / 1143). The f32 kernels are bound by their MFMAs and LDS fragment reads (6 MFMAs
// per 3 fragments of 1 KiB), the 16-bit ones by the VALU work per score (exponential and split).
//
// One source file per element type (attention_g_f32.hip, attention_g_f16.hip, attention_g_bf16.hip)
// includes this one and instantiates its launchers: 84 kernels each, which then build side by side.
#pragma once
#include <algorithm>
#include <cmath>
#include <mutex>

#include "attention_g.h"

namespace reels {

// bf16 parts of an input element
template <int ELT> constexpr int kParts = ELT == REELS_HIP_F32 ? 3 : (ELT == REELS_HIP_F16 ? 2 : 1);

template <int ELT>
__device__ __forceinline__ void attg_st(void* p, int64_t i, float x) {
  if constexpr (ELT == REELS_HIP_F32) static_cast<float*>(p)[i] = x;
  else static_cast<uint16_t*>(p)[i] = (uint16_t)Elt<ELT>::bits(x);
}

namespace attg {
constexpr int QW = 16;  // queries (forward, dQ) or keys (dK / dV) per wave
}  // namespace attg

// visibility modes as in attention.hip: 0 bounds only, 1 causal, 2 mask (and causal if set)
template <int VM>
__device__ __forceinline__ bool attg_visible(const AttgArgs& a, int64_t qi, int64_t kj, uint32_t mask) {
  bool in = (kj < a.Sk) & (qi < a.Sq);
  if constexpr (VM == 1) in = in & (kj <= qi);
  if constexpr (VM == 2) in = in & (mask != 0) & ((a.causal == 0) | (kj <= qi));
  return in;
}
// the mask bytes of keys kj .. kj + 3 for query qi, one byte each (0 past the ends)
__device__ __forceinline__ uint32_t mask_keys(const AttgArgs& a, int64_t qi, int64_t kj) {
  typedef uint32_t u32_any __attribute__((aligned(1)));
  if (qi >= a.Sq) return 0u;
  const uint8_t* p = a.mask + qi * a.Sk + kj;
  if (kj + 4 <= a.Sk) return *reinterpret_cast<const u32_any*>(p);
  uint32_t m = 0u;
  for (int e = 0; kj + e < a.Sk; ++e) m |= (uint32_t)p[e] << (8 * e);
  return m;
}
// the same of queries qi .. qi + 3 for key kj: byte loads from the tile's mask rows (rows q0 .. of
// rs), branch-free, or one by one where 32-bit offsets would not reach
__device__ __forceinline__ uint32_t mask_queries(const AttgArgs& a, const __amdgpu_buffer_rsrc_t& rs,
                                                 int64_t q0, int row, int64_t kj) {
  uint32_t m = 0u;
  if (a.Sk < (1 << 24)) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t off = kj < a.Sk ? (uint32_t)((row + e) * a.Sk + kj) : 0x80000000u;
      m |= ((uint32_t)__builtin_amdgcn_raw_buffer_load_b8(rs, off, 0, 0) & 0xffu) << (8 * e);
    }
  } else {
    for (int e = 0; e < 4; ++e)
      if (kj < a.Sk && q0 + row + e < a.Sq) m |= (uint32_t)a.mask[(q0 + row + e) * a.Sk + kj] << (8 * e);
  }
  return m;
}

__device__ __forceinline__ f32x4 mfma_bf(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t pk_bf16(float a, float b) { return Elt<REELS_HIP_BF16>::pack2_fast(a, b); }

// 8 f32 values into three bf16 parts (nearest; finite values below bf16's range end: probabilities
// and dS)
__device__ __forceinline__ void split8(const float* x, u32x4 (&o)[3]) {
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const float a = x[2 * d], b = x[2 * d + 1];
    const uint32_t h = pk_bf16(a, b);
    const float ra = a - bf16_lo(h), rb = b - bf16_hi(h);
    const uint32_t m = pk_bf16(ra, rb);
    o[0][d] = h;
    o[1][d] = m;
    o[2][d] = pk_bf16(ra - bf16_lo(m), rb - bf16_hi(m));
  }
}
// the same for input elements; NaN stays NaN. Of two parts (f16) the first is taken by truncation, so that
// the second has the element's sign, and an Inf is in the first. Of three the first is the nearest bf16
// value, or the truncated one where nearest would pass the end of the range, and an Inf is all in the
// last, which is only multiplied by first parts (nonzero unless the element is). That selection runs
// only where some lane of the wave meets an Inf, a NaN or such a value.
template <int NI>
__device__ __forceinline__ void split8_in(const float* x, u32x4 (&o)[NI]) {
  uint32_t top = 0u;  // largest magnitude pattern of the 8
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t u = __float_as_uint(x[e]) & 0x7fffffffu;
    top = u > top ? u : top;
  }
  auto parts = [&](auto special) {
    constexpr bool SP = decltype(special)::value;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      float r[2];
      uint32_t h[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float v = x[2 * d + e];
        if (NI > 2 && !SP) continue;
        const bool inf = SP && __builtin_isinf(v);
        h[e] = NI > 2 && inf ? 0u : __float_as_uint(v) & 0xffff0000u;
        r[e] = NI > 2 || !inf ? v - __uint_as_float(h[e]) : 0.0f;
      }
      if constexpr (NI > 2 && !SP) {
        o[0][d] = pk_bf16(x[2 * d], x[2 * d + 1]);
        r[0] = x[2 * d] - bf16_lo(o[0][d]);
        r[1] = x[2 * d + 1] - bf16_hi(o[0][d]);
      } else {
        o[0][d] = __builtin_amdgcn_perm(h[1], h[0], 0x07060302u);
      }
      if constexpr (NI == 2) o[1][d] = pk_bf16(r[0], r[1]);
      if constexpr (NI > 2) {
        const float m0 = SP && __builtin_isinf(r[0]) ? 0.0f : r[0], m1 = SP && __builtin_isinf(r[1]) ? 0.0f : r[1];
        o[1][d] = pk_bf16(m0, m1);
        o[2][d] = pk_bf16(r[0] - bf16_lo(o[1][d]), r[1] - bf16_hi(o[1][d]));
      }
    }
  };
  if (__builtin_amdgcn_ballot_w64(top >= (NI > 2 ? 0x7f7f8000u : 0x7f800000u))) parts(std::true_type{});
  else parts(std::false_type{});
}

// dS: infinite where dY or V is (finite it stays below half of the range). As for input elements an Inf is
// then all in the last part, so that it meets first parts only.
__device__ __forceinline__ void split8_ds(const float* x, u32x4 (&o)[3]) {
  float top = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) top = fmaxf(top, fabsf(x[e]));
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(top == INFINITY) != 0, 0)) split8_in<3>(x, o);
  else split8(x, o);
}

// 8 consecutive elements of a row: raw from memory, then as bf16 parts. Buffer loads, so rows and
// elements past the end read zeros without a branch. VEC (rows 16-byte aligned, decided on the
// host): 16-byte loads, of which D % 4 (f32) or D % 8 elements are never split; else one by one.
template <int ELT> struct Raw8 {
  static constexpr int NI = kParts<ELT>;
  u32x4 r[ELT == REELS_HIP_F32 ? 2 : 1];
  __device__ __forceinline__ void load(const __amdgpu_buffer_rsrc_t& rs, bool row_ok, uint32_t row_off,
                                       int d0, int D, bool vec) {
    constexpr uint32_t OOB = 0x80000000u;
    if constexpr (ELT == REELS_HIP_F32) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int d = d0 + 4 * i;
        if (vec) {
          r[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                               rs, row_ok && d < D ? row_off + 4 * d : OOB, 0, 0));
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            r[i][e] = __builtin_amdgcn_raw_buffer_load_b32(rs, row_ok && d + e < D ? row_off + 4 * (d + e) : OOB, 0, 0);
        }
      }
    } else {
      if (vec) {
        r[0] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                             rs, row_ok && d0 < D ? row_off + 2 * d0 : OOB, 0, 0));
      } else {
        uint32_t v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)
          v[e] = __builtin_amdgcn_raw_buffer_load_b16(rs, row_ok && d0 + e < D ? row_off + 2 * (d0 + e) : OOB, 0, 0) & 0xffffu;
#pragma unroll
        for (int e = 0; e < 4; ++e) r[0][e] = v[2 * e] | (v[2 * e + 1] << 16);
      }
    }
  }
  __device__ __forceinline__ void parts(u32x4 (&o)[NI]) const {
    if constexpr (ELT == REELS_HIP_BF16) {
      o[0] = r[0];
    } else {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if constexpr (ELT == REELS_HIP_F32) x[e] = __uint_as_float(r[e >> 2][e & 3]);
        else x[e] = (e & 1) ? Elt<ELT>::hi(r[0][e >> 1]) : Elt<ELT>::lo(r[0][e >> 1]);
      }
      split8_in<NI>(x, o);
    }
  }
};

// one (batch, head) of a [B][S][H][D] tensor
struct GRows {
  __amdgpu_buffer_rsrc_t rs;
  uint32_t stride;  // bytes from one token to the next
  int64_t S;
};
template <int ELT>
__device__ __forceinline__ GRows attg_rows(const void* p, int64_t b, int64_t h, int64_t S, int64_t H, int64_t D) {
  constexpr int ES = ELT == REELS_HIP_F32 ? 4 : 2;
  GRows g;
  const uint8_t* base = static_cast<const uint8_t*>(p) + (b * S * H + h) * D * ES;
  g.rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), (short)0,
                                           S > 0 ? (int)(((S - 1) * H + 1) * D * ES) : 0, 0x00020000);
  g.stride = (uint32_t)(H * D * ES);
  g.S = S;
  return g;
}

// An LDS tile of R rows in NI parts: part p of row r starts at (p R + r) PITCH bytes. The 32 bytes
// added to a row put 8 consecutive rows on all 64 banks for the 32-byte pieces of the transposed
// reads, and the fragment reads of 16 rows (two 8-lane groups per pass, one chunk apart) on distinct
// banks. A thread moves pieces of 8 elements: registers first (load), then parts to LDS (store).
template <int ELT, int R, int DP, int NT> struct GTile {
  static constexpr int NI = kParts<ELT>, PITCH = DP * 2 + 32, BYTES = NI * R * PITCH;
  static constexpr int CPR = DP / 8, N = R * CPR, PT = (N + NT - 1) / NT;
  Raw8<ELT> raw[PT];
  __device__ __forceinline__ void load(const GRows& g, int64_t row0, int D, bool vec) {
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int id = threadIdx.x + NT * i, row = id / CPR;
      const bool ok = id < N && row0 + row < g.S;
      raw[i].load(g.rs, ok, (uint32_t)(row0 + row) * g.stride, id % CPR * 8, D, vec);
    }
  }
  __device__ __forceinline__ void store(uint8_t* lds) const {
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int id = threadIdx.x + NT * i, row = id / CPR;
      if (N % NT != 0 && id >= N) break;
      u32x4 o[NI];
      raw[i].parts(o);
#pragma unroll
      for (int p = 0; p < NI; ++p)
        *reinterpret_cast<u32x4*>(lds + (p * R + row) * PITCH + id % CPR * 16) = o[p];
    }
  }
  // fragment of row r, elements 32 kb + 8 g ..
  static __device__ __forceinline__ u32x4 frag(const uint8_t* lds, int p, int r, int kb, int g) {
    return *reinterpret_cast<const u32x4*>(lds + (p * R + r) * PITCH + kb * 64 + g * 16);
  }
  // transposed fragment: lane i16 gets column c + i16 of rows r0 .. r0 + 3 and r0 + 16 .. r0 + 19
  static __device__ __forceinline__ u32x4 frag_tr(const uint8_t* lds, int p, int r0, int c, int i16) {
    const uint8_t* q = lds + (p * R + r0 + (i16 >> 2)) * PITCH + (c + 4 * (i16 & 3)) * 2;
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(i16x4, q));
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(i16x4, q + 16 * PITCH));
    const u32x2 l = __builtin_bit_cast(u32x2, lo), h = __builtin_bit_cast(u32x2, hi);
    return u32x4{l[0], l[1], h[0], h[1]};
  }
};

// The products of 32 rows of a tile, read transposed, with the parts b of P or dS, over the NDT 16-wide
// blocks of the head dim in groups: run calls add(block, i + j, tile part i, b[j]) for the pairs of parts
// i + j <= 2, smallest first; first loads the first group's fragments ahead of it.
template <typename T, int NI, int NDT> struct GProducts {
  static constexpr int G = NI == 1 ? 4 : 2;
  u32x4 head[G][NI];
  static __device__ __forceinline__ void load(const uint8_t* tile, int row, int l16, int d0, u32x4 (&f)[G][NI]) {
#pragma unroll
    for (int i = 0; i < G; ++i)
#pragma unroll
      for (int q = 0; q < NI; ++q)
        if (d0 + i < NDT) f[i][q] = T::frag_tr(tile, q, row, 16 * (d0 + i), l16);
  }
  __device__ __forceinline__ void first(const uint8_t* tile, int row, int l16) { load(tile, row, l16, 0, head); }
  template <typename Add>
  __device__ __forceinline__ void run(const uint8_t* tile, int row, int l16, const u32x4 (&b)[3], Add&& add) {
    auto group = [&](int d0, const u32x4 (&f)[G][NI]) {
#pragma unroll
      for (int s = 2; s >= 0; --s)
#pragma unroll
        for (int q = 0; q < NI; ++q)
#pragma unroll
          for (int i = 0; i < G; ++i)
            if (s - q >= 0 && d0 + i < NDT) add(d0 + i, s, f[i][q], b[s - q]);
    };
    group(0, head);
#pragma unroll
    for (int d0 = G; d0 < NDT; d0 += G) {
      u32x4 f[G][NI];
      load(tile, row, l16, d0, f);
      group(d0, f);
    }
  }
};

// acc_hi + acc_lo += A B over the pairs of parts i + j <= 2: the pair (0, 0) into hi, the others,
// smallest first, into lo
template <int NA, int NB>
__device__ __forceinline__ void mfma_parts2(const u32x4 (&a)[NA], const u32x4 (&b)[NB], f32x4& hi, f32x4& lo) {
#pragma unroll
  for (int s = 2; s > 0; --s)
#pragma unroll
    for (int i = 0; i < NA; ++i)
      if (s - i >= 0 && s - i < NB) lo = mfma_bf(a[i], b[s - i], lo);
  hi = mfma_bf(a[0], b[0], hi);
}

// The score (or dP) of the two accumulators. Of two-part operands an infinite element lies in a first
// part, and its product with a second part of zero is NaN: a sum of first parts that is not finite is the
// score by itself (a first part is zero only where the element is, so its infinities and NaNs are the
// score's). 1 to 2% of the backward; the forward, where it took 5%, makes its second parts nonzero instead.
template <int NI>
__device__ __forceinline__ float score(float hi, float lo) {
  if constexpr (NI == 1) return hi;
  if constexpr (NI == 2) return __builtin_isfinite(hi) ? hi + lo : hi;
  return hi + lo;
}

// Probabilities are powers of two: 2^(s ch + s cl - off) of a raw score s, scale log2(e) in two parts
// (one f32 constant would be off by up to 2^-24 of the exponent for every score alike). cl > 0, so a
// score of -Inf stays -Inf. v_exp_f32 is within an ulp (results below the f32 normal range are zero).
__device__ __forceinline__ float exp2_f(float x) { return __builtin_amdgcn_exp2f(x); }
// lse log2(e) in two parts, for the exponents of the backward
__device__ __forceinline__ float lse2_hi(float lse) { return lse * 1.44269502f; }
__device__ __forceinline__ float lse2_lo(float lse, float hi) {
  return fmaf(lse, 1.92596299e-8f, fmaf(lse, 1.44269502f, -hi));
}

// own rows of a wave as MFMA operands: row of lane l16, parts x 32-element blocks. NONZERO: the second of
// two parts is 2^-126 with the element's sign where it would be zero (and the element is not), which
// leaves the sum of two f16 products as it is and an infinity times it the infinity it is times the
// element.
template <int ELT, int DP, bool NONZERO = false>
__device__ __forceinline__ void attg_frags(const GRows& g, int64_t row, int lq, int D, bool vec,
                                           u32x4 (&f)[DP / 32][kParts<ELT>]) {
#pragma unroll
  for (int kb = 0; kb < DP / 32; ++kb) {
    Raw8<ELT> r;
    r.load(g.rs, row < g.S, (uint32_t)row * g.stride, kb * 32 + lq * 8, D, vec);
    r.parts(f[kb]);
    if constexpr (NONZERO && kParts<ELT> == 2) {
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const uint32_t a = f[kb][0][d], b = f[kb][1][d];
        uint32_t lo = b & 0xffffu, hi = b >> 16;
        if ((lo & 0x7fffu) == 0u && (a & 0x7fffu) != 0u) lo = (a & 0x8000u) | 0x0080u;
        if ((hi & 0x7fffu) == 0u && (a & 0x7fff0000u) != 0u) hi = ((a >> 16) & 0x8000u) | 0x0080u;
        f[kb][1][d] = lo | (hi << 16);
      }
    }
  }
}

// keys (forward, dQ) or queries (dK / dV) per LDS tile: the parts of a wider type fill the LDS of a
// longer tile of a narrower one
template <int ELT> constexpr int kTileRows = ELT == REELS_HIP_BF16 ? 64 : 32;

// The two streamed tensors' tiles pass through two LDS stages: in step j the waves multiply stage
// j % 2, put tile j + 1 (in registers since step j - 1) into the other stage and start loading tile
// j + 2; one barrier ends the step. The older half of the waves fills the stage before it multiplies,
// the younger half after, so that on each SIMD one wave's splitting runs beside the other's MFMAs.
// step(stage, row0) multiplies; extra(stage, row0, load) moves whatever else a tile carries.
template <typename T, typename Step, typename Extra>
__device__ __forceinline__ void attg_stream(const GRows& r0, const GRows& r1, int64_t beg, int64_t end, int rows,
                                            int D, bool vec, uint8_t* smem, bool fill_first, Step&& step,
                                            Extra&& extra) {
  if (beg >= end) return;  // uniform over the workgroup
  T t0, t1;
  auto load = [&](int64_t row) {
    t0.load(r0, row, D, vec);
    t1.load(r1, row, D, vec);
    extra(0, row, true);
  };
  auto store = [&](int stage, int64_t row) {
    t0.store(smem + stage * 2 * T::BYTES);
    t1.store(smem + (stage * 2 + 1) * T::BYTES);
    extra(stage, row, false);
  };
  load(beg);
  store(0, beg);
  if (beg + rows < end) load(beg + rows);
  __syncthreads();
  int stage = 0;
  for (int64_t row = beg; row < end; row += rows, stage ^= 1) {
    const bool more = row + rows < end;
    auto fill = [&]() {
      store(stage ^ 1, row + rows);
      if (row + 2 * rows < end) load(row + 2 * rows);
    };
    if (more && fill_first) fill();
    step(smem + stage * 2 * T::BYTES, smem + (stage * 2 + 1) * T::BYTES, stage, row);
    if (more && !fill_first) fill();
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------------------------
// forward: a workgroup takes 16 NW queries of one (batch, head), 16 per wave, and streams the keys.
// Online softmax (attention.jl:136-160): probabilities at most 1, so that values up to the end of the
// range cannot overflow the sums; the rescale runs only when some query of the wave meets a new
// maximum.
template <int ELT, int DP, int VM, int NW>
__global__ __launch_bounds__(NW * 64, 2) void attng_fwd_kernel(AttgArgs a, int vec) {
  using namespace attg;
  constexpr int NI = kParts<ELT>, KT = kTileRows<ELT>, NKB = DP / 32, NDT = DP / 16, WB = NW * QW;
  using T = GTile<ELT, KT, DP, NW * 64>;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int t = threadIdx.x, lane = t & 63, l16 = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int64_t b = blockIdx.z, h = blockIdx.y, H = a.H, Sq = a.Sq, Sk = a.Sk;
  const int D = (int)a.D;
  const int64_t qi = (int64_t)blockIdx.x * WB + w * QW + l16;  // this lane's query
  const GRows rq = attg_rows<ELT>(a.q, b, h, Sq, H, D), rk = attg_rows<ELT>(a.k, b, h, Sk, H, D),
              rv = attg_rows<ELT>(a.v, b, h, Sk, H, D);
  u32x4 qf[NKB][NI];
  attg_frags<ELT, DP, true>(rq, qi, g, D, vec, qf);
  f32x4 oacc[NDT];  // O^T: lane holds d = 16 dt + 4 g + v of query qi
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) oacc[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // the running maximum of the raw scores, the exponents' offset, this lane's part of the sum
  float m = -INFINITY, off = 0.0f, l = 0.0f;
  // keys past the last one any query of this workgroup can see (causal) need no tile
  const int64_t kvis = (int64_t)(blockIdx.x + 1) * WB;
  const int64_t kend = a.causal && kvis < Sk ? kvis : Sk;
  // FIRST: the pass over the keys; else the second one (below), which keeps m and adds the first
  // parts of P only
  // FULL: every key of the tile exists and is visible (no mask, not causal)
  auto step = [&](const uint8_t* sk, const uint8_t* sv, int64_t k0, auto first, auto full) {
    constexpr bool FIRST = decltype(first)::value, FULL = decltype(full)::value;
    uint32_t mk[KT / 16];
#pragma unroll
    for (int u = 0; u < KT / 16; ++u) mk[u] = VM == 2 ? mask_keys(a, qi, k0 + 16 * u + 4 * g) : 0u;
    // S^T per 16-key tile u: lane holds keys k0 + 16 u + 4 g + v of query qi
    float sc[KT / 16][4];
    float bmax = -INFINITY;
#pragma unroll
    for (int u0 = 0; u0 < KT / 16; u0 += 2) {
      f32x4 sh[2], sl[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) sh[u] = sl[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          u32x4 kf[NI];
#pragma unroll
          for (int p = 0; p < NI; ++p) kf[p] = T::frag(sk, p, 16 * (u0 + u) + l16, kb, g);
          mfma_parts2(kf, qf[kb], sh[u], sl[u]);
        }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int64_t kj = k0 + 16 * (u0 + u) + 4 * g + v;
          const float s = NI > 1 ? sh[u][v] + sl[u][v] : sh[u][v];
          sc[u0 + u][v] = FULL || attg_visible<VM>(a, qi, kj, (mk[u0 + u] >> (8 * v)) & 0xffu) ? s : -INFINITY;
          bmax = fmaxf(bmax, sc[u0 + u][v]);
        }
    }
    // with no visible key so far (m = -Inf) there is nothing to rescale; the reference's
    // exp(-Inf - -Inf) = NaN there would only reach queries that see no key at all
    if (FIRST && __builtin_amdgcn_ballot_w64(bmax > m)) {
      const float nmax = fmaxf(m, wave_max16(bmax));
      // the exponents' offset: about the new maximum's exponent. It stays finite while a query has seen
      // scores of -Inf alone, whose probabilities then come out as zero
      const float noff = nmax == -INFINITY ? 0.0f : nmax * a.ch;
      const float ps = nmax == -INFINITY || m == -INFINITY ? (nmax == -INFINITY ? 1.0f : 0.0f) : exp2_f(off - noff);
      m = nmax;
      off = noff;
      l *= ps;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int v = 0; v < 4; ++v) oacc[dt][v] *= ps;
    }
#pragma unroll
    for (int kb = 0; kb < KT / 32; ++kb) {
      float p[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = sc[2 * kb + (e >> 2)][e & 3];
        const float pe = exp2_f(fmaf(x, a.ch, fmaf(x, a.cl, -off)));
        p[e] = !FULL && x == -INFINITY ? 0.0f : pe;
        if (FIRST) l += p[e];
      }
      u32x4 pb[3];
      split8(p, pb);
      // O^T += V^T P^T, smallest pairs of parts first
      constexpr int G = NI == 1 ? 4 : 2;
#pragma unroll
      for (int d0 = 0; d0 < NDT; d0 += G) {
        u32x4 vf[G][NI];
#pragma unroll
        for (int i = 0; i < G; ++i)
#pragma unroll
          for (int q = 0; q < NI; ++q)
            if (d0 + i < NDT) vf[i][q] = T::frag_tr(sv, q, 32 * kb + 4 * g, 16 * (d0 + i), l16);
#pragma unroll
        for (int s = 2; s >= 0; --s)
#pragma unroll
          for (int q = 0; q < NI; ++q)
#pragma unroll
            for (int i = 0; i < G; ++i)
              if (s - q >= 0 && (FIRST || s == q) && d0 + i < NDT)
                oacc[d0 + i] = mfma_bf(vf[i][q], pb[s - q], oacc[d0 + i]);
      }
    }
  };
  const auto none_extra = [](int, int64_t, bool) {};
  attg_stream<T>(rk, rv, 0, kend, KT, D, vec, smem, w < NW / 2,
                 [&](const uint8_t* sk, const uint8_t* sv, int, int64_t k0) {
                   if (VM == 0 && k0 + KT <= Sk) step(sk, sv, k0, std::true_type{}, std::true_type{});
                   else step(sk, sv, k0, std::true_type{}, std::false_type{});
                 },
                 none_extra);
  // An infinite value times a low part of P (zero or negative) is NaN where P times it is that
  // infinity. If any output of the workgroup is NaN, its keys are walked again with P rounded to its
  // first part, which is positive wherever P is, and a NaN that is an infinity there becomes it.
  bool bad = false;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int v = 0; v < 4; ++v) bad |= oacc[dt][v] != oacc[dt][v];
  if (__syncthreads_or(bad && qi < Sq && m != -INFINITY)) {
    f32x4 keep[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
      keep[dt] = oacc[dt];
      oacc[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    attg_stream<T>(rk, rv, 0, kend, KT, D, vec, smem, w < NW / 2,
                   [&](const uint8_t* sk, const uint8_t* sv, int, int64_t k0) {
                   if (VM == 0 && k0 + KT <= Sk) step(sk, sv, k0, std::false_type{}, std::true_type{});
                   else step(sk, sv, k0, std::false_type{}, std::false_type{});
                 },
                   none_extra);
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (keep[dt][v] == keep[dt][v]) oacc[dt][v] = keep[dt][v];
  }
  l = wave_sum16(l);
  if (qi >= Sq) return;
  // out = acc / l, lse = off ln(2) + log(l); a query without a visible key: NaN output, lse NaN (-Inf
  // without keys: the reference's -Inf + log(0))
  const bool none = m == -INFINITY;
  const int64_t ob = ((b * Sq + qi) * H + h) * D;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int d = 16 * dt + 4 * g + v;
      if (d < D) attg_st<ELT>(a.o, ob + d, none ? NAN : oacc[dt][v] / l);
    }
  if (g == 0 && a.lse_out) a.lse_out[(b * H + h) * Sq + qi] = none ? (Sk == 0 ? -INFINITY : NAN) : fmaf(off, 0.693147182f, fmaf(off, -1.90465421e-9f, logf(l)));
}

// correction[q] = sum(dy .* out) over the head dim (attention.jl:190), in f32: 16 lanes per row,
// each the elements l16, l16 + 16, .. in order, then a fixed tree over the lanes
template <int ELT>
__global__ __launch_bounds__(256) void attng_corr_kernel(AttgArgs a, int64_t B) {
  const int l16 = threadIdx.x & 15;
  const int64_t i = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);  // (b, q, h) in memory order
  const bool in = i < B * a.Sq * a.H;
  float s = 0.0f;
  for (int64_t d = l16; in && d < a.D; d += 16) {
    float x, y;
    if constexpr (ELT == REELS_HIP_F32) {
      x = static_cast<const float*>(a.dy)[i * a.D + d];
      y = static_cast<const float*>(a.out)[i * a.D + d];
    } else {
      x = Elt<ELT>::to_f32(static_cast<const uint16_t*>(a.dy)[i * a.D + d]);
      y = Elt<ELT>::to_f32(static_cast<const uint16_t*>(a.out)[i * a.D + d]);
    }
    s += x * y;
  }
#pragma unroll
  for (int k = 1; k < 16; k <<= 1) s += __shfl_xor(s, k);
  if (!in || l16 != 0) return;
  const int64_t h = i % a.H, q = (i / a.H) % a.Sq, b = i / (a.H * a.Sq);
  a.corr[(b * a.H + h) * a.Sq + q] = s;
}

// dK and dV: a workgroup takes 16 NW keys of one (batch, head), 16 per wave, their K and V parts in
// registers, and streams the queries (from the first that can see them when causal). With
// S = Q K^T a lane holds queries 4 g + v of a 16-query tile for key kj, and the dV / dK products take
// queries {4 g ..} and {16 + 4 g ..} of a 32-query block in its k slots: dV^T += dY^T P, dK^T += Q^T
// dS with dS = P (dP - correction), dP = dY V^T.
template <int ELT, int DP, int VM, int NW, bool SPLIT>
__global__ __launch_bounds__(NW * 64, 2) void attng_dkdv_kernel(AttgArgs a, int vec) {
  using namespace attg;
  constexpr int NI = kParts<ELT>, QT = kTileRows<ELT>, NKB = DP / 32, NDT = DP / 16, WB = NW * QW;
  using T = GTile<ELT, QT, DP, NW * 64>;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  __shared__ __attribute__((aligned(16))) float slse[2][2][QT], scorr[2][QT];  // lse log2(e): high, low part
  const int t = threadIdx.x, lane = t & 63, l16 = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int sp = SPLIT ? (int)blockIdx.z % a.qsplits : 0;
  const int64_t b = SPLIT ? blockIdx.z / a.qsplits : blockIdx.z, h = blockIdx.y, H = a.H, Sq = a.Sq, Sk = a.Sk;
  const int D = (int)a.D;
  const int64_t kb0 = (int64_t)blockIdx.x * WB;
  const int64_t kj = kb0 + w * QW + l16;  // this lane's key
  const GRows rq = attg_rows<ELT>(a.q, b, h, Sq, H, D), rdy = attg_rows<ELT>(a.dy, b, h, Sq, H, D),
              rk = attg_rows<ELT>(a.k, b, h, Sk, H, D), rv = attg_rows<ELT>(a.v, b, h, Sk, H, D);
  u32x4 kf[NKB][NI], vf[NKB][NI];
  attg_frags<ELT, DP>(rk, kj, g, D, vec, kf);
  attg_frags<ELT, DP>(rv, kj, g, D, vec, vf);
  // 16-bit dY: an infinite element is (in) a first part, and times a low part of P (zero or negative) no
  // number or of the other sign. dV's pairs of parts past the first have sums of their own, which count
  // where the first pair's is finite. (The first part of P is zero only where P is.)
  constexpr bool LOW = NI < 3;
  f32x4 dka[NDT], dva[NDT], dvl[LOW ? NDT : 1];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) dka[dt] = dva[dt] = dvl[LOW ? dt : 0] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // causal: queries before the workgroup's first key see none of its keys
  int64_t qstart = a.causal ? kb0 / QT * QT : 0, qend = Sq;
  if constexpr (SPLIT) {  // this workgroup's range of tiles
    const int64_t lo = (int64_t)sp * a.qper * QT, hi = lo + (int64_t)a.qper * QT;
    qstart = qstart > lo ? qstart : lo;
    qend = qend < hi ? qend : hi;
  }
  float plse = 0.0f, pcorr = 0.0f;  // a tile's lse and correction on their way to LDS (threads 0 .. QT - 1)
  auto extra = [&](int stage, int64_t q0, bool load) {
    if (t >= QT) return;
    if (load) {
      const bool in = q0 + t < Sq;
      plse = in ? a.lse[(b * H + h) * Sq + q0 + t] : 0.0f;
      pcorr = in ? a.corr[(b * H + h) * Sq + q0 + t] : 0.0f;
    } else {
      const float hi = lse2_hi(plse);
      slse[stage][0][t] = hi;
      slse[stage][1][t] = lse2_lo(plse, hi);
      scorr[stage][t] = pcorr;
    }
  };
  auto step = [&](const uint8_t* sq, const uint8_t* sdy, int stage, int64_t q0) {
    uint32_t mk[QT / 16];
    const int64_t left = Sq - q0 < QT ? Sq - q0 : QT;
    const __amdgpu_buffer_rsrc_t rm = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(VM == 2 ? a.mask + q0 * Sk : nullptr), (short)0, VM == 2 ? (int)(left * Sk) : 0, 0x00020000);
#pragma unroll
    for (int u = 0; u < QT / 16; ++u) mk[u] = VM == 2 ? mask_queries(a, rm, q0, 16 * u + 4 * g, kj) : 0u;
#pragma unroll
    for (int qb = 0; qb < QT; qb += 32) {
      float p[8], ds[8];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        f32x4 sh = {0.0f, 0.0f, 0.0f, 0.0f}, sl = sh, dh = sh, dl = sh;
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
          u32x4 qf[NI], df[NI];
#pragma unroll
          for (int q = 0; q < NI; ++q) {
            qf[q] = T::frag(sq, q, qb + 16 * u + l16, kb, g);
            df[q] = T::frag(sdy, q, qb + 16 * u + l16, kb, g);
          }
          mfma_parts2(qf, kf[kb], sh, sl);
          mfma_parts2(df, vf[kb], dh, dl);
        }
        // a hidden pair adds nothing (its query's correction is NaN when that query sees no key)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int qq = qb + 16 * u + 4 * g + v;
          const bool vis = VM == 0 || attg_visible<VM>(a, q0 + qq, kj, (mk[qb / 16 + u] >> (8 * v)) & 0xffu);
          const float s = score<NI>(sh[v], sl[v]), dp = score<NI>(dh[v], dl[v]);
          const float pv = exp2_f(fmaf(s, a.ch, -slse[stage][0][qq]) + fmaf(s, a.cl, -slse[stage][1][qq]));
          p[4 * u + v] = vis ? pv : 0.0f;
          ds[4 * u + v] = vis ? pv * (dp - scorr[stage][qq]) : 0.0f;
        }
      }
      // without a mask only the queries past Sq need hiding (their zero rows times infinite keys and
      // values are no numbers; a key past Sk is not stored): a branch that the last tile alone takes
      // (the step a second time, with bounds checks, spilled in f32: 420 -> 685 us at head dim 128)
      if (VM == 0 && left < QT) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const bool in = qb + 16 * (e >> 2) + 4 * g + (e & 3) < (int)left;
          p[e] = in ? p[e] : 0.0f;
          ds[e] = in ? ds[e] : 0.0f;
        }
      }
      // dV^T += dY^T P and dK^T += Q^T dS. dK's first fragments are on their way before the branch of
      // split8_ds, which the compiler moves no load across
      GProducts<T, NI, NDT> pr;
      u32x4 pb[3], db[3];
      split8(p, pb);
      pr.first(sdy, qb + 4 * g, l16);
      pr.run(sdy, qb + 4 * g, l16, pb, [&](int dt, int s, u32x4 t, u32x4 b) {
        if (LOW && s > 0) dvl[LOW ? dt : 0] = mfma_bf(t, b, dvl[LOW ? dt : 0]);
        else dva[dt] = mfma_bf(t, b, dva[dt]);
      });
      pr.first(sq, qb + 4 * g, l16);
      split8_ds(ds, db);
      pr.run(sq, qb + 4 * g, l16, db, [&](int dt, int, u32x4 t, u32x4 b) { dka[dt] = mfma_bf(t, b, dka[dt]); });
    }
  };
  attg_stream<T>(rq, rdy, qstart, qend, QT, D, vec, smem, w < NW / 2, step, extra);
  if (kj >= Sk) return;
  if constexpr (LOW) {
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int v = 0; v < 4; ++v) dva[dt][v] = __builtin_isfinite(dva[dt][v]) ? dva[dt][v] + dvl[dt][v] : dva[dt][v];
  }
  const int64_t ob = ((b * Sk + kj) * H + h) * D;
  if constexpr (SPLIT) {
    const int64_t plane = (int64_t)(gridDim.z / a.qsplits) * Sk * H * D;
    float* p = a.part + sp * 2 * plane + ob;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int d = 16 * dt + 4 * g + v;
        if (d < D) {
          p[d] = dva[dt][v];
          p[plane + d] = dka[dt][v];
        }
      }
    return;
  }
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int d = 16 * dt + 4 * g + v;
      if (d < D) {
        attg_st<ELT>(a.dk, ob + d, dka[dt][v] * a.scale);
        attg_st<ELT>(a.dv, ob + d, dva[dt][v]);
      }
    }
}

// dv = sum over splits of dV's partials, dk = scale times the sum of dK's, in split order, rounded to
// the element type (n elements per tensor)
template <int ELT>
__global__ __launch_bounds__(256) void attng_dkdv_sum_kernel(AttgArgs a, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float v = 0.0f, k = 0.0f;
#pragma unroll 4
  for (int sp = 0; sp < a.qsplits; ++sp) {
    v += a.part[2 * sp * n + i];
    k += a.part[(2 * sp + 1) * n + i];
  }
  attg_st<ELT>(a.dv, i, v);
  attg_st<ELT>(a.dk, i, k * a.scale);
}

// dQ: a workgroup takes 16 NW queries, 16 per wave, and streams the keys: dQ^T += K^T dS^T with
// dS^T = P^T (dP^T - correction), dP^T = V dY^T (the forward's orientation).
template <int ELT, int DP, int VM, int NW>
__global__ __launch_bounds__(NW * 64, 2) void attng_dq_kernel(AttgArgs a, int vec) {
  using namespace attg;
  constexpr int NI = kParts<ELT>, KT = kTileRows<ELT>, NKB = DP / 32, NDT = DP / 16, WB = NW * QW;
  using T = GTile<ELT, KT, DP, NW * 64>;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int t = threadIdx.x, lane = t & 63, l16 = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int64_t b = blockIdx.z, h = blockIdx.y, H = a.H, Sq = a.Sq, Sk = a.Sk;
  const int D = (int)a.D;
  const int64_t qi = (int64_t)blockIdx.x * WB + w * QW + l16;
  const GRows rq = attg_rows<ELT>(a.q, b, h, Sq, H, D), rdy = attg_rows<ELT>(a.dy, b, h, Sq, H, D),
              rk = attg_rows<ELT>(a.k, b, h, Sk, H, D), rv = attg_rows<ELT>(a.v, b, h, Sk, H, D);
  u32x4 qf[NKB][NI], df[NKB][NI];
  attg_frags<ELT, DP>(rq, qi, g, D, vec, qf);
  attg_frags<ELT, DP>(rdy, qi, g, D, vec, df);
  const float lse = qi < Sq ? a.lse[(b * H + h) * Sq + qi] : 0.0f;
  const float lh = lse2_hi(lse), ll = lse2_lo(lse, lh);
  const float corr = qi < Sq ? a.corr[(b * H + h) * Sq + qi] : 0.0f;
  f32x4 dqa[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) dqa[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // causal: keys past the workgroup's last query are seen by none of its queries
  const int64_t kvis = (int64_t)(blockIdx.x + 1) * WB;
  const int64_t kend = a.causal && kvis < Sk ? kvis : Sk;
  auto step = [&](const uint8_t* sk, const uint8_t* sv, int64_t k0, auto full) {
    constexpr bool FULL = decltype(full)::value;
    uint32_t mk[KT / 16];
#pragma unroll
    for (int u = 0; u < KT / 16; ++u) mk[u] = VM == 2 ? mask_keys(a, qi, k0 + 16 * u + 4 * g) : 0u;
#pragma unroll
    for (int kb2 = 0; kb2 < KT; kb2 += 32) {
      float ds[8];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        f32x4 sh = {0.0f, 0.0f, 0.0f, 0.0f}, sl = sh, dh = sh, dl = sh;
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
          u32x4 kf[NI], vf[NI];
#pragma unroll
          for (int q = 0; q < NI; ++q) {
            kf[q] = T::frag(sk, q, kb2 + 16 * u + l16, kb, g);
            vf[q] = T::frag(sv, q, kb2 + 16 * u + l16, kb, g);
          }
          mfma_parts2(kf, qf[kb], sh, sl);
          mfma_parts2(vf, df[kb], dh, dl);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int64_t kk = k0 + kb2 + 16 * u + 4 * g + v;
          const float s = score<NI>(sh[v], sl[v]), dp = score<NI>(dh[v], dl[v]);
          const float x = exp2_f(fmaf(s, a.ch, -lh) + fmaf(s, a.cl, -ll)) * (dp - corr);
          ds[4 * u + v] = FULL || attg_visible<VM>(a, qi, kk, (mk[kb2 / 16 + u] >> (8 * v)) & 0xffu) ? x : 0.0f;
        }
      }
      GProducts<T, NI, NDT> pr;
      u32x4 db[3];
      pr.first(sk, kb2 + 4 * g, l16);
      split8_ds(ds, db);
      pr.run(sk, kb2 + 4 * g, l16, db, [&](int dt, int, u32x4 t, u32x4 b) { dqa[dt] = mfma_bf(t, b, dqa[dt]); });
    }
  };
  attg_stream<T>(rk, rv, 0, kend, KT, D, vec, smem, w < NW / 2,
                 [&](const uint8_t* sk, const uint8_t* sv, int, int64_t k0) {
                   if (VM == 0 && k0 + KT <= Sk) step(sk, sv, k0, std::true_type{});
                   else step(sk, sv, k0, std::false_type{});
                 },
                 [](int, int64_t, bool) {});
  if (qi >= Sq) return;
  const int64_t ob = ((b * Sq + qi) * H + h) * D;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int d = 16 * dt + 4 * g + v;
      if (d < D) attg_st<ELT>(a.o, ob + d, dqa[dt][v] * a.scale);
    }
}

// ---------------------------------------------------------------------------------------------
// host side (attn_generic_fwd / _bwd, attention_g.hip)
template <typename F>
static int attg_dispatch(const AttgArgs& a, F&& f) {
  auto by_vm = [&](auto dp) {
    if (a.mask != nullptr) return f(dp, std::integral_constant<int, 2>{});
    if (a.causal) return f(dp, std::integral_constant<int, 1>{});
    return f(dp, std::integral_constant<int, 0>{});
  };
  if (a.D <= 32) return by_vm(std::integral_constant<int, 32>{});
  if (a.D <= 64) return by_vm(std::integral_constant<int, 64>{});
  if (a.D <= 96) return by_vm(std::integral_constant<int, 96>{});
  return by_vm(std::integral_constant<int, 128>{});
}

// rows start on 16-byte boundaries in every tensor the kernels read
static int attg_vec(const AttgArgs& a, int esz) {
  const int64_t row = a.D * esz;
  return row % 16 == 0 && aligned16(a.q) && aligned16(a.k) && aligned16(a.v) && aligned16(a.dy);
}

// Waves per workgroup over S own rows: eight (128 rows share each streamed tile, so its splitting
// and copies cost half per row; one workgroup per CU) unless four put no more than one workgroup on
// each CU (the grid is then the shorter the smaller its pieces). 1560 tokens x 12 heads x 128, f32,
// forward and backward 706 us with four waves everywhere (one LDS stage), 620 us with this rule.
template <typename F>
static int attg_waves(int64_t S, const AttgArgs& a, int64_t B, F&& f) {
  if (ceil_div(S, 4 * attg::QW) * a.H * B <= 256) return f(std::integral_constant<int, 4>{});
  return f(std::integral_constant<int, 8>{});
}

template <auto KERN, int ELT, int DP, int NW>
static int attg_launch(const char* name, int64_t S, const AttgArgs& a, int64_t B, hipStream_t st, int splits = 1) {
  constexpr int lds = 4 * GTile<ELT, kTileRows<ELT>, DP, NW * 64>::BYTES;
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  std::call_once(once, [] {
    attr_err = hipFuncSetAttribute((const void*)KERN, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  });
  if (attr_err != hipSuccess)
    return fail(REELS_HIP_EHIP, std::string(name) + ": hipFuncSetAttribute: " + hipGetErrorString(attr_err));
  const dim3 grid((unsigned)ceil_div(S, NW * attg::QW), (unsigned)a.H, (unsigned)(B * splits));
  { TraceScope _ts(st, name); KERN<<<grid, NW * 64, lds, st>>>(a, attg_vec(a, ELT == REELS_HIP_F32 ? 4 : 2)); }
  return check_launch(name);
}

// scale log2(e) in two f32 parts, the first rounded down
static void set_exponent(AttgArgs& a) {
  const double c = (double)a.scale * 1.4426950408889634;
  a.ch = (float)c;
  if ((double)a.ch >= c) a.ch = nextafterf(a.ch, 0.0f);
  a.cl = (float)(c - (double)a.ch);
}

template <int ELT>
int attng_fwd(const AttgArgs& args, int64_t B, hipStream_t st) {
  AttgArgs a = args;
  set_exponent(a);
  return attg_dispatch(a, [&](auto dp, auto vm) {
    constexpr int DP = decltype(dp)::value, VM = decltype(vm)::value;
    return attg_waves(a.Sq, a, B, [&](auto nw) {
      constexpr int NW = decltype(nw)::value;
      return attg_launch<attng_fwd_kernel<ELT, DP, VM, NW>, ELT, DP, NW>("attng_fwd_kernel", a.Sq, a, B, st);
    });
  });
}

// Query splits of the dK / dV pass: with fewer key blocks than CUs, as many as fill them, while the
// walk they shorten (about 2 us per tile at head dim 128) is worth the partials' traffic (16 bytes
// per element of dK and dV and split at 5 TB/s) and a launch; the partials lie in dQ's buffer, as in
// attention.hip. 2048 queries x 16 heads x 128 on 64 keys, f32:
// 297 us unsplit, 38 + 7 us on 16 splits (forward and backward 338 -> 94 us).
static int attg_splits(const AttgArgs& a, int64_t B, int esz, int rows) {
  const int64_t n = ceil_div(a.Sk, 4 * attg::QW) * a.H * B, tiles = ceil_div(a.Sq, rows);
  const int64_t one = 2 * B * a.Sk * a.H * a.D * 4;
  if (n <= 0 || n > 128) return 1;
  const int64_t room = dq_scratch_bytes(a, B, a.D, esz) / one;
  const int64_t s = std::min<int64_t>({256 / n, room, tiles / 4, 16});
  if (s < 2) return 1;
  const double walk = tiles * 2.0 * a.D / 128, cost = s * one * 2 / 5e6 + 5.0;
  return walk - walk / s > 1.5 * cost ? (int)s : 1;
}

template <int ELT>
int attng_bwd(const AttgArgs& args, int64_t B, hipStream_t st) {
  AttgArgs a = args;
  set_exponent(a);
  return attg_dispatch(a, [&](auto dp, auto vm) {
    constexpr int DP = decltype(dp)::value, VM = decltype(vm)::value;
    {
      TraceScope _ts(st, "attng_corr_kernel");
      attng_corr_kernel<ELT><<<(unsigned)ceil_div(B * a.Sq * a.H, 16), 256, 0, st>>>(a, B);
    }
    if (int rc = check_launch("attng_corr_kernel")) return rc;
    if (a.Sk > 0) {
      const int splits = attg_splits(a, B, ELT == REELS_HIP_F32 ? 4 : 2, kTileRows<ELT>);
      int rc;
      if (splits > 1) {  // fewer key blocks than CUs: four waves each
        a.part = static_cast<float*>(a.o);
        a.qsplits = splits;
        a.qper = (int)ceil_div(ceil_div(a.Sq, kTileRows<ELT>), splits);
        rc = attg_launch<attng_dkdv_kernel<ELT, DP, VM, 4, true>, ELT, DP, 4>("attng_dkdv_kernel", a.Sk, a, B, st, splits);
        if (rc) return rc;
        const int64_t n = B * a.Sk * a.H * a.D;
        { TraceScope _ts(st, "attng_dkdv_sum_kernel");
          attng_dkdv_sum_kernel<ELT><<<(unsigned)ceil_div(n, 256), 256, 0, st>>>(a, n); }
        rc = check_launch("attng_dkdv_sum_kernel");
      } else {
        rc = attg_waves(a.Sk, a, B, [&](auto nw) {
          constexpr int NW = decltype(nw)::value;
          return attg_launch<attng_dkdv_kernel<ELT, DP, VM, NW, false>, ELT, DP, NW>("attng_dkdv_kernel", a.Sk, a, B, st);
        });
      }
      if (rc) return rc;
    }
    return attg_waves(a.Sq, a, B, [&](auto nw) {
      constexpr int NW = decltype(nw)::value;
      return attg_launch<attng_dq_kernel<ELT, DP, VM, NW>, ELT, DP, NW>("attng_dq_kernel", a.Sq, a, B, st);
    });
  });
}

}  // namespace reels
