// fp32 compute with int8 frozen weights: the reference's Float32 path (_dequantize_for_compute
// with T = Float32, src/layers/quantization.jl:61-64: W = Float32.(values) .* scales; lora_forward
// and lora_backward in Float32, src/layers/lora.jl:56-118). Every operand, intermediate and
// result is fp32.
//
// The weight product runs on bf16 MFMA without giving up a bit of its operands: an int8 code is
// exact in bf16, and an f32 activation is the exact sum of three bf16 values (8 significant bits
// each). With s = mant 2^e, the weight operand is q 2^e (exact in bf16) and
// mant multiplies the f32 sum (forward, one output column) or the activation before it is taken
// apart (dX, fl32(dy mant): one rounding, where fl32(q s) rounded the weight before). See the
// bf16-plane form of bfgemm_kernel (i8gemm.hip) for the order of the sums and their error. The
// rank-r products (h, u, dA, dB and the adapter term) stay on fp32 MFMA (v_mfma_f32_16x16x4_f32).
//
// Fast path: any K, N (below 2^20; N K below 2^30), any rank, 4-byte aligned operands, a 16-byte
// aligned workspace. The rest takes the one-output-per-thread kernels at the end of this file.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "i8gemm.h"

namespace reels {

// ---------------------------------------------------------------------------------------------
// s = mant 2^e, mant in [0.5, 1) where it multiplies the activation (dX), in [1, 2) where it multiplies
// the sum (forward), so that neither passes the end of the range before the product with s does (0 for
// s = 0). e stays in [-126, 120], where q 2^e is exact in bf16 for every code; outside it mant takes the
// rest (s below 2^-126: mant below that).
template <bool FORWARD>
__device__ __forceinline__ float scale_mant(float s, int& e) {
  int x = 0;
  (void)frexpf(s, &x);
  if (FORWARD) --x;
  e = x < -126 ? -126 : (x > 120 ? 120 : x);
  if (!(fabsf(s) < INFINITY)) e = 0;
  return ldexpf(s, -e);
}
// bf16 bits of q 2^e, p2 = 2^e
__device__ __forceinline__ uint32_t code_bits(uint32_t byte, float p2) {
  return __float_as_uint((float)(int8_t)byte * p2) >> 16;
}
__device__ __forceinline__ float pow2f(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }

// Operands of one call in one launch, by block range:
//   [0, nbw)  the weight operand: rows w[n][k] (TRANS 0, row stride Kp) or transposed wt[k][n]
//             (TRANS 1, row stride Np), q 2^e in bf16, zeros past the matrix up to the padded
//             length, and mant [N];
//   then nba blocks: at [r][Kp] = A^T (zeros past K); then nbb blocks: bt [N][r] = B^T.
struct OperandArgs {
  const int8_t* q;
  const float* s;
  uint16_t* w;
  float* mant;
  const float* A;
  const float* B;
  float* at;
  float* bt;
  int64_t N, K, Kp, Np;
  int r, nbw, nba, nbb;
  bool qvec;  // rows of q are 16-byte aligned
};
constexpr int kOpGroups = 4;  // 16-code groups per thread: their loads are in flight together

__device__ __forceinline__ u32x4 load_codes(const OperandArgs& a, int64_t n, int64_t k) {
  u32x4 v = {0u, 0u, 0u, 0u};
  if (n >= a.N) return v;
  const int8_t* p = a.q + n * a.K + k;
  if (a.qvec) {
    if (k < a.K) v = *reinterpret_cast<const u32x4*>(p);
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (k + i < a.K) v[i >> 2] |= (uint32_t)(uint8_t)p[i] << (8 * (i & 3));
  }
  return v;
}

// out[c][row] = in[row][c] for one 32 x 32 tile, zeros for rows..rows_pad
__device__ __forceinline__ void transpose_tile(const float* in, int64_t rows, int64_t cols,
                                               int64_t rows_pad, int64_t r0, int64_t c0, float* out,
                                               float (*tile)[33]) {
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int i = ty; i < 32; i += 8)
    tile[i][tx] = (r0 + i < rows && c0 + tx < cols) ? in[(r0 + i) * cols + c0 + tx] : 0.0f;
  __syncthreads();
  for (int i = ty; i < 32; i += 8)
    if (c0 + i < cols && r0 + tx < rows_pad) out[(c0 + i) * rows_pad + r0 + tx] = tile[tx][i];
}

template <bool TRANS>
__global__ __launch_bounds__(256) void f32_operands_kernel(OperandArgs a) {
  constexpr int G = kOpGroups;
  __shared__ union {
    float f[32][33];
    uint16_t w[64][66];  // [k][n], rows padded to 132 bytes
  } sm;
  const int t = threadIdx.x, b = blockIdx.x;
  if (b >= a.nbw) {
    const int c = b - a.nbw;
    if (c < a.nba) {  // A [K][r]: tiles of 32 k x 32 j, j fastest
      const int gx = (a.r + 31) / 32;
      transpose_tile(a.A, a.K, a.r, a.Kp, (int64_t)(c / gx) * 32, (int64_t)(c % gx) * 32, a.at, sm.f);
    } else {          // B [r][N]: tiles of 32 j x 32 n, n fastest
      const int d = c - a.nba, gx = (int)((a.N + 31) / 32);
      transpose_tile(a.B, a.r, a.N, a.r, (int64_t)(d / gx) * 32, (int64_t)(d % gx) * 32, a.bt, sm.f);
    }
    return;
  }
  if constexpr (!TRANS) {
    const int64_t groups = a.Kp >> 4, total = a.N * groups;
    const int64_t base = (int64_t)b * (256 * G) + t;
    u32x4 v[G];
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const int64_t i = base + 256 * j, n = i / groups;
      v[j] = load_codes(a, n, (i - n * groups) * 16);  // rows past N read as zeros
    }
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const int64_t i = base + 256 * j;
      if (i >= total) break;
      const int64_t n = i / groups, c = i - n * groups;
      int e;
      const float m = scale_mant<true>(a.s[n], e), p2 = pow2f(e);
      if (c == 0) a.mant[n] = m;
      u32x4 o[2];
#pragma unroll
      for (int d = 0; d < 8; ++d) {
        const uint32_t x = v[j][d >> 1] >> (16 * (d & 1));
        o[d >> 2][d & 3] = code_bits(x & 0xff, p2) | (code_bits((x >> 8) & 0xff, p2) << 16);
      }
      u32x4* dst = reinterpret_cast<u32x4*>(a.w + n * a.Kp + c * 16);
      dst[0] = o[0];
      dst[1] = o[1];
    }
  } else {
    // 64 x 64 tiles through LDS, G consecutive ones along k per block
    const int nkb = (int)((a.K + 64 * G - 1) / (64 * G));
    const int64_t n0 = (int64_t)(b / nkb) * 64, kb = (int64_t)(b % nkb) * 64 * G;
    const int nl = t >> 2, kl = (t & 3) * 16;
    u32x4 v[G];
#pragma unroll
    for (int i = 0; i < G; ++i) v[i] = load_codes(a, n0 + nl, kb + 64 * i + kl);
    float p2 = 0.0f;
    if (n0 + nl < a.N) {
      int e;
      const float m = scale_mant<false>(a.s[n0 + nl], e);
      p2 = pow2f(e);
      if (kb == 0 && kl == 0) a.mant[n0 + nl] = m;
    }
    const int kr = t >> 2, nc = (t & 3) * 16;
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int64_t k0 = kb + 64 * i;
      if (k0 >= a.K) break;        // uniform over the block
      if (i > 0) __syncthreads();  // the previous tile's rows have been read
#pragma unroll
      for (int j = 0; j < 16; ++j)
        sm.w[kl + j][nl] = (uint16_t)code_bits((v[i][j >> 2] >> (8 * (j & 3))) & 0xff, p2);
      __syncthreads();
      if (k0 + kr < a.K) {
        const uint32_t* row = reinterpret_cast<const uint32_t*>(&sm.w[kr][nc]);
        u32x4* dst = reinterpret_cast<u32x4*>(a.w + (k0 + kr) * a.Np + n0 + nc);
        dst[0] = u32x4{row[0], row[1], row[2], row[3]};
        dst[1] = u32x4{row[4], row[5], row[6], row[7]};
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// One pass over f32 rows src [M][Kd]: the rank-r projection out[m][j] = sum_k src[m][k] P[j][k]
// (JT 16-wide rank tiles, JT = 0: none) and, with PLANES, the three bf16 planes of the rows
// (of fl32(src mant) with mant set), planes[m][low | middle | high], each of Kp columns, zeros
// past Kd. HBM-bound (4 B read, 6 B written per element): the projection rides on the read.
// A block takes 32 rows and walks them in chunks of KC columns (256, or 128 at ranks above 32: LDS):
// every wave instruction loads a whole row segment of 1 KiB (512 B) and stores whole segments of
// the planes; the chunk and the same columns of P go to LDS while the next two chunks are in
// flight in registers (buffer loads: dword-aligned rows suffice, and rows past M and offsets past
// the buffer read zeros without a branch). Wave w multiplies columns [w KC / 4, (w + 1) KC / 4) (MFMA
// A = rows of P, B = tokens); the four partial sums are added in wave order. blockIdx.y splits the
// columns when there are few rows (partials [split][M][r], added in split order by
// f32_sum_kernel).
// 4680 tokens, r 32: x (1536) and dy (8960) together 132 us; loading each lane's MFMA operand
// straight from memory (32 rows by 64 columns per wave) took 194-207 us, one wave per 16 tokens
// over the whole reduction without the planes 466 us.
struct ProjArgs {
  const float* src;
  int64_t M, Kd, Kp;
  const float* P;      // [r][ldp]
  int64_t ldp;
  int r;               // ranks of this launch (at most 128)
  float* out;          // [M][ldo]; with part set: partials [gridDim.y][M][r] instead
  int64_t ldo;
  float* part;
  const float* mant;   // [Kd] or nullptr
  uint16_t* planes;
};

// the three bf16 values of x as the top halves of three f32 patterns (truncation; their sum is x).
// Inf keeps low parts of zero, NaN is made quiet so that its top half stays a NaN.
__device__ __forceinline__ void split3(float x, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  const uint32_t u = __float_as_uint(x);
  const bool fin = (u & 0x7f800000u) != 0x7f800000u;
  hi = (x == x ? u : 0x7fc00000u) & 0xffff0000u;
  const float r = fin ? x - __uint_as_float(hi) : 0.0f;
  mid = __float_as_uint(r) & 0xffff0000u;
  lo = __float_as_uint(r - __uint_as_float(mid));
}

template <int JT> struct ProjCfg {
  static constexpr int KC = JT <= 2 ? 256 : 128;  // columns per chunk
  static constexpr int LROW = KC + 4;             // LDS row: the rows read together start 4 banks apart
};

template <int JT, bool PLANES>
__global__ __launch_bounds__(256) void f32_project_kernel(ProjArgs a) {
  constexpr int KC = ProjCfg<JT>::KC, LROW = ProjCfg<JT>::LROW, ROWS = 32;
  constexpr int C4 = KC / 4;                 // 16-byte pieces per row of a chunk
  constexpr int NX = ROWS * C4 / 256;        // x pieces per thread (rows t / C4 + i 256 / C4)
  constexpr int NP = 16 * JT * C4 / 256;     // P pieces per thread
  constexpr int JN = JT > 0 ? JT : 1;
  constexpr int SM = JT > 0 ? (ROWS + 16 * JT) * LROW : 1;
  static_assert(JT == 0 || SM >= 4 * ROWS * 16 * JT, "the wave partials reuse the operand tiles");
  __shared__ __attribute__((aligned(16))) float sm[SM];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int l16 = lane & 15, lq = lane >> 4;
  const int64_t mb = (int64_t)blockIdx.x * ROWS, Kd = a.Kd;
  const int rows = (int)(a.M - mb < ROWS ? a.M - mb : ROWS);
  const int nch = (int)((a.Kp + KC - 1) / KC), ks = (int)gridDim.y, sp = (int)blockIdx.y;
  const int cbeg = (int)((int64_t)sp * nch / ks), cend = (int)((int64_t)(sp + 1) * nch / ks);
  auto rsrc = [](const float* p, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), (short)0, (int)bytes, 0x00020000);
  };
  const __amdgpu_buffer_rsrc_t rx = rsrc(a.src + mb * Kd, rows * Kd * 4);
  const __amdgpu_buffer_rsrc_t rm = rsrc(a.mant, a.mant != nullptr ? Kd * 4 : 0);
  const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
      a.planes + (PLANES ? mb * 3 * a.Kp : 0), (short)0, PLANES ? (int)(rows * 6 * a.Kp) : 0, 0x00020000);
  const __amdgpu_buffer_rsrc_t rp = rsrc(JT > 0 ? a.P : a.src, JT > 0 ? a.r * a.ldp * 4 : 0);
  auto ld = [](const __amdgpu_buffer_rsrc_t& rs, uint32_t off) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
  };
  const int c4 = t % C4, row0 = t / C4;
  typedef f32x4 XV[NX];
  typedef f32x4 PV[NP > 0 ? NP : 1];
  auto load = [&](int ck, XV& x, PV& p, f32x4& mt) {  // chunks past the split's last read zeros
    const int64_t k = (int64_t)ck * KC + 4 * c4;
    const bool in = ck < cend && k < Kd;
#pragma unroll
    for (int i = 0; i < NX; ++i)
      x[i] = ld(rx, in ? (uint32_t)(((row0 + i * (256 / C4)) * Kd + k) * 4) : 0x80000000u);
#pragma unroll
    for (int i = 0; i < NP; ++i)
      p[i] = ld(rp, in ? (uint32_t)(((row0 + i * (256 / C4)) * a.ldp + k) * 4) : 0x80000000u);
    if constexpr (PLANES) mt = ld(rm, in ? (uint32_t)(k * 4) : 0x80000000u);
  };
  // a chunk's registers to LDS, and its planes to memory
  auto stash = [&](int ck, XV& x, PV& p, const f32x4& mt) {
    const int64_t k = (int64_t)ck * KC + 4 * c4;
    if (k + 4 > Kd) {  // the piece across the end of a row holds the next row's first elements
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int i = 0; i < NX; ++i) x[i][e] = k + e < Kd ? x[i][e] : 0.0f;
#pragma unroll
        for (int i = 0; i < NP; ++i) p[i][e] = k + e < Kd ? p[i][e] : 0.0f;
      }
    }
    if constexpr (JT > 0) {
#pragma unroll
      for (int i = 0; i < NX; ++i)
        *reinterpret_cast<f32x4*>(&sm[(row0 + i * (256 / C4)) * LROW + 4 * c4]) = x[i];
#pragma unroll
      for (int i = 0; i < NP; ++i)
        *reinterpret_cast<f32x4*>(&sm[(ROWS + row0 + i * (256 / C4)) * LROW + 4 * c4]) = p[i];
    }
    if constexpr (PLANES) {
      if (ck < cend && k < a.Kp) {
#pragma unroll
        for (int i = 0; i < NX; ++i) {
          const int row = row0 + i * (256 / C4);
          u32x2 o[3];
#pragma unroll
          for (int d = 0; d < 2; ++d) {
            const float y0 = a.mant != nullptr ? x[i][2 * d] * mt[2 * d] : x[i][2 * d];
            const float y1 = a.mant != nullptr ? x[i][2 * d + 1] * mt[2 * d + 1] : x[i][2 * d + 1];
            uint32_t h0, m0, l0, h1, m1, l1;
            split3(y0, h0, m0, l0);
            split3(y1, h1, m1, l1);
            o[0][d] = __builtin_amdgcn_perm(l1, l0, 0x07060302u);
            o[1][d] = __builtin_amdgcn_perm(m1, m0, 0x07060302u);
            o[2][d] = __builtin_amdgcn_perm(h1, h0, 0x07060302u);
          }
          // rows past M lie past the buffer: nothing is stored
          const uint32_t off = (uint32_t)((row * 3 * a.Kp + k) * 2);
#pragma unroll
          for (int pl = 0; pl < 3; ++pl)
            __builtin_amdgcn_raw_buffer_store_b64(o[pl], ro, off + pl * (uint32_t)(2 * a.Kp), 0, 0);
        }
      }
    }
  };
  f32x4 acc[2][JN];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < JN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto compute = [&]() {
#pragma unroll
    for (int s = 0; s < KC / 64; ++s) {  // 16 columns: a lane's 4 (lq) feed 4 MFMAs
      const int col = w * (KC / 4) + s * 16 + lq * 4;
      f32x4 xf[2], pf[JN];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) xf[tt] = *reinterpret_cast<const f32x4*>(&sm[(tt * 16 + l16) * LROW + col]);
#pragma unroll
      for (int j = 0; j < JT; ++j) pf[j] = *reinterpret_cast<const f32x4*>(&sm[(ROWS + j * 16 + l16) * LROW + col]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < JT; ++j)
#pragma unroll
          for (int tt = 0; tt < 2; ++tt)
            acc[tt][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(pf[j][e], xf[tt][e], acc[tt][j], 0, 0, 0);
    }
  };
  auto step = [&](int ck, XV& x, PV& p, f32x4& mt) {
    stash(ck, x, p, mt);
    if constexpr (JT > 0) __syncthreads();
    load(ck + 2, x, p, mt);
    if constexpr (JT > 0) {
      compute();
      __syncthreads();
    }
  };
  XV x0, x1;
  PV p0, p1;
  f32x4 mt0 = {1.0f, 1.0f, 1.0f, 1.0f}, mt1 = mt0;
  load(cbeg, x0, p0, mt0);
  load(cbeg + 1, x1, p1, mt1);
  // in pairs, the second unconditional (a chunk past the end is all zeros and stores nothing): a
  // branch around it would make the compiler's waits drain both register stages
  for (int ck = cbeg; ck < cend; ck += 2) {
    step(ck, x0, p0, mt0);
    step(ck + 1, x1, p1, mt1);
  }
  if constexpr (JT > 0) {
    // the waves' sums [wave][token][16 JT], then one sum per output in wave order
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int j = 0; j < JT; ++j)
        *reinterpret_cast<f32x4*>(&sm[((w * ROWS + tt * 16 + l16) * JT + j) * 16 + lq * 4]) = acc[tt][j];
    __syncthreads();
    for (int i = t; i < ROWS * 16 * JT; i += 256) {
      const int row = i / (16 * JT), jj = i % (16 * JT);
      if (row >= rows || jj >= a.r) continue;
      constexpr int PL = ROWS * 16 * JT;
      const float s = ((sm[i] + sm[PL + i]) + sm[2 * PL + i]) + sm[3 * PL + i];
      if (a.part) a.part[((int64_t)sp * a.M + mb + row) * a.r + jj] = s;
      else a.out[(mb + row) * a.ldo + jj] = s;
    }
  }
}

// out[m][j] (row stride ldo) = sum over splits of part[sp][m][j] in split order
__global__ __launch_bounds__(256) void f32_sum_kernel(const float* __restrict__ part, int ks, int64_t M,
                                                      int r, float* __restrict__ out, int64_t ldo) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, n = M * r;
  if (i >= n) return;
  float s = 0.0f;
#pragma unroll 4
  for (int sp = 0; sp < ks; ++sp) s += part[sp * n + i];
  out[i / r * ldo + i % r] = s;
}

// ---------------------------------------------------------------------------------------------
// Column gradients c sum_m src[m][o] Lm[m][j] (src [M][Od], Lm rows of ldl floats), split over
// tokens: up to two passes (dA over x with u, dB over dy with h) in one launch, job 0 taking the
// first nb0 blocks (column block fastest). HBM-bound (src is read once). A block takes 256 columns
// of one token range, a wave 64 of them: a lane loads 16 bytes of src (columns 4 l16 .. + 3 of
// token 4 i + lq) and one element of Lm per rank tile, and element e of its 4 columns feeds the
// e-th MFMA (A = Lm^T rows j, B = columns o0 + 4 l16 + e), so nothing passes through LDS; eight
// token groups of loads are in flight per wave. Each wave writes its own sums: partials
// [split][Od][ldp], or the scaled result where one range covers all tokens.
// With BS, one job's column sums of src (the bias gradient) come from the same read: a lane adds up
// its token group's elements, the four groups are added at the end in a fixed order; JT 0 is that
// pass alone, with the same sums, so the bias gradient does not depend on the other outputs.
// 4680 tokens, r 32: both passes and the column sums 69 us, against 205 us for 64-column blocks staged
// through LDS and 33 us for column sums in passes of their own.
struct CgF32Job {
  const float* src;
  const float* Lm;
  float* part;
  float* out;  // not nullptr: one split, written directly
  int64_t Od, tps;
  int nbx, trans;
  float* bpart;  // column sums: split partials [split][Od], or (bout) the result with one split
  float* bout;
};
namespace f32c {
constexpr int BO = 256, UT = 8;  // columns per block, token groups of 4 in flight
}
template <int JT, bool BS>
__global__ __launch_bounds__(256) void colgrad_f32_kernel(CgF32Job j0, CgF32Job j1, int nb0, int64_t M,
                                                          int r, int64_t ldl, int64_t ldp, int rall,
                                                          float c) {
  using namespace f32c;
  const bool second = (int)blockIdx.x >= nb0;
  const CgF32Job& jb = second ? j1 : j0;
  const int b = second ? (int)blockIdx.x - nb0 : (int)blockIdx.x;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int l16 = lane & 15, lq = lane >> 4;
  const int64_t Od = jb.Od, o = (int64_t)(b % jb.nbx) * BO + w * 64 + 4 * l16;
  const int sp = b / jb.nbx;
  const int64_t mbeg = (int64_t)sp * jb.tps;
  const int rows = (int)(M - mbeg < jb.tps ? M - mbeg : jb.tps);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(jb.src + mbeg * Od), (short)0, (int)(rows * Od * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t rl = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(JT > 0 ? jb.Lm + mbeg * ldl : jb.src), (short)0,
      JT > 0 ? (int)(((rows - 1) * ldl + r) * 4) : 0, 0x00020000);
  f32x4 acc[4][JT > 0 ? JT : 1], bs = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int j = 0; j < JT; ++j) acc[e][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int t0 = 0; t0 < rows; t0 += 4 * UT) {
    f32x4 xv[UT];
    float lv[UT][JT > 0 ? JT : 1];
#pragma unroll
    for (int i = 0; i < UT; ++i) {
      const int tok = t0 + 4 * i + lq;
      const bool in = tok < rows && o < Od;  // columns past Od (the next row's) are not stored
      xv[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                            rs, in ? (uint32_t)((tok * Od + o) * 4) : 0x80000000u, 0, 0));
#pragma unroll
      for (int j = 0; j < JT; ++j) {
        const bool inl = tok < rows && j * 16 + l16 < r;
        lv[i][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                 rl, inl ? (uint32_t)((tok * ldl + j * 16 + l16) * 4) : 0x80000000u, 0, 0));
      }
    }
    if constexpr (BS) {
#pragma unroll
      for (int i = 0; i < UT; ++i) bs += xv[i];
    }
#pragma unroll
    for (int i = 0; i < UT; ++i)
#pragma unroll
      for (int j = 0; j < JT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[e][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(lv[i][j], xv[i][e], acc[e][j], 0, 0, 0);
  }
  if constexpr (BS) {
    if (jb.bpart != nullptr || jb.bout != nullptr) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float s = wave_sum16(bs[e]);  // over the four token groups
        if (lq == 0 && o + e < Od) {
          if (jb.bout != nullptr) jb.bout[o + e] = s;
          else jb.bpart[(int64_t)sp * Od + o + e] = s;
        }
      }
    }
  }
  // D: lane holds j = 16 jt + 4 lq + v of column o + e
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (o + e >= Od) continue;
#pragma unroll
    for (int j = 0; j < JT; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int jj = j * 16 + lq * 4 + v;
        if (jj >= r) continue;
        if (jb.out == nullptr) jb.part[((int64_t)sp * Od + o + e) * ldp + jj] = acc[e][j][v];
        else if (jb.trans) jb.out[jj * Od + o + e] = c * acc[e][j][v];
        else jb.out[(o + e) * rall + jj] = c * acc[e][j][v];
      }
  }
}

// ---------------------------------------------------------------------------------------------
// generic kernels (any shape / alignment): one output per thread, f32 sums in k order
__global__ void gf_rowproj_kernel(const float* __restrict__ src, int64_t M, int64_t Kd,
                                  const float* __restrict__ P, int64_t ps_k, int64_t ps_j, int r,
                                  float* __restrict__ out) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= M * r) return;
  const int64_t m = idx / r, j = idx % r;
  float acc = 0.0f;
  for (int64_t k = 0; k < Kd; ++k) acc += src[m * Kd + k] * P[k * ps_k + j * ps_j];
  out[idx] = acc;
}

// y = (sum_k x w + bias) + c sum_j h B, w = fl32(q s)
__global__ void gf_fwd_kernel(const float* __restrict__ x, const int8_t* __restrict__ q,
                              const float* __restrict__ s, const float* __restrict__ h,
                              const float* __restrict__ B, const float* __restrict__ bias,
                              int64_t M, int64_t K, int64_t N, int r, float c,
                              float* __restrict__ y) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= M * N) return;
  const int64_t m = idx / N, n = idx % N;
  float acc = 0.0f;
  for (int64_t k = 0; k < K; ++k) acc += x[m * K + k] * ((float)q[n * K + k] * s[n]);
  float lo = 0.0f;
  for (int j = 0; j < r; ++j) lo += h[m * r + j] * B[(int64_t)j * N + n];
  y[idx] = (acc + (bias ? bias[n] : 0.0f)) + c * lo;
}

// dx = sum_n dy w + c sum_j u A, w = fl32(q s)
__global__ void gf_dx_kernel(const float* __restrict__ dy, const int8_t* __restrict__ q,
                             const float* __restrict__ s, const float* __restrict__ u,
                             const float* __restrict__ A, int64_t M, int64_t K, int64_t N, int r,
                             float c, float* __restrict__ dx) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= M * K) return;
  const int64_t m = idx / K, k = idx % K;
  float acc = 0.0f;
  for (int64_t n = 0; n < N; ++n) acc += dy[m * N + n] * ((float)q[n * K + k] * s[n]);
  float lo = 0.0f;
  for (int j = 0; j < r; ++j) lo += u[m * r + j] * A[k * r + j];
  dx[idx] = acc + c * lo;
}

// out[o][j] (or [j][o] when TRANS) = c * sum_m src[m][o] Lm[m][j]
template <bool TRANS>
__global__ void gf_colgrad_kernel(const float* __restrict__ src, int64_t M, int64_t Od,
                                  const float* __restrict__ Lm, int r, float c,
                                  float* __restrict__ out) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= Od * r) return;
  int64_t o, j;
  if (TRANS) { j = idx / Od; o = idx % Od; } else { o = idx / r; j = idx % r; }
  float acc = 0.0f;
  for (int64_t m = 0; m < M; ++m) acc += src[m * Od + o] * Lm[m * r + j];
  out[idx] = c * acc;
}

__global__ void zero_f32_kernel(float* __restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.0f;
}

__global__ void gelu_f32_kernel(const float* __restrict__ x, float* __restrict__ y, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = gelu_f(x[i]);
}
__global__ void gelu_bwd_f32_kernel(const float* __restrict__ x, const float* __restrict__ dy,
                                    float* __restrict__ dx, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dx[i] = dy[i] * gelu_grad_f(x[i]);
}

// ---------------------------------------------------------------------------------------------
// host side
static unsigned g1(int64_t n) { return (unsigned)ceil_div(n, 256); }

// rank chunk of the projection and gradient kernels (accumulators for 128 ranks)
constexpr int kRankChunk = 128;

struct PlanF32 {
  bool fast;
  int64_t Kp, Np;        // reduction lengths padded to the GEMM's step of 64
  int64_t chf, chb;      // tokens per chunk (forward over K, dX over N)
  int psf, psb;          // column splits of the projections over K and N
  int64_t tpsa, tpsb;    // tokens per split of dA (columns K) and dB (columns N)
  int spa, spb;
};

// Tokens per chunk. The planes of one chunk take up to kPlaneBytes of the workspace (the GEMM's copies
// would address up to 2 GiB), so that a call needs no more than that beside the 16-bit weight copy. Longer
// calls run as chunks of as many 256-row tiles as give the least time: rounds of 256 x 256 tiles over the
// CUs at 2.4 us per 64-deep step and 4 for the epilogue, split partials at 5 TB/s, 3 us per chunk.
// Forward / backward and forward workspace, one chunk of up to 2 GiB against chunks: 32760 tokens on 5120 x
// 5120 4036 / 4297 us, 1015 MiB -> 4127 / 4400, 303; 16384 on 3072 x 3072 781 / 859, 307 -> 835 / 940,
// 162; 32760 on 8960 -> 1536 2476 / 2598, 1711 -> 2762 / 2640, 345; 9360 there 791 / 841 -> 795 / 842.
constexpr int64_t kPlaneBytes = (int64_t)256 << 20;
static int64_t plane_chunk(int64_t M, int64_t Kp, int64_t Ncols) {
  const int64_t most = std::max<int64_t>(kPlaneBytes / (6 * Kp) / 256, 1), tm = ceil_div(M, 256);
  if (tm <= most) return std::max<int64_t>(tm, 1) * 256;
  const int64_t tn = ceil_div(Ncols, 256);
  const double round = 2.4 * (double)(Kp / 64) + 4.0;
  auto chunk_us = [&](int64_t rows) {
    if (rows == 0) return 0.0;
    const int64_t ks = planegemm_splits(rows * 256, Ncols, Kp);
    return 3.0 + round * (double)ceil_div(rows * tn * ks, 256) / (double)ks +
           (ks > 1 ? (double)(2 * ks * rows * 256 * Ncols * 4) / 5e6 : 0.0);
  };
  int64_t best = most;
  double tbest = 1e300;
  for (int64_t t = most; t > most / 4; --t) {
    const double time = (double)(tm / t) * chunk_us(t) + chunk_us(tm % t);
    if (time < tbest) { tbest = time; best = t; }
  }
  return best * 256;
}
// most bytes of split partials of a chunk: the last, shorter one has a split of its own
static size_t plane_partials(int64_t M, int64_t chunk, int64_t Kp, int64_t Ncols) {
  size_t most = 0;
  for (int64_t m : {std::min(M, chunk), M % chunk}) {
    const int64_t ks = m > 0 ? planegemm_splits(m, Ncols, Kp) : 1;
    if (ks > 1) most = std::max(most, (size_t)(ks * m * ((Ncols + 3) / 4 * 16)));
  }
  return most;
}
// column splits of a projection: 32-row blocks, about 512 of them (two per CU)
static int project_splits(int64_t M, int64_t Kp) {
  const int64_t s = 512 / ceil_div(M > 0 ? M : 1, 32);
  return (int)std::max<int64_t>(1, std::min<int64_t>({s, ceil_div(Kp, 256), 16}));
}
// token splits of a gradient pass: about 512 blocks, at least 128 tokens each, and buffers of one
// split below 2^31 bytes
static void colgrad_split(int64_t M, int64_t Od, int64_t r, int64_t& tps, int& sp) {
  int64_t s = 512 / ceil_div(Od, f32c::BO);
  s = std::max<int64_t>(1, std::min<int64_t>({s, ceil_div(M, 128), 64}));
  tps = std::max<int64_t>(32, ceil_div(ceil_div(M, s), 32) * 32);
  const int64_t most = (((int64_t)1 << 31) - 1) / (4 * std::max<int64_t>(Od, r)) / 32 * 32;
  tps = std::min(tps, most);
  sp = (int)std::max<int64_t>(1, ceil_div(M, tps));
}

static PlanF32 plan_f32(int64_t M, int64_t K, int64_t N, int64_t r, bool aligned) {
  PlanF32 p{};
  p.Kp = (K + 63) / 64 * 64;
  p.Np = (N + 63) / 64 * 64;
  p.fast = aligned && K > 0 && N > 0 && p.Kp <= (1 << 20) && p.Np <= (1 << 20) &&
           p.Kp * p.Np * 2 < ((int64_t)1 << 31);
  if (!p.fast) return p;
  p.chf = plane_chunk(M, p.Kp, N);
  p.chb = plane_chunk(M, p.Np, K);
  p.psf = project_splits(std::min(M, p.chf), p.Kp);
  p.psb = project_splits(std::min(M, p.chb), p.Np);
  colgrad_split(M, K, r, p.tpsa, p.spa);
  colgrad_split(M, N, r, p.tpsb, p.spb);
  return p;
}

struct WsF32 {
  size_t at, bt, h, wd, mant, planes, kp, rq, u, pa, pb, pbias, total;
};

static WsF32 ws_f32(int64_t M, int64_t K, int64_t N, int64_t r, int which, const PlanF32& p) {
  WsF32 w{};
  size_t off = 0;
  auto take = [&](size_t bytes) { size_t o = off; off = align_up(off + bytes, 256); return o; };
  w.at = take((size_t)r * (p.fast ? p.Kp : K) * 4);
  w.h = take((size_t)M * r * 4);
  if (p.fast) {
    const bool fwd = which == REELS_HIP_WS_FWD;
    const int64_t ch = std::min(M, fwd ? p.chf : p.chb);
    w.wd = take((size_t)(fwd ? N * p.Kp : K * p.Np) * 2);
    w.mant = take((size_t)N * 4);
    w.planes = take((size_t)ch * 6 * (fwd ? p.Kp : p.Np));
    w.kp = take(fwd ? plane_partials(M, p.chf, p.Kp, N) : plane_partials(M, p.chb, p.Np, K));
    // split partials of the projections (the backward also recomputes h)
    const size_t rc = (size_t)std::min<int64_t>(r, kRankChunk);
    const size_t pf = p.psf > 1 ? (size_t)p.psf * std::min(M, p.chf) * rc * 4 : 0;
    const size_t pb = p.psb > 1 ? (size_t)p.psb * std::min(M, p.chb) * rc * 4 : 0;
    w.rq = take(fwd ? pf : std::max(pf, pb));
  }
  if (which == REELS_HIP_WS_FWD) {
    w.bt = take((size_t)N * r * 4);
  } else {
    w.u = take((size_t)M * r * 4);
    w.pa = take(p.fast && r > 0 && p.spa > 1 ? (size_t)p.spa * K * r * 4 : 0);
    w.pb = take(p.fast && r > 0 && p.spb > 1 ? (size_t)p.spb * N * r * 4 : 0);
    // the bias gradient's split partials
    w.pbias = take(p.fast ? (size_t)p.spb * N * 4 : colsum_partial_bytes(M, N));
  }
  w.total = off == 0 ? 256 : off;
  return w;
}

// at (A^T) and bt (B^T) only when set
static int launch_operands(bool trans, const int8_t* q, const float* s, int64_t N, int64_t K,
                           const PlanF32& p, uint16_t* w, float* mant, const float* A,
                           const float* B, int64_t r, float* at, float* bt, hipStream_t st) {
  OperandArgs a{};
  a.q = q; a.s = s; a.w = w; a.mant = mant; a.A = A; a.B = B; a.at = at; a.bt = bt;
  a.N = N; a.K = K; a.Kp = p.Kp; a.Np = p.Np; a.r = (int)r;
  a.qvec = K % 16 == 0 && aligned16(q);
  if (w) a.nbw = (int)(trans ? ceil_div(K, 64 * kOpGroups) * (p.Np / 64) : ceil_div(N * (p.Kp / 16), 256 * kOpGroups));
  if (at) a.nba = (int)(ceil_div(p.Kp, 32) * ceil_div(r, 32));
  if (bt) a.nbb = (int)(ceil_div(r, 32) * ceil_div(N, 32));
  const unsigned grid = (unsigned)(a.nbw + a.nba + a.nbb);
  if (grid == 0) return REELS_HIP_OK;
  { TraceScope _ts(st, "f32_operands_kernel");
    if (trans) f32_operands_kernel<true><<<grid, 256, 0, st>>>(a);
    else f32_operands_kernel<false><<<grid, 256, 0, st>>>(a); }
  return check_launch("f32_operands_kernel");
}

// out [M][r] = src P^T (out nullptr: no projection) and the planes of src (planes nullptr: none),
// for one token chunk; ks column splits through part
static int launch_project(const float* src, int64_t M, int64_t Kd, int64_t Kp, const float* P,
                          int64_t ldp, int r, float* out, float* part, int ks, const float* mant,
                          uint16_t* planes, hipStream_t st) {
  for (int c0 = 0; c0 == 0 || (out && c0 < r); c0 += kRankChunk) {
    ProjArgs a{};
    const int rc = out ? std::min(r - c0, kRankChunk) : 0;
    a.src = src; a.M = M; a.Kd = Kd; a.Kp = Kp; a.P = rc > 0 ? P + c0 * ldp : nullptr; a.ldp = ldp; a.r = rc;
    a.out = rc > 0 ? out + c0 : nullptr; a.ldo = r; a.part = rc > 0 && ks > 1 ? part : nullptr;
    a.mant = mant; a.planes = c0 == 0 ? planes : nullptr;
    const dim3 grid((unsigned)ceil_div(M, 32), (unsigned)ks);
    const int jt = (rc + 15) / 16;
    { TraceScope _ts(st, a.planes ? "f32_project_kernel<planes>" : "f32_project_kernel");
      auto go = [&](auto pl) {
        constexpr bool PL = decltype(pl)::value;
        if (jt == 0) f32_project_kernel<0, PL><<<grid, 256, 0, st>>>(a);
        else if (jt == 1) f32_project_kernel<1, PL><<<grid, 256, 0, st>>>(a);
        else if (jt == 2) f32_project_kernel<2, PL><<<grid, 256, 0, st>>>(a);
        else if (jt <= 4) f32_project_kernel<4, PL><<<grid, 256, 0, st>>>(a);
        else f32_project_kernel<8, PL><<<grid, 256, 0, st>>>(a);
      };
      if (a.planes) go(std::true_type{});
      else go(std::false_type{}); }
    if (int e = check_launch("f32_project_kernel")) return e;
    if (a.part) {
      { TraceScope _ts(st, "f32_sum_kernel");
        f32_sum_kernel<<<g1(M * rc), 256, 0, st>>>(part, ks, M, rc, out + c0, r); }
      if (int e = check_launch("f32_sum_kernel")) return e;
    }
  }
  return REELS_HIP_OK;
}

// dA = c x^T u, dB = c (dy^T h)^T (r ranks) and dbias = sum_m dy (each may be absent)
static int launch_colgrad_f32(const float* x, int64_t K, const float* u, float* dA, const float* dy,
                              int64_t N, const float* h, float* dB, float* dbias, int64_t M, int r,
                              float c, const PlanF32& p, float* pa, float* pb, float* pbias,
                              hipStream_t st) {
  if (!dA && !dB && !dbias) return REELS_HIP_OK;
  const int rr = dA || dB ? r : 0;
  for (int c0 = 0; c0 == 0 || c0 < rr; c0 += kRankChunk) {
    const int rc = std::min(rr - c0, kRankChunk);
    const bool bias = dbias && c0 == 0;  // rides on the first rank chunk's read of dy
    CgF32Job j[2] = {};
    int nb[2] = {0, 0}, n = 0;
    if (dA) {
      j[n].src = x; j[n].Lm = u + c0; j[n].part = pa + c0; j[n].out = p.spa == 1 ? dA + c0 : nullptr;
      j[n].Od = K; j[n].tps = p.tpsa; j[n].nbx = (int)ceil_div(K, f32c::BO); j[n].trans = 0;
      nb[n] = j[n].nbx * p.spa; ++n;
    }
    auto dyjob = [&](CgF32Job& q, int& blocks) {
      q.src = dy; q.Od = N; q.tps = p.tpsb; q.nbx = (int)ceil_div(N, f32c::BO); q.trans = 1;
      if (bias) (p.spb == 1 ? q.bout : q.bpart) = p.spb == 1 ? dbias : pbias;
      blocks = q.nbx * p.spb;
    };
    if (dB) {
      j[n].Lm = h + c0; j[n].part = pb + c0;
      j[n].out = p.spb == 1 ? dB + (int64_t)c0 * N : nullptr;
      dyjob(j[n], nb[n]);
      ++n;
    }
    const int jt = (rc + 15) / 16;
    if (n > 0) {
      const unsigned grid = (unsigned)(nb[0] + nb[1]);
      TraceScope _ts(st, "colgrad_f32_kernel");
      auto go = [&](auto b) {
        constexpr bool BS = decltype(b)::value;
        if (jt <= 1) colgrad_f32_kernel<1, BS><<<grid, 256, 0, st>>>(j[0], j[1], nb[0], M, rc, r, r, r, c);
        else if (jt == 2) colgrad_f32_kernel<2, BS><<<grid, 256, 0, st>>>(j[0], j[1], nb[0], M, rc, r, r, r, c);
        else if (jt <= 4) colgrad_f32_kernel<4, BS><<<grid, 256, 0, st>>>(j[0], j[1], nb[0], M, rc, r, r, r, c);
        else colgrad_f32_kernel<8, BS><<<grid, 256, 0, st>>>(j[0], j[1], nb[0], M, rc, r, r, r, c);
      };
      if (bias && dB) go(std::true_type{});
      else go(std::false_type{});
    }
    if (int e = check_launch("colgrad_f32_kernel")) return e;
    if (bias && !dB) {  // no dB pass to ride on
      CgF32Job q{};
      int blocks = 0;
      dyjob(q, blocks);
      { TraceScope _ts(st, "colgrad_f32_kernel<bias>");
        colgrad_f32_kernel<0, true><<<(unsigned)blocks, 256, 0, st>>>(q, q, blocks, M, 0, 0, 0, 0, c); }
      if (int e = check_launch("colgrad_f32_kernel")) return e;
    }
  }
  const bool ra = dA && p.spa > 1, rb = dB && p.spb > 1, rbias = dbias && p.spb > 1;
  if (ra && rb)
    return launch_reduce_partials2(pa, p.spa, K, dA, pb, p.spb, N, dB, r, r, c, rbias ? pbias : nullptr, dbias, st);
  if (ra)
    if (int e = launch_reduce_partials(pa, p.spa, K, r, r, c, dA, false, st)) return e;
  if (rb)
    if (int e = launch_reduce_partials(pb, p.spb, N, r, r, c, dB, true, st)) return e;
  // column sums alone: one "rank" of N outputs
  if (rbias) return launch_reduce_partials(pbias, p.spb, N, 1, 1, 1.0f, dbias, false, st);
  return REELS_HIP_OK;
}

// every f32 pointer on its natural alignment (NULL counts)
static bool aligned4(std::initializer_list<const void*> ps) {
  for (const void* q : ps)
    if ((reinterpret_cast<uintptr_t>(q) & 3u) != 0) return false;
  return true;
}

static int i8lora_fwd_f32_impl(const float* x, const int8_t* q, const float* scales, const float* A,
                               const float* B, const float* bias, int64_t M, int64_t K, int64_t N,
                               int64_t r, float c, float* y, float* h_save, void* workspace,
                               size_t ws_bytes, hipStream_t st) {
  const char* fn = "reels_hip_i8lora_fwd_f32";
  if (M < 0 || K <= 0 || N <= 0 || r < 0 || r > 4096)
    return fail(REELS_HIP_EINVAL, std::string(fn) + ": need M >= 0, K > 0, N > 0, 0 <= r <= 4096");
  if (!(c == c)) return fail(REELS_HIP_EINVAL, std::string(fn) + ": lora_scale is NaN");
  if (M == 0) return REELS_HIP_OK;
  if (!x || !q || !scales || !y || (r > 0 && (!A || !B)))
    return fail(REELS_HIP_EINVAL, std::string(fn) + ": NULL x, q, scales, y, or A/B with r > 0");
  const bool aligned = aligned4({x, scales, A, B, bias, y, h_save}) && aligned16(workspace);
  const PlanF32 p = plan_f32(M, K, N, r, aligned);
  const WsF32 w = ws_f32(M, K, N, r, REELS_HIP_WS_FWD, p);
  if (!workspace || ws_bytes < w.total)
    return fail(REELS_HIP_EWORKSPACE, std::string(fn) + ": workspace NULL or smaller than "
                                      "reels_hip_i8lora_workspace_bytes_f32(..., REELS_HIP_WS_FWD)");
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  float* h = h_save ? h_save : reinterpret_cast<float*>(ws + w.h);
  int rc;
  if (!p.fast) {
    if (r > 0) {
      // h = x A (A [K][r]: P(j, k) = A[k * r + j])
      { TraceScope _ts(st, "gf_rowproj_kernel"); gf_rowproj_kernel<<<g1(M * r), 256, 0, st>>>(x, M, K, A, r, 1, (int)r, h); }
      if ((rc = check_launch("gf_rowproj_kernel"))) return rc;
    }
    { TraceScope _ts(st, "gf_fwd_kernel"); gf_fwd_kernel<<<g1(M * N), 256, 0, st>>>(x, q, scales, h, B, bias, M, K, N, (int)r, c, y); }
    return check_launch("gf_fwd_kernel");
  }
  float* at = r > 0 ? reinterpret_cast<float*>(ws + w.at) : nullptr;
  float* bt = r > 0 ? reinterpret_cast<float*>(ws + w.bt) : nullptr;
  uint16_t* wd = reinterpret_cast<uint16_t*>(ws + w.wd);
  uint16_t* planes = reinterpret_cast<uint16_t*>(ws + w.planes);
  float* mant = reinterpret_cast<float*>(ws + w.mant);
  if ((rc = launch_operands(false, q, scales, N, K, p, wd, mant, A, B, r, at, bt, st))) return rc;
  for (int64_t m0 = 0; m0 < M; m0 += p.chf) {
    const int64_t mc = std::min(M - m0, p.chf);
    float* hc = r > 0 ? h + m0 * r : nullptr;
    if ((rc = launch_project(x + m0 * K, mc, K, p.Kp, at, p.Kp, (int)r, hc,
                             reinterpret_cast<float*>(ws + w.rq), p.psf, nullptr, planes, st)))
      return rc;
    GemmArgs g{};
    g.act = planes; g.colscale = mant; g.fL = hc; g.fR = bt; g.fbias = bias; g.fout = y + m0 * N;
    g.M = mc; g.Ncols = N; g.Kred = p.Kp; g.fr = (int)r; g.c = c;
    g.fvout = N % 4 == 0;
    g.ksplit = planegemm_splits(mc, N, p.Kp); g.part = reinterpret_cast<float*>(ws + w.kp); g.ldp = (N + 3) / 4 * 4;
    if ((rc = launch_planegemm(0, g, wd, st))) return rc;
  }
  return REELS_HIP_OK;
}

static int i8lora_bwd_f32_impl(const char* fn, const float* dy, const float* x, const float* hh,
                               const int8_t* q, const float* scales, const float* A,
                               const float* B, int64_t M, int64_t K, int64_t N, int64_t r, float c,
                               float* dx, float* dA, float* dB, float* dbias, void* workspace,
                               size_t ws_bytes, hipStream_t st) {
  if (M < 0 || K <= 0 || N <= 0 || r < 0 || r > 4096)
    return fail(REELS_HIP_EINVAL, std::string(fn) + ": need M >= 0, K > 0, N > 0, 0 <= r <= 4096");
  if (!(c == c)) return fail(REELS_HIP_EINVAL, std::string(fn) + ": lora_scale is NaN");
  if (r == 0) { dA = nullptr; dB = nullptr; }
  int rc;
  if (M == 0) {  // empty token set: the reductions over tokens are zero
    if (dA && K * r > 0) {
      { TraceScope _ts(st, "zero_f32_kernel"); zero_f32_kernel<<<g1(K * r), 256, 0, st>>>(dA, K * r); }
      if ((rc = check_launch("zero_f32_kernel"))) return rc;
    }
    if (dB && N * r > 0) {
      { TraceScope _ts(st, "zero_f32_kernel"); zero_f32_kernel<<<g1(N * r), 256, 0, st>>>(dB, N * r); }
      if ((rc = check_launch("zero_f32_kernel"))) return rc;
    }
    if (dbias) {
      { TraceScope _ts(st, "zero_f32_kernel"); zero_f32_kernel<<<g1(N), 256, 0, st>>>(dbias, N); }
      if ((rc = check_launch("zero_f32_kernel"))) return rc;
    }
    return REELS_HIP_OK;
  }
  if (!dy || !q || !scales || (r > 0 && (!A || !B)) || ((dA || (dB && !hh)) && !x))
    return fail(REELS_HIP_EINVAL, std::string(fn) + ": NULL dy, q, scales, A/B with r > 0, or x "
                                  "needed for dA / recomputing h");
  if (!dx && !dA && !dB && !dbias) return REELS_HIP_OK;
  const bool aligned = aligned4({dy, x, hh, scales, A, B, dx, dA, dB, dbias}) && aligned16(workspace);
  const PlanF32 p = plan_f32(M, K, N, r, aligned);
  const WsF32 w = ws_f32(M, K, N, r, REELS_HIP_WS_BWD, p);
  if (!workspace || ws_bytes < w.total)
    return fail(REELS_HIP_EWORKSPACE, std::string(fn) + ": workspace NULL or smaller than "
                                      "reels_hip_i8lora_workspace_bytes_f32(..., REELS_HIP_WS_BWD)");
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  float* u = reinterpret_cast<float*>(ws + w.u);
  if (!p.fast) {
    if (r > 0) {
      // u = dy B^T (B [r][N]: P(j, n) = B[j * N + n])
      { TraceScope _ts(st, "gf_rowproj_kernel"); gf_rowproj_kernel<<<g1(M * r), 256, 0, st>>>(dy, M, N, B, 1, N, (int)r, u); }
      if ((rc = check_launch("gf_rowproj_kernel"))) return rc;
    }
    if (dx) {
      { TraceScope _ts(st, "gf_dx_kernel"); gf_dx_kernel<<<g1(M * K), 256, 0, st>>>(dy, q, scales, u, A, M, K, N, (int)r, c, dx); }
      if ((rc = check_launch("gf_dx_kernel"))) return rc;
    }
    if (dA) {
      { TraceScope _ts(st, "gf_colgrad_kernel<false>"); gf_colgrad_kernel<false><<<g1(K * r), 256, 0, st>>>(x, M, K, u, (int)r, c, dA); }
      if ((rc = check_launch("gf_colgrad_kernel"))) return rc;
    }
    if (dB) {
      const float* hp = hh;
      if (!hp) {
        float* hw = reinterpret_cast<float*>(ws + w.h);
        { TraceScope _ts(st, "gf_rowproj_kernel"); gf_rowproj_kernel<<<g1(M * r), 256, 0, st>>>(x, M, K, A, r, 1, (int)r, hw); }
        if ((rc = check_launch("gf_rowproj_kernel"))) return rc;
        hp = hw;
      }
      { TraceScope _ts(st, "gf_colgrad_kernel<true>"); gf_colgrad_kernel<true><<<g1(N * r), 256, 0, st>>>(dy, M, N, hp, (int)r, c, dB); }
      if ((rc = check_launch("gf_colgrad_kernel"))) return rc;
    }
    if (dbias)
      return launch_colsum(REELS_HIP_F32, dy, M, N, reinterpret_cast<float*>(ws + w.pbias), dbias, st);
    return REELS_HIP_OK;
  }
  float* rq = reinterpret_cast<float*>(ws + w.rq);
  uint16_t* wt = dx ? reinterpret_cast<uint16_t*>(ws + w.wd) : nullptr;
  float* mant = reinterpret_cast<float*>(ws + w.mant);
  uint16_t* planes = dx ? reinterpret_cast<uint16_t*>(ws + w.planes) : nullptr;
  float* at = dB && !hh ? reinterpret_cast<float*>(ws + w.at) : nullptr;  // to recompute h
  if ((rc = launch_operands(true, q, scales, N, K, p, wt, mant, A, B, r, at, nullptr, st))) return rc;
  // 1. u = dy B^T (B [r][N] rows are the projection rows) with the planes of dy mant from the same
  // read; 2. dx = (dy mant) (q 2^e) + c u A^T
  float* up = r > 0 && (dx || dA) ? u : nullptr;
  if (dx || up) {
    for (int64_t m0 = 0; m0 < M; m0 += p.chb) {
      const int64_t mc = std::min(M - m0, p.chb);
      float* uc = up ? up + m0 * r : nullptr;
      if ((rc = launch_project(dy + m0 * N, mc, N, p.Np, B, N, (int)r, uc, rq, p.psb, mant, planes, st)))
        return rc;
      if (!dx) continue;
      GemmArgs g{};
      g.act = planes; g.fL = uc; g.fR = A; g.fout = dx + m0 * K;
      g.M = mc; g.Ncols = K; g.Kred = p.Np; g.fr = (int)r; g.c = c;
      g.fvout = K % 4 == 0;
      g.ksplit = planegemm_splits(mc, K, p.Np); g.part = reinterpret_cast<float*>(ws + w.kp); g.ldp = (K + 3) / 4 * 4;
      if ((rc = launch_planegemm(1, g, wt, st))) return rc;
    }
  }
  // 3. dA = c x^T u ; dB = c (dy^T h)^T (h recomputed first when not given)
  const float* hp = hh;
  if (dB && !hp) {
    float* hw = reinterpret_cast<float*>(ws + w.h);
    for (int64_t m0 = 0; m0 < M; m0 += p.chf) {
      const int64_t mc = std::min(M - m0, p.chf);
      if ((rc = launch_project(x + m0 * K, mc, K, p.Kp, at, p.Kp, (int)r, hw + m0 * r, rq, p.psf, nullptr, nullptr, st)))
        return rc;
    }
    hp = hw;
  }
  return launch_colgrad_f32(x, K, u, dA, dy, N, hp, dB, dbias, M, (int)r, c, p,
                            reinterpret_cast<float*>(ws + w.pa), reinterpret_cast<float*>(ws + w.pb),
                            reinterpret_cast<float*>(ws + w.pbias), st);
}

}  // namespace reels

using namespace reels;

extern "C" size_t reels_hip_i8lora_workspace_bytes_f32(int64_t M, int64_t K, int64_t N, int64_t r,
                                                       int which) {
  if (M < 0 || K < 0 || N < 0 || r < 0) return 0;
  if (which != REELS_HIP_WS_FWD && which != REELS_HIP_WS_BWD) return 0;
  const PlanF32 p = plan_f32(M, K, N, r, true);  // the fast layout is never smaller
  return ws_f32(M, K, N, r, which, p).total;
}

extern "C" int reels_hip_i8lora_fwd_f32(const float* x, const int8_t* q, const float* scales,
                                        const float* A, const float* B, const float* bias,
                                        int64_t M, int64_t K, int64_t N, int64_t r,
                                        float lora_scale, float* y, float* h_save, void* workspace,
                                        size_t ws_bytes, void* stream) {
  clear_error();
  return i8lora_fwd_f32_impl(x, q, scales, A, B, bias, M, K, N, r, lora_scale, y, h_save,
                             workspace, ws_bytes, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int reels_hip_i8lora_bwd_f32(const float* dy, const float* x, const float* h,
                                        const int8_t* q, const float* scales, const float* A,
                                        const float* B, int64_t M, int64_t K, int64_t N, int64_t r,
                                        float lora_scale, float* dx, float* dA, float* dB,
                                        void* workspace, size_t ws_bytes, void* stream) {
  clear_error();
  return i8lora_bwd_f32_impl("reels_hip_i8lora_bwd_f32", dy, x, h, q, scales, A, B, M, K, N, r,
                             lora_scale, dx, dA, dB, nullptr, workspace, ws_bytes,
                             reinterpret_cast<hipStream_t>(stream));
}

extern "C" int reels_hip_i8lora_bwd_bias_f32(const float* dy, const float* x, const float* h,
                                             const int8_t* q, const float* scales, const float* A,
                                             const float* B, int64_t M, int64_t K, int64_t N,
                                             int64_t r, float lora_scale, float* dx, float* dA,
                                             float* dB, float* dbias, void* workspace,
                                             size_t ws_bytes, void* stream) {
  clear_error();
  return i8lora_bwd_f32_impl("reels_hip_i8lora_bwd_bias_f32", dy, x, h, q, scales, A, B, M, K, N,
                             r, lora_scale, dx, dA, dB, dbias, workspace, ws_bytes,
                             reinterpret_cast<hipStream_t>(stream));
}

extern "C" int reels_hip_gelu_tanh_f32(const float* x, float* y, int64_t n, void* stream) {
  clear_error();
  if (n < 0) return fail(REELS_HIP_EINVAL, "reels_hip_gelu_tanh_f32: n < 0");
  if (n == 0) return REELS_HIP_OK;
  if (!x || !y) return fail(REELS_HIP_EINVAL, "reels_hip_gelu_tanh_f32: NULL pointer");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  { TraceScope _ts(st, "gelu_f32_kernel"); gelu_f32_kernel<<<g1(n), 256, 0, st>>>(x, y, n); }
  return check_launch("gelu_f32_kernel");
}

extern "C" int reels_hip_gelu_tanh_bwd_f32(const float* x, const float* dy, float* dx, int64_t n,
                                           void* stream) {
  clear_error();
  if (n < 0) return fail(REELS_HIP_EINVAL, "reels_hip_gelu_tanh_bwd_f32: n < 0");
  if (n == 0) return REELS_HIP_OK;
  if (!x || !dy || !dx) return fail(REELS_HIP_EINVAL, "reels_hip_gelu_tanh_bwd_f32: NULL pointer");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  { TraceScope _ts(st, "gelu_bwd_f32_kernel"); gelu_bwd_f32_kernel<<<g1(n), 256, 0, st>>>(x, dy, dx, n); }
  return check_launch("gelu_bwd_f32_kernel");
}
