// Legacy (reference-format) kernels: the arithmetic of the reference's torch forms.
//
//   encode  torch_low_rank_addition_fuse_compression_quantization
//           (low_rank_extraction_fuse_compression_quantization.py:153-171)
//             xr = bf16(x - bf16(l @ r));  o = xr if |xr| > bf16(tau) else 0;
//             c  = clamp(rint(bf16((xr - o) / s)), -2^(b-1), 2^(b-1)-1) + 2^(b-1)
//             q  = row-planar packing: byte j of a row holds column j + p*N/NP in bits
//                  p*b .. p*b+b-1 of plane p (NP = 8/b planes)
//   decode  torch_low_rank_addition_fuse_decompression_dequantization
//           (low_rank_extraction_fuse_decompression_dequantization.py:155-165)
//             x_hat = bf16(bf16(bf16((c - 2^(b-1)) * s) + o) + bf16(l @ r))
//   fused   decode without outliers, then store / SiLU backward / product with y
//           (extraction_fuse_silu_backward.py:192-216, extraction_fuse_hadamard.py:185-209)
//   add     torch_low_rank_addition (low_rank_extraction_speed.py:106-107): bf16(x + bf16(l @ r))
//   hist    histogram of the 15-bit magnitudes |bf16(x - bf16(l @ r))| (the encode's residual), for
//           the outlier threshold torch.kthvalue(|x[0] - l @ r|, k) of
//           low_rank_system_profile_forward.py:45: a 256-bin pass over the top 8 bits, then a
//           128-bin pass over the low 7 bits of the keys in the selected bin.
//
// l is [M, K] and rt = r^T is [N, K] (K = 16 or 32, zero-padded by the caller as the reference
// pads K < 16); s is [1 or B, N].  bf16(l @ r) is the fp32 rounding of the exact sum, then bf16
// (what an fp32-accumulating GEMM returns up to the order of its additions).
//
// Two implementations with identical results:
//   * on MFMA — when every plane is a whole number of 64-column units and the operands are 16-byte
//     aligned: k_legacy_encode (encode), k_legacy_apply (decode with sparse or no outliers, fused
//     consumers), k_legacy_rows (decode, denser sparse outliers of large tensors), k_legacy_mfma
//     (decode from dense outliers, add, histogram), k_legacy_gemm (the product).  The unit layout of lrq_common.h (lane (j, g) owns 16 consecutive
//     columns of its row in every plane) with l @ r rebuilt on MFMA exactly like the
//     group-mode reconstruction (V = rt).
//   * k_legacy_scalar — any shape: one thread per packed byte, l @ r summed in fp64 (the
//     products of bf16 values are exact and so is their fp64 sum for K <= 32).
#include "lrq_common.h"
#include "lrq_coo.h"
#include "lrq_host.h"
#include "lrq_math.h"

namespace lrq {

enum LegacyMode : int { kEncode = 0, kDecode = 1, kFusedStore = 2, kFusedSilu = 3, kFusedMul = 4, kAdd = 5, kHist = 6 };

struct LegacyArgs {
  const uint16_t* l;    // [M, K]
  const uint16_t* rt;   // [N, K]
  const uint16_t* x;    // encode / add input [B, M, N] with strides (ldx_b, ldx_m, 1)
  int64_t ldx_b, ldx_m;
  const uint16_t* s;    // [s_rows, N]
  int64_t s_rows;
  const uint8_t* qin;   // decode / fused codes [B, M, N/NP]
  const uint16_t* oin;  // decode outliers, dense [B, M, N], or null
  const int64_t* optr;  // decode outliers as COO: first entry of each 64-column piece of a row,
  const int64_t* ocol;  //   [B * M * npc + 1]; the entries' column indices and bf16 values, in
  const uint16_t* oval; //   row-major order (lrq_coo_compact's output)
  int64_t npc;          // 64-column pieces per row, ceil(N / 64)
  int64_t* pcnt;        // staged encode: each 64-column piece's record (lrq_coo.h), [B * M * npc]
  int64_t ncap;         // entries the COO arrays hold: reads are clamped to [0, ncap)
  uint32_t* hist;       // hist: 256 global bins
  const int64_t* sel;   // hist: sel[0] = the selected top-8-bit bin, or -1 in the first pass
  const uint16_t* y;    // fused SiLU dy / product operand [B, M, N]
  uint16_t* out;        // decode / fused / add output [B, M, N]
  uint16_t* oout;       // encode outliers, dense [B, M, N]
  uint8_t* qout;        // encode codes [B, M, N/NP]
  int64_t M, N;
  float tau;            // outlier threshold, already rounded to bf16
  int rb;               // MFMA path: 64-row blocks per workgroup
};

// Encode of one element given its bf16 input x, bf16(l @ r) lr and scale sc: returns the code
// (0 .. 2^b - 1) and writes the outlier value (0 unless an outlier).
// big: |xr| > tau, i.e. o = xr; with tau >= 0 that is exactly an outlier entry the compaction
// keeps (o's bf16 bits not +-0).
template <int BITS>
__device__ __forceinline__ uint32_t legacy_code(float x, float lr, float sc, float tau, float& o, bool& big) {
  constexpr float half = (float)(1 << (BITS - 1));
  const float xr = bf16r(x - lr);
  big = fabsf(xr) > tau;
  o = big ? xr : 0.f;
  const float d = bf16r((xr - o) / sc);  // IEEE division, then the bf16 rounding of the torch op
  const float c = __builtin_amdgcn_fmed3f(rintf(d), -half, half - 1.f);
  return (uint32_t)(int)(c + half);
}

// The MFMA encode's forms of legacy_code, with the same codes:
// - the quotient: for scales with 2^-100 <= |sc| <= 2^100 (rc_scale_ok) a product with 1/sc as two
//   bf16 terms (legacy_codes_mfma) instead of the IEEE division: its code equals the IEEE quotient's at
//   every bit width for every finite bf16 numerator a (a and sc are bf16 values, so a / sc never comes
//   near a code boundary within the product's error); other scales take the IEEE division;
// - bf16_roundtrip2 rounds two values to bf16 with one conversion;
// - the code of a bf16 quotient d is legacy_code_biased(d) - kCodeBias + half, where
//   legacy_code_biased(d) = bits(d + 1.5 * 2^23) clamped to [kCodeBias - half, kCodeBias + half - 1]:
//   for |d| < 2^22 the sum lies in [2^23, 2^24), where the fp32 ulp is 1, so the add rounds d to the
//   nearest integer, ties to even (1.5 * 2^23 is even), as rint does, and the bits are kCodeBias +
//   rint(d); for d >= 2^22 the sum is at least 2^24 and clamps to the top code; for d <= -2^22 it is
//   at most 2^23, +0 or negative (a negative int32) and clamps to the bottom code, as the clamp of
//   rint(d) does (infinities included).  A byte starting from legacy_code_base (the sum of
//   (half - kCodeBias) << BITS p over its planes, mod 2^32) and adding legacy_code_biased << BITS p
//   per plane holds the planes' codes in its low 8 bits;
// - at 1 bit the code is 1 exactly when bf16(q) >= -0.5, i.e. when q >= -(0.5 + 2^-9) (below
//   -0.5 the bf16 spacing is 2^-8, and the tie at -0.5 - 2^-9 rounds to the even -0.5): one
//   compare of the quotient, no rounding.
// The host check tests/legacy_code_check.c compares the code forms with the reference's over every fp32
// quotient but NaN, and the two-term product's codes with the IEEE quotient's over every finite bf16
// numerator and every scale served.
constexpr uint32_t kCodeBias = 0x4B400000u;  // bits of 1.5 * 2^23
template <int BITS>
__device__ __forceinline__ uint32_t legacy_code_biased(float d) {
  constexpr int half = 1 << (BITS - 1);
  const int v = (int)__float_as_uint(d + 0x1.8p23f);
  return (uint32_t)min(max(v, (int)kCodeBias - half), (int)kCodeBias + half - 1);
}
constexpr float kOneBitLow = -(0.5f + 0x1p-9f);
template <int BITS>
constexpr uint32_t legacy_code_base() {
  if (BITS == 1) return 0u;  // the complements of the 1-bit codes are or-ed in
  uint32_t k = 0;
  for (int p = 0; p < 8 / BITS; ++p) k += ((1u << (BITS - 1)) - kCodeBias) << (BITS * p);
  return k;
}

// legacy_code of two elements in the forms above, with the IEEE division and one bf16 conversion per
// rounding step of the pair: at 1 bit the code itself (an outlier leaves a = 0, whose code is 1;
// otherwise a = xr), at 2, 4 and 8 bits biased (legacy_code_biased).
template <int BITS>
__device__ __forceinline__ void legacy_code_mfma2(const float* x, const float* lr, const float* sc, float tau, float* o,
                                                  bool* big, uint32_t* code) {
  float xr[2] = {x[0] - lr[0], x[1] - lr[1]}, q[2];
  bf16_roundtrip2(xr[0], xr[1]);
  if constexpr (BITS == 1) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      big[k] = fabsf(xr[k]) > tau;
      o[k] = big[k] ? xr[k] : 0.f;
      code[k] = (big[k] || xr[k] / sc[k] >= kOneBitLow) ? 1u : 0u;
    }
    return;
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    big[k] = fabsf(xr[k]) > tau;
    o[k] = big[k] ? xr[k] : 0.f;
    q[k] = (xr[k] - o[k]) / sc[k];
  }
  bf16_roundtrip2(q[0], q[1]);
  code[0] = legacy_code_biased<BITS>(q[0]);
  code[1] = legacy_code_biased<BITS>(q[1]);
}
// (At 1 bit the code comes as a word whose sign bit is its complement, gathered complemented.)
template <int BITS>
__device__ __forceinline__ void legacy_accumulate(uint32_t& byte, uint32_t code, int p) {
  if constexpr (BITS == 1) byte |= (code >> (31 - p)) & (1u << p);
  else byte += code << (BITS * p);
}

// The bf16 bits of element i (0 .. 15) of the 16 packed in w0 (elements 0 .. 7) and w1: a select
// tree, no indexed register access.
__device__ __forceinline__ uint32_t bf16_at(const u32x4& w0, const u32x4& w1, uint32_t i) {
  const u32x4 w = (i & 8u) ? w1 : w0;
  const uint32_t lo = (i & 2u) ? w[1] : w[0], hi = (i & 2u) ? w[3] : w[2];
  const uint32_t d = (i & 4u) ? hi : lo;
  return (d >> (16u * (i & 1u))) & 0xffffu;
}

// The encode's element work on the matrix pipe.  Per element the VALU only rounds, tests and packs:
// every widening, subtraction and product goes through 4x4x4 MFMA steps (16 blocks of 4 lanes each),
// whose B operand is 4 elements of the lane itself and whose A operand is diagonal (lane l holds row
// l % 4, the coefficient of element l % 4), which makes them elementwise:
//   x - bf16(l r)       A = I on x, then A = -I on bf16(l r) with that as C: one fp32 rounding
//   q = a r1 + a r2     A = diag r1, then diag r2; 1/s = r1 + r2 to 2^-18 (legacy_rc_split), a r1 exact
//   d + 1.5 * 2^23      A = I, C = 1.5 * 2^23: the code's biased bits (legacy_code_biased)
//   q + (0.5 + 2^-9)    at 1 bit the threshold is the first product's C operand, the sign bit the code
//                       (rounding 17-bit sums to fp32 changes no sign)
// A sum of two bf16 values (or of two products with a common bf16 factor) is rounded once, so every
// value is the one the VALU forms above give.  The bf16 tests and masks are packed 16-bit integer
// operations (two elements each).  An infinite or NaN x would spread over its 4 elements through the
// zeros of A, and a residual so large that a r2 overflows would meet a r1's infinity: the wave redoes
// a plane with such a magnitude (mag_limit) with legacy_code_mfma2.  tau >= +0 here (legacy_tau).
// (The packed operations are asm: written as vector code the compiler splits a saturated difference
// and its test into per-half compares and selects.)
__device__ __forceinline__ uint32_t pk_sub_sat_u16(uint32_t a, uint32_t b) {
  uint32_t r;
  asm("v_pk_sub_u16 %0, %1, %2 clamp" : "=v"(r) : "v"(a), "s"(b));
  return r;
}
__device__ __forceinline__ uint32_t pk_min1_u16(uint32_t a, uint32_t one2) {
  uint32_t r;
  asm("v_pk_min_u16 %0, %1, %2" : "=v"(r) : "v"(a), "s"(one2));
  return r;
}
__device__ __forceinline__ uint32_t pk_max_u16(uint32_t a, uint32_t b) {
  uint32_t r;
  asm("v_pk_max_u16 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ uint32_t pk_neg_u16(uint32_t a) {
  uint32_t r;
  asm("v_pk_sub_u16 %0, 0, %1" : "=v"(r) : "v"(a));
  return r;
}

// D(4x4) += A(4x4) * B(4x4) in each of 16 blocks of 4 lanes, bf16 inputs, fp32 accumulate: lane l holds
// row l % 4 of A, column l % 4 of B and of D.
__device__ __forceinline__ f32x4 mfma_4x4x4(u32x2 a, u32x2 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0, 0);
}
// The diagonal A operand of that step with bf16 bits `v` in this lane's row.
__device__ __forceinline__ u32x2 diag4_aop(int lane, uint32_t v) {
  const uint32_t d = v << (16u * (lane & 1));
  return (lane & 2) ? u32x2{0u, d} : u32x2{d, 0u};
}
// Selectors (v_perm_b32) that place the low (hi = 0) or high half of a dword as diag4_aop does.
__device__ __forceinline__ u32x2 diag4_sel(int lane, int hi) {
  const uint32_t h = hi ? 0x0302u : 0x0100u, d = (lane & 1) ? (h << 16) | 0x0c0cu : 0x0c0c0000u | h;
  return (lane & 2) ? u32x2{0x0c0c0c0cu, d} : u32x2{d, 0x0c0c0c0cu};
}
// 1/s as the sum of two bf16 terms (relative error at most 2^-18 + 2^-24: a quotient of two bf16
// values is at least 2^-17 from a code boundary, relative).
__device__ __forceinline__ void legacy_rc_split(float sc, uint32_t& r1, uint32_t& r2) {
  const float rc = 1.0f / sc;
  r1 = pack_bf16x2(rc, 0.f);
  r2 = pack_bf16x2(rc - __uint_as_float(r1 << 16), 0.f);
}

// fp32(l r) of the lane's 16 columns of one plane (step q: elements 4q .. 4q + 3).
template <int K>
__device__ __forceinline__ void legacy_lowrank_mfma(const u32x2 (&vop)[4][K / 16], const u32x2* lop, f32x4 (&t)[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if constexpr (K == 16) {
      t[q] = mfma_16x16x16(vop[q][0], lop[0], zero4());
    } else {
      t[q] = mfma_16x16x32(u32x4{vop[q][0][0], vop[q][0][1], vop[q][1][0], vop[q][1][1]},
                           u32x4{lop[0][0], lop[0][1], lop[1][0], lop[1][1]}, zero4());
    }
  }
}

// The plane's outlier test and codes from the packed residuals w (w[k]: elements 2k, 2k + 1): hm bit e =
// element e is an outlier, w becomes the outlier values (0 elsewhere), code[16] the codes
// (legacy_code_biased; at 1 bit a word whose sign bit is the code's complement).  Returns whether some
// magnitude of the lane reaches mag_limit (bf16 bits): hm, w and code are then unspecified.
// rc[q]: r1 | r2 << 16 of column 4q + lane % 4 (legacy_rc_split), the two diagonals' bf16 bits in this lane's row.
template <int BITS>
__device__ __forceinline__ bool legacy_codes_mfma(uint32_t (&w)[8], uint32_t tau2, uint32_t mag_limit, u32x4 rc, int lane,
                                                  uint32_t (&code)[16], uint32_t& hm) {
  uint32_t a[8], mag[8], h2 = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) mag[k] = w[k] & 0x7fff7fffu;
  const uint32_t t0 = pk_max_u16(pk_max_u16(mag[0], mag[1]), pk_max_u16(mag[2], mag[3]));
  const uint32_t t1 = pk_max_u16(pk_max_u16(mag[4], mag[5]), pk_max_u16(mag[6], mag[7]));
  const uint32_t top = pk_max_u16(t0, t1);
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const uint32_t one = pk_min1_u16(pk_sub_sat_u16(mag[k], tau2), 0x00010001u);  // 1 where |xr| > tau
    h2 |= one << (2 * k);  // bits 2k (element 2k) and 16 + 2k (element 2k + 1)
    const uint32_t m = pk_neg_u16(one);
    a[k] = w[k] & ~m;
    w[k] &= m;
  }
  hm = (h2 & 0xffffu) | (h2 >> 15);
  f32x4 t[4];
  constexpr float c0 = BITS == 1 ? -kOneBitLow : 0.f;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const u32x2 sel = diag4_sel(lane, h);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const u32x2 ra = u32x2{__builtin_amdgcn_perm(rc[q], rc[q], sel[0]), __builtin_amdgcn_perm(rc[q], rc[q], sel[1])};
      t[q] = mfma_4x4x4(ra, u32x2{a[2 * q], a[2 * q + 1]}, h == 0 ? f32x4{c0, c0, c0, c0} : t[q]);
    }
  }
  if constexpr (BITS == 1) {
#pragma unroll
    for (int e = 0; e < 16; ++e) code[e] = __float_as_uint(t[e >> 2][e & 3]);
  } else {
    constexpr float mg = 0x1.8p23f;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      t[q] = mfma_4x4x4(diag4_aop(lane, 0x3f80u), u32x2{pack_bf16x2(t[q][0], t[q][1]), pack_bf16x2(t[q][2], t[q][3])},
                        f32x4{mg, mg, mg, mg});
    constexpr int half = 1 << (BITS - 1);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int v = (int)__float_as_uint(t[e >> 2][e & 3]);
      code[e] = (uint32_t)min(max(v, (int)kCodeBias - half), (int)kCodeBias + half - 1);
    }
  }
  return (top >> 16) >= mag_limit || (top & 0xffffu) >= mag_limit;
}

// Scales whose two-term reciprocal gives legacy_code's codes, 2^-100 <= |sc| <= 2^100: compared as bits, so
// that a NaN is above (this build's float comparisons take no NaN).
__device__ __forceinline__ bool rc_scale_ok(float sc) {
  const uint32_t m = __float_as_uint(sc) & 0x7fffffffu;
  return m >= 0x0d800000u && m <= 0x71800000u;
}

// Decode of one element: bf16(bf16(bf16((code - 2^(b-1)) * s) + o) + lr); with !HAS_O the add
// of o (exact zero) is skipped.  The outliers come as a dense tensor (OSRC 1) or as COO pieces
// (OSRC 2); both feed the same per-element add, so the two give the same bits.
template <int BITS, bool HAS_O>
__device__ __forceinline__ float legacy_value(uint32_t code, float sc, float o, float lr) {
  float a = bf16r((float)((int)code - (1 << (BITS - 1))) * sc);
  if constexpr (HAS_O) a = bf16r(a + o);
  return bf16r(a + lr);
}

// Histogram bin of a residual xr (bf16 value) for the pass that sel selects, or -1 if the key
// is not counted in this pass.
__device__ __forceinline__ int hist_bin(float xr, int64_t sel) {
  const uint32_t key = (__float_as_uint(xr) >> 16) & 0x7fffu;
  if (sel < 0) return (int)(key >> 7);
  return (int64_t)(key >> 7) == sel ? (int)(key & 127u) : -1;
}

template <int MODE>
__device__ __forceinline__ float legacy_consume(float xh, float yv) {
  if constexpr (MODE == kFusedSilu) return silu_bwd_f32(xh, yv);
  else if constexpr (MODE == kFusedMul) return xh * yv;
  else return xh;
}

// ------------------------------------------------------------------ MFMA path
// Grid: ceil(M / (64 * rb)) * (N / (64 * NP)) * B workgroups (one dimension); 4 waves; the
// workgroup's tile t = (b, bx, u), units fastest, is xcd_tile of its index: the workgroups of one
// XCD that run together cover neighbouring units of the same rows, which share L2 lines of the COO
// entries (a piece's entries do not start on a line boundary), of the code rows and of the output
// rows.  Wave w walks row blocks (bx * rb + i) * 64 + w * 16, i < rb, of unit u.  Decodes from dense
// outliers, adds and histograms (the other decodes: k_legacy_apply, k_legacy_rows).
template <int MODE, int BITS, int K>
__global__ __launch_bounds__(256) void k_legacy_mfma(LegacyArgs a) {
  constexpr int NP = (MODE == kAdd || MODE == kHist) ? 1 : 8 / BITS, G = 64, E = 16, RT = K / 16;
  __shared__ uint32_t lh[MODE == kHist ? 256 : 1];
  int64_t sel = -1;
  if constexpr (MODE == kHist) {
    lh[threadIdx.x] = 0u;
    sel = a.sel[0];
    __syncthreads();
  }
  constexpr uint32_t kMask = BITS == 8 ? 0xffu : (1u << BITS) - 1u;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  const int j = lane & 15, g = lane >> 4;
  const int M = (int)a.M, N = (int)a.N;
  // tile t = (batch, 64-row chunk, unit), units fastest
  const int nu = N / NP / G, gx = (M + 64 * a.rb - 1) / (64 * a.rb);
  const int t = __builtin_amdgcn_readfirstlane(xcd_tile(blockIdx.x, gridDim.x));
  const int u = __builtin_amdgcn_readfirstlane(t % nu);
  const int bx = __builtin_amdgcn_readfirstlane((t / nu) % gx);
  const int b = __builtin_amdgcn_readfirstlane(t / (nu * gx));
  const int64_t NB = N / NP;  // bytes per code row
  const uint16_t* srow = a.s + (a.s_rows == 1 ? 0 : (int64_t)b * N);

  u32x2 vop[NP][G / 16][RT];
#pragma unroll
  for (int p = 0; p < NP; ++p) load_vops<G, K>(a.rt, unit_base(p, u, N, NP, G), j, g, vop[p]);
  const float zero[E] = {};

  // the unit's scales in LDS for every row block of the workgroup (the same columns throughout)
  constexpr bool kScales = MODE == kDecode;
  __shared__ __attribute__((aligned(16))) float stab[kScales ? NP * G : 4];
  if constexpr (kScales) {
    for (int i = threadIdx.x; i < NP * G; i += 256) stab[i] = bf_lo(srow[unit_base(i / G, u, N, NP, G) + i % G]);
    __syncthreads();
  }

  for (int i = 0; i < a.rb; ++i) {
    const int row0 = (bx * a.rb + i) * 64 + w * 16;  // wave-uniform: a scalar exit
    if (row0 >= M) break;  // whole 16-row block past the end
    const int row = row0 + j;
    const int64_t rr = min(row, M - 1);
    const int64_t erow = ((int64_t)b * M + rr) * N;  // element offset of the row in [B, M, N] outputs
    u32x2 lop[RT];
    u32x4 qb = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int t = 0; t < RT; ++t) lop[t] = ld8(a.l + rr * K + 16 * t + 4 * g);
    if constexpr (MODE == kDecode) qb = ld16(a.qin + ((int64_t)b * M + rr) * NB + u * G + E * g);

#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int c0 = unit_base(p, u, N, NP, G) + E * g;
      float lr[E];
      residual_unit<G, K>(vop[p], lop, zero, lr);
#pragma unroll
      for (int e = 0; e < E; e += 2) bf16_roundtrip2(lr[e], lr[e + 1]);
      float sc[E];
      if constexpr (kScales) {
        const float* sp = stab + p * G + E * g;
#pragma unroll
        for (int k = 0; k < E; k += 4) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(sp + k);
#pragma unroll
          for (int e = 0; e < 4; ++e) sc[k + e] = v[e];
        }
      }
      if constexpr (MODE == kHist) {
        float xv[E];
        const uint16_t* xp = a.x + rr * a.ldx_m + c0;
        unpack8(ld16(xp), xv);
        unpack8(ld16(xp + 8), xv + 8);
        if (row < M) {
#pragma unroll
          for (int e = 0; e < E; ++e) {
            const int bin = hist_bin(bf16r(xv[e] - lr[e]), sel);
            if (bin >= 0) atomicAdd(&lh[bin], 1u);
          }
        }
      } else if constexpr (MODE == kAdd) {
        const uint16_t* xp = a.x + (int64_t)b * a.ldx_b + rr * a.ldx_m + c0;
        float xv[E];
        unpack8(ld16(xp), xv);
        unpack8(ld16(xp + 8), xv + 8);
        float ov[E];
#pragma unroll
        for (int e = 0; e < E; ++e) ov[e] = xv[e] + lr[e];  // fp32 add, then bf16 (pack8), as torch
        st16(a.out + erow + c0, pack8(ov));
        st16(a.out + erow + c0 + 8, pack8(ov + 8));
      } else {
        float ov[E], oo[E];
        unpack8(ld16(a.oin + erow + c0), oo);
        unpack8(ld16(a.oin + erow + c0 + 8), oo + 8);
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const uint32_t code = (qb[e >> 2] >> (8 * (e & 3) + BITS * p)) & kMask;
          ov[e] = legacy_value<BITS, true>(code, sc[e], oo[e], lr[e]);
        }
        st16(a.out + erow + c0, pack8(ov));
        st16(a.out + erow + c0 + 8, pack8(ov + 8));
      }
    }
  }
  if constexpr (MODE == kHist) {
    __syncthreads();
    if (lh[threadIdx.x] != 0u) atomicAdd(&a.hist[threadIdx.x], lh[threadIdx.x]);
  }
}

// ------------------------------------------------------------------ MFMA encode
// Independent waves (no barrier), four to a workgroup on four neighbouring units of the same rows: wave
// w of tile (batch, run, unit group), unit groups fastest, in XCD order (xcd_tile), takes unit 4 * group +
// w over RBW 16-row blocks.  x streams through a private LDS ring of four (row block, plane) slots,
// 16 rows x 128 bytes each, straight from HBM (two 1 KB loads of eight whole lines; slot position c of
// row r holds chunk c ^ (r % 8), so that reading it back in the MFMA layout spreads over the banks); a
// slot is requested again, four planes on, as soon as the wave has read it.  A skeleton with these
// accesses and stores moves the 604 MB of [4, 8192, 8192] at 2 bits in 126 us; loads in the MFMA
// layout, four row blocks of one unit per workgroup, took 162 - 176 us.  The encode itself runs 152 us
// there (218 us in that layout with the element work on the VALU; 184 us with it on the matrix pipe),
// 155 us at 1 bit (202 us); 13.4 vector instructions per element at 1 bit, matrix steps included (22.4
// before, without any).
// STAGED: each 64-column piece's record (lrq_coo.h) goes to a.pcnt and the dense outliers only of the
// pieces it cannot hold; else the dense outliers.  A block's 16 NP records are gathered in LDS, each
// lane writing the entries it holds (usually none or one: the or of its masked values), and leave
// as one 8-byte store per record.
// At 1 bit and rank 32 the r^T operands of eight planes (128 registers) spilled inside the loop, and the
// reloads waited in the ring's memory queue: the last LP planes' live in LDS (with 3 one workgroup per CU
// would be left).  With the compaction [4, 4096, 4096] 82.5 -> 59.6 us, [4, 8192, 8192] 229 -> 186 us.
template <int BITS, int K>
struct LegacyEnc {
  static constexpr int NP = 8 / BITS, NW = 4, RING = 4, SLOT = 16 * 128, NREC = 16 * NP;
  static constexpr int LP = BITS == 1 && K == 32 ? 2 : 0;
  static constexpr int TAB = NP * 64 * 4, WAVE = RING * SLOT + TAB + NREC * 8 + LP * 4 * 64 * 16;  // bytes per wave
  static constexpr int kStepOps = 4;  // memory operations per step: two loads, two (dense outlier) stores
};
template <int BITS, int K, bool STAGED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(!STAGED ? 1 : BITS >= 2 && K == 16 ? 3 : 2))) void k_legacy_encode(
    LegacyArgs a, int RBW, int ug) {
  using Le = LegacyEnc<BITS, K>;
  constexpr int NP = Le::NP, G = 64, E = 16, RT = K / 16, RING = Le::RING, SLOT = Le::SLOT, NREC = Le::NREC, VREG = NP - Le::LP;
  __shared__ __attribute__((aligned(16))) unsigned char lds[Le::NW][Le::WAVE];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  const int j = lane & 15, g = lane >> 4;
  const int M = (int)a.M, N = (int)a.N, nrb = (M + 15) / 16, nrun = (nrb + RBW - 1) / RBW;
  const int t = __builtin_amdgcn_readfirstlane(xcd_tile(blockIdx.x, gridDim.x));
  const int u = __builtin_amdgcn_readfirstlane(t % ug) * Le::NW + w;
  const int run = __builtin_amdgcn_readfirstlane((t / ug) % nrun), b = __builtin_amdgcn_readfirstlane(t / (ug * nrun));
  const int64_t NB = N / NP;  // bytes per code row
  if (u * G >= NB) return;    // the group's last units (this wave only)
  const int rb0 = run * RBW, nblk = min(RBW, nrb - rb0);
  unsigned char* const ring = lds[w];
  uint32_t* const rtab = reinterpret_cast<uint32_t*>(ring + RING * SLOT);  // [NP][16 (g, j % 4)][4 steps]
  u32x2* const recs = reinterpret_cast<u32x2*>(ring + RING * SLOT + Le::TAB);
  const uint16_t* srow = a.s + (a.s_rows == 1 ? 0 : (int64_t)b * N);

  // step st = (block st / NP, plane st % NP): slot st % RING.  Load k covers rows 8k .. 8k + 7 of the
  // block (rows past the end clamp to the last), lane l chunk (l % 8) ^ (row % 8) of row 8k + l / 8.
  const uint16_t* const xbase = a.x + (int64_t)b * a.ldx_b + u * G + 8 * ((lane & 7) ^ (lane >> 3));
  auto request = [&](int i, int p, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int64_t row = min((rb0 + i) * 16 + 8 * k + (lane >> 3), M - 1);
      ld16_to_lds(xbase + row * a.ldx_m + p * NB, ring + slot * SLOT + 1024 * k);
    }
  };
#pragma unroll
  for (int st = 0; st < RING; ++st) request(min(st / NP, nblk - 1), st % NP, st);
  u32x2 nl[RT];
  auto fetch_l = [&](int i) __attribute__((always_inline)) {
    const int64_t rn = min((rb0 + i) * 16 + j, M - 1);
#pragma unroll
    for (int k = 0; k < RT; ++k) nl[k] = ld8(a.l + rn * K + 16 * k + 4 * g);
  };
  fetch_l(0);
  u32x2 vop[VREG][4][RT];
#pragma unroll
  for (int p = 0; p < VREG; ++p) load_vops<G, K>(a.rt, unit_base(p, u, N, NP, G), j, g, vop[p]);
  u32x4* const vlds = reinterpret_cast<u32x4*>(ring + RING * SLOT + Le::TAB + NREC * 8) + lane;  // [LP][4][64]
  if constexpr (Le::LP > 0) {
#pragma unroll 1
    for (int p = 0; p < Le::LP; ++p) {
      u32x2 v[4][RT];
      load_vops<G, K>(a.rt, unit_base(VREG + p, u, N, NP, G), j, g, v);
#pragma unroll
      for (int q = 0; q < 4; ++q) vlds[(p * 4 + q) * 64] = u32x4{v[q][0][0], v[q][0][1], v[q][RT - 1][0], v[q][RT - 1][1]};
    }
  }
  auto lowrank = [&](auto pc, const u32x2* lo, f32x4 (&t)[4]) __attribute__((always_inline)) {  // plane pc's fp32(l r)
    constexpr int p = decltype(pc)::value;
    if constexpr (p < VREG) {
      legacy_lowrank_mfma<K>(vop[p], lo, t);
    } else {
      u32x2 v[4][RT];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const u32x4 d = vlds[((p - VREG) * 4 + q) * 64];
        v[q][0] = u32x2{d[0], d[1]};
        v[q][RT - 1] = u32x2{d[2], d[3]};
      }
      legacy_lowrank_mfma<K>(v, lo, t);
    }
  };
  // fast: the estimate serves every scale of the unit and the threshold is not negative
  int ok = a.tau >= 0.f ? 1 : 0;
  float smin = INFINITY;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const float sv = bf_lo(srow[unit_base(p, u, N, NP, G) + lane]);
    smin = fminf(smin, fabsf(sv));
    uint32_t r1, r2;
    legacy_rc_split(sv, r1, r2);
    // column c = 16g' + 4q + v of the unit: entry [g'][v][q]
    rtab[p * 64 + ((lane >> 4) * 4 + (lane & 3)) * 4 + ((lane >> 2) & 3)] = r1 | (r2 << 16);
    ok &= rc_scale_ok(sv) ? 1 : 0;
  }
  const bool fast = __builtin_amdgcn_ballot_w64(ok == 0) == 0;  // wave-uniform
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) smin = fminf(smin, __shfl_xor(smin, d));
  // magnitudes below 2^118 min |s| keep every quotient below 2^119 (at most the bits of infinity)
  const uint32_t mag_limit = __builtin_amdgcn_readfirstlane(__float_as_uint(smin * 0x1p118f) >> 16);
  const u32x2 ida = diag4_aop(lane, 0x3f80u), idn = diag4_aop(lane, 0xbf80u);  // I, -I
  const uint32_t tau2 = (__float_as_uint(a.tau) >> 16) * 0x10001u;
  // the prologue's loads have landed (the counted waits below start from none outstanding)
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  __builtin_amdgcn_sched_barrier(0);

#pragma unroll 1
  for (int i = 0; i < nblk; ++i) {
    const int row0 = (rb0 + i) * 16;
    const int row = row0 + j;
    const int64_t rr = min(row, M - 1);
    u32x2 lop[RT];
#pragma unroll
    for (int k = 0; k < RT; ++k) lop[k] = nl[k];
    fetch_l(min(i + 1, nblk - 1));
    uint32_t byte[E];
#pragma unroll
    for (int e = 0; e < E; ++e) byte[e] = legacy_code_base<BITS>();
    if constexpr (STAGED) {
#pragma unroll
      for (int k = 0; k < (NREC + 63) / 64; ++k)
        if (64 * k + lane < NREC) recs[64 * k + lane] = u32x2{0u, 0u};
    }
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, NP>([&](auto pc) {
      constexpr int p = decltype(pc)::value;
      const int c0 = unit_base(p, u, N, NP, G) + E * g;
      const int slot = (i * NP + p) % RING;
      // The slot's loads were issued RING steps ago; the RING - 1 steps between issued kStepOps memory
      // operations each (and the blocks' own loads and stores besides), and memory operations retire
      // in issue order.
      __builtin_amdgcn_s_waitcnt(vmcnt_imm((RING - 1) * Le::kStepOps));
      __builtin_amdgcn_sched_barrier(0);
      const unsigned char* xs = ring + slot * SLOT + 128 * j;
      const u32x4 x0 = *reinterpret_cast<const u32x4*>(xs + 16 * ((2 * g) ^ (j & 7)));
      const u32x4 x1 = *reinterpret_cast<const u32x4*>(xs + 16 * ((2 * g + 1) ^ (j & 7)));
      const u32x4 rc = *reinterpret_cast<const u32x4*>(rtab + p * 64 + (g * 4 + (j & 3)) * 4);
      f32x4 tl[4], tx[4];
      lowrank(pc, lop, tl);
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the slot is read
      __builtin_amdgcn_sched_barrier(0);
      // (past the run the last block is requested again: unused)
      request(min(i + (p + RING) / NP, nblk - 1), (p + RING) % NP, slot);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const u32x4 x = q < 2 ? x0 : x1;
        tx[q] = mfma_4x4x4(ida, u32x2{x[2 * (q & 1)], x[2 * (q & 1) + 1]}, zero4());
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
        tx[q] = mfma_4x4x4(idn, u32x2{pack_bf16x2(tl[q][0], tl[q][1]), pack_bf16x2(tl[q][2], tl[q][3])}, tx[q]);
      uint32_t ow[8];   // the residuals, then the outlier values, packed
      uint32_t hm = 0;  // bit e: element e is an outlier entry
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        ow[2 * q] = pack_bf16x2(tx[q][0], tx[q][1]);
        ow[2 * q + 1] = pack_bf16x2(tx[q][2], tx[q][3]);
      }
      uint32_t code[E];
      bool slow = true;
      if (fast) slow = __builtin_amdgcn_ballot_w64(legacy_codes_mfma<BITS>(ow, tau2, mag_limit, rc, lane, code, hm)) != 0;
      if (slow) {
        // scales the estimate does not serve, a negative threshold, or an x (or residual) that is not
        // finite in the wave's plane: legacy_code of each element, two at a time
        float lr[E], xv[E], ov[E];
        const uint16_t* xp = a.x + (int64_t)b * a.ldx_b + rr * a.ldx_m + c0;
        unpack8(ld16(xp), xv);
        unpack8(ld16(xp + 8), xv + 8);
        lowrank(pc, lop, tl);
        hm = 0;
#pragma unroll
        for (int e = 0; e < E; ++e) lr[e] = tl[e >> 2][e & 3];
#pragma unroll
        for (int e = 0; e < E; e += 2) {
          const uint32_t sw = ld4(srow + c0 + e);
          const float sc[2] = {bf_lo(sw), bf_hi(sw)};
          bool hit[2];
          uint32_t cd[2];
          bf16_roundtrip2(lr[e], lr[e + 1]);
          legacy_code_mfma2<BITS>(xv + e, lr + e, sc, a.tau, ov + e, hit, cd);
          code[e] = BITS == 1 ? (cd[0] ^ 1u) << 31 : cd[0];
          code[e + 1] = BITS == 1 ? (cd[1] ^ 1u) << 31 : cd[1];
          hm |= (hit[0] ? 1u << e : 0u) | (hit[1] ? 2u << e : 0u);
          ow[e / 2] = pack_bf16x2(ov[e], ov[e + 1]);
        }
      }
#pragma unroll
      for (int e = 0; e < E; ++e) {
        legacy_accumulate<BITS>(byte[e], code[e], p);
        asm("" : "+v"(byte[e]));  // accumulated here, not kept as a code per plane until the end
      }
      const u32x4 ow0 = u32x4{ow[0], ow[1], ow[2], ow[3]}, ow1 = u32x4{ow[4], ow[5], ow[6], ow[7]};
      if constexpr (STAGED) {
        // the lane's entries: hits pre .. pre + n - 1 of its row's piece (lane g: columns 16g .. 16g + 15)
        static_assert(kCooSlots == 2, "two entries per record");
        const uint32_t n = __builtin_popcount(hm);
        uint32_t pre, total;
        row_prefix4(n, g, pre, total);
        uint32_t* rec = reinterpret_cast<uint32_t*>(&recs[p * 16 + j]);
        const uint32_t col = (uint32_t)(16 * g);
        if (__builtin_amdgcn_ballot_w64(n > 1u) != 0) {  // (wave-uniform)
          const uint32_t i0 = __builtin_ctz(hm | 0x10000u) & 15u, h1 = hm & (hm - 1u);
          const uint32_t i1 = __builtin_ctz(h1 | 0x10000u) & 15u;
          if (n > 0u && pre < 2u) rec[pre] = (col + i0) | (bf16_at(ow0, ow1, i0) << 16) | (pre == 0u ? total << 8 : 0u);
          if (n > 1u && pre == 0u) rec[1] = (col + i1) | (bf16_at(ow0, ow1, i1) << 16);
        } else {
          // at most one hit in the lane: its value is the or of the masked ones
          const uint32_t o = (ow[0] | ow[1] | ow[2]) | (ow[3] | ow[4] | ow[5]) | (ow[6] | ow[7]);
          const uint32_t v = (o & 0xffff0000u) | (o << 16);
          if (n > 0u && pre < 2u) rec[pre] = (col + __builtin_ctz(hm)) | v | (pre == 0u ? total << 8 : 0u);
        }
        uint16_t* orow = a.oout + ((int64_t)b * M + row0) * N;
        const uint32_t olen = (uint32_t)(16 * N * 2), ooff = (uint32_t)(((rr - row0) * N + c0) * 2);
        const bool dense = total > (uint32_t)kCooSlots && row < M;
        st16_pred(orow, olen, ooff, ow0, dense);
        st16_pred(orow, olen, ooff + 16, ow1, dense);
      } else {
        uint16_t* op = a.oout + ((int64_t)b * M + rr) * N + c0;
        st16(op, ow0);
        st16(op + 8, ow1);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    uint32_t word[E / 4];
#pragma unroll
    for (int k = 0; k < E / 4; ++k) {
      word[k] = gather_bytes(byte[4 * k], byte[4 * k + 1], byte[4 * k + 2], byte[4 * k + 3]);
      if constexpr (BITS == 1) word[k] = ~word[k];
    }
    st16(a.qout + ((int64_t)b * M + rr) * NB + u * G + E * g, u32x4{word[0], word[1], word[2], word[3]});
    if constexpr (STAGED) {
      // record 64 k + lane: plane (64 k + lane) / 16, row lane % 16 (range-checked stores: no branch)
      int64_t* prow = a.pcnt + ((int64_t)b * M + row0) * a.npc;  // the block's first row
#pragma unroll
      for (int k = 0; k < (NREC + 63) / 64; ++k) {
        const int q = min(64 * k + lane, NREC - 1);
        st8_pred(prow, (uint32_t)(16 * a.npc * 8), (uint32_t)((j * a.npc + (q >> 4) * (NB / 64) + u) * 8), recs[q],
                 64 * k + lane < NREC && row < M);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // the requests past the run have landed before the LDS can go to another workgroup
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
}

// ------------------------------------------------------------------ MFMA decode and fused consumers
// x_hat without outliers or with sparse COO outliers (COO), stored (kDecode / kFusedStore) or consumed
// with y (kFusedSilu, kFusedMul).  Independent waves as in k_legacy_encode (wave w of a tile: unit
// 4 * group + w, RBW 16-row blocks); a step is one plane of one block.
// - y streams through the same LDS ring of whole 128-byte lines; the result goes through a private LDS
//   tile and leaves as two 1 KB stores of whole lines (a skeleton of the MFMA-layout accesses that
//   these replace reaches 3.9 TB/s, of these 5.1).
// - Element work on the matrix pipe (diagonal 4x4x4 steps, see legacy_codes_mfma): the codes enter as
//   the bf16 values 128 + c (a byte permute, no conversion), a = s (128 + c) - s (128 + h) is exact in
//   fp32 (h = 2^(b-1); at 8 bits c = 16 hi + lo takes two steps); then a's bf16 rounding (4 and 8 bits),
//   + o and + bf16(l r) are identity steps with one rounding each, as in legacy_value.  The 2-bit COO
//   decode issues 8.4 vector instructions per element, matrix steps included (row-tile decode 15.7).
//   2-bit decode of [4, 8192, 8192] with 0.6 % outliers 209 -> 114 us, 1-bit 319 -> 115 us; SiLU gradient
//   at [4, 4096, 4096] 97 -> 57.6 us a call.
// - COO: the block's pieces (one per (row, plane)) take LPP lanes each; a lane's piece bounds are
//   requested two blocks ahead and its SLOTS entries one block ahead, as range-checked loads (an absent
//   entry reads nothing); they go into the wave's zeroed tile [NP][16][64] at the block's start and are
//   cleared from it at its end.  Pieces with more entries take further rounds on the spot.
// A diagonal step sums over four elements, so nothing in it may overflow or be infinite: scales below
// 2^100, |o| below 2^126 and max |l| max |r| K below 2^120 (legacy_value's sums are then all finite);
// a block beyond that takes legacy_value element by element.
template <int MODE, int BITS, int COO>
struct LegacyApply {
  static constexpr int NP = 8 / BITS, NW = 4, RING = 4, SLOT = 16 * 128, NREC = 16 * NP;
  static constexpr bool HASY = MODE == kFusedSilu || MODE == kFusedMul;
  static constexpr int TAB = NP * 64 * 4;
  static constexpr int OFF_TAB = HASY ? RING * SLOT : 0, OFF_OUT = OFF_TAB + TAB, OFF_O = OFF_OUT + SLOT;
  static constexpr int WAVE = OFF_O + (COO ? NP * SLOT : 0);  // bytes per wave
  static constexpr int kStepOps = 4;                          // with y: two loads, two stores per step
  static constexpr int64_t kWindow = (int64_t)1 << 27;        // entries of a block within reach of its first
  static constexpr int LPP = NREC <= 64 ? 64 / NREC : 1, PPL = NREC <= 64 ? 1 : NREC / 64;
  // entries of a piece per lane and round (2 bits, 16 % outliers: [4, 3072, 3072] 49.7 us at 8, 58.5 at
  // 12, 61.3 at 20)
  static constexpr int SLOTS = COO == 2 ? (PPL > 1 ? 4 : LPP == 1 ? 8 : 20 / LPP) : PPL == 1 && LPP < 4 ? 4 : 2;
};
template <int MODE, int BITS, int K, int COO>
__global__ __launch_bounds__(256) void k_legacy_apply(LegacyArgs a, int RBW, int ug) {
  using La = LegacyApply<MODE, BITS, COO>;
  constexpr int NP = La::NP, G = 64, E = 16, RT = K / 16, RING = La::RING, SLOT = La::SLOT;
  constexpr bool HASY = La::HASY;
  __shared__ __attribute__((aligned(16))) unsigned char lds[La::NW][La::WAVE];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  const int j = lane & 15, g = lane >> 4;
  const int M = (int)a.M, N = (int)a.N, nrb = (M + 15) / 16, nrun = (nrb + RBW - 1) / RBW;
  const int t = __builtin_amdgcn_readfirstlane(xcd_tile(blockIdx.x, gridDim.x));
  const int u = __builtin_amdgcn_readfirstlane(t % ug) * La::NW + w;
  const int run = __builtin_amdgcn_readfirstlane((t / ug) % nrun), b = __builtin_amdgcn_readfirstlane(t / (ug * nrun));
  const int64_t NB = N / NP;  // bytes per code row
  if (u * G >= NB) return;    // the group's last units (this wave only)
  const int rb0 = run * RBW, nblk = min(RBW, nrb - rb0);
  const int64_t bm0 = (int64_t)b * M;
  unsigned char* const ring = lds[w];
  uint32_t* const stab = reinterpret_cast<uint32_t*>(ring + La::OFF_TAB);  // [NP][16 (g, j % 4)][4 steps]
  unsigned char* const otile = ring + La::OFF_O;
  unsigned char* const xtile = ring + La::OFF_OUT;
  const uint16_t* srow = a.s + (a.s_rows == 1 ? 0 : (int64_t)b * N);

  // y: step st = (block st / NP, plane st % NP) in slot st % RING (see k_legacy_encode)
  const uint16_t* const ybase = HASY ? a.y + bm0 * N + u * G + 8 * ((lane & 7) ^ (lane >> 3)) : nullptr;
  auto request = [&](int i, int p, int slot) __attribute__((always_inline)) {
    if constexpr (HASY) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int64_t row = min((rb0 + i) * 16 + 8 * k + (lane >> 3), M - 1);
        ld16_to_lds(ybase + row * N + p * NB, ring + slot * SLOT + 1024 * k);
      }
    }
  };
#pragma unroll
  for (int st = 0; st < RING; ++st) request(min(st / NP, nblk - 1), st % NP, st);
  u32x2 nl[RT];
  u32x4 nq;
  auto fetch = [&](int i) __attribute__((always_inline)) {  // block i's codes and l operand
    const int64_t rn = min((rb0 + i) * 16 + j, M - 1);
#pragma unroll
    for (int k = 0; k < RT; ++k) nl[k] = ld8(a.l + rn * K + 16 * k + 4 * g);
    nq = ld16(a.qin + (bm0 + rn) * NB + u * G + E * g);
  };
  fetch(0);

  // COO: lane -> piece pi = lane / LPP + 64 q' of the block (plane pi / 16, row pi % 16), place lane % LPP
  constexpr int LPP = La::LPP, PPL = La::PPL, SL = La::SLOTS;
  struct Bnd {
    int64_t s0, s1;
  };
  struct Ent {
    uint32_t col[SL];
    uint32_t val[SL];
  };
  Bnd bnd[PPL], bnd_n[PPL];  // of the block whose entries are in flight, and of the one after
  Ent ent[PPL];
  int64_t ebase = 0;  // the entry buffers' first entry (wave-uniform)
  auto bounds = [&](int i, Bnd (&d)[PPL]) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < PPL; ++h) {
      const int pi = lane / LPP + 64 * h;
      const int64_t rn = min((rb0 + i) * 16 + (pi & 15), M - 1);
      const int64_t pc = (bm0 + rn) * a.npc + (pi >> 4) * (NB / G) + u;
      d[h].s0 = max(a.optr[pc], (int64_t)0);
      d[h].s1 = min(a.optr[pc + 1], a.ncap);
    }
  };
  // entries s0 + LPP * (SL * round + k) + lane % LPP, k < SL, of the lane's pieces; an entry past the
  // piece (or kWindow entries past the block's first) is outside the range and reads as column 0, value 0
  auto load_entries = [&](const Bnd (&d)[PPL], int round, Ent (&en)[PPL]) __attribute__((always_inline)) {
    const int64_t left = max(min(a.ncap - ebase, La::kWindow), (int64_t)0);
    const __amdgpu_buffer_rsrc_t rc = uniform_rsrc(const_cast<int64_t*>(a.ocol + ebase), (uint32_t)(left * 8));
    const __amdgpu_buffer_rsrc_t rv = uniform_rsrc(const_cast<uint16_t*>(a.oval + ebase), (uint32_t)(left * 2));
#pragma unroll
    for (int h = 0; h < PPL; ++h)
#pragma unroll
      for (int k = 0; k < SL; ++k) {
        const int64_t e = d[h].s0 + LPP * (SL * round + k) + lane % LPP;
        const int64_t rel = e - ebase;
        const bool in = e < d[h].s1 && rel >= 0 && rel < left;
        en[h].col[k] = __builtin_amdgcn_raw_buffer_load_b32(rc, in ? (uint32_t)rel * 8u : 0x7ffffff0u, 0, 0);
        en[h].val[k] = __builtin_amdgcn_raw_buffer_load_b16(rv, in ? (uint32_t)rel * 2u : 0x7ffffff0u, 0, 0);
      }
  };
  // writes the entries of a round into the tile (or clears them from it); returns whether an entry's
  // magnitude is 2^126 or more (or not finite)
  auto put = [&](const Bnd (&d)[PPL], int round, const Ent (&en)[PPL], bool clear) __attribute__((always_inline)) -> bool {
    bool big = false;
#pragma unroll
    for (int h = 0; h < PPL; ++h) {
      const int pi = lane / LPP + 64 * h;
      const int cbase = (pi >> 4) * (int)NB + u * G;
#pragma unroll
      for (int k = 0; k < SL; ++k) {
        const int64_t e = d[h].s0 + LPP * (SL * round + k) + lane % LPP;
        const int64_t rel = e - ebase;
        const uint32_t c = en[h].col[k] - (uint32_t)cbase;
        if (e < d[h].s1 && rel >= 0 && rel < La::kWindow && c < 64u) {
          // (chunk c / 8 of row r at position (c / 8) ^ (r % 8))
          uint16_t* o = reinterpret_cast<uint16_t*>(otile + pi * 128 + 16 * ((c >> 3) ^ (pi & 7)));
          o[c & 7u] = clear ? (uint16_t)0 : (uint16_t)en[h].val[k];
          big |= (en[h].val[k] & 0x7fffu) >= 0x7e80u;
        }
      }
    }
    return big;
  };
  auto zero_tile = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2 * NP; ++k) *reinterpret_cast<u32x4*>(otile + 1024 * k + 16 * lane) = u32x4{0u, 0u, 0u, 0u};
  };
  auto first_entry = [&](const Bnd (&d)[PPL]) __attribute__((always_inline)) -> int64_t {
    const uint64_t v = (uint64_t)d[0].s0;  // lane 0: plane 0 of the block's first row, the smallest
    return (int64_t)(((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(v >> 32)) << 32) |
                     (uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)v));
  };
  if constexpr (COO != 0) {
    bounds(0, bnd);
    bounds(min(1, nblk - 1), bnd_n);
    zero_tile();
    ebase = first_entry(bnd);
    load_entries(bnd, 0, ent);
  }

  u32x2 vop[NP][4][RT];
  uint32_t rtop = 0;  // the largest magnitude of the lane's r^T operands (bf16 bits, both halves)
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    load_vops<G, K>(a.rt, unit_base(p, u, N, NP, G), j, g, vop[p]);
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int k = 0; k < RT; ++k)
        rtop = pk_max_u16(pk_max_u16(rtop, vop[p][q][k][0] & 0x7fff7fffu), vop[p][q][k][1] & 0x7fff7fffu);
  }
  bool s_ok = true;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const float sv = bf_lo(srow[unit_base(p, u, N, NP, G) + lane]);
    s_ok &= (__float_as_uint(sv) & 0x7fffffffu) < 0x71800000u;  // |s| < 2^100 (as bits: a NaN is above)
    // bf16(s) | bf16(16 s) << 16: the second term serves the high nibble at 8 bits
    stab[p * 64 + ((lane >> 4) * 4 + (lane & 3)) * 4 + ((lane >> 2) & 3)] = pack_bf16x2(sv, 16.f * sv);
  }
  uint32_t rmax = max(rtop >> 16, rtop & 0xffffu);
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) rmax = max(rmax, (uint32_t)__shfl_xor((int)rmax, d));
  // K max |r| of the unit, infinite or NaN when an operand is
  const float rbound = (float)K * __uint_as_float(__builtin_amdgcn_readfirstlane(rmax) << 16);
  const bool unit_ok = __builtin_amdgcn_ballot_w64(!s_ok) == 0;  // wave-uniform
  const u32x2 ida = diag4_aop(lane, 0x3f80u);
  constexpr uint32_t kMask = (BITS == 8 ? 0x0fu : (1u << BITS) - 1u) * 0x01010101u;
  constexpr int kHalf = 1 << (BITS - 1);
  // -(128 + h) as bf16 pairs (at 8 bits -(16 * 128 + 128 + 128)): exact
  const uint32_t koff = pack_bf16x2_exact(-(float)(BITS == 8 ? 2304 : 128 + kHalf), -(float)(BITS == 8 ? 2304 : 128 + kHalf));
  if constexpr (HASY) {
    // the prologue's loads have landed (the counted waits below start from none outstanding)
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    __builtin_amdgcn_sched_barrier(0);
  }

#pragma unroll 1
  for (int i = 0; i < nblk; ++i) {
    const int row0 = (rb0 + i) * 16;
    u32x2 lop[RT];
#pragma unroll
    for (int k = 0; k < RT; ++k) lop[k] = nl[k];
    const u32x4 qb = nq;
    bool big = false, rest = false;
    Bnd cur[PPL];
    Ent cure[PPL];
    int64_t cbase_e = ebase;
    if constexpr (COO != 0) {
      big = put(bnd, 0, ent, false);
#pragma unroll
      for (int h = 0; h < PPL; ++h) {
        rest |= bnd[h].s1 - bnd[h].s0 > (int64_t)LPP * SL;
        cur[h] = bnd[h];
        if constexpr (COO == 1) cure[h] = ent[h];
        bnd[h] = bnd_n[h];
      }
      rest = __builtin_amdgcn_ballot_w64(rest) != 0;  // (wave-uniform)
      if (rest) {
        for (int round = 1;; ++round) {
          bool more = false;
          Ent en[PPL];
          load_entries(cur, round, en);
          big |= put(cur, round, en, false);
#pragma unroll
          for (int h = 0; h < PPL; ++h) more |= cur[h].s1 - cur[h].s0 > (int64_t)LPP * SL * (round + 1);
          if (__builtin_amdgcn_ballot_w64(more) == 0) break;
        }
      }
      ebase = first_entry(bnd);
      load_entries(bnd, 0, ent);
      bounds(min(i + 2, nblk - 1), bnd_n);
    }
    fetch(min(i + 1, nblk - 1));
    // max |l| K max |r| < 2^120: every l r is finite and small enough
    uint32_t lt = 0;
#pragma unroll
    for (int k = 0; k < RT; ++k) lt = pk_max_u16(lt, pk_max_u16(lop[k][0] & 0x7fff7fffu, lop[k][1] & 0x7fff7fffu));
    const float lmax = __uint_as_float(max(lt & 0xffff0000u, lt << 16));
    // (as bits: an infinity or a NaN in either is above)
    const uint32_t lrb = __float_as_uint(lmax * rbound) & 0x7fffffffu;
    const bool lr_big = lrb >= 0x7b800000u || __float_as_uint(lmax) >= 0x7f800000u || __float_as_uint(rbound) >= 0x7f800000u;
    const bool fast = unit_ok && __builtin_amdgcn_ballot_w64(lr_big || big) == 0;  // wave-uniform
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, NP>([&](auto pc) {
      constexpr int p = decltype(pc)::value;
      const int slot = (i * NP + p) % RING;
      u32x4 yw[2];
      if constexpr (HASY) {
        // (the slot's loads: RING steps ago, kStepOps memory operations in each step since)
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((RING - 1) * La::kStepOps));
        __builtin_amdgcn_sched_barrier(0);
        const unsigned char* ys = ring + slot * SLOT + 128 * j;
        yw[0] = *reinterpret_cast<const u32x4*>(ys + 16 * ((2 * g) ^ (j & 7)));
        yw[1] = *reinterpret_cast<const u32x4*>(ys + 16 * ((2 * g + 1) ^ (j & 7)));
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the slot is read
        __builtin_amdgcn_sched_barrier(0);
        request(min(i + (p + RING) / NP, nblk - 1), (p + RING) % NP, slot);
        __builtin_amdgcn_sched_barrier(0);
      }
      u32x4 ov[2] = {u32x4{0u, 0u, 0u, 0u}, u32x4{0u, 0u, 0u, 0u}};
      if constexpr (COO != 0) {
        const unsigned char* os = otile + (p * 16 + j) * 128;
        ov[0] = *reinterpret_cast<const u32x4*>(os + 16 * ((2 * g) ^ (j & 7)));
        ov[1] = *reinterpret_cast<const u32x4*>(os + 16 * ((2 * g + 1) ^ (j & 7)));
      }
      uint32_t xo[8];  // x_hat, packed
      f32x4 tl[4], tv[4];
      legacy_lowrank_mfma<K>(vop[p], lop, tl);
      if (fast) {
        const u32x4 st = *reinterpret_cast<const u32x4*>(stab + p * 64 + (g * 4 + (j & 3)) * 4);
        const u32x2 sel = diag4_sel(lane, 0), selh = diag4_sel(lane, 1);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const u32x2 sa = u32x2{__builtin_amdgcn_perm(st[q], st[q], sel[0]), __builtin_amdgcn_perm(st[q], st[q], sel[1])};
          // elements 4q .. 4q + 3: 128 + code as bf16 (bytes code, 0x43)
          const uint32_t m = BITS == 8 ? qb[q] & kMask : (qb[q] >> (BITS * p)) & kMask;
          const u32x2 cb = u32x2{__builtin_amdgcn_perm(0x43434343u, m, 0x04010400u), __builtin_amdgcn_perm(0x43434343u, m, 0x04030402u)};
          f32x4 v = mfma_4x4x4(sa, u32x2{koff, koff}, zero4());
          v = mfma_4x4x4(sa, cb, v);
          if constexpr (BITS == 8) {
            const u32x2 sb = u32x2{__builtin_amdgcn_perm(st[q], st[q], selh[0]), __builtin_amdgcn_perm(st[q], st[q], selh[1])};
            const uint32_t mh = (qb[q] >> 4) & kMask;
            v = mfma_4x4x4(sb, u32x2{__builtin_amdgcn_perm(0x43434343u, mh, 0x04010400u), __builtin_amdgcn_perm(0x43434343u, mh, 0x04030402u)}, v);
          }
          tv[q] = v;
        }
        auto rounded = [&](f32x4 v) __attribute__((always_inline)) {
          return u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        };
        if constexpr (BITS > 2) {  // (already a bf16 value at 1 and 2 bits)
#pragma unroll
          for (int q = 0; q < 4; ++q) tv[q] = mfma_4x4x4(ida, rounded(tv[q]), zero4());
        }
        if constexpr (COO != 0) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const u32x4 o = ov[q >> 1];
            tv[q] = mfma_4x4x4(ida, u32x2{o[2 * (q & 1)], o[2 * (q & 1) + 1]}, tv[q]);
          }
#pragma unroll
          for (int q = 0; q < 4; ++q) tv[q] = mfma_4x4x4(ida, rounded(tv[q]), zero4());
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) tv[q] = mfma_4x4x4(ida, rounded(tl[q]), tv[q]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const u32x2 r = rounded(tv[q]);
          xo[2 * q] = r[0];
          xo[2 * q + 1] = r[1];
        }
      } else {
        const uint16_t* sp = srow + unit_base(p, u, N, NP, G) + E * g;
#pragma unroll
        for (int e = 0; e < E; e += 2) {
          const uint32_t sw = ld4(sp + e), ow = ov[e >> 3][(e >> 1) & 3];
          const uint32_t c0 = (qb[e >> 2] >> (8 * (e & 3) + BITS * p)) & ((1u << BITS) - 1u);
          const uint32_t c1 = (qb[e >> 2] >> (8 * ((e + 1) & 3) + BITS * p)) & ((1u << BITS) - 1u);
          xo[e / 2] = pack_bf16x2_exact(
              legacy_value<BITS, COO != 0>(c0, bf_lo(sw), bf_lo(ow), bf16r(tl[e >> 2][e & 3])),
              legacy_value<BITS, COO != 0>(c1, bf_hi(sw), bf_hi(ow), bf16r(tl[e >> 2][(e + 1) & 3])));
        }
      }
      if constexpr (HASY) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const uint32_t y = yw[k >> 2][k & 3];
          xo[k] = pack_bf16x2(legacy_consume<MODE>(bf_lo(xo[k]), bf_lo(y)), legacy_consume<MODE>(bf_hi(xo[k]), bf_hi(y)));
        }
      }
      // through the tile (this wave's LDS operations run in order) to two stores of eight whole lines;
      // rows past the end fall outside the store range
      unsigned char* xs = xtile + 128 * j;
      *reinterpret_cast<u32x4*>(xs + 16 * ((2 * g) ^ (j & 7))) = u32x4{xo[0], xo[1], xo[2], xo[3]};
      *reinterpret_cast<u32x4*>(xs + 16 * ((2 * g + 1) ^ (j & 7))) = u32x4{xo[4], xo[5], xo[6], xo[7]};
      uint16_t* orow = a.out + (bm0 + row0) * N;
      const int c = u * G + p * (int)NB + 8 * ((lane & 7) ^ (lane >> 3));
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int r = 8 * k + (lane >> 3);
        const u32x4 v = *reinterpret_cast<const u32x4*>(xtile + 1024 * k + 16 * lane);
        st16_pred_stream(orow, (uint32_t)(16 * N * 2), (uint32_t)((r * N + c) * 2), v, row0 + r < M);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (COO != 0) {
      if (COO == 2 || rest) {
        zero_tile();
      } else {
        const int64_t keep = ebase;
        ebase = cbase_e;
        put(cur, 0, cure, true);
        ebase = keep;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // the requests past the run have landed before the LDS can go to another workgroup
  if constexpr (HASY) __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
}

// ------------------------------------------------------------------ scalar path
// One thread per packed byte position c of one row; grid.x enumerates (b, m, 256-byte chunk).
template <int MODE, int BITS, int OSRC>
__global__ __launch_bounds__(256) void k_legacy_scalar(LegacyArgs a, int K, int64_t chunks) {
  constexpr int NP = (MODE == kAdd) ? 1 : 8 / BITS;
  constexpr uint32_t kMask = BITS == 8 ? 0xffu : (1u << BITS) - 1u;
  const int64_t M = a.M, N = a.N, NB = N / NP;
  const int64_t blk = blockIdx.x;
  const int64_t bm = blk / chunks;
  const int64_t c = (blk - bm * chunks) * 256 + threadIdx.x;
  if (c >= NB) return;
  const int64_t b = bm / M, m = bm - b * M;
  const uint16_t* srow = a.s + (a.s_rows == 1 ? 0 : b * N);
  const uint16_t* lrow = a.l + m * K;
  const int64_t erow = bm * N;
  uint32_t byte = 0u;
  if constexpr (MODE == kDecode || MODE == kFusedStore || MODE == kFusedSilu || MODE == kFusedMul)
    byte = a.qin[bm * NB + c];
  uint32_t qout = 0u;
  for (int p = 0; p < NP; ++p) {
    const int64_t col = p * NB + c;
    const uint16_t* rrow = a.rt + col * K;
    double acc = 0.0;
    for (int k = 0; k < K; ++k)
      acc = __builtin_fma((double)__uint_as_float((uint32_t)lrow[k] << 16),
                          (double)__uint_as_float((uint32_t)rrow[k] << 16), acc);
    const float lr = bf16r((float)acc);
    if constexpr (MODE == kEncode) {
      const float xv = __uint_as_float((uint32_t)a.x[b * a.ldx_b + m * a.ldx_m + col] << 16);
      const float sc = __uint_as_float((uint32_t)srow[col] << 16);
      float o;
      bool hit;
      qout |= legacy_code<BITS>(xv, lr, sc, a.tau, o, hit) << (BITS * p);
      a.oout[erow + col] = (uint16_t)pack_bf16x2(o, 0.f);
    } else if constexpr (MODE == kAdd) {
      const float xv = __uint_as_float((uint32_t)a.x[b * a.ldx_b + m * a.ldx_m + col] << 16);
      a.out[erow + col] = (uint16_t)pack_bf16x2(xv + lr, 0.f);
    } else {
      const float sc = __uint_as_float((uint32_t)srow[col] << 16);
      const uint32_t code = (byte >> (BITS * p)) & kMask;
      float o = 0.f, yv = 0.f;
      if constexpr (MODE == kDecode && OSRC == 1) o = __uint_as_float((uint32_t)a.oin[erow + col] << 16);
      if constexpr (MODE == kDecode && OSRC >= 2) {  // COO pieces (both lookups give the same values)
        const int64_t pc = bm * a.npc + col / 64, e1 = min(a.optr[pc + 1], a.ncap);
        for (int64_t k = max(a.optr[pc], (int64_t)0); k < e1; ++k)
          if (a.ocol[k] == col) o = __uint_as_float((uint32_t)a.oval[k] << 16);
      }
      if constexpr (MODE == kFusedSilu || MODE == kFusedMul) yv = __uint_as_float((uint32_t)a.y[erow + col] << 16);
      const float xh = legacy_value<BITS, MODE == kDecode && OSRC != 0>(code, sc, o, lr);
      a.out[erow + col] = (uint16_t)pack_bf16x2(legacy_consume<MODE>(xh, yv), 0.f);
    }
  }
  if constexpr (MODE == kEncode) a.qout[bm * NB + c] = (uint8_t)qout;
}

// ------------------------------------------------------------------ row-tile decode
// Decode from denser COO outliers of large tensors (2, 4 or 8 bits; legacy_rows_pays), staged through an LDS
// tile so that the output leaves as whole row segments.  A workgroup of 4 waves owns 4 units
// (wave w: unit u0 + w, i.e. 64 columns in every plane) of one batch over a run of RBW 16-row
// blocks, with the unit's r^T operands in registers and the units' scales in LDS for the whole
// run (in registers they pushed the 2-bit kernel past 256 VGPRs: one wave per SIMD).  The tile is
// [16 rows][NP planes][256 columns] bf16 (rows padded by 16 bytes, so the lanes of a column
// quarter reach different banks), two of them in turn.  Per block b:
//   B1 | x_hat of block b: each lane reads its 16 outlier values per plane from tile b, forms
//   x_hat (the reconstruction MFMA for l @ r, the decode's roundings two columns at a time) and
//   writes it over them; the workers zero the other tile | B2 | tile b leaves as row segments
//   (non-temporal 16-byte stores of whole lines) and the codes and l operand of block b + PD are
//   requested (PD = 2; 4 measured slower); the workers write block b + 1's COO entries, requested
//   a block earlier, into the zeroed tile and request the entries of block b + 2 and the COO
//   bounds of block b + 4.
// COO ranges: the entries of one (row, plane) of the workgroup's units are contiguous (row-major
// COO, 64-column pieces in order): [piece_ptr[pc], piece_ptr[pc + units]).  The
// workgroup has 4 more waves, COO workers (their loads and waits stay out of the decoding waves'
// in-order memory queues): worker w takes ranges w * RPW .. w * RPW + RPW - 1 (range q: row q % 16,
// plane q / 16), LPR = 64 / RPW lanes each; lane l of range r loads its own bounds and entries
// start + l % LPR + LPR i for the i < ns the wave's longest range needs (64 entries of a range per
// pass); a range of more than 64 entries takes further passes right away.  An entry outside the
// units' columns, or past the entry capacity, is not written.  (Four waves per SIMD, two
// workgroups per CU: 128 VGPRs with a small spill measured faster than 136 VGPRs and one
// workgroup.)  Blocks are taken PD at a time
// (ring slots by position); the positions past the run compute on the last block's inputs and
// store nothing (a zero-length store range).
template <int BITS>
struct LegacyRows {
  static constexpr int NP = 8 / BITS, NW = 4, G = 64, SEG = NW * G, PD = 2;
  static constexpr int RSTR = NP * SEG + 8;  // bf16 per tile row
  static constexpr int TILE = 16 * RSTR;     // bf16 per tile
  static constexpr int NR = 16 * NP, RPW = NR / NW;
  static constexpr size_t LDS = (2 * (size_t)TILE + 64 + NP * SEG) * 2;  // two tiles, a 64-lane dummy row, the scales
  static_assert(BITS == 2 || BITS == 4 || BITS == 8, "2, 4 or 8 bits");
};

template <int BITS, int K>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void k_legacy_rows(LegacyArgs a, int RBW, int ug) {
  using Lr = LegacyRows<BITS>;
  constexpr int NP = Lr::NP, NW = Lr::NW, G = 64, E = 16, RT = K / 16, SEG = Lr::SEG, RSTR = Lr::RSTR;
  constexpr int TILE = Lr::TILE, RPW = Lr::RPW, PD = Lr::PD, T = 512;
  constexpr uint32_t kMask = BITS == 8 ? 0xffu : (1u << BITS) - 1u;
  extern __shared__ __attribute__((aligned(16))) uint16_t lt[];  // [2][TILE] + dummy[64]
  uint16_t* const dummy = lt + 2 * TILE;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, g = lane >> 4;
  const int M = (int)a.M, N = (int)a.N;
  const int64_t NB = N / NP;
  const int nu = (int)(NB / G), nrb = (M + 15) / 16, nrun = (nrb + RBW - 1) / RBW;
  // tile (batch, run, unit group), unit groups fastest, in XCD-aware order: the workgroups that
  // run together on an XCD take neighbouring unit groups of the same rows (their COO ranges and
  // code rows share L2 lines)
  const int t = __builtin_amdgcn_readfirstlane(xcd_tile(blockIdx.x, gridDim.x));
  const int ugi = t % ug, run = (t / ug) % nrun, b = t / (ug * nrun);
  const int u0 = ugi * NW, nuw = min(NW, nu - u0), u = min(u0 + w % NW, nu - 1);
  // waves NW .. 2 NW - 1 are COO workers: they zero the tiles and write the
  // entries into them, so that their loads and waits never hold up the decoding waves' block ring
  // (memory operations retire in issue order, per wave)
  const bool worker = w >= NW;  // (uniform)
  const int rb0 = run * RBW, nblk = min(RBW, nrb - rb0);
  const int64_t bm0 = (int64_t)b * M;  // first row of the batch in [B * M] rows
  const uint16_t* srow = a.s + (a.s_rows == 1 ? 0 : (int64_t)b * N);

  // resident: the unit's r^T operands and its 16 scales per plane (bf16 pairs)
  u32x2 vop[NP][G / 16][RT];
  uint16_t* const stab = lt + 2 * TILE + 64;  // [NP][SEG] scales of the workgroup's units (bf16)
  if (!worker) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int base = unit_base(p, u, N, NP, G);
      load_vops<G, K>(a.rt, base, j, g, vop[p]);
    }
  }
  for (int i = threadIdx.x; i < NP * SEG; i += T) {
    const int p = i / SEG, c = min(i % SEG, nuw * G - 1);
    stab[i] = srow[p * (int)NB + u0 * G + c];
  }

  // per block: codes (16 bytes per lane) and the l operand, PD blocks ahead
  struct Blk {
    u32x4 cb;
    u32x2 lop[RT];
  };
  auto load_blk = [&](int i, Blk& d) __attribute__((always_inline)) {
    const int64_t rr = min(min(rb0 + i, nrb - 1) * 16 + j, M - 1);
    d.cb = ld16_stream(a.qin + (bm0 + rr) * NB + u * G + E * g);
#pragma unroll
    for (int k = 0; k < RT; ++k) d.lop[k] = ld8(a.l + rr * K + 16 * k + 4 * g);
  };
  // COO (workers): this lane's range (row rq, plane pq) and its place among the range's LPR lanes
  constexpr int LPR = 64 / RPW;
  const int wq = w % NW;
  const int rq = (wq * RPW + lane / LPR) % 16, pq = (wq * RPW + lane / LPR) / 16, lr_ = lane % LPR;
  const int cbase = pq * (int)NB + u0 * G;  // the range's first column
  struct Bnd {
    int64_t s0, s1;
  };
  auto load_bounds = [&](int i) __attribute__((always_inline)) -> Bnd {
    const int64_t rr = min(min(rb0 + i, nrb - 1) * 16 + rq, M - 1);
    const int64_t pc = (bm0 + rr) * a.npc + (int64_t)pq * (NB / G) + u0;
    return Bnd{a.optr[pc], a.optr[pc + nuw]};
  };
  uint32_t ecol[RPW], eval[RPW];
  // the entry slots a pass needs: the wave's longest range over LPR lanes (wave-uniform)
  auto slots = [&](const Bnd& bd, int pass) __attribute__((always_inline)) -> int {
    int len = (int)min(min(bd.s1, a.ncap) - max(bd.s0, (int64_t)0) - (int64_t)64 * pass, (int64_t)64);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) len = max(len, __shfl_xor(len, m));
    return __builtin_amdgcn_readfirstlane(min(max(len, 0) + LPR - 1, 64) / LPR);
  };
  // entries start + 64 pass + lr_ + LPR i, i < ns, of the lane's range (indices clamped to the capacity)
  auto load_entries = [&](const Bnd& bd, int pass, int ns) __attribute__((always_inline)) {
    const int64_t s0 = max(bd.s0, (int64_t)0) + 64 * pass + lr_;
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      if (i < ns) {  // (uniform)
        const int64_t k = min(s0 + LPR * i, a.ncap - 1);
        ecol[i] = reinterpret_cast<const uint32_t*>(a.ocol)[2 * k];  // the column's low dword
        eval[i] = a.oval[k];
      }
    }
  };
  auto scatter = [&](uint16_t* tb, const Bnd& bd, int pass, int ns) __attribute__((always_inline)) {
    const int64_t s0 = max(bd.s0, (int64_t)0) + 64 * pass + lr_, s1 = min(bd.s1, a.ncap);
    uint16_t* row = tb + rq * RSTR + pq * SEG;
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      if (i < ns) {  // (uniform)
        const int d = (int)ecol[i] - cbase;
        const bool ok = s0 + LPR * i < s1 && d >= 0 && d < nuw * G;
        uint16_t* dst = ok ? row + d : dummy + lane;
        *dst = (uint16_t)eval[i];
      }
    }
  };
  // the passes after the first, for ranges of more than 64 entries (rare), loaded and written in turn
  auto scatter_rest = [&](uint16_t* tb, const Bnd& bd) __attribute__((always_inline)) {
    const int64_t len = min(bd.s1, a.ncap) - max(bd.s0, (int64_t)0);
    for (int pass = 1; __builtin_amdgcn_ballot_w64(len > (int64_t)64 * pass) != 0; ++pass) {  // (uniform)
      const int ns = slots(bd, pass);
      load_entries(bd, pass, ns);
      scatter(tb, bd, pass, ns);
    }
  };
  // (the workers' 256 threads)
  auto zero_tile = [&](uint16_t* tb) __attribute__((always_inline)) {
    for (int i = (int)threadIdx.x - 256; i < TILE / 8; i += 256) *reinterpret_cast<u32x4*>(tb + 8 * i) = u32x4{0u, 0u, 0u, 0u};
  };

  const float zero[E] = {};
  constexpr float kHalf = (float)(1 << (BITS - 1));
  // x_hat of a block from tile tb (the lane's own 16 columns of every plane: outlier values in,
  // x_hat out): bf16(bf16(bf16((code - 2^(b-1)) s) + o) + bf16(l @ r)), as legacy_value
  auto compute = [&](const Blk& d, uint16_t* tb) __attribute__((always_inline)) {
    static_for<0, NP>([&](auto pc) {
      constexpr int p = decltype(pc)::value;
      float lr[E];
      residual_unit<G, K>(vop[p], d.lop, zero, lr);
      uint16_t* tp = tb + j * RSTR + p * SEG + w * G + E * g;
      u32x4 ov[2] = {u32x4{0u, 0u, 0u, 0u}, u32x4{0u, 0u, 0u, 0u}};
      ov[0] = *reinterpret_cast<const u32x4*>(tp);
      ov[1] = *reinterpret_cast<const u32x4*>(tp + 8);
      u32x4 xo[2];
      const uint16_t* sp = stab + p * SEG + w * G + E * g;
      const u32x4 scp[2] = {*reinterpret_cast<const u32x4*>(sp), *reinterpret_cast<const u32x4*>(sp + 8)};
#pragma unroll
      for (int e = 0; e < E; e += 2) {
        const uint32_t sw = scp[e >> 3][(e >> 1) & 3], lp = pack_bf16x2(lr[e], lr[e + 1]);
        float av[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint32_t code = (d.cb[(e + h) >> 2] >> (8 * ((e + h) & 3) + BITS * p)) & kMask;
          const float s = h ? bf_hi(sw) : bf_lo(sw);
          av[h] = __builtin_fmaf((float)code, s, -kHalf * s);  // (code - 2^(b-1)) * s, exact in fp32
        }
        if constexpr (BITS > 2) {  // (already a bf16 value at 1 and 2 bits)
          const uint32_t ap = pack_bf16x2(av[0], av[1]);
          av[0] = bf_lo(ap);
          av[1] = bf_hi(ap);
        }
        const uint32_t ow = ov[e >> 3][(e >> 1) & 3];
        const uint32_t ao = pack_bf16x2(av[0] + bf_lo(ow), av[1] + bf_hi(ow));
        av[0] = bf_lo(ao);
        av[1] = bf_hi(ao);
        xo[e >> 3][(e >> 1) & 3] = pack_bf16x2(av[0] + bf_lo(lp), av[1] + bf_hi(lp));
      }
      *reinterpret_cast<u32x4*>(tp) = xo[0];
      *reinterpret_cast<u32x4*>(tp + 8) = xo[1];
    });
  };
  // tile tb -> the rows of block i: 16 rows x NP planes x the units' 64 nuw columns (16 bytes a
  // lane; rows past M and blocks past the run fall outside the store range)
  auto store_tile = [&](const uint16_t* tb, int i) __attribute__((always_inline)) {
    const int rb = rb0 + min(i, nblk - 1);
    const uint32_t rows = i < nblk ? (uint32_t)min(16, M - rb * 16) : 0u;
    const __amdgpu_buffer_rsrc_t rs = uniform_rsrc(a.out + (bm0 + (int64_t)rb * 16) * N, rows * (uint32_t)N * 2u);
    constexpr int CH = SEG / 8;  // 16-byte chunks per (row, plane)
    static_assert((16 * NP * CH) % 256 == 0, "whole store passes");
#pragma unroll
    for (int c0 = 0; c0 < 16 * NP * CH; c0 += 256) {
      const int c = c0 + (int)threadIdx.x;
      const int r = c / (NP * CH), rem = c % (NP * CH), p = rem / CH, k = rem % CH;
      const u32x4 v = *reinterpret_cast<const u32x4*>(tb + r * RSTR + p * SEG + 8 * k);
      const uint32_t off = (uint32_t)((r * N + p * (int)NB + u0 * G + 8 * k) * 2);
      __builtin_amdgcn_raw_buffer_store_b128(v, rs, 8 * k < nuw * G ? off : 0x7ffffff0u, 0, 2);
    }
  };

  Blk ring[PD];
  const int npos = (nblk + PD - 1) / PD * PD;  // positions, whole ring rounds
  if (worker) {
    // block 0's entries into tile 0, block 1's requested; per position: zero the next tile
    // (between the barriers), then write the next block's entries into it and request those
    // of the block after
    const Bnd bnd0 = load_bounds(0);
    Bnd bnd_c = load_bounds(1), bnd_n = load_bounds(2), bnd_nn = load_bounds(3);
    zero_tile(lt);
    zero_tile(lt + TILE);
    int ns = slots(bnd0, 0);
    load_entries(bnd0, 0, ns);
    lds_barrier();  // B0: both tiles zeroed
    scatter(lt, bnd0, 0, ns);
    scatter_rest(lt, bnd0);
    int ns_c = slots(bnd_c, 0);
    load_entries(bnd_c, 0, ns_c);  // block 1's
#pragma unroll 1
    for (int bi = 0; bi < npos; ++bi) {
      uint16_t* tn = lt + ((bi + 1) & 1) * TILE;
      lds_barrier();  // B1: tn's previous rows have left
      zero_tile(tn);
      lds_barrier();  // B2: tn zeroed
      scatter(tn, bnd_c, 0, ns_c);  // block bi + 1
      scatter_rest(tn, bnd_c);
      bnd_c = bnd_n;
      bnd_n = bnd_nn;
      ns_c = slots(bnd_c, 0);
      load_entries(bnd_c, 0, ns_c);  // block bi + 2
      bnd_nn = load_bounds(bi + 4);
    }
  } else {
    static_for<0, PD>([&](auto kc) { load_blk(decltype(kc)::value, ring[decltype(kc)::value]); });
    lds_barrier();  // B0
#pragma unroll 1
    for (int bb = 0; bb < npos; bb += PD)
      static_for<0, PD>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        const int bi = bb + k;
        uint16_t* tc = lt + (bi & 1) * TILE;
        lds_barrier();  // B1: block bi's outliers are in tc
        compute(ring[k], tc);
        lds_barrier();  // B2: x_hat of block bi in tc
        store_tile(tc, bi);
        __builtin_amdgcn_sched_barrier(0);
        load_blk(bi + PD, ring[k]);
        __builtin_amdgcn_sched_barrier(0);
      });
  }
}

// ------------------------------------------------------------------ dequant-GEMM
// out[b, m, c] = bf16( sum_n x_hat[b, m, n] * y[b, n, c] ), the sum in fp32, with x_hat the
// fused decode's value bf16(bf16(bf16((code - 2^(b-1)) * s) + bf16(l @ r))): the reference's
// triton_matmul_decompress (extraction_fuse_matmul.py:224-249, kernel :151-221) on the torch form
// of its decode.  x_hat never leaves the registers.
struct LegacyGemmArgs {
  const uint16_t* l;   // [M, K]
  const uint16_t* rt;  // [N, K]
  const uint8_t* q;    // [B, M, N/NP]
  const uint16_t* s;   // [s_rows, N]
  int64_t s_rows;
  const uint16_t* y;   // [B, N, ldy]: columns c0 .. c0 + NOUT - 1 for this launch (y points at c0)
  int64_t ldy;
  uint16_t* out;       // [B, M, ldo] (out points at column c0)
  int64_t ldo;
  int64_t M, N;
  int n_out;           // scalar path: output columns
};

// MFMA path (every plane a whole number of 64-column units).  Grid: B * ceil(row blocks / RB)
// workgroups of 8 waves; a workgroup owns RB 16-row blocks of one batch.  Work items are
// (unit, plane) pairs, unit-major, so the waves that run together share a unit's code rows in
// L2; wave w takes items w, w + 8, ...  An item's operands (rt and y rows of the plane's 64
// columns in the reconstruction layout, the scales, the RB blocks' code vectors) sit in
// one of two register slots, loaded while the other item is computed (wave-uniform bases and 32-bit lane
// offsets).  Per item the y operands are transposed once (identity MFMA); per row block x_hat is formed on
// the matrix pipe by diagonal 4x4x4 steps as in k_legacy_apply (the -s (128 + h) term once per item), and
// x_hat (bf16, exact) is the B operand of the product MFMA.  The 8 waves' partial tiles are then summed
// through LDS in wave order.
// An item whose scales or l r could overflow inside a diagonal step (the limits of k_legacy_apply) is
// formed element by element.
// Bound by the operands' loads (every CU reads all of y and rt through L2: 512 KB at [4096, 32] each,
// against 64 KB of codes) and their latency, two waves a SIMD: [4, 4096, 4096] 2 bits @ [4, 4096, 32], K = 32:
// 32.9 -> 28.8 us, a call 36.9 -> 31.7: x_hat on the matrix pipe (5.5 vector instructions per element in all,
// matrix steps included) with wave-uniform address bases gave 2.7 of that, y and the scales as 16-byte loads 2.5.
template <int BITS, int K, int NOUT, int RB>
__global__ __launch_bounds__(512) void k_legacy_gemm(LegacyGemmArgs a) {
  constexpr int NP = 8 / BITS, G = 64, E = 16, RT = K / 16, TO = NOUT / 16, NW = 8;
  constexpr uint32_t kMask = (BITS == 8 ? 0x0fu : (1u << BITS) - 1u) * 0x01010101u;
  constexpr int kHalf = 1 << (BITS - 1);
  __shared__ f32x4 part[NW][TO][64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, g = lane >> 4;
  const int M = (int)a.M, N = (int)a.N;
  const int nrb = (M + 15) / 16, gx = (nrb + RB - 1) / RB;
  const int b = __builtin_amdgcn_readfirstlane(blockIdx.x / gx);
  const int rb0 = (blockIdx.x - b * gx) * RB;
  const int nu = N / NP / G, ni = nu * NP;
  const int64_t NB = N / NP;
  const uint16_t* srow = a.s + (a.s_rows == 1 ? 0 : (int64_t)b * N);
  const uint16_t* yb = a.y + (int64_t)b * N * a.ldy;
  const uint8_t* qb = a.q + ((int64_t)b * M + rb0 * 16) * NB;  // the workgroup's first code row
  const u32x2 ident = identity_bop(j, g);
  const u32x2 ida = diag4_aop(lane, 0x3f80u), dmask = diag4_aop(lane, 0xffffu);
  const uint32_t koff = pack_bf16x2_exact(-(float)(BITS == 8 ? 2304 : 128 + kHalf), -(float)(BITS == 8 ? 2304 : 128 + kHalf));

  f32x4 acc[RB][TO];
  u32x2 lop[RB][RT];
  uint32_t qoff[RB];  // the lane's code rows
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const int row = min(min(rb0 + i, nrb - 1) * 16 + j, M - 1);
    qoff[i] = (uint32_t)(row - rb0 * 16) * (uint32_t)NB + (uint32_t)(E * g);
#pragma unroll
    for (int t = 0; t < TO; ++t) acc[i][t] = zero4();
#pragma unroll
    for (int t = 0; t < RT; ++t) lop[i][t] = ld8(a.l + (int64_t)row * K + 16 * t + 4 * g);
  }
  // byte offsets of the lane's rt and y rows (row q of the layout is 4 q rows on)
  const uint32_t voff = (uint32_t)(2 * (vrow_res<G>(0, j, 0) * K + 4 * g));
  const uint32_t ldy2 = 2u * (uint32_t)a.ldy, yoff = (uint32_t)vrow_res<G>(0, j, 0) * ldy2 + (uint32_t)(8 * TO * g);
  const uint32_t soff = (uint32_t)(2 * E * g);
  struct Item {
    u32x4 cb[RB];           // the lane's 16 code bytes of each row block
    u32x2 ya[G / 16][TO];   // y rows of the item's columns (reconstruction layout): columns 4 TO g .. + 4 TO - 1
    u32x2 vop[G / 16][RT];  // rt rows of the item's columns (reconstruction A operand)
    u32x4 sw[2];            // the lane's 16 scales (bf16)
  };
  auto load_item = [&](int it, Item& d) __attribute__((always_inline)) {
    const int u = it / NP, p = it % NP;
    const int base = unit_base(p, u, N, NP, G);
    const uint8_t* qu = qb + u * G;
    const unsigned char* yu = reinterpret_cast<const unsigned char*>(yb + (int64_t)base * a.ldy);
    const unsigned char* vu = reinterpret_cast<const unsigned char*>(a.rt + (int64_t)base * K);
    const unsigned char* su = reinterpret_cast<const unsigned char*>(srow + base);
#pragma unroll
    for (int i = 0; i < RB; ++i) d.cb[i] = ld16_stream(qu + qoff[i]);
#pragma unroll
    for (int q = 0; q < G / 16; ++q)
#pragma unroll
      for (int t = 0; t < TO; ++t) d.ya[q][t] = ld8(yu + (yoff + (uint32_t)(4 * q) * ldy2) + 8 * t);
#pragma unroll
    for (int q = 0; q < G / 16; ++q)
#pragma unroll
      for (int t = 0; t < RT; ++t) d.vop[q][t] = ld8(vu + voff + (8 * q * K + 32 * t));
    d.sw[0] = ld16(su + soff);
    d.sw[1] = ld16(su + soff + 16);
  };
  Item ring[2];
#pragma unroll
  for (int sl = 0; sl < 2; ++sl) load_item(min(w + sl * NW, ni - 1), ring[sl]);
  __builtin_amdgcn_sched_barrier(0);
  uint32_t ltop = 0;  // the largest |l| of the workgroup's rows (bf16 bits)
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int t = 0; t < RT; ++t)
      ltop = pk_max_u16(pk_max_u16(ltop, lop[i][t][0] & 0x7fff7fffu), lop[i][t][1] & 0x7fff7fffu);
  uint32_t lmax = max(ltop >> 16, ltop & 0xffffu);
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) lmax = max(lmax, (uint32_t)__shfl_xor((int)lmax, d));
  const float lbound = (float)K * __uint_as_float(lmax << 16);  // infinite or NaN when an operand is
  auto compute_item = [&](const Item& d, int p) __attribute__((always_inline)) {
    // (the scales are the item's last loads: every load of the item has landed before the branch)
    uint32_t rtop = 0, stop = 0, sc[4];  // sc: the scales of columns 4q + j % 4 / 2 * 2 and the next
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      sc[q] = (j & 2) ? d.sw[q >> 1][2 * (q & 1) + 1] : d.sw[q >> 1][2 * (q & 1)];
      stop = pk_max_u16(stop, sc[q] & 0x7fff7fffu);
#pragma unroll
      for (int t = 0; t < RT; ++t)
        rtop = pk_max_u16(pk_max_u16(rtop, d.vop[q][t][0] & 0x7fff7fffu), d.vop[q][t][1] & 0x7fff7fffu);
    }
    // |s| < 2^100 and K max |l| |r| < 2^120, as bits (a NaN or an infinity is above)
    const float rmax = __uint_as_float(max(rtop & 0xffff0000u, rtop << 16));
    const bool big = max(stop & 0xffff0000u, stop << 16) >= 0x71800000u || __float_as_uint(rmax) >= 0x7f800000u ||
                     __float_as_uint(lbound) >= 0x7f800000u ||
                     (__float_as_uint(lbound * rmax) & 0x7fffffffu) >= 0x7b800000u;
    const bool fast = __builtin_amdgcn_ballot_w64(big) == 0;  // wave-uniform
    u32x4 yt[G / 32][TO];
    transpose_vops<G, NOUT>(d.ya, ident, yt);
    if (fast) {
      u32x2 sa[4], sb[4];
      f32x4 off[4];  // -(128 + h) s
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        sa[q] = u32x2{sc[q] & dmask[0], sc[q] & dmask[1]};
        if constexpr (BITS == 8) {  // 16 s for the codes' high nibbles
          const uint32_t s16 = pack_bf16x2(16.f * bf_lo(sc[q]), 16.f * bf_hi(sc[q]));
          sb[q] = u32x2{s16 & dmask[0], s16 & dmask[1]};
        }
        off[q] = mfma_4x4x4(sa[q], u32x2{koff, koff}, zero4());
      }
      auto rounded = [&](f32x4 v) __attribute__((always_inline)) {
        return u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      };
      auto code_op = [&](uint32_t m) __attribute__((always_inline)) {  // 128 + code as bf16 (bytes code, 0x43)
        return u32x2{__builtin_amdgcn_perm(0x43434343u, m, 0x04010400u), __builtin_amdgcn_perm(0x43434343u, m, 0x04030402u)};
      };
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        f32x4 tl[4], tv[4];
        legacy_lowrank_mfma<K>(d.vop, lop[i], tl);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t c = d.cb[i][q];
          tv[q] = mfma_4x4x4(sa[q], code_op(BITS == 8 ? c & kMask : (c >> (BITS * p)) & kMask), off[q]);
          if constexpr (BITS == 8) tv[q] = mfma_4x4x4(sb[q], code_op((c >> 4) & kMask), tv[q]);
        }
        if constexpr (BITS > 2) {  // (already a bf16 value at 1 and 2 bits)
#pragma unroll
          for (int q = 0; q < 4; ++q) tv[q] = mfma_4x4x4(ida, rounded(tv[q]), zero4());
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) tv[q] = mfma_4x4x4(ida, rounded(tl[q]), tv[q]);
        u32x4 xb[G / 32];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const u32x2 r = rounded(tv[q]);
          xb[q >> 1][2 * (q & 1)] = r[0];
          xb[q >> 1][2 * (q & 1) + 1] = r[1];
        }
        project_unit_vt<G, NOUT>(yt, xb, acc[i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        f32x4 tl[4];
        legacy_lowrank_mfma<K>(d.vop, lop[i], tl);
        u32x4 xb[G / 32];
#pragma unroll
        for (int e = 0; e < E; e += 2) {
          float v[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const uint32_t code = (d.cb[i][(e + h) >> 2] >> (8 * ((e + h) & 3) + BITS * p)) & ((1u << BITS) - 1u);
            const uint32_t sw = d.sw[e >> 3][(e >> 1) & 3];
            const float sv = h ? bf_hi(sw) : bf_lo(sw);
            v[h] = legacy_value<BITS, false>(code, sv, 0.f, bf16r(tl[e >> 2][(e + h) & 3]));
          }
          xb[e / 8][(e / 2) % 4] = pack_bf16x2_exact(v[0], v[1]);
        }
        project_unit_vt<G, NOUT>(yt, xb, acc[i]);
      }
    }
  };
  // Items w, w + NW, ... through the two slots.  The loop body requests and computes unconditionally (an
  // item's loads that land under a branch make the compiler wait for every outstanding load, the other
  // slot's included, at the join); an odd last item runs after the loop.  NW is a multiple of NP, so every item of a wave
  // is in plane w % NP.
  static_assert(NW % NP == 0, "one plane per wave");
  const int nit = w < ni ? (ni - w + NW - 1) / NW : 0, pw = w % NP;
  int i0 = 0;
  for (; i0 + 1 < nit; i0 += 2) {
    compute_item(ring[0], pw);
    __builtin_amdgcn_sched_barrier(0);
    load_item(min(w + (i0 + 2) * NW, ni - 1), ring[0]);
    __builtin_amdgcn_sched_barrier(0);
    compute_item(ring[1], pw);
    __builtin_amdgcn_sched_barrier(0);
    load_item(min(w + (i0 + 3) * NW, ni - 1), ring[1]);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (i0 < nit) compute_item(ring[0], pw);  // wave-uniform

  // acc[i][t] in lane (j, g), component v: out[row j][4 TO g + 4t + v] (partial over this wave's items)
  constexpr int F = TO * 256 / NW, S = 64 / F, PPL = NW / S;
  static_assert(F >= 1 && F <= 64 && 64 % F == 0 && NW % S == 0, "out reduction split");
  const float* partf = reinterpret_cast<const float*>(&part[0][0][0]);
  uint16_t* ob = a.out + (int64_t)b * M * a.ldo;
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    if (rb0 + i >= nrb) break;  // uniform
#pragma unroll
    for (int t = 0; t < TO; ++t) part[w][t][lane] = acc[i][t];
    __syncthreads();
    const int f = lane % F, pg = lane / F;
    const int fi = w * F + f;
    const int t = fi >> 8, src = (fi >> 2) & 63, v = fi & 3;
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < PPL; ++k) s += partf[(((pg * PPL + k) * TO + t) * 64 + src) * 4 + v];
#pragma unroll
    for (int m = F; m < 64; m <<= 1) s += __shfl_xor(s, m);
    const int row = (rb0 + i) * 16 + (src & 15);
    const int col = 4 * TO * (src >> 4) + 4 * t + v;
    if (pg == 0 && row < M) ob[(int64_t)row * a.ldo + col] = (uint16_t)pack_bf16x2(s, 0.f);
    __syncthreads();
  }
}

// Scalar path (any shape): one workgroup per row (b, m); thread t decodes columns t, t + 256, ...
// (l @ r in fp64, exact, as k_legacy_scalar) and multiplies them into up to 32 fp32 sums; the 256
// threads' sums are added through LDS in thread order.  Output columns in chunks of 32.
template <int BITS>
__global__ __launch_bounds__(256) void k_legacy_gemm_scalar(LegacyGemmArgs a, int K) {
  constexpr int NP = 8 / BITS, OC = 32;
  constexpr uint32_t kMask = BITS == 8 ? 0xffu : (1u << BITS) - 1u;
  __shared__ float red[OC][257];
  const int64_t M = a.M, N = a.N, NB = N / NP;
  const int64_t bm = blockIdx.x, b = bm / M, m = bm - b * M;
  const uint16_t* srow = a.s + (a.s_rows == 1 ? 0 : b * N);
  const uint16_t* lrow = a.l + m * K;
  const uint16_t* yb = a.y + b * N * a.ldy;
  const int t = threadIdx.x;
  for (int o0 = 0; o0 < a.n_out; o0 += OC) {
    const int nc = min(OC, a.n_out - o0);
    float acc[OC];
#pragma unroll
    for (int o = 0; o < OC; ++o) acc[o] = 0.f;
    for (int64_t col = t; col < N; col += 256) {
      const int64_t c = col % NB;
      const int p = (int)(col / NB);
      const uint16_t* rrow = a.rt + col * K;
      double dot = 0.0;
      for (int k = 0; k < K; ++k)
        dot = __builtin_fma((double)__uint_as_float((uint32_t)lrow[k] << 16),
                            (double)__uint_as_float((uint32_t)rrow[k] << 16), dot);
      const uint32_t code = ((uint32_t)a.q[bm * NB + c] >> (BITS * p)) & kMask;
      const float sc = __uint_as_float((uint32_t)srow[col] << 16);
      const float xh = legacy_value<BITS, false>(code, sc, 0.f, bf16r((float)dot));
      const uint16_t* yr = yb + col * a.ldy + o0;
#pragma unroll
      for (int o = 0; o < OC; ++o)
        if (o < nc) acc[o] = __builtin_fmaf(xh, __uint_as_float((uint32_t)yr[o] << 16), acc[o]);
    }
#pragma unroll
    for (int o = 0; o < OC; ++o) red[o][t] = acc[o];
    __syncthreads();
    if (t < nc) {
      float s = 0.f;
      for (int i = 0; i < 256; ++i) s += red[t][i];
      a.out[bm * a.ldo + o0 + t] = (uint16_t)pack_bf16x2(s, 0.f);
    }
    __syncthreads();
  }
}

// Scalar form of the hist pass: one thread per column of one row (any shape).
__global__ __launch_bounds__(256) void k_hist_scalar(LegacyArgs a, int K, int64_t chunks) {
  __shared__ uint32_t lh[256];
  lh[threadIdx.x] = 0u;
  const int64_t sel = a.sel[0];
  __syncthreads();
  const int64_t m = blockIdx.x / chunks;
  const int64_t c = (blockIdx.x - m * chunks) * 256 + threadIdx.x;
  if (c < a.N) {
    const uint16_t* lrow = a.l + m * K;
    const uint16_t* rrow = a.rt + c * K;
    double acc = 0.0;
    for (int k = 0; k < K; ++k)
      acc = __builtin_fma((double)__uint_as_float((uint32_t)lrow[k] << 16),
                          (double)__uint_as_float((uint32_t)rrow[k] << 16), acc);
    const float xv = __uint_as_float((uint32_t)a.x[m * a.ldx_m + c] << 16);
    const int bin = hist_bin(bf16r(xv - bf16r((float)acc)), sel);
    if (bin >= 0) atomicAdd(&lh[bin], 1u);
  }
  __syncthreads();
  if (lh[threadIdx.x] != 0u) atomicAdd(&a.hist[threadIdx.x], lh[threadIdx.x]);
}

// hist[0..255] = 0, sel = {-1, k}.
__global__ __launch_bounds__(256) void k_kth_init(uint32_t* __restrict__ hist, int64_t* __restrict__ sel, int64_t k) {
  hist[threadIdx.x] = 0u;
  if (threadIdx.x == 0) {
    sel[0] = -1;
    sel[1] = k;
  }
}

// The bin holding the sel[1]-th smallest key (1-based) of the histogram.  First pass: sel =
// {bin, rank within it}, histogram cleared for the second pass.  Second pass (fine): the key
// (sel[0] << 7 | bin) as an fp32 value in out.  256 threads, one bin each.
__global__ __launch_bounds__(256) void k_kth_select(uint32_t* __restrict__ hist, int64_t* __restrict__ sel, int fine,
                                                    float* __restrict__ out) {
  __shared__ uint64_t wsum[4];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const uint64_t h = (fine && t >= 128) ? 0u : hist[t];
  const uint64_t k = (uint64_t)sel[1];
  uint64_t incl = h;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint64_t o = __shfl_up(incl, d);
    if (lane >= d) incl += o;
  }
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  for (int i = 0; i < w; ++i) incl += wsum[i];
  const int64_t prev = sel[0];
  __syncthreads();  // every thread has read sel before it is rewritten
  if (incl >= k && incl - h < k) {  // exactly one bin: the cumulative count first reaches k
    if (!fine) {
      sel[0] = t;
      sel[1] = (int64_t)(k - (incl - h));
    } else {
      out[0] = __uint_as_float((uint32_t)((prev << 7) | t) << 16);
    }
  }
  hist[t] = 0u;
}

// ------------------------------------------------------------------ host side
// 64-row blocks per workgroup of the MFMA path: 4, or 2 / 1 where 4 would give fewer than two
// workgroups per CU (small M or few units: the reference speed tests' M = 512 gives 8).
static int legacy_rows_per_wg(int64_t M, int64_t wg_cols) {
  const int64_t want = 2 * (int64_t)cu_count();
  for (int rb = 4; rb > 1; rb /= 2)
    if ((M + 64 * rb - 1) / (64 * rb) * wg_cols >= want) return rb;
  return 1;
}

// Row blocks per run of k_legacy_encode and k_legacy_apply (up to 16): the length that gives the busiest CU
// the fewest blocks, a run's set-up (operands, tables, the first loads) counted as 3/4 of one, with at least
// two workgroups per CU where there is the work (three from 24 blocks a CU up: at [4, 8192, 8192], 1 bit,
// runs of 16 leave two, SiLU gradient 223 -> 232 us).  A length taken from the mean alone left CUs with one run
// more than the others: [4, 3072, 3072], us with the mean's length -> with this one (before the streamed
// kernels): staged encode + compaction 8 bits 55.0 -> 47.2 (42.4), 4 bits 46.7 -> 42.3 (44.3), 1 bit of rank
// 32 77.1 -> 58.7 (61.3; 50.2 without its spills), 2 bits 44.1 -> 39.6 (52.5); SiLU gradient 1 bit 44.7 -> 36.4 (39.5).
static int64_t legacy_run_blocks(int64_t B, int64_t ug, int64_t nrb) {
  const int64_t cus = cu_count();
  int64_t best = 1, least = INT64_MAX;
  for (int64_t r = 1; r <= 16; ++r) {
    const int64_t per_cu = (B * ug * ((nrb + r - 1) / r) + cus - 1) / cus;
    if (r > 1 && per_cu < (B * ug * nrb >= 24 * cus ? 3 : 2)) break;
    if (per_cu * (4 * r + 3) < least) {
      least = per_cu * (4 * r + 3);
      best = r;
    }
  }
  return best;
}

// Whether k_legacy_rows decodes n COO entries in E elements faster than k_legacy_apply: where the codes and
// entries come from HBM, its longer contiguous entry ranges pay.  Times in us of both, inputs that are not
// in the caches / inputs of the pass before (rank 16):
//   4 bits  [4, 4096, 4096] 2 %: 56 and 59 / 57 and 36;  5 %: 57 and 71 / 59 and 44;  16 %: 70 and 79 / 69 and 63
//           [4, 8192, 8192] 2 %: 198 and 216 / 202 and 128;  3.5 %: 203 and 230 / 206 and 222
//           [4, 2048, 4096] 8 %: 34 and 36 / 34 and 28;  30 %: 54 and 65 / 47 and 57
//   2 bits  [4, 4096, 4096] 16 %: 89 and 94 / 77 and 68;  [4, 8192, 4096] 8 %: 139 and 132 / 122 and 90;
//           16 %: 169 and 181 / 148 and 168
//   8 bits  [4, 8192, 4096] 8 %: 139 and 134 / 144 and 128;  16 %: 151 and 155 / 143 and 155
static bool legacy_rows_pays(int bits, int64_t E, int64_t n) {
  if (bits == 4) return (E >= ((int64_t)1 << 26) && n * 32 > E) || (E >= ((int64_t)1 << 25) && n * 6 > E);
  return (bits == 2 || bits == 8) && E >= ((int64_t)1 << 27) && n * 8 > E;
}

// The row-tile decode (k_legacy_rows), in runs of whole ring rounds (PD blocks).  Returns false where it does
// not apply.
template <int MODE, int BITS, int OSRC>
static bool legacy_rows_launch(const LegacyArgs& a, int K, int64_t B, hipStream_t st, int* status) {
  if constexpr (MODE != kDecode || OSRC != 3 || BITS == 1) {
    return false;
  } else {
    using Lr = LegacyRows<BITS>;
    const int64_t NB = a.N / Lr::NP, nu = NB / 64, nrb = (a.M + 15) / 16;
    if (!legacy_rows_pays(BITS, B * a.M * a.N, a.ncap)) return false;
    if (NB % 64 != 0 || nu < Lr::NW || 16 * a.N * 2 >= ((int64_t)1 << 31)) return false;
    const int64_t ug = (nu + Lr::NW - 1) / Lr::NW, tiles = B * ug;
    const int64_t want = 2 * (int64_t)cu_count();
    if (tiles * nrb < want * 2 * Lr::PD) return false;  // under two ring rounds per workgroup
    int64_t runs = std::max<int64_t>(1, want / tiles);
    int64_t rbw = (nrb + runs - 1) / runs;
    rbw = (rbw + Lr::PD - 1) / Lr::PD * Lr::PD;
    runs = (nrb + rbw - 1) / rbw;
    const int64_t nwg = tiles * runs;
    if (nwg > INT32_MAX) return false;
    auto go = [&](auto kern) __attribute__((always_inline)) {
      (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Lr::LDS);
      *status = launch(kern, dim3((unsigned)nwg), dim3(512), Lr::LDS, st, a, (int)rbw, (int)ug);
    };
    if (K == 16) go(k_legacy_rows<BITS, 16>);
    else go(k_legacy_rows<BITS, 32>);
    return true;
  }
}

template <int MODE, int BITS, int OSRC>
static int legacy_launch(const LegacyArgs& a, int K, int64_t B, bool mfma_ok, hipStream_t st) {
  constexpr int NP = (MODE == kAdd) ? 1 : 8 / BITS;
  if (mfma_ok) {
    int status = LRQ_OK;
    if (legacy_rows_launch<MODE, BITS, OSRC>(a, K, B, st, &status)) return status;
  }
  const int64_t NB = a.N / NP;
  const int rb = legacy_rows_per_wg(a.M, NB / 64 * B);
  const int64_t nwg = (a.M + 64 * rb - 1) / (64 * rb) * (NB / 64) * B;
  // k_legacy_apply's store range covers 16 rows of fewer than 2^26 columns (32-bit offsets, past which a
  // dropped lane's offset lies), its entry range kWindow entries of those.  Other shapes take the scalar
  // kernel (at [64, 2^21] 2 bits 140 us against 3.8 ms)
  constexpr bool kApply = (MODE == kDecode && OSRC != 1) || MODE == kFusedStore || MODE == kFusedSilu ||
                          MODE == kFusedMul;
  constexpr int64_t kWindow = LegacyApply<kDecode, BITS, 1>::kWindow;
  const bool fits = !kApply || (32 * a.N <= 0x7ffffff0 && (OSRC == 0 || 16 * a.N <= kWindow || a.ncap <= kWindow));
  if (mfma_ok && fits && NB % 64 == 0 && nwg <= INT32_MAX) {
    // 4 row blocks per workgroup, fewer where that would leave under two workgroups per CU
    LegacyArgs la = a;
    la.rb = rb;
    const dim3 grid((unsigned)nwg);
    if constexpr (MODE == kEncode) {
      const int64_t ug = (NB / 64 + 3) / 4, nrb = (a.M + 15) / 16;
      const int64_t rbw = legacy_run_blocks(B, ug, nrb);
      const int64_t wgs = (nrb + rbw - 1) / rbw * ug * B;
      if (wgs > INT32_MAX) return LRQ_ERR_SHAPE;
      const dim3 eg((unsigned)wgs);
      if (K == 16) return launch((k_legacy_encode<BITS, 16, OSRC == 1>), eg, dim3(256), 0, st, a, (int)rbw, (int)ug);
      return launch((k_legacy_encode<BITS, 32, OSRC == 1>), eg, dim3(256), 0, st, a, (int)rbw, (int)ug);
    } else if constexpr (kApply) {
      const int64_t ug = (NB / 64 + 3) / 4, nrb = (a.M + 15) / 16;
      const int64_t rbw = legacy_run_blocks(B, ug, nrb);
      const int64_t wgs = (nrb + rbw - 1) / rbw * ug * B;
      if (wgs > INT32_MAX) return LRQ_ERR_SHAPE;
      const dim3 eg((unsigned)wgs);
      constexpr int kMode = MODE == kFusedStore ? (int)kDecode : MODE;
      constexpr int kCoo = OSRC >= 2 ? OSRC - 1 : 0;
      if (kCoo != 0 && a.ncap > 0) {
        if (K == 16) return launch((k_legacy_apply<kMode, BITS, 16, kCoo>), eg, dim3(256), 0, st, a, (int)rbw, (int)ug);
        return launch((k_legacy_apply<kMode, BITS, 32, kCoo>), eg, dim3(256), 0, st, a, (int)rbw, (int)ug);
      }
      if (K == 16) return launch((k_legacy_apply<kMode, BITS, 16, 0>), eg, dim3(256), 0, st, a, (int)rbw, (int)ug);
      return launch((k_legacy_apply<kMode, BITS, 32, 0>), eg, dim3(256), 0, st, a, (int)rbw, (int)ug);
    } else {
      if (K == 16) return launch((k_legacy_mfma<MODE, BITS, 16>), grid, dim3(256), 0, st, la);
      return launch((k_legacy_mfma<MODE, BITS, 32>), grid, dim3(256), 0, st, la);
    }
  } else {
    const int64_t chunks = (NB + 255) / 256;
    if (B * a.M * chunks > INT32_MAX) return LRQ_ERR_SHAPE;
    LRQ_TRY(launch((k_legacy_scalar<MODE, BITS, OSRC>), dim3((unsigned)(B * a.M * chunks)), dim3(256), 0, st, a,
                       K, chunks));
  }
  return LRQ_OK;
}

template <int MODE, int OSRC>
static int legacy_bits(const LegacyArgs& a, int K, int64_t B, int bits, bool mfma_ok, hipStream_t st) {
  switch (bits) {
    case 1: return legacy_launch<MODE, 1, OSRC>(a, K, B, mfma_ok, st);
    case 2: return legacy_launch<MODE, 2, OSRC>(a, K, B, mfma_ok, st);
    case 4: return legacy_launch<MODE, 4, OSRC>(a, K, B, mfma_ok, st);
    case 8: return legacy_launch<MODE, 8, OSRC>(a, K, B, mfma_ok, st);
    default: return LRQ_ERR_UNSUPPORTED;
  }
}

// The outlier threshold as the kernels compare with it: rounded to bf16, and -0 (also what a tiny negative
// threshold rounds to) as +0, which compares alike but whose bits the encode's packed-integer test can take.
static float legacy_tau(float outlier) {
  const uint16_t h = bf16_bits_host(outlier);
  return bf16_value_host(h == 0x8000u ? (uint16_t)0 : h);
}

// Shape / argument checks common to every legacy entry point.
static int legacy_check(const void* l, const void* rt, int32_t K, int64_t B, int64_t M, int64_t N, int32_t bits,
                        const void* s, int64_t s_rows, bool need_s) {
  if (l == nullptr || rt == nullptr) return LRQ_ERR_NULL;
  if (need_s && s == nullptr) return LRQ_ERR_NULL;
  if (K != 16 && K != 32) return LRQ_ERR_UNSUPPORTED;
  if (bits != 1 && bits != 2 && bits != 4 && bits != 8) return LRQ_ERR_UNSUPPORTED;
  if (B < 0 || M < 0 || N <= 0 || M > INT32_MAX || N > INT32_MAX) return LRQ_ERR_SHAPE;
  if (N % (8 / bits) != 0) return LRQ_ERR_SHAPE;
  if (need_s && s_rows != 1 && s_rows != B) return LRQ_ERR_SHAPE;
  if (!aligned(l, 2) || !aligned(rt, 2) || (need_s && !aligned(s, 2))) return LRQ_ERR_ALIGN;
  return LRQ_OK;
}

// The MFMA path reads and writes 16-byte vectors and 8-byte L / V operands.
static bool vec_ok(std::initializer_list<const void*> ptrs) {
  for (const void* p : ptrs)
    if (p != nullptr && !aligned(p, 16)) return false;
  return true;
}

}  // namespace lrq

using namespace lrq;

extern "C" int lrq_legacy_encode(const void* l, const void* rt, int32_t K, const void* x, int64_t B, int64_t M,
                                 int64_t N, int64_t ldx_b, int64_t ldx_m, const void* s, int64_t s_rows,
                                 int32_t bits, float outlier, void* o, void* q, void* stream) {
  int st = legacy_check(l, rt, K, B, M, N, bits, s, s_rows, true);
  if (st) return st;
  if (x == nullptr || o == nullptr || q == nullptr) return LRQ_ERR_NULL;
  if (ldx_m < N || (M > 1 && B > 1 && ldx_b < ldx_m * (M - 1) + N)) return LRQ_ERR_SHAPE;
  if (!aligned(x, 2) || !aligned(o, 2)) return LRQ_ERR_ALIGN;
  if (B == 0 || M == 0) return LRQ_OK;
  LegacyArgs a{};
  a.l = (const uint16_t*)l, a.rt = (const uint16_t*)rt, a.x = (const uint16_t*)x, a.ldx_b = ldx_b, a.ldx_m = ldx_m;
  a.s = (const uint16_t*)s, a.s_rows = s_rows, a.oout = (uint16_t*)o, a.qout = (uint8_t*)q, a.M = M, a.N = N;
  a.tau = legacy_tau(outlier);
  const bool mfma_ok = vec_ok({l, rt, x, s, o, q}) && ldx_b % 8 == 0 && ldx_m % 8 == 0 && N % 8 == 0;
  return legacy_bits<kEncode, 0>(a, K, B, bits, mfma_ok, (hipStream_t)stream);
}

// lrq_legacy_encode whose outlier compaction starts from the staged piece records the encode
// writes (the MFMA path: each 64-column piece's count and first entries, its dense values only
// when it has more entries than a record holds), so the dense outliers are neither written nor
// read whole; other shapes take the encode and the full compaction.
extern "C" int lrq_legacy_encode_coo(const void* l, const void* rt, int32_t K, const void* x, int64_t B, int64_t M,
                                     int64_t N, int64_t ldx_b, int64_t ldx_m, const void* s, int64_t s_rows,
                                     int32_t bits, float outlier, void* o, void* q, int64_t* indices, int64_t ld_idx,
                                     void* values, int64_t cap, int64_t* nnz, int64_t* piece_ptr, void* workspace,
                                     int64_t workspace_bytes, void* stream) {
  int st = legacy_check(l, rt, K, B, M, N, bits, s, s_rows, true);
  if (st) return st;
  if (x == nullptr || o == nullptr || q == nullptr) return LRQ_ERR_NULL;
  if (ldx_m < N || (M > 1 && B > 1 && ldx_b < ldx_m * (M - 1) + N)) return LRQ_ERR_SHAPE;
  if (!aligned(x, 2) || !aligned(o, 2)) return LRQ_ERR_ALIGN;
  st = coo_compact_check(o, B, M, N, indices, ld_idx, values, cap, nnz, piece_ptr, workspace, workspace_bytes);
  if (st) return st;
  const int NP = 8 / bits;
  const bool mfma_ok = vec_ok({l, rt, x, s, o, q}) && ldx_b % 8 == 0 && ldx_m % 8 == 0 && N % 8 == 0;
  const int64_t NB = N / NP;
  const float tau = legacy_tau(outlier);
  // (with tau >= 0 an element's |xr| > tau is exactly "an entry"; a negative threshold keeps every
  // element but the +-0 ones, counted by the compaction's own pass)
  const bool counted = mfma_ok && NB % 64 == 0 && NB / 64 <= 65535 && B <= 65535 && aligned(o, 16) && tau >= 0.f;
  if (!counted || B == 0 || M == 0) {
    LRQ_TRY(lrq_legacy_encode(l, rt, K, x, B, M, N, ldx_b, ldx_m, s, s_rows, bits, outlier, o, q, stream));
    return lrq_coo_compact(o, B, M, N, indices, ld_idx, values, cap, nnz, piece_ptr, workspace, workspace_bytes,
                           stream);
  }
  LegacyArgs a{};
  a.l = (const uint16_t*)l, a.rt = (const uint16_t*)rt, a.x = (const uint16_t*)x, a.ldx_b = ldx_b, a.ldx_m = ldx_m;
  a.s = (const uint16_t*)s, a.s_rows = s_rows, a.oout = (uint16_t*)o, a.qout = (uint8_t*)q, a.M = M, a.N = N;
  a.tau = tau;
  a.npc = (N + 63) / 64, a.pcnt = piece_ptr;
  LRQ_TRY((legacy_bits<kEncode, 1>(a, K, B, bits, true, (hipStream_t)stream)));
  return coo_compact_staged(o, B, M, N, indices, ld_idx, values, cap, nnz, piece_ptr, workspace, (hipStream_t)stream);
}

extern "C" int lrq_legacy_decode(const void* l, const void* rt, int32_t K, const void* q, const void* o,
                                 const void* s, int64_t s_rows, int64_t B, int64_t M, int64_t N, int32_t bits,
                                 void* out, void* stream) {
  int st = legacy_check(l, rt, K, B, M, N, bits, s, s_rows, true);
  if (st) return st;
  if (q == nullptr || out == nullptr) return LRQ_ERR_NULL;
  if (!aligned(out, 2) || (o != nullptr && !aligned(o, 2))) return LRQ_ERR_ALIGN;
  if (B == 0 || M == 0) return LRQ_OK;
  LegacyArgs a{};
  a.l = (const uint16_t*)l, a.rt = (const uint16_t*)rt, a.s = (const uint16_t*)s, a.s_rows = s_rows;
  a.qin = (const uint8_t*)q, a.oin = (const uint16_t*)o, a.out = (uint16_t*)out, a.M = M, a.N = N;
  const bool mfma_ok = vec_ok({l, rt, q, o, s, out}) && N % 8 == 0;
  if (o != nullptr) return legacy_bits<kDecode, 1>(a, K, B, bits, mfma_ok, (hipStream_t)stream);
  return legacy_bits<kDecode, 0>(a, K, B, bits, mfma_ok, (hipStream_t)stream);
}

extern "C" int lrq_legacy_fused(const void* l, const void* rt, int32_t K, const void* q, const void* s,
                                int64_t s_rows, int64_t B, int64_t M, int64_t N, int32_t bits, int32_t op,
                                const void* y, void* out, void* stream) {
  int st = legacy_check(l, rt, K, B, M, N, bits, s, s_rows, true);
  if (st) return st;
  if (op < 0 || op > 2) return LRQ_ERR_UNSUPPORTED;
  if (q == nullptr || out == nullptr || (op != 0 && y == nullptr)) return LRQ_ERR_NULL;
  if (!aligned(out, 2) || (y != nullptr && !aligned(y, 2))) return LRQ_ERR_ALIGN;
  if (B == 0 || M == 0) return LRQ_OK;
  LegacyArgs a{};
  a.l = (const uint16_t*)l, a.rt = (const uint16_t*)rt, a.s = (const uint16_t*)s, a.s_rows = s_rows;
  a.qin = (const uint8_t*)q, a.y = (const uint16_t*)y, a.out = (uint16_t*)out, a.M = M, a.N = N;
  const bool mfma_ok = vec_ok({l, rt, q, s, y, out}) && N % 8 == 0;
  hipStream_t hs = (hipStream_t)stream;
  switch (op) {
    case 0: return legacy_bits<kFusedStore, 0>(a, K, B, bits, mfma_ok, hs);
    case 1: return legacy_bits<kFusedSilu, 0>(a, K, B, bits, mfma_ok, hs);
    default: return legacy_bits<kFusedMul, 0>(a, K, B, bits, mfma_ok, hs);
  }
}

namespace lrq {
template <int BITS, int K, int NOUT>
static int legacy_gemm_chunk(const LegacyGemmArgs& a, int64_t B, hipStream_t st) {
  // 16-row blocks per workgroup: 4, or 2 / 1 where 4 would leave CUs without a workgroup
  const int64_t nrb = (a.M + 15) / 16, cu = cu_count();
  auto launch_rb = [&](auto rb) __attribute__((always_inline)) {
    constexpr int RB = decltype(rb)::value;
    const int64_t nwg = B * ((nrb + RB - 1) / RB);
    if (nwg > INT32_MAX) return (int)LRQ_ERR_SHAPE;
    return launch((k_legacy_gemm<BITS, K, NOUT, RB>), dim3((unsigned)nwg), dim3(512), 0, st, a);
  };
  if (B * ((nrb + 3) / 4) >= cu) return launch_rb(std::integral_constant<int, 4>{});
  if (B * ((nrb + 1) / 2) >= cu) return launch_rb(std::integral_constant<int, 2>{});
  return launch_rb(std::integral_constant<int, 1>{});
}

template <int BITS>
static int legacy_gemm_bits(LegacyGemmArgs a, int K, int64_t B, bool mfma_ok, hipStream_t st) {
  if (!mfma_ok) {
    if (B * a.M > INT32_MAX) return LRQ_ERR_SHAPE;
    return launch(k_legacy_gemm_scalar<BITS>, dim3((unsigned)(B * a.M)), dim3(256), 0, st, a, K);
  }
  // output columns in chunks of 32 (then 16); each chunk is one pass over the codes
  const uint16_t* y0 = a.y;
  uint16_t* o0 = a.out;
  for (int c0 = 0; c0 < a.n_out;) {
    const int nc = a.n_out - c0 >= 32 ? 32 : 16;
    a.y = y0 + c0;
    a.out = o0 + c0;
    int r;
    if (K == 16) r = nc == 32 ? legacy_gemm_chunk<BITS, 16, 32>(a, B, st) : legacy_gemm_chunk<BITS, 16, 16>(a, B, st);
    else r = nc == 32 ? legacy_gemm_chunk<BITS, 32, 32>(a, B, st) : legacy_gemm_chunk<BITS, 32, 16>(a, B, st);
    LRQ_TRY(r);
    c0 += nc;
  }
  return LRQ_OK;
}
}  // namespace lrq

extern "C" int lrq_legacy_dequant_gemm(const void* l, const void* rt, int32_t K, const void* q, const void* s,
                                       int64_t s_rows, int64_t B, int64_t M, int64_t N, int32_t bits, const void* y,
                                       int64_t ldy, int32_t n_out, void* out, int64_t ldo, void* stream) {
  int st = legacy_check(l, rt, K, B, M, N, bits, s, s_rows, true);
  if (st) return st;
  if (q == nullptr || y == nullptr || out == nullptr) return LRQ_ERR_NULL;
  if (n_out < 1 || ldy < n_out || ldo < n_out) return LRQ_ERR_SHAPE;
  if (!aligned(y, 2) || !aligned(out, 2)) return LRQ_ERR_ALIGN;
  if (B == 0 || M == 0) return LRQ_OK;
  LegacyGemmArgs a{};
  a.l = (const uint16_t*)l, a.rt = (const uint16_t*)rt, a.q = (const uint8_t*)q, a.s = (const uint16_t*)s;
  a.s_rows = s_rows, a.y = (const uint16_t*)y, a.ldy = ldy, a.out = (uint16_t*)out, a.ldo = ldo, a.M = M, a.N = N;
  a.n_out = n_out;
  const int64_t NB = N / (8 / bits);
  const bool mfma_ok = vec_ok({l, rt, q, s}) && NB % 64 == 0 && n_out % 16 == 0 && aligned(y, 8) && ldy % 4 == 0 &&
                       NB <= (int64_t)1 << 26 && ldy <= (int64_t)1 << 25;  // (32-bit lane offsets: 63 rows)
  hipStream_t hs = (hipStream_t)stream;
  switch (bits) {
    case 1: return legacy_gemm_bits<1>(a, K, B, mfma_ok, hs);
    case 2: return legacy_gemm_bits<2>(a, K, B, mfma_ok, hs);
    case 4: return legacy_gemm_bits<4>(a, K, B, mfma_ok, hs);
    default: return legacy_gemm_bits<8>(a, K, B, mfma_ok, hs);
  }
}

extern "C" int lrq_lowrank_add(const void* l, const void* rt, int32_t K, const void* x, int64_t B, int64_t M,
                               int64_t N, void* out, void* stream) {
  int st = legacy_check(l, rt, K, B, M, N, 8, nullptr, 1, false);
  if (st) return st;
  if (x == nullptr || out == nullptr) return LRQ_ERR_NULL;
  if (!aligned(x, 2) || !aligned(out, 2)) return LRQ_ERR_ALIGN;
  if (B == 0 || M == 0) return LRQ_OK;
  LegacyArgs a{};
  a.l = (const uint16_t*)l, a.rt = (const uint16_t*)rt, a.x = (const uint16_t*)x, a.ldx_b = M * N, a.ldx_m = N;
  a.out = (uint16_t*)out, a.M = M, a.N = N;
  const bool mfma_ok = vec_ok({l, rt, x, out}) && N % 8 == 0;
  return legacy_launch<kAdd, 8, 0>(a, K, B, mfma_ok, (hipStream_t)stream);
}

extern "C" int lrq_legacy_decode_coo(const void* l, const void* rt, int32_t K, const void* q, const int64_t* piece_ptr,
                                     const int64_t* cols, const void* vals, int64_t n_entries, const void* s,
                                     int64_t s_rows, int64_t B, int64_t M, int64_t N, int32_t bits, void* out,
                                     void* stream) {
  int st = legacy_check(l, rt, K, B, M, N, bits, s, s_rows, true);
  if (st) return st;
  if (q == nullptr || out == nullptr || piece_ptr == nullptr) return LRQ_ERR_NULL;
  if (n_entries < 0) return LRQ_ERR_SHAPE;
  if (n_entries > 0 && (cols == nullptr || vals == nullptr)) return LRQ_ERR_NULL;
  if (!aligned(out, 2) || !aligned(piece_ptr, 8) || !aligned(cols, 8) || !aligned(vals, 2)) return LRQ_ERR_ALIGN;
  if (B == 0 || M == 0) return LRQ_OK;
  LegacyArgs a{};
  a.l = (const uint16_t*)l, a.rt = (const uint16_t*)rt, a.s = (const uint16_t*)s, a.s_rows = s_rows;
  a.qin = (const uint8_t*)q, a.out = (uint16_t*)out, a.M = M, a.N = N;
  a.optr = piece_ptr, a.ocol = cols, a.oval = (const uint16_t*)vals, a.npc = (N + 63) / 64, a.ncap = n_entries;
  const bool mfma_ok = vec_ok({l, rt, q, s, out}) && N % 8 == 0;
  // more than about 4 entries per 64-column piece (1/16 of the elements): more of a piece's entries are
  // requested ahead (k_legacy_apply), or the row-tile decode (legacy_rows_pays)
  if (mfma_ok && (n_entries * 16 > B * M * N || legacy_rows_pays(bits, B * M * N, n_entries))) return legacy_bits<kDecode, 3>(a, K, B, bits, mfma_ok, (hipStream_t)stream);
  return legacy_bits<kDecode, 2>(a, K, B, bits, mfma_ok, (hipStream_t)stream);
}

extern "C" int lrq_legacy_kth_residual(const void* l, const void* rt, int32_t K, const void* x, int64_t M, int64_t N,
                                       int64_t ldx_m, int64_t k, float* out, void* workspace, int64_t workspace_bytes,
                                       void* stream) {
  int st = legacy_check(l, rt, K, 1, M, N, 8, nullptr, 1, false);
  if (st) return st;
  if (x == nullptr || out == nullptr || workspace == nullptr) return LRQ_ERR_NULL;
  if (ldx_m < N) return LRQ_ERR_SHAPE;
  if (M * N >= ((int64_t)1 << 32) || k < 1 || k > M * N) return LRQ_ERR_SHAPE;
  if (workspace_bytes < 2048) return LRQ_ERR_WORKSPACE;
  if (!aligned(x, 2) || !aligned(out, 4) || !aligned(workspace, 16)) return LRQ_ERR_ALIGN;
  hipStream_t hs = (hipStream_t)stream;
  uint32_t* hist = reinterpret_cast<uint32_t*>(workspace);
  int64_t* sel = reinterpret_cast<int64_t*>(hist + 256);
  LegacyArgs a{};
  a.l = (const uint16_t*)l, a.rt = (const uint16_t*)rt, a.x = (const uint16_t*)x, a.ldx_b = 0, a.ldx_m = ldx_m;
  a.M = M, a.N = N, a.hist = hist, a.sel = sel;
  const bool mfma_ok = vec_ok({l, rt, x}) && ldx_m % 8 == 0 && N % 64 == 0;
  LRQ_TRY(launch(k_kth_init, dim3(1), dim3(256), 0, hs, hist, sel, k));
  for (int fine = 0; fine < 2; ++fine) {
    if (mfma_ok) {
      a.rb = legacy_rows_per_wg(M, N / 64);
      const dim3 grid((unsigned)((M + 64 * a.rb - 1) / (64 * a.rb) * (N / 64)));  // < 2^26 (M * N < 2^32)
      if (K == 16) LRQ_TRY(launch((k_legacy_mfma<kHist, 8, 16>), grid, dim3(256), 0, hs, a));
      else LRQ_TRY(launch((k_legacy_mfma<kHist, 8, 32>), grid, dim3(256), 0, hs, a));
    } else {
      const int64_t chunks = (N + 255) / 256;
      if (M * chunks > INT32_MAX) return LRQ_ERR_SHAPE;
      LRQ_TRY(launch(k_hist_scalar, dim3((unsigned)(M * chunks)), dim3(256), 0, hs, a, (int)K, chunks));
    }
    LRQ_TRY(launch(k_kth_select, dim3(1), dim3(256), 0, hs, hist, sel, fine, out));
  }
  return LRQ_OK;
}
