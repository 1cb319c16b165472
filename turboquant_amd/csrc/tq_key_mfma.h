// What the matrix-core key quantisers share: MFMA wrappers, the exact split of fp32 values into bf16 terms, and the
// reductions over the lanes that hold one vector.
#pragma once

#include "tq_quantize.h"

namespace tq {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x4 mfma_bf16(const u32x4& rows, const u32x4& cols, f32x4 c) {
  bf16x8 av, bv;
  __builtin_memcpy(&av, &rows, 16);
  __builtin_memcpy(&bv, &cols, 16);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, c, 0, 0, 0);
}

// fp6 (A: 16 rows x 128) x fp4 (B: 128 x 16) MFMA with per-lane power-of-two block scales (E8M0 codes); SEL
// picks the byte of scale_a that holds the code.  Only six dwords of `a` and the four of `b` are read.
template <int SEL>
__device__ __forceinline__ f32x4 mfma_fp6_fp4(const i32x8& a, const u32x4& b, f32x4 c, int scale_a, int scale_b) {
  const i32x8 bv = {(int)b[0], (int)b[1], (int)b[2], (int)b[3], 0, 0, 0, 0};
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, bv, c, 2 /*A: fp6 e2m3*/, 4 /*B: fp4*/, SEL, scale_a, 0, scale_b);
}

// two fp32 -> packed bf16 (first value in the low half), round to nearest even
__device__ __forceinline__ uint32_t cvt_pk_bf16(float a, float b) {
  f32x2 v = {a, b};
  bf16x2 r = __builtin_convertvector(v, bf16x2);
  uint32_t u;
  __builtin_memcpy(&u, &r, 4);
  return u;
}

// (v0, v1) = t[0] + t[1] + t[2] lane-wise, each term a packed pair of bf16: a term is
// the rounding of what the previous terms left, and every remainder is exact in fp32
__device__ __forceinline__ void split3_pk(float v0, float v1, uint32_t (&t)[3]) {
  t[0] = cvt_pk_bf16(v0, v1);
  float r0 = v0 - __uint_as_float(t[0] << 16), r1 = v1 - __uint_as_float(t[0] & 0xffff0000u);
  t[1] = cvt_pk_bf16(r0, r1);
  r0 -= __uint_as_float(t[1] << 16);
  r1 -= __uint_as_float(t[1] & 0xffff0000u);
  t[2] = cvt_pk_bf16(r0, r1);
}

// N consecutive elements of the input dtype from LDS (16-byte aligned) as fp32
template <int DT, int N>
__device__ __forceinline__ void load_run(const typename Elem<DT>::storage* p, float (&out)[N]) {
  if constexpr (DT == TQ_F32) {
#pragma unroll
    for (int c = 0; c < N; c += 4) {
      const f32x4 v = *(const f32x4*)(p + c);
      out[c] = v.x; out[c + 1] = v.y; out[c + 2] = v.z; out[c + 3] = v.w;
    }
  } else if constexpr (N % 8 == 0) {
#pragma unroll
    for (int c = 0; c < N; c += 8) {
      const u32x4 v = *(const u32x4*)(p + c);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        out[c + 2 * k] = Elem<DT>::load(&v, 2 * k);
        out[c + 2 * k + 1] = Elem<DT>::load(&v, 2 * k + 1);
      }
    }
  } else {
    static_assert(N == 4, "runs of 4 or a multiple of 8");
    const u32x2 v = *(const u32x2*)p;
#pragma unroll
    for (int k = 0; k < 4; ++k) out[k] = Elem<DT>::load(&v, k);
  }
}

template <int DT> struct InTerms;                       // bf16 terms that represent a value of the input dtype exactly
template <> struct InTerms<TQ_BF16> { static constexpr int N = 1; };
template <> struct InTerms<TQ_F16> { static constexpr int N = 2; };
template <> struct InTerms<TQ_F32> { static constexpr int N = 3; };

// OR / sum of a value over the four lanes that hold the same vector (lane & 15 equal); the result is valid in
// the first of them (lanes 0..15).  The lane-swap instructions move rows of 16 / halves of 32 lanes through
// the vector ALU: no LDS round trip and nothing to wait for.
__device__ __forceinline__ uint32_t or_over_kb(uint32_t v) {
  v |= (uint32_t)__builtin_amdgcn_permlane32_swap(v, v, false, false)[1];       // lanes 0..31: | lane + 32
  v |= (uint32_t)__builtin_amdgcn_permlane16_swap(v, v, false, false)[1];       // lanes 0..15: | lane + 16
  return v;
}
// sum over groups of N neighbouring lanes (N = 4, 8 or 16, inside a row of 16) with DPP moves: quad swaps,
// then half-row / row mirrors (every lane of a quad already holds the quad's sum, so a mirror pairs the quads)
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
template <int N>
__device__ __forceinline__ float sum_lanes(float v) {
  static_assert(N == 4 || N == 8 || N == 16, "4, 8 or 16 lanes");
  v += dpp_mov<0xB1>(v);
  v += dpp_mov<0x4E>(v);
  if (N >= 8) v += dpp_mov<0x141>(v);
  if (N >= 16) v += dpp_mov<0x140>(v);
  return v;
}
__device__ __forceinline__ float sum_over_kb(float f) {
  f += __uint_as_float(__builtin_amdgcn_permlane32_swap(__float_as_uint(f), __float_as_uint(f), false, false)[1]);
  f += __uint_as_float(__builtin_amdgcn_permlane16_swap(__float_as_uint(f), __float_as_uint(f), false, false)[1]);
  return f;
}

}  // namespace tq
