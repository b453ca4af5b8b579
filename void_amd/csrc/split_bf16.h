// split_bf16.h — fp32 products on the bf16 matrix cores, for the SDDMM
// kernels.
//
// An fp32 value is the exact sum of three bf16 values (8 + 8 + 8 significant
// bits): hi, truncated; mid, the rest rounded to nearest; lo, what then
// remains.  A product a b is taken as the six partial products of order 2^-16
// and above (hi hi, hi mid, mid hi, mid mid, hi lo, lo hi); the three left out
// are below 2^-23 |a b| together, of either sign.  Every partial product is
// exact in fp32, and hi hi has an accumulator of its own, so that the running
// sum is rounded once per 16 terms (v_mfma_f32_32x32x2_f32: once per 2): the
// result is closer to the exact one than the fp32 MFMA's (relative error over
// N = 1024 terms 1.9e-7 against 5.7e-7, over 2048 2.7e-7 against 8.1e-7).
// Twelve 32-cycle MFMAs replace sixteen of 64 cycles per 32 terms (SDDMM, 3277
// tiles, N = 1024: 76.6 -> 69.9 us; 14336 tiles, N = 2048: 550 -> 494; the float
// SpMM, whose waves wait for issue and not for the MFMA, gained nothing); the splits
// cost 5.5 VALU instructions a value (v_dot2_f32_bf16 in
// place of the mask and subtraction, 3.5, takes as long).
// Infinities, NaN and sums that overflow: the callers look for a non-finite
// accumulator at the end and compute that block again on the fp32 MFMA, so
// such results are those of fp32 arithmetic.  Values below 2^-110 lose bits
// that bf16 cannot hold (absolute error below 2^-133 per value).

#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace {

typedef int s3_v4i __attribute__((ext_vector_type(4)));
typedef float s3_v16f __attribute__((ext_vector_type(16)));
typedef __bf16 s3_v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 s3_v2bf __attribute__((ext_vector_type(2)));

// 8 H values of one lane in three bf16 parts; part [h] holds values 8 h .. 8 h + 7.
template <int H>
struct Split3 {
  s3_v4i hi[H], mid[H], lo[H];
};

__device__ __forceinline__ uint32_t upper_halves(float x0, float x1) {
  return __builtin_amdgcn_perm(__float_as_uint(x1), __float_as_uint(x0), 0x07060302u);
}

template <int H>
__device__ __forceinline__ Split3<H> split3(const float (&x)[8 * H]) {
  Split3<H> s;
#pragma unroll
  for (int h = 0; h < H; ++h)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float x0 = x[8 * h + 2 * q], x1 = x[8 * h + 2 * q + 1];
      const float r0 = x0 - __uint_as_float(__float_as_uint(x0) & 0xffff0000u);
      const float r1 = x1 - __uint_as_float(__float_as_uint(x1) & 0xffff0000u);
      const s3_v2bf m = {(__bf16)r0, (__bf16)r1};
      const uint32_t mb = __builtin_bit_cast(uint32_t, m);
      s.hi[h][q] = (int)upper_halves(x0, x1);
      s.mid[h][q] = (int)mb;
      s.lo[h][q] = (int)upper_halves(r0 - __uint_as_float(mb << 16), r1 - __uint_as_float(mb & 0xffff0000u));
    }
  return s;
}

__device__ __forceinline__ s3_v16f mfma_bf16(const s3_v4i& a, const s3_v4i& b, const s3_v16f& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(s3_v8bf, a), __builtin_bit_cast(s3_v8bf, b), c, 0,
                                                 0, 0);
}

// big += sum of hi hi, small += the five corrections, over the lanes' 8 H
// values (the same k on both sides; the two lane halves hold different k).
template <int H>
__device__ __forceinline__ void mfma_split3(const Split3<H>& a, const Split3<H>& b, s3_v16f& big, s3_v16f& small) {
#pragma unroll
  for (int h = 0; h < H; ++h) {
    big = mfma_bf16(a.hi[h], b.hi[h], big);
    small = mfma_bf16(a.lo[h], b.hi[h], small);
    small = mfma_bf16(a.hi[h], b.lo[h], small);
    small = mfma_bf16(a.mid[h], b.mid[h], small);
    small = mfma_bf16(a.mid[h], b.hi[h], small);
    small = mfma_bf16(a.hi[h], b.mid[h], small);
  }
}

// Whether any of the wave's accumulators is infinite or NaN.
__device__ __forceinline__ bool any_nonfinite(const s3_v16f& acc) {
  float t = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) t = __builtin_fmaf(acc[r], 0.f, t);
  return __builtin_amdgcn_ballot_w64(t != t) != 0;
}

}  // namespace
