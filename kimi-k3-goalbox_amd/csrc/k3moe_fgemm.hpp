// Grouped expert GEMMs on the scaled FP4 MFMA (v_mfma_scale_f32_16x16x128_f8f6f4)
// for prefill-sized steps: the MXFP4 weights go to the MFMA as they are stored
// (E2M1 nibbles and their E8M0 block scales), the activations as two E4M3
// terms with E8M0 block scales.
//
// Activation format ("two-term MXFP8"): a block of 32 values v (bf16-exact)
// is stored as hi = E4M3(v / 2^eh) and lo = E4M3((v - hi 2^eh) / 2^el), where
// eh = floor(log2 max|v|) - 7 and el the same for the remainders, each scale
// one E8M0 byte per block. The MFMA runs once on hi and once on lo into the
// same fp32 accumulator. A bf16 value has 8 significant bits and E4M3 4, so
// hi + lo equals v for every element within 2^8 of its block's maximum
// (smaller ones lose only bits below 2^-16 of it): the products, accumulated
// in fp32, are those of the bf16 operands. A single E4M3 term would leave the
// reference's band (kimi.py:413-429) by a factor of about 7.
//
// Operand layouts of the 16x16x128 MFMA (one wave; measured on gfx950):
//   A (16 weight rows x 128 k, FP4): lane (row i = l % 16, q = l / 16) holds
//     k 32q .. 32q + 31 in 16 bytes, element 2j in the low nibble of byte j:
//     exactly MXFP4 block q of the k-step; its scale byte is that block's.
//   B (128 k x 16 token columns, FP8): lane (column j, q) holds k 16q .. 16q+15
//     in bytes 0-15 and k 64 + 16q .. 64 + 16q + 15 in bytes 16-31; its scale
//     byte is the one of block q (k 32q .. 32q + 31), whatever lane holds it.
//   D (16 x 16 fp32): lane (column j, q) holds rows 4q .. 4q + 3.
//
// The GEMMs themselves are k_sgemm's FP4 instantiations (k3moe_sgemm.hpp): MFMA on hi
// then on lo into the same accumulator, in place of the decode and the bf16 MFMAs.
// Their gate/up epilogue takes the activation from the hardware exponential and
// reciprocal (fast_act), rounds h to bf16 (kimi.py:322) and splits it into two E4M3
// terms per 32 columns of I (two gate tiles are one block) for the down GEMM.
#pragma once

#include "k3moe_device.hpp"
#include "k3moe_plan.hpp"

namespace k3moe {

typedef __attribute__((ext_vector_type(8))) int i32x8;

// ------------------------------------------------------ two-term MXFP8 --

// E8M0 byte of 2^(floor(log2 amax) - 7) for a block maximum amax >= 0 (0 for
// a zero or subnormal maximum).
__device__ __forceinline__ uint32_t mx8_scale(float amax) {
  const int be = (int)((__float_as_uint(amax) >> 23) & 255u);
  return be > 7 ? (uint32_t)(be - 7) : 0u;
}
// 2^(127 - s) and 2^(s - 127) for an E8M0 byte s <= 248.
__device__ __forceinline__ float mx8_inv(uint32_t s) { return __uint_as_float((254u - s) << 23); }
__device__ __forceinline__ float mx8_val(uint32_t s) { return s ? __uint_as_float(s << 23) : __uint_as_float(0x00400000u); }

// E4M3 bytes (round to nearest even) of four values, packed little-endian.
__device__ __forceinline__ uint32_t e4m3x4(float a, float b, float c, float d) {
  int w = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c, d, w, true);
}
__device__ __forceinline__ float e4m3_f32(uint32_t word, int byte) {
  switch (byte) {
    case 0: return __builtin_amdgcn_cvt_f32_fp8((int)word, 0);
    case 1: return __builtin_amdgcn_cvt_f32_fp8((int)word, 1);
    case 2: return __builtin_amdgcn_cvt_f32_fp8((int)word, 2);
    default: return __builtin_amdgcn_cvt_f32_fp8((int)word, 3);
  }
}

// Lane-group maximum of |v| over the lanes that xor-differ in `mask` bits
// (Masks: the xor distances, ascending).
template <int... Masks>
__device__ __forceinline__ float group_amax(float m) {
  ((m = fmaxf(m, shfl_xor(m, Masks))), ...);
  return m;
}

// Two-term split of the four values v of a lane; the block spans the lanes
// reached by Masks. Returns the hi and lo E4M3 words and the block's scale
// bytes.
template <int... Masks>
__device__ __forceinline__ void mx8_split4(const float v[4], uint32_t &hi, uint32_t &lo, uint32_t &sh, uint32_t &sl) {
  float m = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
  sh = mx8_scale(group_amax<Masks...>(m));
  const float ih = mx8_inv(sh), vh = mx8_val(sh);
  hi = e4m3x4(v[0] * ih, v[1] * ih, v[2] * ih, v[3] * ih);
  float r[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) r[t] = __fsub_rn(v[t], __fmul_rn(e4m3_f32(hi, t), vh));  // exact
  m = fmaxf(fmaxf(fabsf(r[0]), fabsf(r[1])), fmaxf(fabsf(r[2]), fabsf(r[3])));
  sl = mx8_scale(group_amax<Masks...>(m));
  const float il = mx8_inv(sl);
  lo = e4m3x4(r[0] * il, r[1] * il, r[2] * il, r[3] * il);
}

// Expert inputs [n_rows, K] bf16 -> hi, lo [n_rows, K] E4M3 and shi, slo
// [n_rows, K/32] E8M0. 8 lanes per block of 32 (4 values each).
__global__ __launch_bounds__(256) void k_quant(const uint16_t *__restrict__ x, long n_blocks, uint8_t *__restrict__ hi,
                                               uint8_t *__restrict__ lo, uint8_t *__restrict__ shi,
                                               uint8_t *__restrict__ slo) {
  const int s = threadIdx.x & 7;
  const long stride = (long)gridDim.x * 32;
  for (long blk = (long)blockIdx.x * 32 + (threadIdx.x >> 3); blk < n_blocks; blk += stride) {
    const u32x2 w = *reinterpret_cast<const u32x2 *>(x + blk * 32 + 4 * s);
    const float v[4] = {bf16_bits_to_f32(w[0] & 0xFFFFu), bf16_bits_to_f32(w[0] >> 16),
                        bf16_bits_to_f32(w[1] & 0xFFFFu), bf16_bits_to_f32(w[1] >> 16)};
    uint32_t h, l, sh, sl;
    mx8_split4<1, 2, 4>(v, h, l, sh, sl);
    *reinterpret_cast<uint32_t *>(hi + blk * 32 + 4 * s) = h;
    *reinterpret_cast<uint32_t *>(lo + blk * 32 + 4 * s) = l;
    if (s == 0) {
      shi[blk] = (uint8_t)sh;
      slo[blk] = (uint8_t)sl;
    }
  }
}

__device__ __forceinline__ f32x4 mfma_fp4x8(const u32x4 &a, const i32x8 &b, uint32_t sa, uint32_t sb, f32x4 c) {
  const i32x8 a8 = {(int)a[0], (int)a[1], (int)a[2], (int)a[3], 0, 0, 0, 0};
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a8, b, c, 4, 0, 0, (int)sa, 0, (int)sb);
}

// Two-term split of a 32-value block held 8 to a lane by the lanes that differ in
// bits 16 and 32: the hi and lo E4M3 words of each half and the block's scale bytes.
__device__ __forceinline__ void mx8_split8(const float v[2][4], uint32_t hi[2], uint32_t lo[2], uint32_t &sh,
                                           uint32_t &sl) {
  float m = 0.f;
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
    for (int t = 0; t < 4; ++t) m = fmaxf(m, fabsf(v[s2][t]));
  sh = mx8_scale(group_amax<16, 32>(m));
  const float ih = mx8_inv(sh), vh = mx8_val(sh);
  float r[2][4];
  m = 0.f;
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2) {
    hi[s2] = e4m3x4(v[s2][0] * ih, v[s2][1] * ih, v[s2][2] * ih, v[s2][3] * ih);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      r[s2][t] = __fsub_rn(v[s2][t], __fmul_rn(e4m3_f32(hi[s2], t), vh));  // exact
      m = fmaxf(m, fabsf(r[s2][t]));
    }
  }
  sl = mx8_scale(group_amax<16, 32>(m));
  const float il = mx8_inv(sl);
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2) lo[s2] = e4m3x4(r[s2][0] * il, r[s2][1] * il, r[s2][2] * il, r[s2][3] * il);
}

// Activation operand of one GEMM: bf16 rows in `hi`, or rows of two E4M3 terms and their scales.
struct MxAct {
  const uint8_t *hi, *lo, *shi, *slo;
};

}  // namespace k3moe
