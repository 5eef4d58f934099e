// MXFP4 codec on the GPU: unpack_mxfp4 (megabench/tasks/quantization.py:40-51,
// k_decode*) and pack_mxfp4 (:13-37, k_encode), bit for bit with their torch CPU
// chains.
//
// Encoder (fp32 throughout). Per block of 32 values along the last axis:
//   e      = ceil(log2(max(max|x| / 6, 2^-126))), clamped to [-126, 127]
//            (:24-26). log2 is torch's fp32 logarithm, which rounds to the
//            nearest fp32: for a quotient v = 2^n (1 + j 2^-23) with j > 0 the
//            exact ceiling is n + 1, but when log2(v) - n is below half an
//            fp32 step of n the rounded logarithm is n itself and the ceiling
//            stays n. That happens only for small j (j < 23 at |n| < 128), so
//            those quotients take a float64 log2 rounded once to fp32, and
//            every other quotient the exact ceiling from its bits.
//   a      = x * 2^-e as an IEEE fp32 product (:27; subnormal products are
//            rounded, as torch's ldexp rounds them);
//   code   = number of boundaries (0.25 0.75 1.25 1.75 2.5 3.5 5.0) below |a|,
//            plus one at the ties 0.75, 1.75 and 3.5 whose lower code is odd
//            (round to nearest, ties to the even code, :28-34); NaN takes 7
//            (bucketize puts NaN last); | 8 when a < 0 (:35);
//   bytes  = code[2j] | code[2j+1] << 4, scale byte e + 127 (:36-37).
// A block holding a NaN follows torch on x86: its NaN maximum converts to
// int32 as INT_MIN, so the scale byte wraps to 127 and ldexp scales by
// 2^INT_MIN = 0 (NaN and infinite elements then take code 7, finite ones 0).
//
// Layout: a lane takes one 16-byte load, 8 bf16 / fp16 values (4 lanes per
// block) or 4 fp32 values (8 lanes), so a wave reads contiguous 16-byte words
// and writes contiguous packed bytes; the block's maximum magnitude meets in the
// lanes' xor-shuffles as integers (packed 16-bit ones for the 16-bit types),
// whose order is the magnitudes' and which see a NaN as the largest. The values
// are rounded by the hardware's fp32 -> E2M1 conversion (nearest, ties to even,
// saturating), which keeps the sign of a zero: the product is added to +0 first,
// so that -0 and a product that underflows give code 0 as a < 0 does. The
// quotient amax / 6 is only needed where its mantissa is next to a power of two:
// elsewhere amax x (1/6), a few ulps off, has the same exponent.
// HBM-bound: per block 32 input values in, 17 bytes out. A TP8 rank's bf16 gate
// weights [384, 256, 7168]: 320 us, 5.6 TB/s (550 us with the seven
// boundary comparisons per element and the division per lane).
#pragma once

#include "k3moe.h"
#include "k3moe_device.hpp"

namespace k3moe {

constexpr int kEncThreads = 256;
// Workgroups, at most (the rest by a grid stride). The gate weights below in us, encode and
// decode: 2048 workgroups 362 / 359, 16384 398 / 381, 65536 320 / 310, no limit 361 / 316 (one array; why the order is not that of
// the counts is not known). Against the former encoder and decoder no array of 4096 x 32 to
// 90000 x 2048 in any type is slower.
constexpr long kEncGrid = 65536, kDecGrid = 65536;

// The block exponent e (before the +127 bias) of a finite or infinite block
// maximum, as torch's chain computes it (see the file comment).
__device__ __forceinline__ int mx_block_exponent(float amax) {
  // amax x fp32(1/6) is within 2 ulps of the IEEE quotient: 4 mantissa steps away from a power
  // of two, and above the 64 steps past one that need the logarithm, both lie in one binade
  const uint32_t qb = __float_as_uint(__fmul_rn(amax, 1.0f / 6.0f)), qj = qb & 0x7FFFFFu;
  if (qj >= 68u && qj <= 0x7FFFFBu && qb >= 0x01000000u && qb < 0x7F000000u) return (int)(qb >> 23) - 126;
  float v = amax / 6.0f;  // IEEE fp32 division
  if (!(v >= 0x1p-126f)) v = 0x1p-126f;
  const uint32_t b = __float_as_uint(v);
  const int n = (int)(b >> 23) - 127;
  if (n > 127) return 127;  // infinite maximum
  const uint32_t j = b & 0x7FFFFFu;
  int e = j == 0u ? n : n + 1;
  if (j != 0u && j < 64u && n != 0) e = (int)ceilf((float)log2((double)v));
  return e < -126 ? -126 : (e > 127 ? 127 : e);
}

// E2M1 code of one block-normalised value (ties to the even code, NaN -> 7).
__device__ __forceinline__ uint32_t e2m1_code(float a) {
  const float m = fabsf(a);
  uint32_t c = (uint32_t)(m > 0.25f) + (uint32_t)(m > 0.75f) + (uint32_t)(m > 1.25f) + (uint32_t)(m > 1.75f) +
               (uint32_t)(m > 2.5f) + (uint32_t)(m > 3.5f) + (uint32_t)(m > 5.0f);
  c += (uint32_t)((m == 0.75f) | (m == 1.75f) | (m == 3.5f));
  if (m != m) c = 7u;
  return c | (a < 0.f ? 8u : 0u);
}

// 2^-e as an fp32 value, exact for e in [-126, 127] (2^-127 is subnormal).
__device__ __forceinline__ float pow2_neg(int e) {
  return e == 127 ? __uint_as_float(0x00400000u) : __uint_as_float((uint32_t)(127 - e) << 23);
}

// DT: K3MOE_DTYPE_BF16 / _F32 / _F16 (values converted to fp32 exactly)
template <int DT>
__global__ __launch_bounds__(kEncThreads) void k_encode(const void *__restrict__ in, int64_t n_blocks,
                                                        uint8_t *__restrict__ blocks, uint8_t *__restrict__ scales) {
  constexpr int V = DT == K3MOE_DTYPE_F32 ? 4 : 8;  // values per lane
  constexpr int LPB = 32 / V;                       // lanes per block
  const int s = threadIdx.x & (LPB - 1);
  const int64_t stride = (int64_t)gridDim.x * (kEncThreads / LPB);
  for (int64_t blk = (int64_t)blockIdx.x * (kEncThreads / LPB) + threadIdx.x / LPB; blk < n_blocks; blk += stride) {
    const u32x4 w = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const char *>(in) + (blk * LPB + s) * 16);
    // the largest magnitude's bits, in the type's own format
    uint32_t mag;
    if constexpr (DT == K3MOE_DTYPE_F32) {
      mag = max(max(w[0] & 0x7FFFFFFFu, w[1] & 0x7FFFFFFFu), max(w[2] & 0x7FFFFFFFu, w[3] & 0x7FFFFFFFu));
    } else {
      typedef __attribute__((ext_vector_type(2))) uint16_t u16x2;
      u16x2 m = __builtin_bit_cast(u16x2, w[0] & 0x7FFF7FFFu);
#pragma unroll
      for (int t = 1; t < 4; ++t) m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, w[t] & 0x7FFF7FFFu));
      mag = max((uint32_t)m[0], (uint32_t)m[1]);
    }
#pragma unroll
    for (int m = 1; m < LPB; m <<= 1) mag = max(mag, shfl_xor(mag, m));
    float v[V];
#pragma unroll
    for (int t = 0; t < V; ++t) {
      if constexpr (DT == K3MOE_DTYPE_F32) {
        v[t] = __uint_as_float(w[t]);
      } else if constexpr (DT == K3MOE_DTYPE_BF16) {
        v[t] = __uint_as_float(t & 1 ? w[t >> 1] & 0xFFFF0000u : w[t >> 1] << 16);
      } else {
        v[t] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[t >> 1] >> (16 * (t & 1))));
      }
    }
    constexpr uint32_t inf = DT == K3MOE_DTYPE_F32 ? 0x7F800000u : DT == K3MOE_DTYPE_BF16 ? 0x7F80u : 0x7C00u;
    uint32_t sbyte = 127u, packed = 0u;
    if (mag > inf) {  // a NaN in the block
#pragma unroll
      for (int t = 0; t < V; ++t) packed |= e2m1_code(__fmul_rn(v[t], 0.f)) << (4 * t);
    } else {
      const float amax = DT == K3MOE_DTYPE_F32    ? __uint_as_float(mag)
                         : DT == K3MOE_DTYPE_BF16 ? __uint_as_float(mag << 16)
                                                  : (float)__builtin_bit_cast(_Float16, (uint16_t)mag);
      const int e = mx_block_exponent(amax);
      sbyte = (uint32_t)(e + 127);
      const float step = pow2_neg(e);
#pragma unroll
      for (int t = 0; t < V; ++t) v[t] = __fadd_rn(__fmul_rn(v[t], step), 0.f);
      packed = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(packed, v[0], v[1], 1.0f, 0);
      packed = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(packed, v[2], v[3], 1.0f, 1);
      if constexpr (V == 8) {
        packed = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(packed, v[4], v[5], 1.0f, 2);
        packed = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(packed, v[6], v[7], 1.0f, 3);
      }
    }
    if constexpr (V == 8) *reinterpret_cast<uint32_t *>(blocks + blk * 16 + 4 * s) = packed;
    else *reinterpret_cast<uint16_t *>(blocks + blk * 16 + 2 * s) = (uint16_t)packed;
    if (s == 0) scales[blk] = (uint8_t)sbyte;
  }
}

// Exact MXFP4 decode (quantization.py:40-51): a lane takes the codes of one
// 16-byte store, 4 packed bytes for bf16 (8 values) and 2 for fp32 (4), through
// the hardware conversion (exact for every scale byte but 255, whose values are
// the quiet NaN), kDecUnroll of them a grid apart in flight. HBM-bound: 17 bytes
// in, 64 or 128 out per block. A TP8 rank's gate weights to bf16: 301 us, 5.9 TB/s
// (774 us with a byte per thread and the bit construction).
//
// NT: outputs of more than kDecKeep bytes, which the caches do not hold, are stored
// past them (they would only evict the input: the gate weights 310 -> 301 us, 90000
// x 2048 to bf16 83 -> 66); smaller ones stay for the kernel that reads them. us of
// the decode / with a torch amax after it / with a matrix product of 64 rows, kept
// and (past the caches):
//   bf16  16 MB   9.9 / 19.1 / 29.9 (9.6 / 19.1 / 33.7)      fp32  32 MB   9.9 / 30.2 (9.9 / 33.8)
//         64 MB  14.0 / 47.1 / 38.2 (13.8 / 56.5 / 44.3)           64 MB  12.9 / 38.2 (11.5 / 44.5)
//        128 MB  26.0 / 81.8 / 54.3 (26.5 / 103.0 / 65.4)         128 MB  23.8 / 56.3 (25.4 / 70.5)
//        160 MB  37.4 / 104.4 / 69.1 (31.4 / 128.3 / 77.6)        192 MB  33.9 / 76.6 (33.2 / 95.6)
//        256 MB  62.5 / 196.2 / 134.6 (49.9 / 203.2 / 121.7)      256 MB  57.8 / 125.8 (47.9 / 138.5)
constexpr int kDecUnroll = 4;
constexpr int64_t kDecKeep = (int64_t)128 << 20;
template <bool F32, bool NT>
__global__ __launch_bounds__(256) void k_decode(const uint8_t *__restrict__ blocks, const uint8_t *__restrict__ scales,
                                                int64_t n_blocks, void *__restrict__ out) {
  constexpr int LPB = F32 ? 8 : 4;  // lanes per block
  const int64_t n = n_blocks * LPB, stride = (int64_t)gridDim.x * 256;
  for (int64_t u0 = (int64_t)blockIdx.x * 256 + threadIdx.x; u0 < n; u0 += stride * kDecUnroll) {
    uint32_t w[kDecUnroll], s[kDecUnroll];
#pragma unroll
    for (int j = 0; j < kDecUnroll; ++j) {
      const int64_t u = u0 + j * stride < n ? u0 + j * stride : u0;
      if constexpr (F32) w[j] = reinterpret_cast<const uint16_t *>(blocks)[u];
      else w[j] = reinterpret_cast<const uint32_t *>(blocks)[u];
      s[j] = scales[u / LPB];
    }
#pragma unroll
    for (int j = 0; j < kDecUnroll; ++j) {
      const int64_t u = u0 + j * stride;
      if (u >= n) break;
      const float sc = e8m0_to_f32(s[j]);
      u32x4 o;
      if constexpr (F32) {
        typedef __attribute__((ext_vector_type(2))) float f32x2;
        const f32x2 a = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[j], sc, 0);
        const f32x2 b = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w[j], sc, 1);
        o = u32x4{__float_as_uint(a[0]), __float_as_uint(a[1]), __float_as_uint(b[0]), __float_as_uint(b[1])};
      } else {
        o = __builtin_bit_cast(u32x4, fp4x8_to_bf16(w[j], sc));
      }
      if (!scale_is_plain(s[j])) {
        const uint32_t nan = F32 ? 0x7FC00000u : 0x7FC07FC0u;
        o = u32x4{nan, nan, nan, nan};
      }
      if constexpr (NT) __builtin_nontemporal_store(o, reinterpret_cast<u32x4 *>(out) + u);
      else reinterpret_cast<u32x4 *>(out)[u] = o;
    }
  }
}

// The same one byte per thread by bit construction, for arrays that are not
// aligned for k_decode's loads and stores.
__global__ __launch_bounds__(256) void k_decode_bytes(const uint8_t *__restrict__ blocks,
                                                const uint8_t *__restrict__ scales, int64_t n_blocks,
                                                int out_dtype, void *out) {
  const int64_t n = n_blocks * 16;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t byte = blocks[i];
    const uint32_t s = scales[i / 16];
    const uint32_t lo = mxfp4_bits(byte & 15u, s), hi = mxfp4_bits(byte >> 4, s);
    if (out_dtype == K3MOE_DTYPE_F32) {
      reinterpret_cast<u32x2 *>(out)[i] = u32x2{lo, hi};
    } else {
      reinterpret_cast<uint32_t *>(out)[i] = (lo >> 16) | (hi & 0xFFFF0000u);
    }
  }
}

}  // namespace k3moe
