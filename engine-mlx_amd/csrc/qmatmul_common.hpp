// Helpers shared by the affine-quantised matmul kernels (qmatmul.hip, qgemm_ks.hip).
#pragma once

#include "ema_common.hpp"

namespace ema {

struct QmmArgs {
  const uint8_t* x;  // [M, ldx] activations
  const uint8_t* w;  // [N, K * BITS / 8] packed fields
  const uint8_t* s;  // [N, G] scales
  const uint8_t* b;  // [N, G] biases
  uint8_t* y;        // [M, ldy]
  int64_t ldx, ldy;  // row strides in elements
  int M, N, K, G;    // G = K / GS
  int mtiles;        // row tiles of x (16 * MR rows each)
  int remap;         // grid size divisible by 8: give each XCD a contiguous range of tiles
};

// Column and row tiles of 16 of the K-split GEMM (qgemm_ks.hip); mt = 0: it does not apply.
struct KsPlan {
  int mt, nt;
};
KsPlan plan_ks(const QmmArgs& a, int gs, int bits, int cus);
int32_t launch_qgemm_ks(hipStream_t st, const QmmArgs& a, const KsPlan& p, int gs, int bits, bool f16);

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kMaxWaves = 8;
constexpr uint32_t kOffRow = 0xF0000000u;  // a buffer offset past every range: loads return 0

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

template <bool F16>
__device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}

template <bool F16>
__device__ __forceinline__ float act_to_f32(uint32_t bits16) {
  if constexpr (F16)
    return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16);
  else
    return __uint_as_float(bits16 << 16);
}
template <bool F16>
__device__ __forceinline__ uint16_t f32_to_act(float v) {
  if constexpr (F16)
    return __builtin_bit_cast(uint16_t, (_Float16)v);
  else
    return (uint16_t)f32_to_bf16_bits(v);
}

// v_perm_b32 selectors: {lo16(lo), lo16(hi)} and {hi16(lo), hi16(hi)} of two dwords.
constexpr uint32_t kSelLo = 0x05040100u, kSelHi = 0x07060302u;
__device__ __forceinline__ uint32_t pair(uint32_t lo, uint32_t hi, uint32_t sel) {
  return __builtin_amdgcn_perm(hi, lo, sel);
}

// byte I of x as f32 (v_cvt_f32_ubyteI)
template <int I>
__device__ __forceinline__ float ubyte_f32(uint32_t x) { return (float)((x >> (8 * I)) & 0xFFu); }

// Two f32 as a pair of activations (one conversion instruction on gfx950).
template <bool F16>
__device__ __forceinline__ uint32_t pack_act2(float lo, float hi) {
  if constexpr (F16) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 v = {(_Float16)lo, (_Float16)hi};
    return __builtin_bit_cast(uint32_t, v);
  } else {
    return pack_bf16x2(lo, hi);
  }
}

// Eight fields (one word of 4-bit fields, or two words of bytes) as eight activations
// round(fma(sc, q, bc)), one rounding, in field order. The empty asm keeps the two masked
// words as they are, so that every field is one byte conversion of them (the compiler
// otherwise extracts each field on its own: 41 VALU per eight fields instead of 23).
template <int BITS, bool F16>
__device__ __forceinline__ u32x4 dequant8(uint32_t w0, uint32_t w1, float sc, float bc) {
  float q[8];
  if constexpr (BITS == 4) {
    uint32_t lo = w0 & 0x0F0F0F0Fu, hi = (w0 >> 4) & 0x0F0F0F0Fu;  // fields 2i, 2i + 1
    asm("" : "+v"(lo));
    asm("" : "+v"(hi));
    q[0] = ubyte_f32<0>(lo);
    q[1] = ubyte_f32<0>(hi);
    q[2] = ubyte_f32<1>(lo);
    q[3] = ubyte_f32<1>(hi);
    q[4] = ubyte_f32<2>(lo);
    q[5] = ubyte_f32<2>(hi);
    q[6] = ubyte_f32<3>(lo);
    q[7] = ubyte_f32<3>(hi);
  } else {
    q[0] = ubyte_f32<0>(w0);
    q[1] = ubyte_f32<1>(w0);
    q[2] = ubyte_f32<2>(w0);
    q[3] = ubyte_f32<3>(w0);
    q[4] = ubyte_f32<0>(w1);
    q[5] = ubyte_f32<1>(w1);
    q[6] = ubyte_f32<2>(w1);
    q[7] = ubyte_f32<3>(w1);
  }
  u32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    o[e] = pack_act2<F16>(__builtin_fmaf(sc, q[2 * e], bc), __builtin_fmaf(sc, q[2 * e + 1], bc));
  return o;
}

}  // namespace
}  // namespace ema
