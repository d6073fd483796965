// Helpers shared by the affine-quantised matmul kernels (qmatmul.hip, qgemm_ks.hip).
#pragma once

#include "ema_common.hpp"
#include "qmatmul_plan.hpp"

namespace ema {

// Launches of the K-split kernels (qgemm_ks.hip): the GEMM, and exact products of up to 32 rows.
int32_t launch_qgemm_ks(hipStream_t st, const QmmArgs& a, const KsPlan& p, int gs, int bits, bool f16);
int32_t launch_qmv_ks(hipStream_t st, const QmmArgs& a, const KsPlan& p, int gs, int bits, bool f16);

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr uint32_t kOffRow = 0xF0000000u;  // a buffer offset past every range: loads return 0

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

// Between a wave's LDS writes and its reads of what its other lanes wrote: the hardware runs a
// wave's LDS operations in order, and this has the compiler keep that order, which it may not
// otherwise when it can tell a lane's own write and read apart. No instructions.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
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

// (x & m) | c in one v_and_or_b32. gfx950's VOP3 encoding takes no 32-bit literal, so with
// literal masks the compiler splits it into v_and + v_or; the empty asm statements hand the
// constants over as VGPR values (set once per kernel) and the compiler selects the fused
// instruction. The instruction itself is left to the compiler: its result feeds MFMA
// operands, and the hazard recognizer inserts the wait states a VALU write needs before an
// MFMA reads it only for instructions it emits itself, not for an inline-asm VALU
// instruction.
__device__ __forceinline__ uint32_t and_or(uint32_t x, uint32_t m, uint32_t c) {
  asm("" : "+v"(m));
  asm("" : "+v"(c));
  return (x & m) | c;
}

template <int BITS, bool F16>
struct Fields {
  // the weight bits take the mantissa of this constant: value kOff + q, exact
  static constexpr bool kMagic = F16 || BITS == 4;
  static constexpr uint32_t kMagicBits = F16 ? 0x64006400u : 0x43004300u;  // 1024 (f16), 128 (bf16)
  static constexpr float kOff = !kMagic ? 0.0f : (F16 ? 1024.0f : 128.0f);
  static constexpr uint32_t kOnes = F16 ? 0x3C003C00u : 0x3F803F80u;

  // B operand of MFMA step `st`: 8 fields of this lane's weight dwords.
  static __device__ __forceinline__ u32x4 weights(const uint32_t* wd, int st) {
    u32x4 r;
    if constexpr (BITS == 4) {
      const uint32_t w = wd[st];  // fields 0..7; register i holds fields i and i + 4
      r[0] = and_or(w, 0x000F000Fu, kMagicBits);
      r[1] = and_or(w >> 4, 0x000F000Fu, kMagicBits);
      r[2] = and_or(w >> 8, 0x000F000Fu, kMagicBits);
      r[3] = and_or(w >> 12, 0x000F000Fu, kMagicBits);
    } else if constexpr (F16) {
      const uint32_t w0 = wd[2 * st], w1 = wd[2 * st + 1];  // bytes 0..3, 4..7
      r[0] = and_or(w0, 0x00FF00FFu, kMagicBits);           // bytes 0, 2
      r[1] = and_or(w0 >> 8, 0x00FF00FFu, kMagicBits);      // bytes 1, 3
      r[2] = and_or(w1, 0x00FF00FFu, kMagicBits);
      r[3] = and_or(w1 >> 8, 0x00FF00FFu, kMagicBits);
    } else {
      const uint32_t w0 = wd[2 * st], w1 = wd[2 * st + 1];
      // an integer below 256 is exact in the top half of its f32
      const uint32_t f0 = __float_as_uint((float)(w0 & 0xFFu)), f1 = __float_as_uint((float)((w0 >> 8) & 0xFFu));
      const uint32_t f2 = __float_as_uint((float)((w0 >> 16) & 0xFFu)), f3 = __float_as_uint((float)(w0 >> 24));
      const uint32_t f4 = __float_as_uint((float)(w1 & 0xFFu)), f5 = __float_as_uint((float)((w1 >> 8) & 0xFFu));
      const uint32_t f6 = __float_as_uint((float)((w1 >> 16) & 0xFFu)), f7 = __float_as_uint((float)(w1 >> 24));
      r[0] = pair(f0, f1, kSelHi);
      r[1] = pair(f2, f3, kSelHi);
      r[2] = pair(f4, f5, kSelHi);
      r[3] = pair(f6, f7, kSelHi);
    }
    return r;
  }
  // A operand of the same step: 8 consecutive activations (4 dwords) paired as the
  // fields above are.
  static __device__ __forceinline__ u32x4 acts(const uint32_t* d) {
    u32x4 r;
    if constexpr (BITS == 4) {  // {x_i, x_i+4}
      r[0] = pair(d[0], d[2], kSelLo);
      r[1] = pair(d[0], d[2], kSelHi);
      r[2] = pair(d[1], d[3], kSelLo);
      r[3] = pair(d[1], d[3], kSelHi);
    } else if constexpr (F16) {  // {x_0, x_2}, {x_1, x_3}, {x_4, x_6}, {x_5, x_7}
      r[0] = pair(d[0], d[1], kSelLo);
      r[1] = pair(d[0], d[1], kSelHi);
      r[2] = pair(d[2], d[3], kSelLo);
      r[3] = pair(d[2], d[3], kSelHi);
    } else {
      r = u32x4{d[0], d[1], d[2], d[3]};
    }
    return r;
  }
};

}  // namespace
}  // namespace ema
