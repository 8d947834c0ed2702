// Raw MFMA A fragments of low-bit codes: the code values themselves, exact in
// the MFMA input type, block scales left to the f32 accumulator side
// (lowbit_gemv5.cuh, lowbit_skinny.cuh).
#pragma once
#include <type_traits>

#include "gemv_args.h"
#include "illm_device.h"

namespace illm {

// packed-pair nibble extract (x & m) | c as ONE v_and_or_b32: hipcc splits
// the pattern into v_and + v_or where it sees the constants (gfx9 VOP3 takes no
// literal and one constant-bus read), so the mask is a kernel argument (an SGPR)
// and the magic an opaque VGPR (opaque_v).  Not written in asm: beside MFMA the
// compiler places the wait states that a result's register needs before it is
// written again, which it cannot for an asm statement
__device__ __forceinline__ uint32_t and_or(uint32_t x, uint32_t m_s, uint32_t c_v) { return (x & m_s) | c_v; }
__device__ __forceinline__ uint32_t opaque_v(uint32_t x) {
  uint32_t r;
  asm("v_mov_b32 %0, %1" : "=v"(r) : "s"(x));
  return r;
}

template <typename C> struct Raw;
template <> struct Raw<BF16> {
  static constexpr uint32_t k4 = 0x43004300u;   // bf16(128 + q)
  static constexpr float off4 = 128.f;
};
template <> struct Raw<F16> {
  static constexpr uint32_t k4 = 0x64006400u;   // f16(1024 + q)
  static constexpr float off4 = 1024.f;
};

// raw value offset per decoder: value = code_raw - OFF (before scale)
template <int DK, typename C>
__host__ __device__ constexpr float raw_off() {
  return DK == DK_INT4S ? Raw<C>::off4 + 8.f
       : DK == DK_INT4A ? Raw<C>::off4
       : DK == DK_INT8S ? 128.f
       : 0.f;
}

template <int DK, typename C>
__device__ __forceinline__ uint4 raw_a4(uint32_t u, uint32_t mask_s, uint32_t magic_v, const uint32_t* lut2) {
  uint4 r;
  if constexpr (DK == DK_INT4S || DK == DK_INT4A) {
    r.x = and_or(u, mask_s, magic_v);
    r.y = and_or(u >> 4, mask_s, magic_v);
    r.z = and_or(u >> 8, mask_s, magic_v);
    r.w = and_or(u >> 12, mask_s, magic_v);
  } else if constexpr (DK == DK_FP4) {
    if constexpr (std::is_same<C, BF16>::value) {
      r.x = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(u, 1.0f, 0));
      r.y = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(u, 1.0f, 1));
      r.z = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(u, 1.0f, 2));
      r.w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(u, 1.0f, 3));
    } else {
      r.x = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(u, 1.0f, 0));
      r.y = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(u, 1.0f, 1));
      r.z = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(u, 1.0f, 2));
      r.w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(u, 1.0f, 3));
    }
  } else {  // DK_LUT4 (C = F16 pair table)
    r.x = lut2[u & 0xff];
    r.y = lut2[(u >> 8) & 0xff];
    r.z = lut2[(u >> 16) & 0xff];
    r.w = lut2[u >> 24];
  }
  return r;
}

// dword c of raw_a4's fragment
template <int DK, typename C>
__device__ __forceinline__ uint32_t raw_a4_at(uint32_t u, int c, uint32_t mask_s, uint32_t magic_v, const uint32_t* lut2) {
  if constexpr (DK == DK_INT4S || DK == DK_INT4A) return and_or(u >> (4 * c), mask_s, magic_v);
  else if constexpr (DK == DK_LUT4) return lut2[(u >> (8 * c)) & 0xff];
  const uint4 r = raw_a4<DK_FP4, C>(u, mask_s, magic_v, lut2);
  return c == 0 ? r.x : c == 1 ? r.y : c == 2 ? r.z : r.w;
}

template <int DK, typename C>
__device__ __forceinline__ uint32_t raw_pair8(uint32_t u, bool hi) {
  if constexpr (DK == DK_FP8E4) {
    if constexpr (std::is_same<C, BF16>::value)
      return __builtin_bit_cast(uint32_t, hi ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u, 1.0f, true)
                                             : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(u, 1.0f, false));
    else
      return __builtin_bit_cast(uint32_t, hi ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(u, 1.0f, true)
                                             : __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(u, 1.0f, false));
  } else if constexpr (DK == DK_FP8E5) {
    if constexpr (std::is_same<C, BF16>::value)
      return __builtin_bit_cast(uint32_t, hi ? __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(u, 1.0f, true)
                                             : __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(u, 1.0f, false));
    else
      return __builtin_bit_cast(uint32_t, hi ? __builtin_amdgcn_cvt_scalef32_pk_f16_bf8(u, 1.0f, true)
                                             : __builtin_amdgcn_cvt_scalef32_pk_f16_bf8(u, 1.0f, false));
  } else {
    // integer bytes through the exact small-integer float conversion;
    // signed codes are biased by 128 (raw_off = 128)
    if constexpr (DK == DK_INT8S) u ^= 0x80808080u;
    const int sh = hi ? 16 : 0;
    return pack2<C>((float)((u >> sh) & 0xff), (float)((u >> (sh + 8)) & 0xff));
  }
}

// constant of the offset product: -offset for the formats whose codes carry
// one, 1 for unsigned codes with a block minimum (the plain sum of x)
template <int DK, typename T>
__host__ __device__ constexpr uint32_t raw_const2() {
  constexpr bool b = std::is_same<T, BF16>::value;
  // bf16 -136 / -128 / 1, f16 -1032 / -1024 / -128 / 1
  return DK == DK_INT4S ? (b ? 0xC308C308u : 0xE408E408u)
       : DK == DK_INT4A ? (b ? 0xC300C300u : 0xE400E400u)
       : DK == DK_INT8S ? (b ? 0xC300C300u : 0xD800D800u)
       : (b ? 0x3F803F80u : 0x3C003C00u);
}

template <int DK, typename C>
__device__ __forceinline__ uint4 raw_a8(uint32_t lo, uint32_t hi) {
  return make_uint4(raw_pair8<DK, C>(lo, false), raw_pair8<DK, C>(lo, true), raw_pair8<DK, C>(hi, false),
                    raw_pair8<DK, C>(hi, true));
}

// 1 / rms of the rows of a deferred norm from parts of their sums of squares (GemvArgs::xpss_parts): wave w sums rows w, w
// + NW ..  request() comes ahead of the other loads; a launch without parts asks for nothing (an empty descriptor).
template <int NW>
struct RowParts {
  static constexpr int R = 16 / NW;
  f32x4 v[R];
  template <typename A>
  __device__ __forceinline__ void request(const A& a, int wave, int lane) {
    const int n = a.xpss_parts;
    const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc((void*)a.xpss, 0, n > 0 ? a.M * n * 4 : 0, 0x00020000);
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int m = wave + i * NW;
      v[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
          rd, lane * 4 < n ? (uint32_t)(m * n + lane * 4) * 4u : ~0u, 0, 0));
    }
  }
  template <typename A>
  __device__ __forceinline__ void finish(const A& a, int wave, int lane, float* inv) const {
    const int n = a.xpss_parts;
    if (n <= 0) return;
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int m = wave + i * NW;
      if (m >= a.M) continue;
      float s = (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
      for (int j = 256 + lane; j < n; j += 64) s += a.xpss[(size_t)m * n + j];
      s = wave_sum(s);
      if (lane == 0) inv[m] = rsqrtf(s / (float)a.xpss_n + a.xpss_eps);
    }
  }
};

}  // namespace illm
