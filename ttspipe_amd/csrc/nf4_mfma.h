// Device helpers shared by the NF4 matrix-core kernels (nf4_gemm_few.hip,
// nf4_gemm_tile.hip, nf4_gemm_dense.hip): the 32x32x16 product, the 16-bit
// roundings, the epilogue of one value, and the waits around LDS loads.
#pragma once
#include "ttsp_common.h"

namespace ttsp {

typedef __bf16 bf16x8_v __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_v __attribute__((ext_vector_type(8)));
typedef float f32x16_v __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2_v __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_v __attribute__((ext_vector_type(2)));
typedef float f32x2_v __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;

// s_waitcnt: vmcnt n, lgkmcnt 0 (gfx9 encoding; expcnt unbounded)
#define TTSP_WAIT_VM_LGKM0(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (((n) >> 4) << 14) | (7 << 4))
// lgkmcnt 0 alone
#define TTSP_WAIT_LGKM0() __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4))

// Lane l supplies row l % 32 of A and column l % 32 of B, each as 8 consecutive
// k at 8 (l / 32); accumulator r of lane l is D[8 (r / 4) + 4 (l / 32) + r % 4]
// [l % 32]. A and B need only agree on which k a lane carries.
template <int DT>
__device__ __forceinline__ f32x16_v mfma32(u32x4 a, u32x4 b, f32x16_v c) {
  if constexpr (DT == DT_BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_v, a), __builtin_bit_cast(bf16x8_v, b),
                                                   c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_v, a), __builtin_bit_cast(f16x8_v, b), c,
                                                  0, 0, 0);
}

// Two fp32 values, each already rounded to fp32, to the activation type
// (nearest even), one hardware pack-convert; lo in the low half.
template <int DT>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  const f32x2_v v = {opaque(lo), opaque(hi)};
  if constexpr (DT == DT_BF16)
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_v));
  else
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_v));
}

// The epilogue of one value (y already rounded): ep 1 adds r, ep 2 multiplies
// by round(silu(r)); the result rounded.
template <int DT>
__device__ __forceinline__ uint16_t mm_epi(float y, uint16_t r, int ep) {
  float v = y;
  if (ep == 1) v = __fadd_rn(Elem<DT>::load(r), y);
  else if (ep == 2) v = __fmul_rn(Elem<DT>::load(Elem<DT>::store(silu_rn(Elem<DT>::load(r)))), y);
  return Elem<DT>::store(v);
}

// silu_rn's arithmetic with the range tests of its exp as selects: no branch, so
// that several run interleaved.
__device__ __forceinline__ float silu_flat(float a) {
  const float x = -a;
  const float n = __builtin_rintf(__fmul_rn(__builtin_amdgcn_fmed3f(x, -87.0f, 88.72283935546875f),
                                            1.44269502162933349609375f));
  float r = __builtin_fmaf(n, -0.693359375f, x);
  r = __builtin_fmaf(n, 2.12194440e-4f, r);
  const float z = __fmul_rn(r, r);
  float p = 1.9875691500e-4f;
  p = __builtin_fmaf(p, r, 1.3981999507e-3f);
  p = __builtin_fmaf(p, r, 8.3334519073e-3f);
  p = __builtin_fmaf(p, r, 4.1665795894e-2f);
  p = __builtin_fmaf(p, r, 1.6666665459e-1f);
  p = __builtin_fmaf(p, r, 5.0000001201e-1f);
  p = __builtin_fmaf(p, z, r);
  p = __builtin_ldexpf(__fadd_rn(p, 1.0f), (int)n);
  p = x > 88.72283935546875f ? __uint_as_float(0x7f800000u) : x < -87.0f ? 0.0f : p;
  return __fdiv_rn(a, __fadd_rn(1.0f, p));
}

// Eight values of an output row (packed, rounded) through the epilogue with
// their operands. A caller keeps it in a rolled loop: eight silus are ~2 KB.
template <int DT>
__device__ __forceinline__ u32x4 mm_epi8(u32x4 y, u32x4 r, int ep) {
  u32x4 o;
  if (ep == 1) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      o[q] = pack2<DT>(__fadd_rn(Elem<DT>::load(r[q]), Elem<DT>::load(y[q])),
                       __fadd_rn(Elem<DT>::load(r[q] >> 16), Elem<DT>::load(y[q] >> 16)));
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t g = pack2<DT>(silu_flat(Elem<DT>::load(r[q])), silu_flat(Elem<DT>::load(r[q] >> 16)));
      o[q] = pack2<DT>(__fmul_rn(Elem<DT>::load(g), Elem<DT>::load(y[q])),
                       __fmul_rn(Elem<DT>::load(g >> 16), Elem<DT>::load(y[q] >> 16)));
    }
  }
  return o;
}

// Eight values at Y + o (m .. m + 7 of a row of M, full: aligned and all below
// M) with the epilogue: the operand from R where ep needs one, or given (own).
template <int DT>
__device__ __forceinline__ void mm_store8(uint16_t* __restrict__ Y, const uint16_t* __restrict__ R, size_t o, int m,
                                          int M, bool full, int ep, u32x4 y, bool own, u32x4 r) {
  if (ep) {
    if (!own) {
      if (full) {
        r = *reinterpret_cast<const u32x4*>(R + o);
      } else {
        for (int u = 0; u < 8; ++u)
          if (m + u < M) {
            const uint32_t h = (uint32_t)R[o + u] << (16 * (u & 1));
            if (u < 2) r.x |= h;
            else if (u < 4) r.y |= h;
            else if (u < 6) r.z |= h;
            else r.w |= h;
          }
      }
    }
    y = mm_epi8<DT>(y, r, ep);
  }
  if (full) {
    *reinterpret_cast<u32x4*>(Y + o) = y;
  } else {
    for (int u = 0; u < 8; ++u)
      if (m + u < M) {
        const uint32_t w = u < 2 ? y.x : u < 4 ? y.y : u < 6 ? y.z : y.w;
        Y[o + u] = (uint16_t)(w >> (16 * (u & 1)));
      }
  }
}

}  // namespace ttsp
