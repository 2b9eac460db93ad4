// The 32x32x16 matrix operations on 16-bit rows and the transposing LDS read, shared by the
// prefill reads that run on the matrix cores.
#pragma once

#include "lsa_read_dev.h"

namespace lsa {

typedef float f32x16_t __attribute__((ext_vector_type(16)));

template <typename T> struct Mfma;
template <> struct Mfma<bf16_t> {
  typedef bf16x8_t op_t;
  static __device__ __forceinline__ f32x16_t run(op_t a, op_t b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {  // v_cvt_pk_bf16_f32 (RNE)
    typedef __bf16 v2_t __attribute__((ext_vector_type(2)));
    typedef float f2_t __attribute__((ext_vector_type(2)));
    const f2_t f = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, v2_t));
  }
  // c + lo + hi of a packed pair (v_dot2_f32_bf16 against ones)
  static __device__ __forceinline__ float sum2(uint32_t pair, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, pair), __builtin_bit_cast(bf16x2_t, 0x3F803F80u),
                                           c, false);
  }
};
template <> struct Mfma<_Float16> {
  typedef f16x8_t op_t;
  static __device__ __forceinline__ f32x16_t run(op_t a, op_t b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    typedef _Float16 v2_t __attribute__((ext_vector_type(2)));
    typedef float f2_t __attribute__((ext_vector_type(2)));
    const f2_t f = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, v2_t));
  }
  static __device__ __forceinline__ float sum2(uint32_t pair, float c) {
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_t, pair), __builtin_bit_cast(f16x2_t, 0x3C003C00u), c, false);
  }
};

// Four keys of one V column from the row-major V tile, for a V^T MFMA operand, by the
// transposing LDS read (ds_read_b64_tr_b16): in each group of 16 lanes, lane j addresses
// the 8 bytes at key0 + j / 4, dims dim0 + 4 (j % 4) .. + 3, and lane i receives keys
// key0 .. key0 + 3 of dim dim0 + i.
// `lane_base` is this lane's part of the address (key j / 4, dims 4 (j % 4) of the tile);
// the rest is a constant byte offset, which the read's immediate field takes.
typedef short v4i16_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) char lds_char;
__device__ __forceinline__ uint2 v_column4(const lds_char* lane_base, int offset) {
  typedef __attribute__((address_space(3))) v4i16_t lds_v4;
  const v4i16_t r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(lane_base + offset));
  return __builtin_bit_cast(uint2, r);
}

}  // namespace lsa
