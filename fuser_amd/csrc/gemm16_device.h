// Device-side pieces shared by the kernels whose MFMA operands are 16-bit floats (gemm16.hip and its *_kernel.inl files,
// nvfp4_decode.hip).
#pragma once
#include "lds_direct.h"
#include "nvf_internal.h"

namespace nvf {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t pack2(float a, float b, bool out_bf16) {
  if (out_bf16) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    bf16x2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, v);
  }
  f16x2 v = {(_Float16)a, (_Float16)b};
  return __builtin_bit_cast(uint32_t, v);
}

// LDS tile: rows x 64 16-bit elements (128 bytes per row); 16-byte chunk c of row r sits at chunk
// position c ^ ((r >> 1) & 7): two rows fill the 64 banks once, so the MFMA fragment reads (16
// consecutive lanes = 16 consecutive rows, one chunk) are conflict-free.
__device__ __forceinline__ int lds_pos2(int row, int chunk) { return row * 8 + (chunk ^ ((row >> 1) & 7)); }
__device__ __forceinline__ int lds_pos(int row, int chunk) { return lds_pos2(row, chunk); }
// ... for tiles that ds_write_b128 fills with 4 neighbouring lanes writing every other chunk of a row: two neighbouring rows
// differ in the lowest bit of the position as well, so that 8 lanes cover 32 banks, which is what a write is checked for
// (a read is for 64, and stays conflict-free)
__device__ __forceinline__ int lds_pos_staged(int row, int chunk) { return lds_pos2(row, chunk ^ (row & 1)); }

// e4m3 scales of a lane's two blocks -> fp16 pairs; one dword (8 values of one block) -> one MFMA operand
__device__ __forceinline__ void scale_pairs(uint32_t s2, f16x2 sv[2]) {
  const float f0 = __builtin_amdgcn_cvt_f32_fp8((int)s2, 0), f1 = __builtin_amdgcn_cvt_f32_fp8((int)s2, 1);
  sv[0] = __builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_pkrtz(f0, f0));
  sv[1] = __builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_pkrtz(f1, f1));
}
__device__ __forceinline__ u32x4 dequant_dword(uint32_t qw, f16x2 sv) {
  const f16x2 h0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(qw, 1.0f, 0) * sv;
  const f16x2 h1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(qw, 1.0f, 1) * sv;
  const f16x2 h2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(qw, 1.0f, 2) * sv;
  const f16x2 h3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(qw, 1.0f, 3) * sv;
  return u32x4{__builtin_bit_cast(uint32_t, h0), __builtin_bit_cast(uint32_t, h1), __builtin_bit_cast(uint32_t, h2),
               __builtin_bit_cast(uint32_t, h3)};
}

// 32 packed e2m1 values and their two e4m3 block scales -> four MFMA operands of 8 fp16 values
__device__ __forceinline__ void dequant_frags(const u32x4 q, uint32_t s2, u32x4 out[4]) {
  f16x2 sv[2];
  scale_pairs(s2, sv);
#pragma unroll
  for (int w = 0; w < 4; ++w) out[w] = dequant_dword(q[w], sv[w >> 1]);  // dword w = elements 8w..8w+7, scale block w/2
}

}  // namespace
}  // namespace nvf
