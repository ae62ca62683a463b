// Device-side pieces shared by the kernels whose MFMA operands are 16-bit floats (gemm16.hip and its *_kernel.inl files,
// nvfp4_decode.hip).
#pragma once
#include "lds_direct.h"
#include "nvf_internal.h"

namespace nvf {
constexpr int kMaxGroups = 1024;  // same bound as the reference's <<<1, num_experts>>> set-up kernel

struct Params {
  const uint8_t* a;
  const uint8_t* b;
  const uint8_t* sfa;
  const uint8_t* sfb;
  const float* alpha;
  void* out;
  const int32_t* problem_sizes;   // nullptr => dense
  const int32_t* expert_offsets;
  const int32_t* sf_offsets;
  int groups;
  int m, n, k;
  // split of K over workgroups (dense NVFP4 tile kernel only): work item w = tile w / splits, K spans
  // [ (w % splits) * spans_per_split, ... ); fp32 partial tiles go to partial[split][m][n]
  float* partial = nullptr;
  int splits = 1;
  int spans_per_split = 0;
  // NVFP4 tile kernel, grouped: 1 = rows [0, rows & ~255) of every group are computed by the 256x256 kernel,
  // take only the rows after them
  int skip_whole_256 = 0;
  // skinny kernel: first activation row this launch computes (its slabs of 16*TT rows follow in blockIdx.y order)
  int m_base = 0;
  // grouped skinny kernel: the group sizes it serves; the tile kernel skips groups of fewer than min_rows rows
  int rows_lo = 0, rows_hi = 0, min_rows = 0;
  // grouped skinny kernel: 0 = one block of workgroups per group (those of other sizes return at once); otherwise the
  // launch has class_slots blocks and block i looks for the i-th group of rows_lo..rows_hi rows
  int class_slots = 0;
  int tail_done = 0;  // grouped NVFP4 dispatch: the ends of the large groups have been computed by an earlier launch
  // block-scaled result (nvfp4_scaled_mm_blockscale): out = packed e2m1 [m, n/2], out_sf = e4m3 scales in the 128x4
  // layout of [roundUp(m,128), roundUp(n/16,4)], gnorm = the result's global (encode) scale on the device
  uint8_t* out_sf = nullptr;
  const float* gnorm = nullptr;
  // dense weight-streaming kernel: 0 = 16-bit result, 1 = the block-scaled result above, 2 = the fp32 product itself
  int stream_result = 0;
  // ... with stream_result 1: the kernel also zeroes the padding rows and columns of the scale buffer's last 128x4 tiles
  int stream_zero_pad = 0;
  // dense NVFP4 with a 16-bit result: elements between rows of the result; 0: n (a launch that computes some of the
  // columns sets it)
  int ldc = 0;
  __host__ __device__ int out_pitch() const { return ldc ? ldc : n; }
};

// the persistent kernel of nvfp4_persistent.hip: 256x256 (tm = 4) or 128x256 (tm = 2) tiles
enum class Nvfp4Out { kF16, kBf16, kF32, kFp4 };
int launch_nvfp4_persistent(const Params& p, Nvfp4Out out, bool grouped, int tm, int cus, hipStream_t stream);

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
__device__ __forceinline__ int lds_pos(int row, int chunk) { return row * 8 + (chunk ^ ((row >> 1) & 7)); }

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

// Grouped NVFP4: the rows of a group of m_g rows that the 256x256 kernel computes: its whole 256-row tiles, and a
// last tile of more than 128 rows (its missing rows are read as copies of the last one and are not stored).
// The tile kernel takes the rows from there on; a value >= m_g means none are left.
__device__ __forceinline__ int rows_in_256_tiles(int m_g) {
  const int whole = m_g & ~255;
  return m_g - whole > 128 ? whole + 256 : whole;
}

// Block-scaled epilogue of four neighbouring 16x16 accumulator tiles, i.e. of 16 rows and their four blocks: lane (r, g) holds row r, columns
// 16 j + 4 g + e in acc[j][e].  Lane (r, g) works out the scale of block g: the exchanges with the lanes 16 and 32 further on
// hand every lane the other three's maxima of its own block, and their factors back.  q8: the code of block g; h[j]: this
// lane's payload bytes 2 g, 2 g + 1 of block j.  (All four lanes working out all four scales: 2 us more on a 128x256 tile.)
__device__ __forceinline__ void quantize_acc_tiles16(const f32x4 (&acc)[4], float alpha, float gs, float decode, uint32_t& q8, uint32_t (&h)[4]) {
  float x[4][4], m[4];
  bool nonfinite = false;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    m[j] = -INFINITY;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[j][e] = acc[j][e] * alpha;
      m[j] = fmaxf(m[j], fabsf(x[j][e]));  // NaN ignored, as the quantizer does
      nonfinite |= !(fabsf(x[j][e]) < INFINITY);
    }
  }
  const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  const bool odd = (lane & 16) != 0, high = (lane & 32) != 0;
  auto from = [&](float v, int other) { return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ other) << 2, __builtin_bit_cast(int, v))); };
  const float lo = fmaxf(odd ? m[1] : m[0], from(odd ? m[0] : m[1], 16)), hi = fmaxf(odd ? m[3] : m[2], from(odd ? m[2] : m[3], 16));
  const float own = fmaxf(high ? hi : lo, from(high ? lo : hi, 32));  // of block g = 2 high + odd
  float r;
  q8 = nvfp4_block_scale(own, true, gs, decode, true, r);
  const float other = from(r, 32), r_lo = high ? other : r, r_hi = high ? r : other;  // blocks odd and 2 + odd
  const float o_lo = from(r_lo, 16), o_hi = from(r_hi, 16);
  const float f[4] = {odd ? o_lo : r_lo, odd ? r_lo : o_lo, odd ? o_hi : r_hi, odd ? r_hi : o_hi};
  const bool plain = __builtin_amdgcn_ballot_w64(nonfinite) == 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (plain) {
      const uint32_t w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(0u, x[j][0] * f[j], x[j][1] * f[j], 1.0f, 0);
      h[j] = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, x[j][2] * f[j], x[j][3] * f[j], 1.0f, 1);
    } else {  // explicit NaN rule of the narrow cast
      h[j] = f32x2_to_e2m1_byte(x[j][0] * f[j], x[j][1] * f[j]) | f32x2_to_e2m1_byte(x[j][2] * f[j], x[j][3] * f[j]) << 8;
    }
  }
}

}  // namespace
}  // namespace nvf
