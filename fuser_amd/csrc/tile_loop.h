// The K loop of the persistent 256x256 kernels whose operands need no conversion (grouped_mm: bf16 / f16, mxfp8_scaled_mm):
// 4 wavefronts, each a 128x128 part of the tile, operand rows of 128 bytes per step (64 elements of 16 bits, 128 of e4m3).
//
// 16x16 MFMAs: on N(0,1) data the card's power limit, not the matrix pipe, sets the rate, and a 16x16 MFMA moves half the
// accumulator data per flop of a 32x32 one.  Register-only loops, PFLOP/s: bf16 32x32x16 1.81, 16x16x32 2.07; f16 1.68 / 1.93;
// e4m3 32x32x64 4.05, 16x16x128 4.36; on zeros both shapes 2.44 and 4.93.
//
// A step is two phases: tiles 0..3 of A against all 8 tiles of B, then tiles 4..7 of A.  A wavefront holds one step's fragments
// (64 registers per operand) and replaces them in place: A 4..7 of the step are read in its first phase, A 0..3 and B of the
// next step in its second, each B tile once its MFMAs have been issued.  What a phase has read out of LDS is refilled from the
// next barrier on: 12 of the 16 loads of step s + 2 in the first phase of step s, 4 in the second, so that reads and loads
// share the LDS evenly (8 reads and 12 loads, 24 reads and 4 loads; with all 16 loads in one half of a step that half was
// bound by LDS).  A load has at least a whole step to land: the waits are for all but the newest 16 loads, never for all.
//
// LDS: A tile of buffer 0, of buffer 1, B tile of buffer 0, of buffer 1; 256 rows x 128 bytes each, 16-byte chunk c of row r at
// position c ^ ((r >> 1) & 7): the fragment reads (16 consecutive rows, one chunk) are conflict-free.
#pragma once
#include "lds_direct.h"
#include "nvf_internal.h"

namespace nvf {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

enum class Mma { kBf16, kF16, kMxFp8 };

constexpr int kTile256Bytes = 4 * 32768;  // LDS of the operand tiles

template <Mma MMA>
struct Tile256Loop {
  // per tile: lane (r, g) holds chunks g and 4 + g of row 16 * tile + r, the operand of one e4m3 MFMA or of two of 16 bits
  u32x8 fa[8], fb[8];
  f32x4 acc[8][8];  // [tile of A][tile of B], element e: row 16 i + r of A, row 16 j + 4 g + e of B
  uint32_t rd[2][2];  // LDS byte addresses of this lane's chunks: [operand][half], of the buffer being read
  int to_other;       // what takes rd to the other buffer
  uint32_t sa[2], sb[2];  // e4m3: scale bytes of the step's even and odd tiles

  // tile_lds: LDS byte address of the tiles; wm, wn: the wavefront's part of the 256x256 tile
  __device__ __forceinline__ void init(uint32_t tile_lds, int lane, int wm, int wn) {
    const int r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t at = (uint32_t)r * 128u + (uint32_t)((4 * h + g) ^ ((r >> 1) & 7)) * 16u;
      rd[0][h] = tile_lds + (uint32_t)wm * 16384u + at;
      rd[1][h] = tile_lds + 65536u + (uint32_t)wn * 16384u + at;
    }
    to_other = 32768;
  }
  __device__ __forceinline__ void other_buffer() {
#pragma unroll
    for (int op = 0; op < 2; ++op)
#pragma unroll
      for (int h = 0; h < 2; ++h) rd[op][h] += to_other;
    to_other = -to_other;
  }
  __device__ __forceinline__ u32x4 lds_read(uint32_t at) const {
    return *(__attribute__((address_space(3))) const u32x4*)(uintptr_t)at;
  }
  __device__ __forceinline__ static void set_half(u32x8& f, int h, u32x4 v) {
#pragma unroll
    for (int e = 0; e < 4; ++e) f[4 * h + e] = v[e];
  }
  __device__ __forceinline__ static u32x4 half(const u32x8& f, int h) {
    return h ? __builtin_shufflevector(f, f, 4, 5, 6, 7) : __builtin_shufflevector(f, f, 0, 1, 2, 3);
  }
  __device__ __forceinline__ void read_a(int i, int h) { set_half(fa[i], h, lds_read(rd[0][h] + i * 2048)); }
  __device__ __forceinline__ void read_b(int j, int h) { set_half(fb[j], h, lds_read(rd[1][h] + j * 2048)); }

  // In inline assembly, with the accumulator tied to an AGPR tuple: with 4-register accumulators of the builtin the register
  // allocator lets tiles trade places in the loop.  Nothing but LDS reads writes the operands, so that no wait state is due
  // before an MFMA; those between the last MFMA on an accumulator and its first other use are in settle().
  // FIRST: of a tile's first step, whose MFMAs start from zero instead of a zeroed accumulator (256 register writes a tile).
  template <int I, int J, int H, bool FIRST>
  __device__ __forceinline__ void mfma() {
    // e4m3: byte J / 2 of the even or odd tiles' scales of B, byte I / 2 of A's
#define NVF_MFMA16(name)                                                                                                          \
  if constexpr (FIRST && H == 0)                                                                                                  \
    asm volatile(name " %0, %1, %2, 0" : "=a"(acc[I][J]) : "v"(half(fb[J], H)), "v"(half(fa[I], H)));                             \
  else                                                                                                                            \
    asm volatile(name " %0, %1, %2, %0" : "+a"(acc[I][J]) : "v"(half(fb[J], H)), "v"(half(fa[I], H)))
#define NVF_MFMA8(c, constraint)                                                                                                  \
  asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, " c ", %3, %4 op_sel:[%5,%6,0] op_sel_hi:[%7,%8,0]"                 \
               : constraint(acc[I][J])                                                                                            \
               : "v"(fb[J]), "v"(fa[I]), "v"(sb[J & 1]), "v"(sa[I & 1]), "n"((J >> 1) & 1), "n"((I >> 1) & 1), "n"(J >> 2), "n"(I >> 2))
    if constexpr (MMA == Mma::kBf16) {
      NVF_MFMA16("v_mfma_f32_16x16x32_bf16");
    } else if constexpr (MMA == Mma::kF16) {
      NVF_MFMA16("v_mfma_f32_16x16x32_f16");
    } else if constexpr (FIRST) {
      NVF_MFMA8("0", "=a");
    } else {
      NVF_MFMA8("%0", "+a");
    }
#undef NVF_MFMA16
#undef NVF_MFMA8
  }

  __device__ __forceinline__ void pin() {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      asm volatile("" : "+a"(acc[i][0]), "+a"(acc[i][1]), "+a"(acc[i][2]), "+a"(acc[i][3]), "+a"(acc[i][4]), "+a"(acc[i][5]),
                   "+a"(acc[i][6]), "+a"(acc[i][7]));
  }
  // between the accumulators' last MFMA and their use (up to 12 wait states)
  __device__ __forceinline__ void settle() {
    pin();
    asm volatile("s_nop 15" ::: "memory");
  }
  // The fragments that the first step finds in registers (it reads B's last tile itself); the loads of its step have landed.
  __device__ __forceinline__ void first_fragments() {
    static_for<14>([&](auto u) { read_b(decltype(u)::value >> 1, decltype(u)::value & 1); });
    static_for<8>([&](auto u) { read_a(decltype(u)::value >> 1, decltype(u)::value & 1); });
  }

  // One step.  load(u): the load u of the step after the next (u < 12: rows of A's tiles 0..3 and of B; 12..15: A's tiles
  // 4..7; e4m3: 16, the scales, with the first ones); next_scales(part), part 0..3: read, combine and take over the next step's scales, in the second phase.
  // IN_FLIGHT: loads issued per step; FIRST: the first step of a tile.
  template <int IN_FLIGHT, bool FIRST, typename Load, typename Scales>
  __device__ __forceinline__ void step(Load load, Scales next_scales) {
    static_for<2>([&](auto phase_c) {
      constexpr int phase = decltype(phase_c)::value;
      static_for<8>([&](auto j_c) {
        constexpr int j = decltype(j_c)::value;
        static_for<8>([&](auto s_c) {
          constexpr int s = decltype(s_c)::value;
          if constexpr (phase == 0) {
            if constexpr (j == 0 && s < 2) read_b(7, s);
            // every wavefront has read A 0..3 and B of this step and its loads of this step's A 4..7 have landed
            if constexpr (j == 2 && s == 0) fence<IN_FLIGHT>();
            if constexpr (j >= 2 && j < 6 && (s & 3) == 1) read_a(4 + j - 2, s >> 2);
            if constexpr (MMA == Mma::kMxFp8 && j == 5 && s == 4) load(std::integral_constant<int, 16>{});
            if constexpr (j >= 2 && (s & 3) == 2) load(std::integral_constant<int, 2 * (j - 2) + (s >> 2)>{});
          } else {
            // ... has read A 4..7 of this step, and A 0..3 and B of the next have landed
            if constexpr (j == 0 && s == 0) {
              fence<IN_FLIGHT>();
              other_buffer();
            }
            if constexpr (j < 4 && (s & 3) == 1) read_a(j, s >> 2);
            if constexpr (j > 0 && (s & 3) == 3) read_b(j - 1, s >> 2);
            if constexpr (j >= 4 && s == 2) load(std::integral_constant<int, 12 + j - 4>{});
            if constexpr (s == 0 && (j & 1) == 1) next_scales(std::integral_constant<int, j / 2>{});
          }
          if constexpr (MMA != Mma::kMxFp8) mfma<4 * phase + (s & 3), j, (s >> 2), FIRST>();
          else if constexpr (s & 1) mfma<4 * phase + (s >> 1), j, 0, FIRST>();
          __builtin_amdgcn_sched_barrier(0);
        });
      });
    });
  }
  template <int IN_FLIGHT>
  __device__ __forceinline__ void fence() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(IN_FLIGHT) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
};

}  // namespace
}  // namespace nvf
