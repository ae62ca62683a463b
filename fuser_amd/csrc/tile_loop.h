// The K loop of the persistent kernels whose operands need no conversion (grouped_mm: bf16 / f16, mxfp8_scaled_mm): 4
// wavefronts as 2 x 2, each with 16 NI x 16 NJ of the workgroup's 32 NI x 32 NJ tile, operand rows of 128 bytes per step (64
// elements of 16 bits, 128 of e4m3).
//
// 16x16 MFMAs: on N(0,1) data the card's power limit, not the matrix pipe, sets the rate of a large product, and a 16x16 MFMA
// moves half the accumulator data per flop of a 32x32 one.  Register-only loops, PFLOP/s: bf16 32x32x16 1.81, 16x16x32 2.07;
// f16 1.68 / 1.93; e4m3 32x32x64 4.05, 16x16x128 4.36; on zeros both shapes 2.44 and 4.93.
//
// A step is two phases: the first half of a wavefront's tiles of A against all tiles of B, then the second half.  A wavefront
// holds one step's fragments and replaces them in place: A's second half of the step is read in its first phase, A's first
// half and B of the next step in its second, each B tile once its MFMAs have been issued.  What a phase has read out of LDS is
// refilled from the next barrier on: in the first phase of step s the rows of A's first half and of B of step s + NBUF, in the
// second those of A's second half, so that reads and loads share the LDS evenly (256x256: 8 reads and 12 loads, 24 reads and 4
// loads a wavefront; with all 16 loads in one half of a step that half was bound by LDS).  A load has at least NBUF - 1 whole
// steps to land: the waits are for all but the loads of the newest NBUF - 1 steps, never for all.
//
// LDS: NBUF tiles of A, then NBUF tiles of B; rows of 128 bytes, 16-byte chunk c of row r at position c ^ ((r >> 1) & 7): the
// fragment reads (16 consecutive rows, one chunk) are conflict-free.
#pragma once
#include "lds_direct.h"
#include "nvf_internal.h"

namespace nvf {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

enum class Mma { kBf16, kF16, kMxFp8 };

// what the functor that loads is asked for: 8 rows each
constexpr int kLoadB = 100;       // kLoadB + j, j < NJ: the wavefront's rows 8 j .. of its share of B's tile
constexpr int kLoadScales = 200;  // (e4m3) the step's scales; codes below 100, u < NI: rows of A (first half u < NI / 2)

template <Mma MMA, int NI, int NJ, int NBUF>
struct TileLoop {
  static constexpr int kABytes = NI * 4096, kBBytes = NJ * 4096;    // of a step's tiles
  static constexpr int kTileBytes = NBUF * (kABytes + kBBytes);    // LDS of the tiles
  static constexpr bool kFp8 = MMA == Mma::kMxFp8;
  static constexpr int kLoads = NI + NJ + (kFp8 ? 1 : 0);          // loads of a step and wavefront
  static constexpr int kInFlight = (NBUF - 1) * kLoads;
  static constexpr int kFenceGroup = NJ / 4;                       // the group of the first phase before which its barrier is
  static_assert(NI % 4 == 0 && NJ % 4 == 0 && kInFlight < 64, "");

  // per tile: lane (r, g) holds chunks g and 4 + g of row 16 * tile + r, the operand of one e4m3 MFMA or of two of 16 bits
  u32x8 fa[NI], fb[NJ];
  f32x4 acc[NI][NJ];  // [tile of A][tile of B], element e: row 16 i + r of A, row 16 j + 4 g + e of B
  uint32_t rd[2][2];  // LDS byte addresses of this lane's chunks: [operand][half], of the buffer being read
  int rd_buf;
  uint32_t sa[2], sb[2];  // e4m3: scale bytes of the step's even and odd tiles

  // tile_lds: LDS byte address of the tiles; wm, wn: the wavefront's part of the tile
  __device__ __forceinline__ void init(uint32_t tile_lds, int lane, int wm, int wn) {
    const int r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t at = (uint32_t)r * 128u + (uint32_t)((4 * h + g) ^ ((r >> 1) & 7)) * 16u;
      rd[0][h] = tile_lds + (uint32_t)wm * (kABytes / 2) + at;
      rd[1][h] = tile_lds + NBUF * kABytes + (uint32_t)wn * (kBBytes / 2) + at;
    }
    rd_buf = 0;
  }
  __device__ __forceinline__ void next_buffer() {
    const bool wrap = rd_buf == NBUF - 1;
    const int by = wrap ? 1 - NBUF : 1;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      rd[0][h] += by * kABytes;
      rd[1][h] += by * kBBytes;
    }
    rd_buf += by;
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
#ifdef __HIP_DEVICE_COMPILE__  // (the host's compiler does not know the constraints)
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
#endif
  }

  __device__ __forceinline__ void pin() {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; j += 4) asm volatile("" : "+a"(acc[i][j]), "+a"(acc[i][j + 1]), "+a"(acc[i][j + 2]), "+a"(acc[i][j + 3]));
  }
  // between the accumulators' last MFMA and their use (up to 12 wait states): the wait comes after the MFMAs, as volatile
  // statements keep their order, and the uses depend on the pin behind it
  __device__ __forceinline__ void settle() {
    asm volatile("s_nop 15" ::: "memory");
    pin();
  }
  // The fragments that the first step finds in registers (it reads B's last tile itself); the loads of its step have landed.
  __device__ __forceinline__ void first_fragments() {
    static_for<2 * NJ - 2>([&](auto u) { read_b(decltype(u)::value >> 1, decltype(u)::value & 1); });
    static_for<NI>([&](auto u) { read_a(decltype(u)::value >> 1, decltype(u)::value & 1); });
  }

  // f(i) for those of `N` pieces of work that fall to slot T of TOTAL
  template <int N, int T, int TOTAL, typename F>
  __device__ __forceinline__ static void share(F&& f) {
    if constexpr (T < TOTAL) {
      constexpr int first = T * N / TOTAL, count = (T + 1) * N / TOTAL - first;
      static_for<count>([&](auto u) { f(std::integral_constant<int, first + decltype(u)::value>{}); });
    }
  }

  // One step.  load(code): a load of step s + NBUF; next_scales(part), part 0..2: read, combine and take over the next step's
  // scales, in the second phase.  FIRST: the first step of a tile.  A group is a tile of B against half of A's.
  template <bool FIRST, typename Load, typename Scales>
  __device__ __forceinline__ void step(Load load, Scales next_scales) {
    constexpr int kSlots = NI / 2 * (kFp8 ? 1 : 2);  // MFMAs of a group
    static_for<2>([&](auto phase_c) {
      constexpr int phase = decltype(phase_c)::value;
      static_for<NJ>([&](auto j_c) {
        constexpr int j = decltype(j_c)::value;
        static_for<kSlots>([&](auto s_c) {
          constexpr int s = decltype(s_c)::value;
          if constexpr (phase == 0) {
            if constexpr (j == 0) share<2, s, kSlots>([&](auto h) { read_b(NJ - 1, decltype(h)::value); });
            // every wavefront has read A's first half and B of this step, and its loads of this step's second half have landed
            if constexpr (j == kFenceGroup && s == 0) fence();
            if constexpr (j >= kFenceGroup) {
              constexpr int t = (j - kFenceGroup) * kSlots + s, total = (NJ - kFenceGroup) * kSlots;
              // (read in the first two thirds: the next phase starts with them)
              share<NI, t, total * 2 / 3>([&](auto u) { read_a(NI / 2 + decltype(u)::value / 2, decltype(u)::value % 2); });
              share<NI / 2 + NJ + (kFp8 ? 1 : 0), t, total>([&](auto u) {
                constexpr int v = decltype(u)::value;
                load(std::integral_constant<int, v < NI / 2 ? v : v < NI / 2 + NJ ? kLoadB + v - NI / 2 : kLoadScales>{});
              });
            }
          } else {
            // ... has read A's second half of this step, and A's first half and B of the next have landed
            if constexpr (j == 0 && s == 0) {
              fence();
              next_buffer();
            }
            constexpr int t = j * kSlots + s, total = NJ * kSlots;
            share<NI, t, total / 2>([&](auto u) { read_a(decltype(u)::value / 2, decltype(u)::value % 2); });
            if constexpr (j > 0) share<2, s, kSlots>([&](auto h) { read_b(j - 1, decltype(h)::value); });
            if constexpr (t >= total / 2) share<NI / 2, t - total / 2, total / 2>([&](auto u) { load(std::integral_constant<int, NI / 2 + decltype(u)::value>{}); });
            if constexpr (kFp8) {
              if constexpr (t == total / 8) next_scales(std::integral_constant<int, 0>{});
              if constexpr (t == total / 2) next_scales(std::integral_constant<int, 1>{});
              if constexpr (t == total * 3 / 4) next_scales(std::integral_constant<int, 2>{});
            }
          }
          mfma<NI / 2 * phase + s % (NI / 2), j, s / (NI / 2), FIRST>();
          __builtin_amdgcn_sched_barrier(0);
        });
      });
    });
  }
  __device__ __forceinline__ void fence() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kInFlight) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
};

}  // namespace
}  // namespace nvf
