// Grouped NVFP4 GEMM, the groups of 1..32 rows (a decode step, the small experts of a prefill), whose experts' weights are
// read once; in small calls also larger ones, in slabs of 32 rows that each read them.
//   nvfp4_scaled_grouped_mm   (cutlass/nvfp4_scaled_group_mm.cu:714-788, pointer rule :83-155)
//
// Bound by the weight stream, so the kernel is built around keeping it going:
//   * One persistent workgroup per compute unit walks work items - a slab of up to 32 rows of a group against RH x 64
//     weight rows - whose list it derives from problem_sizes.  A wavefront's next loads, those of the next item when the
//     current one has no more, are under way while it converts and multiplies: the memory pipe does not drain at an item's
//     end, as it did with a workgroup per item (first loads, 7 chunks, sums, gone).
//   * A wavefront's step is 256 deep in K: 128 bytes of a weight row, a whole cache line.  Weights that the last-level
//     cache cannot hold are read with non-temporal loads: 64 experts of 7168 x 7168, 2 rows each 288 us (6.4 TB/s), with
//     plain ones 315; 256 of 7168 x 2048 361 / 373.  Where rows do not start on a line (K % 256 != 0) a non-temporal stream
//     fetches lines twice, and plain loads are used: 256 experts of 7168 x 2688 542 us, with non-temporal ones 575.
//   * The wavefronts of a half (RH = 2: four) split K and their partial sums are added in order through LDS.
//     RH = 2 halves the number of sums and barriers per byte and lets both halves read one scale tile (128 weight rows):
//     256 experts of 7168 x 2048, 512 rows with Zipf loads 187 us against 220, of 4096 x 4096 202 / 221, of 2048 x 7168
//     equal.  RH = 1 splits the work finer where there is little of it; there the two items that share a scale tile run at
//     the same time on one XCD, whose L2 then reads it once.
//   * 256 experts, 512 rows with Zipf loads (134 active): N = 2048, K = 7168 232 -> 202 us (6.0 TB/s on the small groups),
//     N = 4096, K = 2048 160 -> 112 us.
// LDS of a wavefront: the weight tile of its step (64 rows of 128 bytes, piece c of row r at position c ^ ((r >> 1) & 7)),
// the activation rows' (32 x 128 bytes, same order) and both operands' scales; loads are LDS-direct, a wavefront reads
// only what it loaded itself.  Fragments and MFMAs as in the weight-streaming kernel: lane (r, g) holds piece g of row r,
// 32 elements, and feeds v_mfma_f32_16x16x32_f16 with 8 of them per step; weight rows are the first operand.
#include <algorithm>

#include "gemm16_device.h"

namespace nvf {
namespace {

constexpr int kWaves = 8;
constexpr int kSlabRows = 32;
constexpr int kMaxEntries = 1024 + 32;  // (group, slab) pairs: every group has one, or 1024 rows in all
constexpr int kWeightBytes = 64 * 128, kRowBytes = kSlabRows * 128, kWeightScaleBytes = 4 * 512, kRowScaleBytes = 4 * 128;
constexpr int kSlotBytes = kWeightBytes + kRowBytes + kWeightScaleBytes + kRowScaleBytes;
constexpr int kSumBytes = kWaves * 4 * 1024;  // one partial 16x16 tile per weight tile, wavefront
constexpr int kLdsBytes = kWaves * kSlotBytes + kSumBytes + kMaxEntries * 8;
static_assert(kLdsBytes <= 160 * 1024, "LDS");

struct DecodeParams {
  const uint8_t *a, *b, *sfa, *sfb;
  const float* alpha;
  uint16_t* out;
  const int32_t *problem_sizes, *expert_offsets, *sf_offsets;
  int groups, n, k;
  int rows_small, rows_large;  // groups of up to rows_small rows and those of rows_large or more are this launch's
};

template <bool OUT_BF16, bool STREAM, int RH>
__global__ __launch_bounds__(kWaves * 64, 2) void persistent_nvfp4_skinny_ring_kernel(const DecodeParams p) {
  extern __shared__ u32x4 lds[];
  char* const lds_bytes = reinterpret_cast<char*>(lds);
  f32x4* const sums = reinterpret_cast<f32x4*>(lds_bytes + kWaves * kSlotBytes);
  u32x2* const entries = reinterpret_cast<u32x2*>(lds_bytes + kWaves * kSlotBytes + kSumBytes);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int kbytes = p.k >> 1;
  const int sf_padded = ((p.k >> 4) + 3) & ~3;
  const int steps = (p.k + 255) >> 8;
  const int tail_pieces = (p.k & 255) >> 5;  // 32-element pieces of a row in a short last step (0: it is whole)

  // ---- the list of (group, slab) pairs: {first row, rows | slab << 6 | group << 16}
  int entry_count;
  {
    int* const wave_total = reinterpret_cast<int*>(lds);
    int before = 0;
    for (int base = 0; base < p.groups; base += kWaves * 64) {
      const int gi = base + tid;
      const int m_g = gi < p.groups ? max(p.problem_sizes[gi * 3], 0) : 0;
      const int slabs = m_g <= p.rows_small || m_g >= p.rows_large ? (m_g + kSlabRows - 1) / kSlabRows : 0;
      int incl = slabs;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(incl, d, 64);
        if (lane >= d) incl += o;
      }
      if (lane == 63) wave_total[wave] = incl;
      __syncthreads();
      int at = before + incl - slabs;
      for (int w = 0; w < kWaves; ++w) {
        if (w < wave) at += wave_total[w];
        before += wave_total[w];
      }
      __syncthreads();
      if (slabs > 0) {
        const uint32_t row0 = (uint32_t)p.expert_offsets[gi];
        for (int s = 0; s < slabs && at + s < kMaxEntries; ++s)
          entries[at + s] = u32x2{row0 + s * kSlabRows, (uint32_t)min(m_g - s * kSlabRows, kSlabRows) | (uint32_t)s << 6 | (uint32_t)gi << 16};
      }
    }
    entry_count = __builtin_amdgcn_readfirstlane(min(before, kMaxEntries));
    __syncthreads();
  }
  constexpr int KS = kWaves / RH;  // wavefronts that split K
  const int half = wave / KS, kpart = wave % KS;
  const int blocks = p.n / (64 * RH);
  const int total = entry_count * blocks;

  struct Item {
    const uint8_t *a, *b, *sfa, *sfb;
    int rows, row0, n0;
    float alpha;
  };
  auto item_info = [&](int t) {
    // 16 consecutive items go to 16 consecutive workgroups, i.e. to XCDs 0..7 twice; the two on one XCD are neighbours
    if constexpr (RH == 1) {
      const int j = t & 15;
      if ((t | 15) < total) t = (t & ~15) + 2 * (j & 7) + (j >> 3);
    }
    const int e = t / blocks, block = t - e * blocks;
    const u32x2 v = entries[e];
    Item it;
    it.row0 = __builtin_amdgcn_readfirstlane((int)v[0]);
    const int packed = __builtin_amdgcn_readfirstlane((int)v[1]);
    const int group = packed >> 16;
    const int sf_row = p.sf_offsets[group] + ((packed >> 6) & 1023) * kSlabRows;
    it.alpha = p.alpha[group];
    it.rows = packed & 63;
    it.n0 = __builtin_amdgcn_readfirstlane(block * (64 * RH) + half * 64);
    const int64_t b_row0 = (int64_t)group * p.n;
    it.a = p.a + (int64_t)it.row0 * kbytes;
    it.b = p.b + (b_row0 + it.n0) * kbytes;
    it.sfa = p.sfa + (int64_t)(sf_row & ~127) * sf_padded + ((sf_row >> 5) & 3) * 4;
    it.sfb = p.sfb + (b_row0 + (it.n0 & ~127)) * sf_padded;
    return it;
  };

  // ---- load side: lane L fetches row L/8 of 8, piece (L%8) ^ ((row >> 1) & 7)
  const uint32_t lds_base = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)lds);
  const uint32_t slot = lds_base + (uint32_t)wave * kSlotBytes;
  const uint32_t piece_even = (uint32_t)((lane & 7) ^ (lane >> 4));  // 8-row blocks 0, 2, ..; the odd ones: ^ 4
  const uint32_t lrow = (uint32_t)(lane >> 3);
  auto issue = [&](const Item& it, int c) {
    uint32_t pe = piece_even, po = piece_even ^ 4u;
    uint32_t tile[2] = {(uint32_t)(lane >> 5), 2u + (uint32_t)(lane >> 5)};  // scale column tiles (64 elements of K)
    if (tail_pieces != 0 && c == steps - 1) {
      // a row's bytes and scale tiles past K do not exist: those lanes fetch its first ones again, unused
      if (pe >= (uint32_t)tail_pieces) pe = 0;
      if (po >= (uint32_t)tail_pieces) po = 0;
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (tile[j] * 2 >= (uint32_t)tail_pieces) tile[j] = 0;
    }
    int rows8 = kbytes * 8;

    const uint8_t* b = it.b + (int64_t)c * 128;
    const uint32_t ve = lrow * (uint32_t)kbytes + pe * 16u, vo = lrow * (uint32_t)kbytes + po * 16u;
    lds_dma16<0, STREAM>(slot, b, ve);
    lds_dma16<1024, STREAM>(slot, b += rows8, vo);
    lds_dma16<2048, STREAM>(slot, b += rows8, ve);
    lds_dma16<3072, STREAM>(slot, b += rows8, vo);
    lds_dma16<4096, STREAM>(slot, b += rows8, ve);
    lds_dma16<5120, STREAM>(slot, b += rows8, vo);
    lds_dma16<6144, STREAM>(slot, b += rows8, ve);
    lds_dma16<7168, STREAM>(slot, b += rows8, vo);
    const uint8_t* a = it.a + (int64_t)c * 128;
    auto a_off = [&](uint32_t first) { return __umul24(min(lrow + first, (uint32_t)(it.rows - 1)), (uint32_t)kbytes); };
    lds_dma16<kWeightBytes>(slot, a, a_off(0) + pe * 16u);
    lds_dma16<kWeightBytes + 1024>(slot, a, a_off(8) + po * 16u);
    if (it.rows > 16) {
      lds_dma16<kWeightBytes + 2048>(slot, a, a_off(16) + pe * 16u);
      lds_dma16<kWeightBytes + 3072>(slot, a, a_off(24) + po * 16u);
    }
    const uint8_t* sb = it.sfb + (int64_t)c * 2048;
    const uint8_t* sa = it.sfa + (int64_t)c * 2048;
    const uint32_t off0 = tile[0] * 512u + (uint32_t)(lane & 31) * 16u, off1 = tile[1] * 512u + (uint32_t)(lane & 31) * 16u;
    constexpr int kScales = kWeightBytes + kRowBytes;
    lds_dma16<kScales>(slot, sb, off0);
    lds_dma16<kScales + 1024>(slot, sb, off1);
    lds_dma4<kScales + kWeightScaleBytes>(slot, sa, off0);
    lds_dma4<kScales + kWeightScaleBytes + 256>(slot, sa, off1);
  };

  // ---- read side
  const char* const sp = lds_bytes + wave * kSlotBytes;
  const int swz = (r >> 1) & 7;
  const int rd_row = r * 128;
  const int sc_shift = (g & 1) * 16;

  if ((int)blockIdx.x >= total) return;
  const bool has_steps = kpart < steps;
  Item it = item_info(blockIdx.x);
  if (has_steps) issue(it, kpart);
  int turn = 0;
  const int half_of_two = wave >> 2;
  for (int t = blockIdx.x; t < total; t += gridDim.x, ++turn) {
    const bool more = t + (int)gridDim.x < total;
    const Item next = more ? item_info(t + gridDim.x) : it;
    auto run = [&](auto tiles_c) {
      constexpr int TILES = decltype(tiles_c)::value, ALL = 4 + TILES;  // row tiles of 16; all tiles of a step
      f32x4 acc[4][TILES];
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int tt = 0; tt < TILES; ++tt) acc[rt][tt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      for (int c = kpart; c < steps; c += KS) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        u32x4 q[2][ALL];
        uint32_t sc[2][ALL];
        const int word0 = (it.n0 & 64) ? 2 : 0;  // which of a piece's 4 scale words: 32-row group of the 128-row tile
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int pos = ((4 * h + g) ^ swz) * 16;
#pragma unroll
          for (int rt = 0; rt < 4; ++rt) q[h][rt] = *reinterpret_cast<const u32x4*>(sp + rt * 2048 + rd_row + pos);
#pragma unroll
          for (int tt = 0; tt < TILES; ++tt) q[h][4 + tt] = *reinterpret_cast<const u32x4*>(sp + kWeightBytes + tt * 2048 + rd_row + pos);
          const char* wsc = sp + kWeightBytes + kRowBytes + (2 * h + (g >> 1)) * 512 + r * 16;
#pragma unroll
          for (int rt = 0; rt < 4; ++rt)
            sc[h][rt] = *reinterpret_cast<const uint32_t*>(wsc + (rt & 1) * 256 + (word0 + (rt >> 1)) * 4) >> sc_shift;
          const char* asc = sp + kWeightBytes + kRowBytes + kWeightScaleBytes + (2 * h + (g >> 1)) * 128 + r * 4;
#pragma unroll
          for (int tt = 0; tt < TILES; ++tt) sc[h][4 + tt] = *reinterpret_cast<const uint32_t*>(asc + tt * 64) >> sc_shift;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read out: may be refilled
        {
          const bool same = c + KS < steps;
          if (same || more) {
            Item to;
            to.a = same ? it.a : next.a;
            to.b = same ? it.b : next.b;
            to.sfa = same ? it.sfa : next.sfa;
            to.sfb = same ? it.sfb : next.sfb;
            to.rows = same ? it.rows : next.rows;
            issue(to, same ? c + KS : kpart);
          }
        }
        if (tail_pieces != 0 && c == steps - 1) {
          // zero scales make the blocks past K count as zero, whatever was fetched for them
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const uint32_t keep = 4 * h + g < tail_pieces ? 0xffffffffu : 0u;
#pragma unroll
            for (int i = 0; i < ALL; ++i) sc[h][i] &= keep;
          }
        }
        // Eight MFMA steps (32 elements of K): the operands of the next one - a dword of every tile - are converted
        // between the MFMAs of the current one.
        f16x2 sv[2][ALL][2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < ALL; ++i) scale_pairs(sc[h][i], sv[h][i]);
        u32x4 f[2][ALL];
        auto convert = [&](int step, int i) {
          const int h = step >> 2, w = step & 3;
          f[step & 1][i] = dequant_dword(q[h][i][w], sv[h][i][w >> 1]);
        };
#pragma unroll
        for (int i = 0; i < ALL; ++i) convert(0, i);
#pragma unroll
        for (int step = 0; step < 8; ++step) {
#pragma unroll
          for (int rt = 0; rt < 4; ++rt) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int tt = 0; tt < TILES; ++tt)
              acc[rt][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, f[step & 1][rt]), __builtin_bit_cast(f16x8, f[step & 1][4 + tt]),
                                                                   acc[rt][tt], 0, 0, 0);
            if (step < 7) {
#pragma unroll
              for (int i = rt * ALL / 4; i < (rt + 1) * ALL / 4; ++i) convert(step + 1, i);
            }
          }
        }
      }
      // ---- the wavefronts' partial tiles, one row tile at a time, summed by alternate halves of the workgroup
      // (those of the first wavefronts also where K = 0 leaves no steps: the result is then zero)
      const int parts = max(min(steps, KS), 1);
#pragma unroll
      for (int tt = 0; tt < TILES; ++tt) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();  // the previous tile has been summed
        asm volatile("" ::: "memory");
        if (kpart < parts) {
#pragma unroll
          for (int rt = 0; rt < 4; ++rt) sums[(wave * 4 + rt) * 64 + lane] = acc[rt][tt];
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (RH == 2 || half_of_two == ((turn + tt) & 1)) {
          const int rt = wave & 3;
          const f32x4* part = sums + half * KS * 256 + rt * 64 + lane;
          f32x4 s = part[0];
          for (int w = 1; w < parts; ++w) s += part[w * 256];
          const int tok = tt * 16 + r;
          if (tok < it.rows) {
            u32x2 v;
            v[0] = pack2(s[0] * it.alpha, s[1] * it.alpha, OUT_BF16);
            v[1] = pack2(s[2] * it.alpha, s[3] * it.alpha, OUT_BF16);
            *reinterpret_cast<u32x2*>(p.out + (int64_t)(it.row0 + tok) * p.n + it.n0 + rt * 16 + 4 * g) = v;
          }
        }
      }
    };
    if (it.rows > 16) run(std::integral_constant<int, 2>{});
    else run(std::integral_constant<int, 1>{});
    it = next;
  }
}

template <bool OUT_BF16, bool STREAM, int RH>
int launch_decode(const DecodeParams& p, int grid, hipStream_t stream) {
  auto kern = persistent_nvfp4_skinny_ring_kernel<OUT_BF16, STREAM, RH>;
  const char* const rows = p.rows_small == 0 ? "129.." : p.rows_large < INT32_MAX ? "1..32,129.." : "1..32";
  const char* const mid = p.rows_small > kSlabRows ? "mid_groups=1," : "";  // and those in between
  if (note_launch("persistent_nvfp4_skinny_ring_kernel<%sstream=%d,halves=%d> grid=%d rows=%s", mid, (int)STREAM, RH, grid, rows))
    return NVF_OK;
  static std::atomic<uint64_t> configured{0};  // one bit per device
  if (const int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), kLdsBytes, configured)) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(kWaves * 64), kLdsBytes, stream, p);
  return check_launch("persistent_nvfp4_skinny_ring_kernel");
}

}  // namespace

int launch_nvfp4_decode(const Gemm16Args& a, int rows_small, bool large_groups, hipStream_t stream) {
  DecodeParams p;
  p.a = static_cast<const uint8_t*>(a.a);
  p.b = static_cast<const uint8_t*>(a.b);
  p.sfa = static_cast<const uint8_t*>(a.sfa);
  p.sfb = static_cast<const uint8_t*>(a.sfb);
  p.alpha = a.alpha;
  p.out = static_cast<uint16_t*>(a.out);
  p.problem_sizes = a.problem_sizes;
  p.expert_offsets = a.expert_offsets;
  p.sf_offsets = a.sf_offsets;
  p.groups = a.groups;
  p.n = (int)a.n;
  p.k = (int)a.k;
  p.rows_small = rows_small;
  p.rows_large = large_groups ? 129 : INT32_MAX;
  const int cus = cu_count();
  const int64_t slabs = a.groups + (rows_small > kSlabRows || large_groups ? a.m / kSlabRows : 0);  // at most
  // two halves of 64 weight rows per workgroup, unless such items cannot fill the compute units
  const bool halves = rows_small != 0 && std::min<int64_t>(a.groups, a.m) * (a.n / 128) >= 4 * (int64_t)cus;
  const int grid = (int)std::min<int64_t>(std::max(cus & ~15, 16), round_up(slabs * (a.n / (halves ? 128 : 64)), 16));
  // weights beyond what the 256 MB last-level cache holds are read past it
  const bool stream_weights = (a.k & 255) == 0 && (double)a.groups * (double)a.n * (double)a.k * (9.0 / 16) > (double)(256 << 20);
  auto launch = [&](auto out_bf16, auto streams) {
    constexpr bool kBf16 = decltype(out_bf16)::value, kStream = decltype(streams)::value;
    return halves ? launch_decode<kBf16, kStream, 2>(p, grid, stream) : launch_decode<kBf16, kStream, 1>(p, grid, stream);
  };
  if (a.dtype == NVF_BF16) return stream_weights ? launch(std::true_type{}, std::true_type{}) : launch(std::true_type{}, std::false_type{});
  return stream_weights ? launch(std::false_type{}, std::true_type{}) : launch(std::false_type{}, std::false_type{});
}

}  // namespace nvf
