// Persistent 256x256 / 128x256 NVFP4 kernel, for gfx950:
//   * nvfp4_scaled_mm          (cutlass/nvfp4_scaled_mm.cu:283-312), its block-scaled form (nvfp4_scaled_mm_blockscale.cu:332-373)
//   * nvfp4_scaled_grouped_mm  (cutlass/nvfp4_scaled_group_mm.cu:714-788, pointer rule :83-155)
// N % 256 == 0, K % 128 == 0 (16-bit results: K % 32 == 0, with a short last step), K >= 256.  Dense: any M, the last row tile
// may hold fewer rows; grouped: the tiles of the launch's groups.
//
// e2m1 x e4m3 is exact in fp16: both operands are converted and multiplied by v_mfma_f32_16x16x32_f16.  The 8 wavefronts of a
// workgroup own 32 columns of the result (weight rows) each, for all rows of the tile:
//   * a weight row is converted once per workgroup, by the wavefront that multiplies it, in registers: it never passes through
//     LDS as fp16.  (Before, wavefronts were 2 x 4 and both operands were staged: LDS writes, which take 13 cycles per KiB and
//     compute unit where reads take 4.5, of all 512 rows of a 256x256 step instead of 256, and of 384 of a 128x256 one instead of 128.)
//   * the activation rows are converted once per workgroup too, 16 NT rows by each wavefront, and go through LDS as fp16 MFMA
//     operands in lane order, [row tile][MFMA step][lane], so that stores and reads are linear.
//   * raw data travels global -> LDS by LDS-direct loads into slots of 128 of K that only the wavefront that loaded them reads;
//     it is in registers long before its slot is refilled, and the stream runs on across tile borders.
//   * two wavefronts per SIMD: one alone cannot issue the conversions, LDS accesses and MFMAs in time (per 4 MFMAs with 8 VALU
//     instructions, a read and a wait 39 ns, two wavefronts 31, MFMAs alone 28).
// A step (128 of K) is two halves of two MFMA steps each.  In a half, dealt out between its MFMAs: the activation operands of
// the next half are converted and stored, the weight operands of the next MFMA step converted, in the second half the next
// step's raw data read out and the slot refilled.  One barrier per half; the operands of the 4 row tiles behind it are in
// registers by then, and none is read in the 3 row tiles in front of it, so that the wait there finds nothing outstanding.
//
// A lane's 16 payload bytes of a row are 32 elements of K and feed four MFMA steps; A and B permute K alike.
//
// Bound by the card's power limit on full chips (8192^3: 693 us on N(0,1) data, 560 on zeros; with the staged operands 726 and
// 634), by instruction issue next to the MFMAs on small ones.  2048 x 14336 x 4096 175.6 -> 165.6 us, 512 x 14336 x 4096 56.1 ->
// 49.3.
#include "gemm16_device.h"
#include "nvf_internal.h"

#include <algorithm>

namespace nvf {
namespace {

constexpr int W = 8, NJ = 2, BR = 16 * NJ;  // wavefronts; 16-row tiles of B of each, their rows

template <int NI, int SLOTS>
struct PersistentLds {
  static constexpr int NT = NI / W;  // row tiles of A that a wavefront converts
  // a slot: 128 of K of a wavefront's data - B's rows of 64 bytes, their scales (dwords [column tile][row]), A's rows, theirs
  static constexpr int kBScales = NJ * 1024, kA = kBScales + 256, kAScales = kA + NT * 1024;
  static constexpr int kSlot = kAScales + 256;
  static constexpr int kHalf = W * NT * 2048;  // a half step's operands of A: [tile][2 MFMA steps][lane]
  static constexpr int kRaw = 2 * kHalf;
  static constexpr int kBytes = kRaw + W * SLOTS * kSlot;
};

// TM: 64-row blocks of a tile: 4 -> 256x256, 2 -> 128x256.
// RAGGED_K: K % 128 = 32, 64 or 96.  In a tile's last step the lanes whose elements lie past K fetch their row's first ones and
// take zero scales, and a zero scale makes a block count as zero.
template <Nvfp4Out OUT, bool GROUPED, int TM, bool RAGGED_K>
__global__ __launch_bounds__(64 * W, 2) void nvfp4_gemm_256_kernel(const Params p) {
  constexpr int NI = 4 * TM, SLOTS = TM == 4 ? 2 : 4;
  using L = PersistentLds<NI, SLOTS>;
  constexpr int NT = L::NT;
  constexpr int BM = 16 * NI, BN = W * BR;
  constexpr int AHEAD = 4;  // groups of NJ MFMAs behind a half step's barrier, whose operands of A are in registers by then
  constexpr int GAP = 3;    // groups in front of it in which no operand is read any more
  extern __shared__ u32x4 lds[];
  __shared__ int tile_prefix[GROUPED ? kMaxGroups + 1 : 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g4 = lane >> 4;

  // ---- persistent tile walk: workgroup ids are dealt round-robin to the 8 XCDs, XCD x owns the tile range
  // [x * chunk, (x + 1) * chunk); with the 8 (m) x 4 (n) blocked numbering the 32 tiles an XCD works on at a time share 8 A
  // panels and 4 B panels in its L2.
  // GROUPED: the 256-row tiles of every group that rows_in_256_tiles() names, the whole ones and a last one of more than 128
  // rows; what is left at the end of a group goes to other launches.  With 128-row tiles (TM == 2) the list is instead one tile
  // per weight panel for every group of rows_lo..rows_hi (<= 128) rows and, if min_rows is set, for the end (what
  // rows_in_256_tiles() leaves) of every group of at least min_rows rows.
  const int tiles_m = (p.m + BM - 1) / BM, tiles_n = p.n / BN;
  int total = tiles_m * tiles_n;
  if constexpr (GROUPED) {
    if (wave == 0) {  // prefix sums of tiles per group, 64 groups per round
      int running = 0;
      for (int base = 0; base < p.groups; base += 64) {
        const int g = base + lane;
        int cnt = 0;
        if (g < p.groups) {
          const int mg = p.problem_sizes[g * 3];
          if constexpr (TM == 4) cnt = (rows_in_256_tiles(mg) / BM) * tiles_n;
          else  // one 128-row tile per weight panel: a group of the class, or (min_rows set) the end of a larger group
            cnt = ((mg >= p.rows_lo && mg <= p.rows_hi) || (p.min_rows && mg >= p.min_rows && mg > rows_in_256_tiles(mg))) ? tiles_n : 0;
        }
        int incl = cnt;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          const int o = __shfl_up(incl, d, 64);
          if (lane >= d) incl += o;
        }
        if (g < p.groups) tile_prefix[g + 1] = running + incl;
        running += __shfl(incl, 63, 64);
      }
      if (lane == 0) tile_prefix[0] = 0;
    }
    __syncthreads();
    total = __builtin_amdgcn_readfirstlane(tile_prefix[p.groups]);
  }
  const int chunk_tiles = (total + 7) >> 3;
  const int xcd = blockIdx.x & 7, slot_id = blockIdx.x >> 3, slots = gridDim.x >> 3;
  const int range_end = min((xcd + 1) * chunk_tiles, total);
  const bool blocked = (tiles_m & 7) == 0 && tiles_n >= 4;
  const int bulk_tiles = tiles_m * (tiles_n & ~3);
  // (n-tiles past the last multiple of 4: blocks of 8 (m) x 1..3 (n) after all the others)
  // tile -> group, first row of the tile among all rows of A (m0), among the rows of the group (gm0), n0, rows that exist
  struct Where { int g; int64_t m0; int gm0, n0, valid; };
  auto tile_where = [&](int t) {
    Where w;
    if constexpr (GROUPED) {
      int lo = 0, hi = p.groups;
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (t < tile_prefix[mid]) hi = mid; else lo = mid;
      }
      w.g = __builtin_amdgcn_readfirstlane(lo);
      const int m_g = __builtin_amdgcn_readfirstlane(p.problem_sizes[w.g * 3]);
      const int64_t row_off = __builtin_amdgcn_readfirstlane(p.expert_offsets[w.g]);
      const int full_m = TM == 4 ? rows_in_256_tiles(m_g) / BM : 1;
      const int local = __builtin_amdgcn_readfirstlane(t - tile_prefix[w.g]);
      // bands of 4 m-tiles, n-major inside a band: 32 consecutive tiles share 4 A and 8 B panels
      const int band = local / (4 * tiles_n), in_band = local - band * 4 * tiles_n;
      const int band_h = min(4, full_m - 4 * band);
      const int nt = in_band / band_h, mt = 4 * band + (in_band - nt * band_h);
      w.gm0 = TM == 4 ? mt * BM : (m_g <= BM ? 0 : rows_in_256_tiles(m_g));
      w.m0 = row_off + w.gm0;
      w.n0 = nt * BN;
      w.valid = min(BM, m_g - w.gm0);
    } else {
      int mt, nt;
      if (blocked && t < bulk_tiles) {
        const int sb = t >> 5, q = t & 31;
        mt = (sb % (tiles_m >> 3)) * 8 + (q & 7);
        nt = (sb / (tiles_m >> 3)) * 4 + (q >> 3);
      } else if (blocked) {
        const int u = t - bulk_tiles, bs = 8 * (tiles_n & 3), sb = u / bs, q = u - sb * bs;
        mt = sb * 8 + (q & 7);
        nt = (tiles_n & ~3) + (q >> 3);
      } else {
        mt = t % tiles_m;
        nt = t / tiles_m;
      }
      w.g = 0;
      w.gm0 = mt * BM;
      w.m0 = w.gm0;
      w.n0 = nt * BN;
      w.valid = min(BM, p.m - w.gm0);
    }
    return w;
  };
  const int first_tile = xcd * chunk_tiles + slot_id;
  if (first_tile >= range_end) return;

  const int kbytes = p.k >> 1;
  const int nsteps = (p.k + 127) >> 7;
  const int sf_padded = ((p.k >> 4) + 3) & ~3;

  // ---- the stream of raw data.  A payload load: lane L fetches row L / 4, piece (L % 4) ^ ((L / 16) % 4) of 16 rows x 64
  // bytes.  A scale load: lane L fetches the 4 codes of row L % R, column tile (L / R) % 2 of the step.
  const int lrow = lane >> 2, lpiece = (lane & 3) ^ ((lane >> 4) & 3);
  constexpr int AR = 16 * NT;  // rows of A a wavefront converts
  uint32_t b_off[NJ], a_off[NT];
#pragma unroll
  for (int j = 0; j < NJ; ++j) b_off[j] = (uint32_t)(16 * j + lrow) * (uint32_t)kbytes + (uint32_t)lpiece * 16u;
  uint32_t sb_off = (uint32_t)(lane & 31) * 16u + (uint32_t)(lane >> 5) * 512u;
  uint32_t sa_off = (uint32_t)(lane & (AR - 1)) * 16u + (uint32_t)((lane / AR) & 1) * 512u;
  // a short last step: the lanes whose elements lie past K fetch their row's first piece, the scales of the first column tile
  const uint32_t tail_back = RAGGED_K && lpiece * 32 >= (p.k & 127) ? (uint32_t)lpiece * 16u : 0u;
  const bool one_sc_tile = (p.k & 127) <= 64;
  int st_tile = first_tile, st_step = 0;
  const uint8_t *st_a, *st_b, *st_sa, *st_sb;
  auto enter_tile = [&](int t) {
    const bool past = t >= range_end;
    const Where w = past ? Where{0, 0, 0, 0, 1} : tile_where(t);
    st_a = p.a + w.m0 * kbytes;
    const int64_t sa_slab = GROUPED && !past ? (int64_t)__builtin_amdgcn_readfirstlane(p.sf_offsets[w.g]) * sf_padded : 0;
    // (rows past the last one are fetched as copies of it, and scales of a row group past the last as its)
    const int a0 = min(w.gm0 + AR * wave, (w.gm0 + w.valid - 1) & ~(AR - 1));
    st_sa = p.sfa + sa_slab + swizzle_128x4(a0, 0, sf_padded);
    const int n_w = w.n0 + BR * wave;
    st_b = p.b + ((int64_t)w.g * p.n + n_w) * kbytes;
    st_sb = p.sfb + (int64_t)w.g * p.n * sf_padded + swizzle_128x4(n_w, 0, sf_padded);
#pragma unroll
    for (int t = 0; t < NT; ++t) a_off[t] = (uint32_t)min(AR * wave + 16 * t + lrow, w.valid - 1) * (uint32_t)kbytes + (uint32_t)lpiece * 16u;
  };
  enter_tile(first_tile);
  const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)lds);
  const uint32_t my_slots = lds0 + L::kRaw + (uint32_t)wave * (SLOTS * L::kSlot);
  int ld_slot = 0;  // byte offset of the slot that is loaded next
  constexpr int kLoads = NJ + NT + 2;
  auto load = [&](auto l_c) {
    constexpr int l = decltype(l_c)::value;
    const bool tail = RAGGED_K && st_step == nsteps - 1;
    const uint32_t at = my_slots + (uint32_t)ld_slot;
    if constexpr (l < NJ) lds_dma16<l * 1024>(at, st_b, tail ? b_off[l] - tail_back : b_off[l]);
    else if constexpr (l == NJ) lds_dma4<L::kBScales>(at, st_sb, tail && one_sc_tile ? sb_off & 511u : sb_off);
    else if constexpr (l <= NJ + NT) lds_dma16<L::kA + (l - NJ - 1) * 1024>(at, st_a, tail ? a_off[l - NJ - 1] - tail_back : a_off[l - NJ - 1]);
    else lds_dma4<L::kAScales>(at, st_sa, tail && one_sc_tile ? sa_off & 511u : sa_off);
  };
  auto advance_stream = [&]() {
    ld_slot = ld_slot == (SLOTS - 1) * L::kSlot ? 0 : ld_slot + L::kSlot;
    st_a += 64, st_b += 64, st_sa += 1024, st_sb += 1024;
    if (++st_step == nsteps) {
      st_step = 0;
      st_tile += slots;
      if (st_tile >= range_end) {
        // Past the last tile nobody reads what is loaded.  From here on every load is of one row's 64 bytes (its own piece by each
        // lane, so that tail_back stays inside the row) and one row's scales, of the first tile of all, which needs no look at the
        // list.  (All rows of the last tile's first steps again: 2048 x 4096 x 256 10.9 -> 10.4 us, x 512 14.0 -> 13.2; 16 groups of
        // 128 rows, N = 2048, K = 512 18.0 -> 16.6 a call.  In assembly: assigned, the offsets are copied at every step.)
#pragma unroll
        for (int j = 0; j < NJ; ++j) asm volatile("v_mov_b32 %0, %1" : "+v"(b_off[j]) : "v"((uint32_t)lpiece * 16u));
        asm volatile("v_mov_b32 %0, 0\n\tv_mov_b32 %1, 0" : "+v"(sa_off), "+v"(sb_off));
      }
      enter_tile(st_tile);
    }
  };

  // ---- LDS addresses of this lane
  auto lds_u32x4 = [](uint32_t at) { return *(__attribute__((address_space(3))) const u32x4*)(uintptr_t)at; };
  auto lds_u16 = [](uint32_t at) { return (uint32_t)*(__attribute__((address_space(3))) const uint16_t*)(uintptr_t)at; };
  const uint32_t rd_payload = my_slots + (uint32_t)(r * 64 + ((g4 ^ ((r >> 2) & 3)) * 16));
  const uint32_t rd_sb = my_slots + (uint32_t)(L::kBScales + ((g4 >> 1) * 32 + r) * 4 + (g4 & 1) * 2);
  const uint32_t rd_sa = my_slots + (uint32_t)(L::kAScales + ((g4 >> 1) * AR + r) * 4 + (g4 & 1) * 2);
  int rd_slot = 0;  // slot of the step that is read out
  const uint32_t frag = lds0 + (uint32_t)lane * 16u;

  f32x4 acc[NI][NJ];
  auto zero_acc = [&](auto ni_c) {
#pragma unroll
    for (int i = 0; i < decltype(ni_c)::value; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  };
  auto pin_acc = [&](auto ni_c) {
    f32x4(&c)[NI][NJ] = acc;
#pragma unroll
    for (int i = 0; i < decltype(ni_c)::value; i += 2) {
#pragma unroll
      for (int j = 0; j < NJ; j += 2) asm volatile("" : "+a"(c[i][j]), "+a"(c[i][j + 1]), "+a"(c[i + 1][j]), "+a"(c[i + 1][j + 1]));
    }
  };
  auto settle_acc = [&](auto ni_c) {
    pin_acc(ni_c);
    asm volatile("s_nop 15" ::: "memory");
    pin_acc(ni_c);
  };
  auto mfma16 = [&](f32x4& c, const u32x4& b, const u32x4& a) { asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(b), "v"(a)); };

  // ---- registers of the pipeline
  u32x4 fa[8];              // operands of A: group m of a step in fa[m & 7]
  u32x4 fb[2][NJ];          // operands of B: MFMA step w of a step in fb[w & 1]
  u32x4 qb[NJ], qa[NT];     // payload: a lane's 32 elements of a row
  uint32_t cb[NJ], ca[NT];  // their two scale codes
  f16x2 vb[NJ], va[NT];     // ... as fp16
  // one operand (dword w of the payload) in eight parts of one instruction; `out` holds the intermediate values
  auto convert_part = [&](u32x4& out, uint32_t q, f16x2 scales, int w, int part) {
    const _Float16 f = scales[w >> 1];
    const f16x2 s = {f, f};
    if (part == 0) out[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(q, 1.0f, 0));
    else if (part == 1) out[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(q, 1.0f, 1));
    else if (part == 2) out[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(q, 1.0f, 2));
    else if (part == 3) out[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(q, 1.0f, 3));
    else out[part - 4] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, (uint32_t)out[part - 4]) * s);
    if (part == 7) asm volatile("" : "+v"(out));  // here, and not in the block where it is used
  };
  const bool lane_in_tail = g4 * 32 < (p.k & 127);
  uint32_t live = ~0u;  // RAGGED_K: 0 in the lanes whose elements of the step being read out lie past K
  auto read_b = [&](int j) {
    qb[j] = lds_u32x4(rd_payload + rd_slot + j * 1024);
    cb[j] = lds_u16(rd_sb + rd_slot + j * 64);
  };
  auto read_a = [&](int t) {
    qa[t] = lds_u32x4(rd_payload + rd_slot + L::kA + t * 1024);
    ca[t] = lds_u16(rd_sa + rd_slot + t * 64);
  };
  auto scales = [&](uint32_t code) {  // exact: every e4m3 value is an fp16 value
    return __builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(RAGGED_K ? code & live : code, 1.0f, false));
  };
  auto write_a = [&](int buf, int t, int o, const u32x4& v) {
    *(__attribute__((address_space(3))) u32x4*)(uintptr_t)(frag + (uint32_t)((NT * wave + t) * 2048 + buf * L::kHalf + o * 1024)) = v;
  };
  auto load_frag = [&](int buf, int m, int i, int o) { fa[m & 7] = lds_u32x4(frag + (uint32_t)(buf * L::kHalf + i * 2048 + o * 1024)); };

  // ---- before the loop: the first SLOTS steps requested, step 0 read out, its first half's operands converted
  static_for<SLOTS>([&](auto) {
    static_for<kLoads>([&](auto l) { load(l); });
    advance_stream();
  });
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SLOTS - 1) * kLoads) : "memory");
  u32x4 conv;  // A's operand in progress
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    read_a(t);
    va[t] = scales(ca[t]);
#pragma unroll
    for (int o = 0; o < 2; ++o) {
#pragma unroll
      for (int q = 0; q < 8; ++q) convert_part(conv, qa[t][o], va[t], o, q);
      write_a(0, t, o, conv);
    }
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    read_b(j);
    vb[j] = scales(cb[j]);
#pragma unroll
    for (int q = 0; q < 8; ++q) convert_part(fb[0][j], qb[j][0], vb[j], 0, q);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  static_for<kLoads>([&](auto l) { load(l); });
  advance_stream();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int m = 0; m < AHEAD; ++m) load_frag(0, m, m, 0);

  // f(u) for those of N pieces of work that fall to slot T of [FROM, TO)
  auto share = [](auto n_c, auto t_c, auto from_c, auto to_c, auto f) {
    constexpr int n = decltype(n_c)::value, t = decltype(t_c)::value, from = decltype(from_c)::value, to = decltype(to_c)::value;
    if constexpr (t >= from && t < to) {
      constexpr int first = (t - from) * n / (to - from), count = (t - from + 1) * n / (to - from) - first;
      static_for<count>([&](auto u) { f(std::integral_constant<int, first + decltype(u)::value>{}); });
    }
  };
#define NVF_C(x) std::integral_constant<int, (x)>{}

  // Half a step: MFMA steps w = 2 h, 2 h + 1 of 32 of K, in groups of the NJ MFMAs of one row tile.
  auto half = [&](auto ni_c, auto h_c) {
    constexpr int NIC = decltype(ni_c)::value, h = decltype(h_c)::value;
    constexpr int TOTAL = 2 * NIC * NJ, BAR = (2 * NIC - AHEAD) * NJ;  // MFMAs of the half, before its barrier
    constexpr int A_GAP = NIC < 8 ? 2 : 4;
    constexpr int LAT = h == 0 ? 0 : NIC < 8 ? 2 : 5;  // MFMAs until the first use of what h = 1 reads out
    if constexpr (h == 1) {
      // the next step's raw data has landed
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SLOTS - 1) * kLoads) : "memory");
      rd_slot = rd_slot == (SLOTS - 1) * L::kSlot ? 0 : rd_slot + L::kSlot;
    }
    uint32_t q3[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) q3[j] = qb[j][3];
    static_for<2 * NIC>([&](auto m_c) {
      constexpr int m = decltype(m_c)::value, i = m % NIC, o = m / NIC;
      if constexpr (NJ * m == BAR) {
        // every wavefront has written its share of the next half step and holds this one's last operands in registers
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      __builtin_amdgcn_sched_barrier(0);
      static_for<NJ>([&](auto j_c) {
        constexpr int j = decltype(j_c)::value, s = NJ * m + j;
        if constexpr (j == 0) {
          // behind the barrier the next half step's first operands, in front of it this one's others
          if constexpr (NJ * m >= BAR) load_frag(h ^ 1, 2 * NIC * (h + 1) + m - BAR / NJ, m - BAR / NJ, 0);
          share(NVF_C(2 * NIC - AHEAD), NVF_C(m), NVF_C(0), NVF_C(2 * NIC - AHEAD - GAP), [&](auto u) {
            constexpr int n = AHEAD + decltype(u)::value;
            load_frag(h, 2 * NIC * h + n, n % NIC, n / NIC);
          });
        }
        if constexpr (h == 1) {
          share(NVF_C(NT), NVF_C(s), NVF_C(0), NVF_C(NT), [&](auto t) { read_a(decltype(t)::value); });
          share(NVF_C(NJ), NVF_C(s), NVF_C(NT), NVF_C(NT + NJ), [&](auto b) { read_b(decltype(b)::value); });
        }
        // B's operands of the next MFMA step: of w = 3 from what has been read before, of w = 0 from what is read now
        constexpr bool fresh = h == 1 && o == 1;
        share(NVF_C((fresh ? 9 : 8) * NJ), NVF_C(s), NVF_C(o ? TOTAL / 2 : 0), NVF_C(o ? TOTAL - 1 : TOTAL / 2 - 1), [&](auto u) {
          constexpr int v = decltype(u)::value, per = fresh ? 9 : 8, b = v / per, q = v % per - (fresh ? 1 : 0);
          if constexpr (q < 0) {
            vb[b] = scales(cb[b]);
            asm volatile("" : "+v"(vb[b]));
          } else {
            constexpr int w = (2 * h + o + 1) & 3;
            convert_part(fb[o ^ 1][b], w == 3 ? q3[b] : (uint32_t)qb[b][w], vb[b], w, q);
          }
        });
        // A's operands of the next half step: w = 2, 3 of this step or 0, 1 of the next
        share(NVF_C((16 + h) * NT), NVF_C(s), NVF_C(LAT), NVF_C(BAR - A_GAP), [&](auto u) {
          constexpr int v = decltype(u)::value, per = 16 + h, t = v / per, q = v % per - h;
          if constexpr (q < 0) {
            va[t] = scales(ca[t]);
            asm volatile("" : "+v"(va[t]));
          } else {
            constexpr int w = 2 * (h ^ 1) + q / 8;
            convert_part(conv, qa[t][w], va[t], w, q % 8);
            if constexpr (q % 8 == 7) write_a(h ^ 1, t, q / 8, conv);
          }
        });
        // the slot that has been read out takes the step SLOTS further on
        if constexpr (h == 1) {
          constexpr int FROM = TOTAL / 2;
          if constexpr (s == FROM) {
#pragma unroll
            for (int b = 0; b < NJ; ++b) asm volatile("" ::"v"(qb[b]), "v"(cb[b]));
#pragma unroll
            for (int t = 0; t < NT; ++t) asm volatile("" ::"v"(qa[t]), "v"(ca[t]));
          }
          share(NVF_C(kLoads), NVF_C(s), NVF_C(FROM), NVF_C(TOTAL), [&](auto l) { load(l); });
        }
        mfma16(acc[i][j], fb[o][j], fa[(2 * NIC * h + m) & 7]);
        __builtin_amdgcn_sched_barrier(0);
      });
    });
    if constexpr (h == 1) advance_stream();
  };

  for (int c_tile = first_tile; c_tile < range_end; c_tile += slots) {
    const Where cw = tile_where(c_tile);
    auto run = [&](auto ni_c) {
    constexpr int NIC = decltype(ni_c)::value;
    zero_acc(ni_c);
    settle_acc(ni_c);
    for (int step = 0; step < nsteps; ++step) {
      half(ni_c, NVF_C(0));
      if (RAGGED_K) live = step + 1 == nsteps - 1 && !lane_in_tail ? 0u : ~0u;
      half(ni_c, NVF_C(1));
    }
    settle_acc(ni_c);
    // ---- epilogue; the next tile's first half step is already in LDS.
    // acc[i][j][e] = C[m = 16 i + r][n = 16 j + 4 g4 + e] of the wavefront's columns.  Results are turned round in the
    // wavefront's own part of A's second half buffer, which it alone writes again, in the next tile's first half step.
    const float alpha = p.alpha[cw.g];
    const int n_w = cw.n0 + BR * wave;
    int elane = lane;
    asm volatile("" : "+v"(elane));  // (worked out here, after the K loop: no registers for these in it)
    uint8_t* const stage = reinterpret_cast<uint8_t*>(lds) + L::kHalf + NT * wave * 2048;
    if constexpr (OUT == Nvfp4Out::kF16 || OUT == Nvfp4Out::kBf16) {
      // 32 rows of 64 bytes at a time, 16-byte chunk c of row y at position c ^ ((y >> 1) & 3)
      const int erow = elane >> 2;
      uint8_t* const wr = stage + (elane & 15) * 64 + ((elane >> 4) & 1) * 8;
      const int wr_chunk = (elane >> 5) ^ ((elane >> 1) & 3);
      const uint8_t* const rd = stage + erow * 64 + ((elane & 3) ^ ((erow >> 1) & 3)) * 16;
      const int ldc = p.out_pitch();
      const uint32_t ooff = ((uint32_t)erow * (uint32_t)ldc + (uint32_t)(elane & 3) * 8u) * 2u;
      uint8_t* const obase = reinterpret_cast<uint8_t*>(static_cast<uint16_t*>(p.out) + cw.m0 * ldc + n_w);
#pragma unroll
      for (int i = 0; i < NIC; i += 2) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {  // the block's four 16x16 tiles
          const f32x4 c = acc[i + (t >> 1)][t & 1];
          u32x2 v;
          v[0] = pack2(c[0] * alpha, c[1] * alpha, OUT == Nvfp4Out::kBf16);
          v[1] = pack2(c[2] * alpha, c[3] * alpha, OUT == Nvfp4Out::kBf16);
          *reinterpret_cast<u32x2*>(wr + (t >> 1) * 1024 + (wr_chunk ^ (2 * (t & 1))) * 16) = v;
        }
        asm volatile("" ::: "memory");  // the reads below see the writes above: one wavefront's LDS accesses stay in order
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const u32x4 v = *reinterpret_cast<const u32x4*>(rd + t * 1024);
          if (16 * (i + t) + erow < cw.valid) *reinterpret_cast<u32x4*>(obase + (int64_t)(16 * (i + t)) * ldc * 2 + ooff) = v;
        }
        asm volatile("" ::: "memory");
      }
    } else if constexpr (OUT == Nvfp4Out::kF32) {
      // 16 rows of 128 bytes at a time, 16-byte chunk c of row y at position c ^ (y & 7), so that whole lines leave.  (Straight
      // from the accumulators, 16 rows' 16 bytes to 16 lanes: a block-scaled call with this dump 512 x 14336 x 4096 114.7 ->
      // 105.2 us, 8192 x 8192 x 256 123.6 -> 116.0.)
      uint8_t* const wr = stage + (elane & 15) * 128;
      const int wr_chunk = (elane >> 4) ^ (elane & 7);
      const int erow = elane >> 3;
      const uint8_t* const rd = stage + erow * 128 + ((elane & 7) ^ erow) * 16;
      const uint32_t ooff = ((uint32_t)erow * (uint32_t)p.n + (uint32_t)(elane & 7) * 4u) * 4u;
      uint8_t* const obase = reinterpret_cast<uint8_t*>(static_cast<float*>(p.out) + cw.m0 * p.n + n_w);
#pragma unroll
      for (int i = 0; i < NIC; ++i) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const f32x4 c = acc[i][j];
          *reinterpret_cast<f32x4*>(wr + (wr_chunk ^ (4 * j)) * 16) = f32x4{c[0] * alpha, c[1] * alpha, c[2] * alpha, c[3] * alpha};
        }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(rd + t * 1024);
          if (16 * i + 8 * t + erow < cw.valid) *reinterpret_cast<f32x4*>(obase + (int64_t)(16 * i + 8 * t) * p.n * 4 + ooff) = v;
        }
        asm volatile("" ::: "memory");
      }
    } else {
      // Block-scaled result.  All wavefronts' parts of the tile are collected in A's second half buffer, rows of 128 payload
      // bytes with 16-byte chunk c of row y at position c ^ (y & 7), and leave as whole rows; the codes behind the slots in the
      // order of the 128x4 layout, where a tile's are 2 KiB in a row for every 128 rows.  Lane (r, g4) works out the scale of row r
      // of block g4 & 1 of row tile g4 >> 1.  Rows past M: the padding rows of the last 128-row scale tile get code zero; a
      // 256-row tile with at most 128 rows has no second scale tile to write.  (Each wavefront its 16 bytes of 32 rows and their two
      // codes at a time, without the barriers: 2048 x 4096 x 256 10.6 -> 10.4 us, 8192 x 8192 x 256 52.6 -> 51.1, x 1024 116 -> 114.)
      const float gs = p.gnorm[0], decode = 1.0f / gs;
      const int er = elane & 15, eg = elane >> 4;
      uint8_t* const rows = reinterpret_cast<uint8_t*>(lds) + L::kHalf;
      uint8_t* const codes = reinterpret_cast<uint8_t*>(lds) + L::kBytes;
      uint8_t* const wr = rows + er * 128 + ((wave ^ (er & 7)) * 16) + eg * 2;
      uint8_t* const wc = codes + (wave >> 1) * 512 + er * 16 + (wave & 1) * 2 + (eg & 1);
#pragma unroll
      for (int i = 0; i < NIC; i += 2) {
        const f32x4 c[4] = {acc[i][0], acc[i][1], acc[i + 1][0], acc[i + 1][1]};
        uint32_t q8, h[4];
        quantize_acc_tiles16(c, alpha, gs, decode, q8, h);
#pragma unroll
        for (int t = 0; t < 4; ++t) *reinterpret_cast<uint16_t*>(wr + (i + (t >> 1)) * 2048 + (t & 1) * 8) = (uint16_t)h[t];
        const int row = 16 * (i + (eg >> 1));
        wc[(row >> 7) * 2048 + (row & 16) * 16 + ((row >> 5) & 3) * 4] = row + er < cw.valid ? (uint8_t)q8 : (uint8_t)0;
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const int erow = elane >> 3;
      const uint8_t* const rd = rows + erow * 128 + ((elane & 7) ^ erow) * 16;
      uint8_t* const obase = static_cast<uint8_t*>(p.out) + (cw.m0 + erow) * (p.n >> 1) + (cw.n0 >> 1) + (elane & 7) * 16;
#pragma unroll
      for (int t = 0; t < NIC / 4; ++t) {
        const int row = (wave * (NIC / 4) + t) * 8;
        if (row + erow < cw.valid) *reinterpret_cast<u32x4*>(obase + (int64_t)row * (p.n >> 1)) = *reinterpret_cast<const u32x4*>(rd + row * 128);
      }
      if (wave < NIC / 4 && (wave >> 1) * 128 < cw.valid)
        *reinterpret_cast<u32x4*>(p.out_sf + (((cw.m0 >> 7) + (wave >> 1)) * (p.n >> 6) + (cw.n0 >> 6)) * 512 + (wave & 1) * 1024 + elane * 16) =
            *reinterpret_cast<const u32x4*>(codes + wave * 1024 + elane * 16);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read out: the next tile's operands may be written
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    };
    // (a group's tile may hold few rows: the MFMAs of row tiles that do not exist are left out)
    if constexpr (GROUPED && TM == 2) {
      if (cw.valid <= 64) run(NVF_C(4));
      else if (cw.valid <= 96) run(NVF_C(6));
      else run(NVF_C(8));
    } else {
      run(NVF_C(NI));
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no LDS-direct load may outlive the workgroup
}
#undef NVF_C

template <Nvfp4Out OUT, bool GROUPED, int TM, bool RAGGED_K>
int launch_cfg(const Params& p, int cus, hipStream_t stream) {
  auto kern = nvfp4_gemm_256_kernel<OUT, GROUPED, TM, RAGGED_K>;
  constexpr int lds_bytes = PersistentLds<4 * TM, TM == 4 ? 2 : 4>::kBytes + (OUT == Nvfp4Out::kFp4 ? 1024 * TM : 0);  // (its scale codes: 16 bytes a row)
  static_assert(lds_bytes + (GROUPED ? (kMaxGroups + 1) * 4 : 4) <= 160 * 1024, "LDS");
  // grouped: an upper bound (128-row tiles: one per weight panel and group of at least rows_lo rows)
  const bool ragged_m = !GROUPED && p.m % (64 * TM) != 0;
  const int64_t tiles_m = (GROUPED && TM == 2) ? std::min<int64_t>(p.groups, p.m / std::max(p.rows_lo, 1)) : (p.m + (ragged_m ? 64 * TM - 1 : 0)) / (64 * TM);
  const int64_t tiles = tiles_m * (p.n / 256);
  const unsigned grid = (unsigned)(tiles >= cus ? (cus & ~7) : ((tiles + 7) / 8) * 8);
  if (grid == 0) return NVF_OK;  // fewer rows in the whole call than the smallest group this launch serves: no work
  if (note_launch("nvfp4_gemm_256_kernel<grouped=%d,TM=%d,f32=%d%s%s%s> grid=%u rows=%d..%d min_rows=%d", (int)GROUPED, TM,
                  (int)(OUT == Nvfp4Out::kF32), OUT == Nvfp4Out::kFp4 ? ",fp4_blockscale" : "", ragged_m ? ",ragged_m" : "",
                  RAGGED_K ? ",ragged_k" : "", grid, p.rows_lo, p.rows_hi, p.min_rows))
    return NVF_OK;
  static std::atomic<uint64_t> configured{0};  // one bit per device
  if (const int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds_bytes, configured)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * W), lds_bytes, stream, p);
  return check_launch("nvfp4_gemm_256_kernel");
}

template <Nvfp4Out OUT, bool GROUPED, int TM>
int launch_tiles(const Params& p, int cus, hipStream_t stream) {
  // (a short last step: 16-bit results; grouped: the 256x256 tiles)
  if constexpr ((OUT == Nvfp4Out::kF16 || OUT == Nvfp4Out::kBf16) && (!GROUPED || TM == 4)) {
    if ((p.k & 127) != 0) return launch_cfg<OUT, GROUPED, TM, true>(p, cus, stream);
  }
  return launch_cfg<OUT, GROUPED, TM, false>(p, cus, stream);
}

template <Nvfp4Out OUT, bool GROUPED>
int launch_out(const Params& p, int tm, int cus, hipStream_t stream) {
  return tm == 4 ? launch_tiles<OUT, GROUPED, 4>(p, cus, stream) : launch_tiles<OUT, GROUPED, 2>(p, cus, stream);
}

}  // namespace

int launch_nvfp4_persistent(const Params& p, Nvfp4Out out, bool grouped, int tm, int cus, hipStream_t stream) {
  switch (out) {
    case Nvfp4Out::kF16: return grouped ? launch_out<Nvfp4Out::kF16, true>(p, tm, cus, stream) : launch_out<Nvfp4Out::kF16, false>(p, tm, cus, stream);
    case Nvfp4Out::kBf16: return grouped ? launch_out<Nvfp4Out::kBf16, true>(p, tm, cus, stream) : launch_out<Nvfp4Out::kBf16, false>(p, tm, cus, stream);
    case Nvfp4Out::kF32: return launch_out<Nvfp4Out::kF32, false>(p, tm, cus, stream);
    case Nvfp4Out::kFp4: return launch_out<Nvfp4Out::kFp4, false>(p, tm, cus, stream);
  }
  return NVF_OK;
}

}  // namespace nvf
