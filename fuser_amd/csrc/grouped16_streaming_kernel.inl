// Persistent weight-streaming kernel for grouped_mm (16-bit operands) of gemm16.hip (included there, inside namespace nvf).
// -------------------------------------------------------------------------------------------------
// grouped_mm with few rows per group (a decode step, a chunk spread over many experts): bound by the weights' way out of
// HBM, which the 128x128 tile kernel - a workgroup barrier per 64-deep step, its pipe drained at every tile's end - drew at
// 4.4 TB/s: 128 rows over 8 experts of 14336 x 4096 213 -> 160 us (5.9 TB/s), 512 rows over 64 experts of 7168 x 2048 415 ->
// 295, 16 rows over 8 experts of 1024 x 4096 55 -> 20.
//   * One persistent workgroup per compute unit walks work items, a slab of up to 64 rows of a group against 16 WT weight
//     rows.  Its 8 wavefronts split K in 64-deep steps and run independently: a step's weights (one 128-byte line per row)
//     and activation rows arrive by LDS-direct loads in the wavefront's own part of LDS, go to registers whole, and the
//     next step's loads - the next item's, when this one has no more - are issued before the MFMAs.
//   * The slabs of a group that use the same weight rows are 8 items apart, on workgroups of one XCD: they run at the same
//     time and its L2 reads the weights once.
//   * The 8 partial sums are added in the order of K through two LDS buffers of one 16x16 tile per wavefront, one barrier a
//     tile: wavefront i sums tile i while the others write tile i + 1.
//   * Any N % 8 and K % 8: weight rows past N repeat the last one and are not stored; pieces of 8 elements past K repeat the
//     row's first one and are zeroed in registers, in both operands.
// LDS order as in the other kernels: 16-byte piece c of row r at position c ^ ((r >> 1) & 7).
// -------------------------------------------------------------------------------------------------
constexpr int kStream16Waves = 8, kStream16Rows = 64;
constexpr int kStream16SumBytes = 2 * kStream16Waves * 1024;
constexpr int stream16_slot_bytes(int wt) { return (16 * wt + kStream16Rows) * 128; }
constexpr int stream16_lds_bytes(int wt) { return kStream16Waves * stream16_slot_bytes(wt) + kStream16SumBytes + kMaxGroups * 8; }
static_assert(stream16_lds_bytes(4) <= 160 * 1024, "LDS");

template <bool BF16, int WT, bool STREAM>
__global__ __launch_bounds__(kStream16Waves * 64, 2) void streaming_gemm16_kernel(const Params p) {
  constexpr int BN = 16 * WT, kSlot = stream16_slot_bytes(WT), kWeights = BN * 128;
  extern __shared__ u32x4 lds[];
  char* const lds_bytes = reinterpret_cast<char*>(lds);
  f32x4* const sums = reinterpret_cast<f32x4*>(lds_bytes + kStream16Waves * kSlot);
  u32x2* const entries = reinterpret_cast<u32x2*>(lds_bytes + kStream16Waves * kSlot + kStream16SumBytes);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int kbytes = p.k * 2;
  const int steps = (p.k + 63) >> 6;
  const int tail_pieces = (p.k & 63) >> 3;  // 8-element pieces of a row in a short last step (0: it is whole)
  const int blocks = (p.n + BN - 1) / BN;

  // ---- the groups that have rows: {first item, group}
  int entry_count, total;
  {
    int* const wave_total = reinterpret_cast<int*>(lds);
    int before_items = 0, before = 0;
    for (int base = 0; base < p.groups; base += kStream16Waves * 64) {
      const int gi = base + tid;
      const int m_g = gi < p.groups ? max(p.problem_sizes[gi * 3], 0) : 0;
      const int items = ((m_g + kStream16Rows - 1) / kStream16Rows) * blocks;
      int incl = items, incl_n = items > 0;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(incl, d, 64), o_n = __shfl_up(incl_n, d, 64);
        if (lane >= d) incl += o, incl_n += o_n;
      }
      if (lane == 63) wave_total[wave] = incl, wave_total[8 + wave] = incl_n;
      __syncthreads();
      int at_item = before_items + incl - items, at = before + incl_n - (items > 0);
      for (int w = 0; w < kStream16Waves; ++w) {
        if (w < wave) at_item += wave_total[w], at += wave_total[8 + w];
        before_items += wave_total[w];
        before += wave_total[8 + w];
      }
      __syncthreads();
      if (items > 0) entries[at] = u32x2{(uint32_t)at_item, (uint32_t)gi};
    }
    total = __builtin_amdgcn_readfirstlane(before_items);
    entry_count = __builtin_amdgcn_readfirstlane(before);
    __syncthreads();
  }
  if ((int)blockIdx.x >= total) return;

  struct Item {
    const uint8_t *a, *b;
    int rows, row0, n0;
  };
  int e = 0;  // the entry of the last item asked for; items are asked for in ascending order
  auto item_info = [&](int t) {
    while (e + 1 < entry_count && __builtin_amdgcn_readfirstlane((int)entries[e + 1][0]) <= t) ++e;
    const int group = __builtin_amdgcn_readfirstlane((int)entries[e][1]);
    const int at = t - __builtin_amdgcn_readfirstlane((int)entries[e][0]);
    const int m_g = __builtin_amdgcn_readfirstlane(p.problem_sizes[group * 3]);
    const int slabs = (m_g + kStream16Rows - 1) / kStream16Rows;
    // runs of 8 weight blocks (fewer in the last run), slab by slab
    const int run = at / (8 * slabs), in_run = at - run * 8 * slabs;
    const int width = min(8, blocks - run * 8);
    const int slab = in_run / width;
    Item it;
    it.row0 = __builtin_amdgcn_readfirstlane(p.expert_offsets[group]) + slab * kStream16Rows;
    it.rows = min(m_g - slab * kStream16Rows, kStream16Rows);
    it.n0 = (run * 8 + in_run - slab * width) * BN;
    it.a = p.a + (int64_t)it.row0 * kbytes;
    it.b = p.b + ((int64_t)group * p.n + it.n0) * kbytes;
    return it;
  };

  // ---- load side: lane L fetches row L/8 of 8, piece (L%8) ^ ((row >> 1) & 7)
  const uint32_t lds_base = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)lds);
  const uint32_t slot = lds_base + (uint32_t)wave * kSlot;
  const uint32_t piece_even = (uint32_t)((lane & 7) ^ (lane >> 4));  // 8-row blocks 0, 2, ..; the odd ones: ^ 4
  const uint32_t lrow = (uint32_t)(lane >> 3);
  auto issue = [&](const Item& it, int c) {
    uint32_t pe = piece_even, po = piece_even ^ 4u;
    if (tail_pieces != 0 && c == steps - 1) {
      if (pe >= (uint32_t)tail_pieces) pe = 0;
      if (po >= (uint32_t)tail_pieces) po = 0;
    }
    const uint8_t* b = it.b + (int64_t)c * 128;
    const uint8_t* a = it.a + (int64_t)c * 128;
    if (it.n0 + BN <= p.n) {
      const uint32_t ve = lrow * (uint32_t)kbytes + pe * 16u, vo = lrow * (uint32_t)kbytes + po * 16u;
#pragma unroll
      for (int j = 0; j < 2 * WT; ++j) lds_dma16<0, STREAM>(slot + j * 1024, b + (int64_t)kbytes * (8 * j), (j & 1) ? vo : ve);
    } else {
      const uint32_t last = (uint32_t)(p.n - it.n0 - 1);
#pragma unroll
      for (int j = 0; j < 2 * WT; ++j)
        lds_dma16<0, STREAM>(slot + j * 1024, b, __umul24(min(lrow + 8 * j, last), (uint32_t)kbytes) + ((j & 1) ? po : pe) * 16u);
    }
#pragma unroll
    for (int j = 0; j < kStream16Rows / 8; ++j) {
      if ((j & 1) == 0 && it.rows <= 8 * j) break;
      lds_dma16(slot + kWeights + j * 1024, a, __umul24(min(lrow + 8 * j, (uint32_t)(it.rows - 1)), (uint32_t)kbytes) + ((j & 1) ? po : pe) * 16u);
    }
  };

  // ---- read side
  const char* const sp = lds_bytes + wave * kSlot;
  const int swz = (r >> 1) & 7;
  const bool has_steps = wave < steps;
  const int parts = min(steps, kStream16Waves);
  Item it = item_info(blockIdx.x);
  if (has_steps) issue(it, wave);
  int turn = 0;
  for (int t = blockIdx.x; t < total; t += gridDim.x, ++turn) {
    const bool more = t + (int)gridDim.x < total;
    const Item next = more ? item_info(t + gridDim.x) : it;
    auto run = [&](auto tiles_c) {
      constexpr int TILES = decltype(tiles_c)::value;  // row tiles of 16
      f32x4 acc[WT][TILES];
#pragma unroll
      for (int rt = 0; rt < WT; ++rt)
#pragma unroll
        for (int tt = 0; tt < TILES; ++tt) acc[rt][tt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      for (int c = wave; c < steps; c += kStream16Waves) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        u32x4 w[2][WT], x[2][TILES];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int pos = r * 128 + ((4 * h + g) ^ swz) * 16;
#pragma unroll
          for (int rt = 0; rt < WT; ++rt) w[h][rt] = *reinterpret_cast<const u32x4*>(sp + rt * 2048 + pos);
#pragma unroll
          for (int tt = 0; tt < TILES; ++tt) x[h][tt] = *reinterpret_cast<const u32x4*>(sp + kWeights + tt * 2048 + pos);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read out: may be refilled
        if (c + kStream16Waves < steps) issue(it, c + kStream16Waves);
        else if (more) issue(next, wave);
        if (tail_pieces != 0 && c == steps - 1) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const uint32_t keep = 4 * h + g < tail_pieces ? 0xffffffffu : 0u;
#pragma unroll
            for (int rt = 0; rt < WT; ++rt) w[h][rt] &= keep;
#pragma unroll
            for (int tt = 0; tt < TILES; ++tt) x[h][tt] &= keep;
          }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int rt = 0; rt < WT; ++rt)
#pragma unroll
            for (int tt = 0; tt < TILES; ++tt) {
              if constexpr (BF16)
                acc[rt][tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[h][rt]), __builtin_bit_cast(bf16x8, x[h][tt]), acc[rt][tt], 0, 0, 0);
              else
                acc[rt][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w[h][rt]), __builtin_bit_cast(f16x8, x[h][tt]), acc[rt][tt], 0, 0, 0);
            }
      }
      // ---- the wavefronts' partial tiles.  An item has an even number of them, so the two buffers alternate across items
      // too; a buffer is written again only after a barrier that follows the reads of its last contents.
#pragma unroll
      for (int i = 0; i < WT * TILES; ++i) {
        const int rt = i % WT, tt = i / WT;
        f32x4* const buffer = sums + (i & 1) * (kStream16Waves * 64);
        if (has_steps) buffer[wave * 64 + lane] = acc[rt][tt];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (wave == ((i + turn * (WT * TILES)) & 7)) {
          f32x4 s = buffer[lane];
          for (int part = 1; part < parts; ++part) s += buffer[part * 64 + lane];
          const int tok = tt * 16 + r, col = it.n0 + rt * 16 + 4 * g;
          if (tok < it.rows && col < p.n) {
            u32x2 v;
            v[0] = pack2(s[0], s[1], BF16);
            v[1] = pack2(s[2], s[3], BF16);
            *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(p.out) + (int64_t)(it.row0 + tok) * p.n + col) = v;
          }
        }
      }
    };
    if (it.rows > 48) run(std::integral_constant<int, 4>{});
    else if (it.rows > 32) run(std::integral_constant<int, 3>{});
    else if (it.rows > 16) run(std::integral_constant<int, 2>{});
    else run(std::integral_constant<int, 1>{});
    it = next;
  }
}

template <bool BF16, int WT, bool STREAM>
int launch_grouped16_streaming_cfg(const Params& p, int grid, hipStream_t stream) {
  auto kern = streaming_gemm16_kernel<BF16, WT, STREAM>;
  if (note_launch("streaming_gemm16_kernel<weight_rows=%d,stream=%d> grid=%d", 16 * WT, (int)STREAM, grid)) return NVF_OK;
  static std::atomic<uint64_t> configured{0};  // one bit per device
  if (const int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), stream16_lds_bytes(WT), configured)) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(kStream16Waves * 64), stream16_lds_bytes(WT), stream, p);
  return check_launch("streaming_gemm16_kernel");
}

template <bool BF16>
int launch_grouped16_streaming(const Params& p, int cus, hipStream_t stream) {
  const int64_t slabs = std::min<int64_t>(p.m, p.groups + p.m / kStream16Rows);  // at most
  // 32 weight rows an item where items of 64 would not go round the compute units twice
  const bool narrow = std::min<int64_t>(p.groups, p.m) * ceil_div(p.n, 64) < 2 * (int64_t)cus;
  const int grid = (int)std::min<int64_t>(std::max(cus & ~7, 8), round_up(slabs * ceil_div(p.n, narrow ? 32 : 64), 8));
  // weights beyond what the 256 MB last-level cache holds are read past it (8 experts of 14336 x 4096, 16 rows each: 159 us,
  // with plain loads 175; 64 of 2048 x 7168, 24 rows 312 / 335)
  const bool past_cache = (p.k & 63) == 0 && 2.0 * p.groups * p.n * p.k > (double)(256 << 20);
  if (narrow) return launch_grouped16_streaming_cfg<BF16, 2, false>(p, grid, stream);
  return past_cache ? launch_grouped16_streaming_cfg<BF16, 4, true>(p, grid, stream) : launch_grouped16_streaming_cfg<BF16, 4, false>(p, grid, stream);
}
