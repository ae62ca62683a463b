// Persistent kernel with 256x256 or 128x128 tiles for grouped_mm (16-bit operands) of gemm16.hip (included there, inside namespace nvf).
// -------------------------------------------------------------------------------------------------
// grouped_mm fast path (16-bit operands): N % 8 == 0, K % 64 == 0.  256x256 tiles:
// Bound by the power limit of the MFMAs (bf16 8192^3 as one group: 1.50..1.57 PFLOP/s, 810..841 -> 703..735 us against a K loop
// of 32x32 MFMAs with all of a step's loads in one half of it; 8 experts, 8192 rows, N = 14336, K = 4096 887..907 -> 766..781).
// 128x128 tiles: groups of fewer rows, or too few 256x256 tiles; any N % 8 == 0.  Bound by the weights' way out of HBM, for which
// four buffers keep three steps' loads in flight.  Against the 128x128 tile kernel (two workgroups per compute unit, a barrier and
// a register stage per step): 64 experts of 2048 x 4096, 2048 rows 288 -> 212 us, 16 of 4096 x 4096, 1000 rows 178 -> 127, 8 of
// 14336 x 4096, 512 rows 220 -> 196, 32 of 2048 x 2048, 2048 rows 86 -> 59, 8 of 2560 x 1600, 474 rows 29 -> 16; 37 shapes of 16 to
// 2048 rows per group, with the 256x256 tiles', 1.22 times as fast in the geometric mean, none slower.  256x256 tiles with a
// short last column tile: 8 experts of 6632 x 4096, 16384 rows 1095 -> 687 us.
//   * Persistent workgroups walk the (group, m-tile, n-tile) list derived on the device from
//     problem_sizes; each XCD owns a contiguous part of the list, whose neighbouring tiles share the
//     group's weight panel in that XCD's L2.
//   * The K loop is TileLoop's.  Its load stream runs NBUF steps ahead of the MFMAs and continues across tile and
//     group borders.  Rows past the end of a group (and weight rows past N) load the last row again (never another group's
//     memory past the tensor) and are not stored.
//   * The groups' rows and places are kept in LDS: a look into global memory at every new tile would wait for all of the
//     stream's loads.
// -------------------------------------------------------------------------------------------------
template <int NI, int NJ, int NBUF>
struct Grouped16Tiles {
  static constexpr int BM = 32 * NI, BN = 32 * NJ;
  static constexpr int kTileBytes = TileLoop<Mma::kF16, NI, NJ, NBUF>::kTileBytes;
  static constexpr int kLdsBytes = kTileBytes + 4 * 4608 + (kMaxGroups + 1) * 4 + kMaxGroups * 8;  // tiles, the epilogue's, groups
  static_assert(kLdsBytes <= 160 * 1024, "LDS");
};

// STREAM_OUT, STREAM_B: results are stored, weights are read past the last-level cache.  RAGGED_N: N is no multiple of the tile's
// columns, but of 8.
template <int NI, int NJ, int NBUF, bool BF16_MMA, bool OUT_BF16, bool STREAM_OUT, bool STREAM_B, bool RAGGED_N>
__global__ __launch_bounds__(256, 1) void grouped16_tile_kernel(const Params p) {
  using T = Grouped16Tiles<NI, NJ, NBUF>;
  constexpr int BM = T::BM, BN = T::BN;
  constexpr int kBand = 4;  // m-tiles that share a weight panel while it is in an XCD's L2 (8: measured no better)
  extern __shared__ u32x4 lds[];
  u32x2* const group_rows = reinterpret_cast<u32x2*>(reinterpret_cast<char*>(lds) + T::kTileBytes + 4 * 4608);  // {rows, first row}
  int* const tile_prefix = reinterpret_cast<int*>(group_rows + kMaxGroups);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int tiles_n = RAGGED_N ? (p.n + BN - 1) / BN : p.n / BN;

  // ---- work list: prefix sums of BM-row tiles per group (one wavefront, 64 groups per round)
  if (wave == 0) {
    int running = 0;
    for (int base = 0; base < p.groups; base += 64) {
      const int g = base + lane;
      int cnt = 0;
      if (g < p.groups) {
        const int mg = p.problem_sizes[g * 3];
        cnt = mg > 0 ? (mg + BM - 1) / BM : 0;
        group_rows[g] = u32x2{(uint32_t)mg, (uint32_t)p.expert_offsets[g]};
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
  // Workgroup ids are dealt round-robin to the 8 XCDs.  The tiles of a group are walked in bands of up to 4 m-tiles,
  // n-major inside a band, so that 32 consecutive tiles share 4 A and 8 B panels in an XCD's L2 and a weight panel
  // comes in from memory once per band.  DEAL (n-tiles a multiple of
  // 8): XCD x takes the n-tiles x, x+8, ... of every band, i.e. its own list of (tiles / 8) tiles of the same make-up as
  // every other XCD's: each expert's weights stream in through all eight XCDs and all of them meet the cheap and
  // the expensive tiles (small groups are bound by streaming their weights once) at the same rate.  Otherwise XCD
  // x owns the contiguous eighth [x*chunk, (x+1)*chunk) of the one list.
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, slots = gridDim.x >> 3;
  const bool deal = (tiles_n & 7) == 0;
  const int per_m = deal ? tiles_n >> 3 : tiles_n;  // list entries per m-tile
  const int total = __builtin_amdgcn_readfirstlane(tile_prefix[p.groups]) * per_m;
  const int chunk_tiles = (total + 7) >> 3;
  const int range_end = deal ? total : min((xcd + 1) * chunk_tiles, total);
  const int first_tile = deal ? slot : xcd * chunk_tiles + slot;
  if (first_tile >= range_end) return;

  const int kb = p.k * 2;   // bytes per operand row
  const int nk = p.k >> 6;  // 64-deep steps

  struct Tile { const uint8_t *a, *b; int valid; int64_t out_row; int n0; };
  auto tile_info = [&](int t) {
    int lo = 0, hi = p.groups;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (t < tile_prefix[mid] * per_m) hi = mid; else lo = mid;
    }
    const int g = __builtin_amdgcn_readfirstlane(lo);
    const u32x2 rows = group_rows[g];
    const int m_g = __builtin_amdgcn_readfirstlane((int)rows[0]);
    const int64_t row_off = __builtin_amdgcn_readfirstlane((int)rows[1]);
    const int tiles_m = (m_g + BM - 1) / BM;
    const int local = __builtin_amdgcn_readfirstlane(t - tile_prefix[g] * per_m);
    // bands of up to kBand m-tiles of near-equal height (9 m-tiles: 3 + 3 + 3), n-major inside a band
    const int nb = (tiles_m + kBand - 1) / kBand, base_h = tiles_m / nb, taller = tiles_m - base_h * nb;  // the first `taller` bands have base_h + 1
    const int mrow = local / per_m;  // m-tiles of the group that lie in earlier bands, plus a remainder
    const int split = taller * (base_h + 1);
    const int band = mrow < split ? mrow / (base_h + 1) : taller + (mrow - split) / base_h;
    const int band_h = band < taller ? base_h + 1 : base_h;
    const int band_m0 = band < taller ? band * (base_h + 1) : split + (band - taller) * base_h;
    const int in_band = local - band_m0 * per_m;
    const int ntl = in_band / band_h, mt = band_m0 + (in_band - ntl * band_h);
    const int nt = deal ? xcd + 8 * ntl : ntl;
    Tile r;
    r.a = p.a + (row_off + (int64_t)mt * BM) * kb;
    r.b = p.b + ((int64_t)g * p.n + (int64_t)nt * BN) * kb;
    r.valid = min(BM, m_g - mt * BM);
    r.out_row = row_off + (int64_t)mt * BM;
    r.n0 = nt * BN;
    return r;
  };

  // ---- LDS-direct loads of a step.  A load is 8 rows: lane L lands at unit +L, i.e. row +(L>>3), chunk position L&7, which
  // must hold global chunk (L&7) ^ ((row>>1)&7) = (L&7) ^ ((L>>4) | ((j&1)<<2)) of load j.
  using Loop = TileLoop<BF16_MMA ? Mma::kBf16 : Mma::kF16, NI, NJ, NBUF>;
  const uint32_t lds_base = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)lds);
  const uint32_t chunk_even = (uint32_t)(((lane & 7) ^ (lane >> 4)) << 4), chunk_odd = chunk_even ^ 64u;
  // the wavefront's share: rows of A's first half (the second's: 8 NI rows further on), of B
  const int a_row0 = wm * (16 * NI) + wn * (4 * NI), b_row0 = wave * (8 * NJ);
  const uint32_t a_lds = lds_base + (uint32_t)a_row0 * 128u, b_lds = lds_base + NBUF * Loop::kABytes + (uint32_t)b_row0 * 128u;
  uint32_t a_off[NI], b_off[NJ];

  // ---- load stream: the step the next loads are issued for (l_ks of the tile lp) and the tile after it (np; past the end
  // of the list: a valid tile, loaded and ignored)
  const Tile first_info = tile_info(first_tile);
  Tile lp = first_info, np;
  int l_ks = 0, l_buf = 0, stream_tile = first_tile;
  uint32_t l_a = a_lds, l_b = b_lds;  // the step's buffer
  auto prepare_next = [&]() {
    stream_tile += slots;
    np = stream_tile < range_end ? tile_info(stream_tile) : first_info;
  };
  prepare_next();
  auto enter_tile = [&](bool first) {
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      const uint32_t row = (uint32_t)(a_row0 + (u < NI / 2 ? 0 : 4 * NI) + 8 * u + (lane >> 3));
      a_off[u] = min(row, (uint32_t)(lp.valid - 1)) * (uint32_t)kb + ((u & 1) ? chunk_odd : chunk_even);
    }
    if (!RAGGED_N && !first) return;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      uint32_t row = (uint32_t)(b_row0 + 8 * j + (lane >> 3));
      if (RAGGED_N) row = min(row, (uint32_t)(p.n - lp.n0 - 1));
      b_off[j] = row * (uint32_t)kb + ((j & 1) ? chunk_odd : chunk_even);
    }
  };
  enter_tile(true);
  auto load = [&](auto code) {
    constexpr int u = decltype(code)::value;
    if constexpr (u >= kLoadB) lds_dma16<(u - kLoadB) * 1024, STREAM_B>(l_b, lp.b, b_off[u - kLoadB]);
    else lds_dma16<(u + (u < NI / 2 ? 0 : NI / 2)) * 1024>(l_a, lp.a, a_off[u]);
  };
  auto load_step = [&]() {  // in the order of the loop's
    static_for<NI / 2>(load);
    static_for<NJ>([&](auto j) { load(std::integral_constant<int, kLoadB + decltype(j)::value>{}); });
    static_for<NI / 2>([&](auto u) { load(std::integral_constant<int, NI / 2 + decltype(u)::value>{}); });
  };
  auto advance = [&]() {
    const int by = l_buf == NBUF - 1 ? 1 - NBUF : 1;
    l_buf += by;
    l_a += by * Loop::kABytes;
    l_b += by * Loop::kBBytes;
    lp.a += 128;
    lp.b += 128;
    if (++l_ks == nk) {
      l_ks = 0;
      lp = np;
      enter_tile(false);
      prepare_next();
    }
  };

  Loop loop;
  loop.init(lds_base, lane, wm, wn);
  auto& acc = loop.acc;

  for (int i = 0; i < NBUF; ++i) {
    load_step();
    advance();
  }
  loop.fence();
  loop.first_fragments();

  for (int c_tile = first_tile; c_tile < range_end; c_tile += slots) {
    loop.template step<true>(load, [](auto) {});
    advance();
    for (int c_ks = 1; c_ks < nk; ++c_ks) {
      loop.template step<false>(load, [](auto) {});
      advance();
    }
    const Tile ct = tile_info(c_tile);
    loop.settle();
    // ---- epilogue of this tile; the loads of the next steps are already in flight.
    // A lane holds 8-byte pieces of 16 rows per tile; stored like that, a tile is 8192 sixteen-byte write
    // requests per compute unit.  Every 32x64 block of the wavefront's tile is therefore turned round in a
    // private 4.5 KiB of LDS (32 rows of 128 bytes at a pitch of 144 bytes) and leaves in 16-byte pieces, 8 lanes
    // to a row's 128 bytes.  One LDS address each for writing and reading (the rest are immediate offsets) and
    // one 32-bit lane offset next to a wave-uniform result address keep the epilogue out of the spill area.
    int elane = lane;
    asm volatile("" : "+v"(elane));
    uint8_t* stage = reinterpret_cast<uint8_t*>(lds) + Loop::kTileBytes + wave * 4608;
    uint8_t* wr = stage + (elane & 15) * 144 + (elane >> 4) * 8;
    const uint8_t* rd = stage + (elane >> 3) * 144 + (elane & 7) * 16;
    const uint32_t ooff = ((uint32_t)(elane >> 3) * (uint32_t)p.n + (uint32_t)(elane & 7) * 8u) * 2u;
    uint8_t* obase = reinterpret_cast<uint8_t*>(static_cast<uint16_t*>(p.out) + (ct.out_row + wm * (16 * NI)) * (int64_t)p.n + ct.n0 + wn * (16 * NJ));
    const int erow = wm * (16 * NI) + (elane >> 3), cols_left = p.n - ct.n0 - wn * (16 * NJ) - (elane & 7) * 8;
#pragma unroll
    for (int i = 0; i < NI / 2; ++i) {
#pragma unroll
      for (int jh = 0; jh < NJ / 4; ++jh) {
#pragma unroll
        for (int t = 0; t < 8; ++t) {  // the block's 2 x 4 tiles
          const f32x4 c = acc[2 * i + (t >> 2)][4 * jh + (t & 3)];
          u32x2 v;
          v[0] = pack2(c[0], c[1], OUT_BF16);
          v[1] = pack2(c[2], c[3], OUT_BF16);
          *reinterpret_cast<u32x2*>(wr + (t >> 2) * 2304 + (t & 3) * 32) = v;
        }
        asm volatile("" ::: "memory");  // the reads below see the writes above: one wavefront's LDS accesses stay in order
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int brow = i * 32 + 8 * t;  // first of the 8 rows of this piece, in the wavefront's tile
          const u32x4 v = *reinterpret_cast<const u32x4*>(rd + t * 1152);
          if (erow + brow < ct.valid && (!RAGGED_N || jh * 64 < cols_left)) {
            u32x4* dst = reinterpret_cast<u32x4*>(obase + ((int64_t)brow * p.n + jh * 64) * 2 + ooff);
            if constexpr (STREAM_OUT) __builtin_nontemporal_store(v, dst);
            else *dst = v;
          }
        }
        asm volatile("" ::: "memory");
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no LDS-direct load may outlive the workgroup
}

template <int NI, int NJ, int NBUF, bool BF16_MMA, bool OUT_BF16, bool STREAM_OUT, bool STREAM_B, bool RAGGED_N>
int launch_grouped16_tiles_cfg(const Params& p, int cus, hipStream_t stream) {
  using T = Grouped16Tiles<NI, NJ, NBUF>;
  auto kern = grouped16_tile_kernel<NI, NJ, NBUF, BF16_MMA, OUT_BF16, STREAM_OUT, STREAM_B, RAGGED_N>;
  if (note_launch("grouped16_tile_kernel<%dx%d,stream_out=%d,stream_weights=%d%s> grid=%d", T::BM, T::BN, (int)STREAM_OUT, (int)STREAM_B,
                  p.n % T::BN ? ",ragged_n" : "", cus & ~7))
    return NVF_OK;
  static std::atomic<uint64_t> configured{0};  // one bit per device
  if (const int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), T::kLdsBytes, configured)) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)(cus & ~7)), dim3(256), T::kLdsBytes, stream, p);
  return check_launch("grouped16_tile_kernel");
}

template <bool BF16_MMA, bool OUT_BF16>
int launch_grouped16_fast(const Params& p, int cus, hipStream_t stream) {
  // Operands and result together beyond what the 256 MB last-level cache holds: the result leaves with
  // non-temporal stores, which keeps it from pushing operand panels out (single 8192-row group, 8192^3: +2.6 %,
  // 16384 x 4096 x 4096: +7 %); smaller problems are better off with plain stores.
  const int64_t bytes = 2 * ((int64_t)p.m * p.k + (int64_t)p.groups * p.n * p.k + (int64_t)p.m * p.n);
  const bool past = bytes > ((int64_t)224 << 20);
  if ((p.n & 255) != 0)
    return past ? launch_grouped16_tiles_cfg<8, 8, 2, BF16_MMA, OUT_BF16, true, false, true>(p, cus, stream)
                : launch_grouped16_tiles_cfg<8, 8, 2, BF16_MMA, OUT_BF16, false, false, true>(p, cus, stream);
  return past ? launch_grouped16_tiles_cfg<8, 8, 2, BF16_MMA, OUT_BF16, true, false, false>(p, cus, stream)
              : launch_grouped16_tiles_cfg<8, 8, 2, BF16_MMA, OUT_BF16, false, false, false>(p, cus, stream);
}

template <bool BF16_MMA, bool OUT_BF16>
int launch_grouped16_small_tiles(const Params& p, int cus, hipStream_t stream) {
  // Weights that the last-level cache cannot hold and that hardly more than one row tile per group reads: past it.
  const bool past = p.m <= 128 * (int64_t)p.groups && 2.0 * p.groups * p.n * p.k > (double)(256 << 20);
  return past ? launch_grouped16_tiles_cfg<4, 4, 4, BF16_MMA, OUT_BF16, false, true, true>(p, cus, stream)
              : launch_grouped16_tiles_cfg<4, 4, 4, BF16_MMA, OUT_BF16, false, false, true>(p, cus, stream);
}
