// mxfp8_scaled_mm for gfx950 (cutlass/mxfp8_scaled_mm.cu:290-319): C = alpha * A * B^T with e4m3
// operands and one e8m0 scale per 32 K-elements, on v_mfma_scale_f32_16x16x128_f8f6f4 (persistent and weight-streaming
// kernels) and v_mfma_scale_f32_32x32x64_f8f6f4 (the tile kernel for the shapes that neither takes).
//
// Operand layout of the latter (fp8 x fp8), measured on hardware:
//   lane l = i + 32*g (i = row of A / column of B, g in {0,1}) supplies 32 bytes:
//     bytes  0..15 = K [16g,      16g + 16)
//     bytes 16..31 = K [32 + 16g, 32 + 16g + 16)
//   and the scale byte of lane i + 32*j applies to row i, K-block j (K [32j, 32j+32)).
// The 128x4 scale layout stores, for 32 consecutive rows, 16 bytes per row position holding
// (rows r, r+32, r+64, r+96) x (4 consecutive K-blocks): one 16-byte load per lane fetches every
// scale a 128-row wave tile needs for a 128-deep K step.
#include "lds_direct.h"
#include "nvf_internal.h"
#include "tile_loop.h"

namespace nvf {
namespace {

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

struct Params {
  const uint8_t* a;
  const uint8_t* b;
  const uint8_t* sfa;
  const uint8_t* sfb;
  const float* alpha;
  void* out;
  int m, n, k;
  int m_base = 0;  // skinny kernel: first activation row this launch computes, a multiple of the slab height (32, 64 or 128)
  int ldc = 0;     // elements between rows of the result; 0: n (a launch that computes some of the columns sets it)
  __host__ __device__ int out_pitch() const { return ldc ? ldc : n; }
};

__device__ __forceinline__ uint32_t pack2(float a, float b, bool out_bf16) {
  if (out_bf16) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    bf16x2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, v);
  }
  f16x2 v = {(_Float16)a, (_Float16)b};
  return __builtin_bit_cast(uint32_t, v);
}

// LDS tile: rows of 128 bytes; 16-byte chunk c of row r sits at chunk position c ^ ((r >> 1) & 7): two rows fill
// the 64 banks once, so the fragment reads (16 consecutive lanes = 16 consecutive rows, one chunk) are conflict-free
__device__ __forceinline__ int lds_pos(int row, int chunk) { return row * 8 + (chunk ^ ((row >> 1) & 7)); }

template <int BM, int BN, bool OUT_BF16>
__global__ __launch_bounds__(256) void mxfp8_gemm_kernel(const Params p) {
  constexpr int BK = 128;  // bytes == elements
  constexpr int WTM = BM / 2, WTN = BN / 2;
  constexpr int TM = WTM / 32, TN = WTN / 32;
  extern __shared__ u32x4 lds[];  // two buffers of (A tile, B tile)
  constexpr int BUF_UNITS = (BM + BN) * 8;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 31, lg = lane >> 5;

  const int tiles_m = (p.m + BM - 1) / BM;
  const int mt = blockIdx.x % tiles_m, nt = blockIdx.x / tiles_m;
  const int m0 = mt * BM, n0 = nt * BN;
  const int sf_cols = p.k / 32;
  const int sf_padded = (sf_cols + 3) & ~3;
  const int nk = (p.k + BK - 1) / BK;

  const uint8_t* a_base = p.a + (int64_t)m0 * p.k;
  const uint8_t* b_base = p.b + (int64_t)n0 * p.k;

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  constexpr int A_TOTAL = BM * 8, B_TOTAL = BN * 8;
  constexpr int A_CH = (A_TOTAL + 255) / 256, B_CH = (B_TOTAL + 255) / 256;
  u32x4 sa[A_CH], sb[B_CH];
  // scale words: [sub-tile] -> 4 e8m0 bytes (K-blocks of this 128-deep step) of row (sub-tile*32 + li)
  uint32_t sca[TM], scb[TN], sca_next[TM], scb_next[TN];

  auto issue_loads = [&](int ks) {
    const int kb0 = ks * BK;
#pragma unroll
    for (int i = 0; i < A_CH; ++i) {
      const int c = tid + 256 * i;
      const int row = c >> 3, chunk = c & 7;
      const bool ok = (c < A_TOTAL) && (m0 + row < p.m) && (kb0 + chunk * 16 < p.k);
      sa[i] = u32x4{0, 0, 0, 0};
      if (ok) sa[i] = *reinterpret_cast<const u32x4*>(a_base + (int64_t)row * p.k + kb0 + chunk * 16);
    }
#pragma unroll
    for (int i = 0; i < B_CH; ++i) {
      const int c = tid + 256 * i;
      const int row = c >> 3, chunk = c & 7;
      const bool ok = (c < B_TOTAL) && (n0 + row < p.n) && (kb0 + chunk * 16 < p.k);
      sb[i] = u32x4{0, 0, 0, 0};
      if (ok) sb[i] = *reinterpret_cast<const u32x4*>(b_base + (int64_t)row * p.k + kb0 + chunk * 16);
    }
    // Scales of rows past m / n and of K-blocks past k belong to zero payload; they are forced to
    // 2^0 (0x7F) so that padding bytes (possibly the NaN code 0xFF) never meet the zeros.
    const int valid_blocks = sf_cols - ks * 4;  // >= 1
    const uint32_t keep = valid_blocks >= 4 ? 0xffffffffu : ((1u << (8 * valid_blocks)) - 1u);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int row = m0 + wm * WTM + i * 32 + li;
      uint32_t w = 0;
      if (row < p.m) w = *reinterpret_cast<const uint32_t*>(p.sfa + swizzle_128x4(row, ks * 4, sf_padded)) & keep;
      else w = 0x7f7f7f7fu & keep;
      sca_next[i] = w | (0x7f7f7f7fu & ~keep);
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int row = n0 + wn * WTN + j * 32 + li;
      uint32_t w = 0;
      if (row < p.n) w = *reinterpret_cast<const uint32_t*>(p.sfb + swizzle_128x4(row, ks * 4, sf_padded)) & keep;
      else w = 0x7f7f7f7fu & keep;
      scb_next[j] = w | (0x7f7f7f7fu & ~keep);
    }
  };

  auto store_lds = [&](int buf) {
    u32x4* lds_a = lds + buf * BUF_UNITS;
    u32x4* lds_b = lds_a + BM * 8;
#pragma unroll
    for (int i = 0; i < A_CH; ++i) {
      const int c = tid + 256 * i;
      if (c < A_TOTAL) lds_a[lds_pos(c >> 3, c & 7)] = sa[i];
    }
#pragma unroll
    for (int i = 0; i < B_CH; ++i) {
      const int c = tid + 256 * i;
      if (c < B_TOTAL) lds_b[lds_pos(c >> 3, c & 7)] = sb[i];
    }
  };

  // K loop: the loads of step ks+1 are in flight under the MFMAs of step ks, then stored into the other
  // LDS buffer; one barrier per step
  issue_loads(0);
  store_lds(0);
  __syncthreads();
  for (int ks = 0; ks < nk; ++ks) {
    const u32x4* lds_a = lds + (ks & 1) * BUF_UNITS;
    const u32x4* lds_b = lds_a + BM * 8;
#pragma unroll
    for (int i = 0; i < TM; ++i) sca[i] = sca_next[i];
#pragma unroll
    for (int j = 0; j < TN; ++j) scb[j] = scb_next[j];
    if (ks + 1 < nk) issue_loads(ks + 1);

#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      i32x8 fa[TM], fb[TN];
      const int c_lo = sub * 4 + lg, c_hi = sub * 4 + 2 + lg;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int row = wm * WTM + i * 32 + li;
        const u32x4 lo = lds_a[lds_pos(row, c_lo)], hi = lds_a[lds_pos(row, c_hi)];
        fa[i] = i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int row = wn * WTN + j * 32 + li;
        const u32x4 lo = lds_b[lds_pos(row, c_lo)], hi = lds_b[lds_pos(row, c_hi)];
        fb[j] = i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
      }
      // K-block of this lane inside the 128-deep step: 2*sub + lg
      const int sh = 8 * (2 * sub + lg);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int s_a = (int)((sca[i] >> sh) & 0xffu);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int s_b = (int)((scb[j] >> sh) & 0xffu);
          // B fragment first: the accumulator then holds 4 consecutive N-elements per register quad
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fb[j], fa[i], acc[i][j], 0, 0, 0, s_b, 0, s_a);
        }
      }
    }
    if (ks + 1 < nk) store_lds((ks + 1) & 1);
    __syncthreads();
  }

  const float alpha = p.alpha[0];
  uint16_t* out = static_cast<uint16_t*>(p.out);
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int mrow = m0 + wm * WTM + i * 32 + li;
    if (mrow >= p.m) continue;
    uint16_t* orow = out + (int64_t)mrow * p.out_pitch();
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        const int ncol = n0 + wn * WTN + j * 32 + rq * 8 + lg * 4;
        if (ncol < p.n) {
          u32x2 v;
          v[0] = pack2(acc[i][j][rq * 4 + 0] * alpha, acc[i][j][rq * 4 + 1] * alpha, OUT_BF16);
          v[1] = pack2(acc[i][j][rq * 4 + 2] * alpha, acc[i][j][rq * 4 + 3] * alpha, OUT_BF16);
          *reinterpret_cast<u32x2*>(orow + ncol) = v;
        }
      }
    }
  }
}


// -------------------------------------------------------------------------------------------------
// Persistent kernel: 256x256, 128x256 or 128x128 tiles, N % 16 == 0, K % 32 == 0, K >= 256.
// -------------------------------------------------------------------------------------------------

// The walk over the tiles.  Workgroup ids are dealt round-robin to the 8 XCDs, so XCD x owns the contiguous tile range
// [x*chunk, (x+1)*chunk) and its workgroups take consecutive tiles of it in each round: with the 8 (m) x 4 (n) blocked tile
// numbering, the 32 tiles an XCD works on at any time share 8 A panels and 4 B panels in that XCD's L2.
// RAGGED: the last row tile holds fewer than BM rows or the last column tile fewer than BN columns (kernels of their own:
// clamping the row of every load costs the others time).  The missing rows load the last row again and are not stored; the
// scale layout is padded to 128 rows, so only a 256-row tile can ask for a scale tile that does not exist (it takes an
// existing one).
template <int BM, int BN, bool RAGGED>
struct TileWalk {
  int tiles_m, tiles_n, first, end, slots, bulk_tiles;
  bool blocked;
  __device__ __forceinline__ explicit TileWalk(const Params& p) {
    tiles_m = RAGGED ? (p.m + BM - 1) / BM : p.m / BM;
    tiles_n = RAGGED ? (p.n + BN - 1) / BN : p.n / BN;
    const int total = tiles_m * tiles_n, chunk = (total + 7) >> 3;
    const int xcd = blockIdx.x & 7;
    slots = gridDim.x >> 3;
    first = xcd * chunk + (blockIdx.x >> 3);
    end = min((xcd + 1) * chunk, total);
    // (n-tiles past the last multiple of 4: blocks of 8 (m) x 1..3 (n) after all the others; 8192 x 29440 x 8192, 115
    // n-tiles: 2.33 -> 2.7 PFLOP/s against the plain m-major order)
    blocked = (tiles_m & 7) == 0 && tiles_n >= 4;
    bulk_tiles = tiles_m * (tiles_n & ~3);
  }
  __device__ __forceinline__ void coords(int t, int& m0, int& n0) const {
    int mt, nt;
    if (blocked && t < bulk_tiles) {
      const int sb = t >> 5, w = t & 31;
      mt = (sb % (tiles_m >> 3)) * 8 + (w & 7);
      nt = (sb / (tiles_m >> 3)) * 4 + (w >> 3);
    } else if (blocked) {
      const int u = t - bulk_tiles, bs = 8 * (tiles_n & 3), sb = u / bs, w = u - sb * bs;
      mt = sb * 8 + (w & 7);
      nt = (tiles_n & ~3) + (w >> 3);
    } else {
      mt = t % tiles_m;
      nt = t / tiles_m;
    }
    m0 = mt * BM;
    n0 = nt * BN;
  }
};

// RAGGED_K: K is a multiple of 32 but not of 128.  The last K step of a tile then holds K % 128 elements per row: the
// lanes whose 16 bytes lie past the end of the row load the row's last ones again, and the scale bytes of the blocks past K
// are replaced by 2^-127 in both operands: what such a lane multiplies is the row's own data (a NaN among them has made the
// row's results NaN already) times 2^-254, below the smallest fp32 number, so that the step adds exact zeros.  No branch in
// the K loop: with the lanes' loads predicated and zeros written instead, every load of every step was a block of code of
// its own (1024 x 5632 x 2880: 31.2 us, against 24.3 for K = 2816; now 29.6 us).

// 256x256 tiles are bound by the power limit of the MFMAs: 8192^3 2.93 PFLOP/s, 394 -> 376 us against a K loop of 32x32 MFMAs
// with all of a step's loads in one half of it.  The smaller tiles, for shapes whose large ones would leave compute units
// idle, move more through LDS per MFMA (a 128x256 step at the rates measured for its parts: 1024 cycles of MFMAs, 1562 of reads
// and loads) and, where the operands come from memory, wait for the loads: three and four buffers.  Weights that change from
// call to call, before (two buffers) and now, us: 1024 x 4096 x 4096 45 -> 22 and 512 x 8192 x 4096 46 -> 23 (128x128), 1979 x
// 7040 x 8416 157 -> 110, 330 x 9856 x 2688 37 -> 17, 1000 x 5760 x 2880 36 -> 27; 336 shapes of 129..8192 rows 1.23 times as
// fast in the geometric mean.
// The scales of a step travel like its operands: 2 KiB of 128x4 tiles (two of A, two of B) by LDS-direct loads, of which
// every wavefront reads the pieces of its rows and keeps its lane group's byte.
template <int NI, int NJ>
struct Tiles {
  static constexpr int BM = 32 * NI, BN = 32 * NJ;
  static constexpr int NBUF = NI + NJ > 12 ? 2 : NI + NJ > 8 ? 3 : 4;
  using Loop = TileLoop<Mma::kMxFp8, NI, NJ, NBUF>;
  static constexpr int kScaleBytes = 2048;                      // of a step: [operand][128-row tile][row % 32][16]
  static constexpr int kStageRows = NBUF == 3 ? 16 : 32;        // rows that the epilogue turns round at a time
  static constexpr int kStageBytes = kStageRows * 144;          // ... of a wavefront
  static constexpr int kLdsBytes = Loop::kTileBytes + NBUF * kScaleBytes + 4 * kStageBytes;
  static_assert(kLdsBytes <= 160 * 1024, "LDS");
};

template <int NI, int NJ, bool OUT_BF16, bool STREAM_OUT, bool RAGGED_K, bool RAGGED>
__global__ __launch_bounds__(256, 1) void mxfp8_tile_kernel(const Params p) {
  using T = Tiles<NI, NJ>;
  using Loop = typename T::Loop;
  constexpr int BM = T::BM, BN = T::BN, NBUF = T::NBUF, kScaleBytes = T::kScaleBytes;
  extern __shared__ u32x4 lds[];  // operand tiles | scales of NBUF steps | the epilogue's
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const TileWalk<BM, BN, RAGGED> walk(p);
  if (walk.first >= walk.end) return;
  const int nk = (p.k + 127) >> 7;
  const int sf_tiles_k = ((p.k >> 5) + 3) >> 2;  // 512-byte scale tiles per 128-row tile
  const int k_tail = p.k & 127;                  // elements of the last step (RAGGED_K: 32, 64 or 96)

  // ---- LDS-direct loads of a step.  A load is 8 rows: lane L lands at unit +L, i.e. row +(L>>3), chunk position L&7, which
  // must hold global chunk (L&7) ^ ((row>>1)&7) = (L&7) ^ ((L>>4) | ((j&1)<<2)) of load j.  The scales: A's by the even
  // wavefronts, B's by the odd ones, lanes 0..31 the first 128-row tile's, lanes 32..63 the second's (where there is one).
  const uint32_t lds_base = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)lds);
  const uint32_t chunk_even = (uint32_t)((lane & 7) ^ (lane >> 4)), chunk_odd = chunk_even ^ 4u;
  // the wavefront's share: rows of A's first half (the second's: 8 NI rows further on), of B
  const int a_row0 = wm * (16 * NI) + wn * (4 * NI), b_row0 = wave * (8 * NJ);
  const uint32_t a_lds = lds_base + (uint32_t)a_row0 * 128u, b_lds = lds_base + NBUF * Loop::kABytes + (uint32_t)b_row0 * 128u;
  const uint32_t s_lds = lds_base + Loop::kTileBytes + (uint32_t)wn * 1024u;
  uint32_t a_off[NI], b_off[NJ], s_off;
  // RAGGED_K: what takes an offset to the row's last chunk in the last step, where the lane's is past it
  const uint32_t last_chunk = (uint32_t)(k_tail >> 4) - 1u;
  const uint32_t tail_even = (min(chunk_even, last_chunk) - chunk_even) * 16u, tail_odd = (min(chunk_odd, last_chunk) - chunk_odd) * 16u;
  uint32_t sub_even = 0, sub_odd = 0;

  // ---- load stream: the step the next loads are issued for (l_ks of the tile lp), and the tile after it
  struct TilePtrs { const uint8_t *a, *b, *s; int rows, cols; };
  auto tile_ptrs = [&](int t) {
    int m0, n0;
    walk.coords(t, m0, n0);
    TilePtrs r;
    r.a = p.a + (int64_t)m0 * p.k;
    r.b = p.b + (int64_t)n0 * p.k;
    r.s = wn ? p.sfb + (int64_t)(n0 >> 7) * sf_tiles_k * 512 : p.sfa + (int64_t)(m0 >> 7) * sf_tiles_k * 512;
    r.rows = p.m - m0;  // rows and columns of the tile that exist (RAGGED: possibly fewer than BM, BN)
    r.cols = p.n - n0;
    return r;
  };
  TilePtrs lp = tile_ptrs(walk.first), np = lp;
  int l_ks = 0, l_buf = 0;
  uint32_t l_a = a_lds, l_b = b_lds, l_s = s_lds;  // the step's buffer
  auto enter_tile = [&]() {
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      uint32_t row = (uint32_t)(a_row0 + (u < NI / 2 ? 0 : 4 * NI) + 8 * u + (lane >> 3));
      if (RAGGED) row = min(row, (uint32_t)(lp.rows - 1));
      a_off[u] = row * (uint32_t)p.k + ((u & 1) ? chunk_odd : chunk_even) * 16u;
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      uint32_t row = (uint32_t)(b_row0 + 8 * j + (lane >> 3));
      if (RAGGED) row = min(row, (uint32_t)(lp.cols - 1));
      b_off[j] = row * (uint32_t)p.k + ((j & 1) ? chunk_odd : chunk_even) * 16u;
    }
    const bool second = (wn ? BN : BM) > 128 && (!RAGGED || (wn ? lp.cols : lp.rows) > 128);
    s_off = (uint32_t)(lane & 31) * 16u + (lane >= 32 && second ? (uint32_t)sf_tiles_k * 512u : 0u);
  };
  enter_tile();
  auto load = [&](auto code) {
    constexpr int u = decltype(code)::value;
    if constexpr (u == kLoadScales) {
      lds_dma16(l_s, lp.s, s_off);
    } else {
      const uint32_t sub = RAGGED_K ? ((u & 1) ? sub_odd : sub_even) : 0u;
      if constexpr (u >= kLoadB) lds_dma16<(u - kLoadB) * 1024>(l_b, lp.b, b_off[u - kLoadB] + sub);
      else lds_dma16<(u + (u < NI / 2 ? 0 : NI / 2)) * 1024>(l_a, lp.a, a_off[u] + sub);
    }
  };
  auto load_step = [&]() {  // in the order of the loop's
    static_for<NI / 2>(load);
    static_for<NJ>([&](auto j) { load(std::integral_constant<int, kLoadB + decltype(j)::value>{}); });
    load(std::integral_constant<int, kLoadScales>{});
    static_for<NI / 2>([&](auto u) { load(std::integral_constant<int, NI / 2 + decltype(u)::value>{}); });
  };
  auto advance = [&]() {
    const int by = l_buf == NBUF - 1 ? 1 - NBUF : 1;
    l_buf += by;
    l_a += by * Loop::kABytes;
    l_b += by * Loop::kBBytes;
    l_s += by * kScaleBytes;
    lp.a += 128;
    lp.b += 128;
    lp.s += 512;
    ++l_ks;
    if (RAGGED_K) {
      sub_even = l_ks == nk - 1 ? tail_even : 0u;
      sub_odd = l_ks == nk - 1 ? tail_odd : 0u;
    }
    if (l_ks == nk) {
      l_ks = 0;
      lp = np;
      if (RAGGED) enter_tile();
    }
  };

  Loop loop;
  loop.init(lds_base, lane, wm, wn);

  // ---- scales of the next step: the lane's rows r (even tiles) and 16 + r (odd ones) of its 128-row tile, whose 16 bytes are
  // 4 words for the rows 32 apart; byte g of each is the lane group's, and those of a wavefront's tiles are one operand register
  uint32_t s_rd[2];
  u32x4 words[2][2];
  uint32_t next_s[2][2];  // [operand][even, odd tiles]
  {
    const uint32_t at = lds_base + Loop::kTileBytes + (uint32_t)(lane & 15) * 16u;
    s_rd[0] = at + (uint32_t)wm * (NI == 8 ? 512u : 8u);  // (4 tiles: the first or second two words of the one scale tile)
    s_rd[1] = at + 1024u + (uint32_t)wn * (NJ == 8 ? 512u : 8u);
  }
  const uint32_t g = (uint32_t)lane >> 4, pick_low = 0x0c0c0400u + g * 0x0101u, pick_high = 0x04000c0cu + g * 0x01010000u;
  const uint32_t tail_keep = (int)g * 32 < k_tail ? 0xffffffffu : 0u;  // RAGGED_K: the lane group's block exists in the last step
  int s_buf = 0;  // of the scales to be read
  auto read_scales = [&]() {
#pragma unroll
    for (int op = 0; op < 2; ++op)
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        if ((op ? NJ : NI) == 8) {
          words[op][o] = loop.lds_read(s_rd[op] + o * 256u);
        } else {
          const u32x2 two = *(__attribute__((address_space(3))) const u32x2*)(uintptr_t)(s_rd[op] + o * 256u);
          words[op][o] = u32x4{two[0], two[1], 0u, 0u};
        }
      }
    const int by = s_buf == NBUF - 1 ? 1 - NBUF : 1;
    s_buf += by;
    s_rd[0] += by * kScaleBytes;
    s_rd[1] += by * kScaleBytes;
  };
  auto combine_scales = [&](int op, bool tail) {
#pragma unroll
    for (int o = 0; o < 2; ++o) {
      const u32x4 w = words[op][o];
      next_s[op][o] = __builtin_amdgcn_perm(w[1], w[0], pick_low);
      if ((op ? NJ : NI) == 8) next_s[op][o] |= __builtin_amdgcn_perm(w[3], w[2], pick_high);
      if (RAGGED_K && tail) next_s[op][o] &= tail_keep;
    }
  };
  auto take_scales = [&]() {
#pragma unroll
    for (int o = 0; o < 2; ++o) {
      loop.sa[o] = next_s[0][o];
      loop.sb[o] = next_s[1][o];
    }
    // two wait states between the registers' writing and the first MFMA
    asm volatile("s_nop 1" : "+v"(loop.sa[0]), "+v"(loop.sa[1]), "+v"(loop.sb[0]), "+v"(loop.sb[1]));
  };

  // The stream runs NBUF steps ahead of the MFMAs: it enters the tile after the next before the next has begun where a tile
  // has that few steps.  (c: the tile being computed, in steps of its list; past the end: a valid tile, loaded and ignored)
  const TilePtrs first_lp = lp;
  int stream_tile = walk.first;
  auto prepare_next = [&]() {
    stream_tile += walk.slots;
    np = stream_tile < walk.end ? tile_ptrs(stream_tile) : first_lp;
  };
  prepare_next();
  auto advance_and_prepare = [&]() {
    advance();
    if (l_ks == 0) prepare_next();
  };
  for (int i = 0; i < NBUF; ++i) {
    load_step();
    advance_and_prepare();
  }
  loop.fence();
  loop.first_fragments();
  read_scales();
  combine_scales(0, nk == 1);
  combine_scales(1, nk == 1);
  take_scales();

  const float alpha = p.alpha[0];
  for (int c_tile = walk.first; c_tile < walk.end; c_tile += walk.slots) {
    auto step = [&](auto first, int c_ks) {
      loop.template step<decltype(first)::value>(load, [&](auto part) {
        if constexpr (decltype(part)::value == 0) read_scales();
        if constexpr (decltype(part)::value == 1) combine_scales(0, c_ks + 2 == nk);
        if constexpr (decltype(part)::value == 2) combine_scales(1, c_ks + 2 == nk);
      });
      take_scales();
      advance_and_prepare();
    };
    step(std::true_type{}, 0);
    for (int c_ks = 1; c_ks < nk; ++c_ks) step(std::false_type{}, c_ks);
    loop.settle();
    // ---- epilogue of this tile; the loads of the next steps are already in flight.
    // A lane holds 8-byte pieces of 16 rows per tile; stored like that, a tile is 8192 sixteen-byte write
    // requests per compute unit and the L2 takes longer over them than over a whole K step of MFMAs.  Every
    // block of 32 (16) rows x 64 columns of the wavefront's tile is therefore turned round in a private piece of LDS (rows of
    // 128 bytes at a pitch of 144 bytes) and leaves in 16-byte pieces, 8 lanes to a row's 128 bytes.  One LDS address
    // each for writing and reading (the rest are immediate offsets) and one 32-bit lane offset next to a
    // wave-uniform result address; the lane number passes through an empty asm statement so that they are worked
    // out here, after the K loop.
    constexpr int kRowTiles = T::kStageRows / 16;
    int m0, n0;
    walk.coords(c_tile, m0, n0);
    int elane = lane;
    asm volatile("" : "+v"(elane));
    uint8_t* stage = reinterpret_cast<uint8_t*>(lds) + Loop::kTileBytes + NBUF * kScaleBytes + wave * T::kStageBytes;
    uint8_t* wr = stage + (elane & 15) * 144 + (elane >> 4) * 8;
    const uint8_t* rd = stage + (elane >> 3) * 144 + (elane & 7) * 16;
    const int ldc = p.out_pitch();
    const uint32_t ooff = ((uint32_t)(elane >> 3) * (uint32_t)ldc + (uint32_t)(elane & 7) * 8u) * 2u;
    uint8_t* obase = reinterpret_cast<uint8_t*>(static_cast<uint16_t*>(p.out) + (int64_t)(m0 + wm * (16 * NI)) * ldc + n0 + wn * (16 * NJ));
    // RAGGED: rows and columns from this lane's first ones to the end
    const int rows_left = p.m - m0 - wm * (16 * NI) - (elane >> 3), cols_left = p.n - n0 - wn * (16 * NJ) - (elane & 7) * 8;
#pragma unroll
    for (int i = 0; i < NI; i += kRowTiles) {
#pragma unroll
      for (int jh = 0; jh < NJ / 4; ++jh) {
#pragma unroll
        for (int t = 0; t < 4 * kRowTiles; ++t) {  // the block's tiles
          const f32x4 c = loop.acc[i + (t >> 2)][4 * jh + (t & 3)];
          u32x2 v;
          v[0] = pack2(c[0] * alpha, c[1] * alpha, OUT_BF16);
          v[1] = pack2(c[2] * alpha, c[3] * alpha, OUT_BF16);
          *reinterpret_cast<u32x2*>(wr + (t >> 2) * 2304 + (t & 3) * 32) = v;
        }
        asm volatile("" ::: "memory");  // the reads below see the writes above: one wavefront's LDS accesses stay in order
#pragma unroll
        for (int t = 0; t < 2 * kRowTiles; ++t) {
          const u32x4 v = *reinterpret_cast<const u32x4*>(rd + t * 1152);
          u32x4* dst = reinterpret_cast<u32x4*>(obase + ((int64_t)(i * 16 + 8 * t) * ldc + jh * 64) * 2 + ooff);
          if (RAGGED && (i * 16 + 8 * t >= rows_left || jh * 64 >= cols_left)) continue;
          if constexpr (STREAM_OUT) __builtin_nontemporal_store(v, dst);
          else *dst = v;
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);  // (the next block's results stay in the accumulators until then)
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no LDS-direct load may outlive the workgroup
}

template <int NI, int NJ, bool OUT_BF16, bool STREAM_OUT, bool RAGGED_K, bool RAGGED>
int launch_tiles_cfg(const Params& p, hipStream_t stream) {
  using T = Tiles<NI, NJ>;
  auto kern = mxfp8_tile_kernel<NI, NJ, OUT_BF16, STREAM_OUT, RAGGED_K, RAGGED>;
  const int64_t tiles = ceil_div(p.m, T::BM) * ceil_div(p.n, T::BN);
  if (!RAGGED && (p.m % T::BM != 0 || p.n % T::BN != 0))
    return fail(NVF_ERR_LAUNCH, "mxfp8_tile_kernel: %d x %d is no multiple of %d x %d", p.m, p.n, T::BM, T::BN);
  const int cus = cu_count() & ~7;  // workgroup ids are dealt round-robin to the 8 XCDs
  const unsigned grid = (unsigned)(tiles >= cus ? cus : ((tiles + 7) / 8) * 8);
  if (note_launch("mxfp8_tile_kernel<%dx%d,stream_out=%d%s%s%s> grid=%u", T::BM, T::BN, (int)STREAM_OUT, RAGGED_K ? ",ragged_k" : "",
                  p.m % T::BM ? ",ragged_m" : "", p.n % T::BN ? ",ragged_n" : "", grid))
    return NVF_OK;
  static std::atomic<uint64_t> configured{0};  // one bit per device (and per instantiation of this launcher)
  if (const int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), T::kLdsBytes, configured)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256), T::kLdsBytes, stream, p);
  return check_launch("mxfp8_tile_kernel");
}

template <int NI, int NJ, bool OUT_BF16>
int launch_tiles(const Params& p, hipStream_t stream) {
  // Operands and result together beyond what the 256 MB last-level cache holds: the result would push the
  // operand panels out of it (and out of the L2s) on its way to memory, so it leaves with non-temporal stores
  // (8192^3: +5 %, 16384 x 16384 x 2048: +17 %; smaller problems lose 1-5 % that way).  128x128 tiles are for small ones.
  const bool ragged = p.m % (32 * NI) != 0 || p.n % (32 * NJ) != 0, ragged_k = (p.k & 127) != 0;
  if constexpr (NJ == 8) {
    if (((int64_t)p.m + p.n) * p.k + 2 * (int64_t)p.m * p.n > (int64_t)224 << 20) {
      if (ragged) return ragged_k ? launch_tiles_cfg<NI, NJ, OUT_BF16, true, true, true>(p, stream) : launch_tiles_cfg<NI, NJ, OUT_BF16, true, false, true>(p, stream);
      return ragged_k ? launch_tiles_cfg<NI, NJ, OUT_BF16, true, true, false>(p, stream) : launch_tiles_cfg<NI, NJ, OUT_BF16, true, false, false>(p, stream);
    }
  }
  if (ragged) return ragged_k ? launch_tiles_cfg<NI, NJ, OUT_BF16, false, true, true>(p, stream) : launch_tiles_cfg<NI, NJ, OUT_BF16, false, false, true>(p, stream);
  return ragged_k ? launch_tiles_cfg<NI, NJ, OUT_BF16, false, true, false>(p, stream) : launch_tiles_cfg<NI, NJ, OUT_BF16, false, false, false>(p, stream);
}

// -------------------------------------------------------------------------------------------------
// Skinny path: slabs of up to 128 activation rows (decode-sized activations; more rows as several slabs, the
// whole ones side by side in one launch, blockIdx.y = slab), K % 32 == 0, N % (16*RT) == 0.  A slab streams
// the weight matrix exactly once, so the op is bound by HBM (by the last-level cache for the slabs after the
// first):
//   * A workgroup owns 16*RT weight rows for the whole of K and all M activation rows; its W = 8 wavefronts
//     (4 in the form of which two workgroups share a compute unit) split K in interleaved 128-element chunks and their partial sums are added in a fixed order through
//     LDS (no atomics, no workspace, deterministic).
//   * v_mfma_scale_f32_16x16x128_f8f6f4, measured operand layout: lane (i, g) = i + 16 g supplies row i,
//     bytes 0..15 = K [16g, 16g+16) and bytes 16..31 = K [64+16g, 64+16g+16); the scale byte of lane
//     (i, j) applies to row i, K-block j.  Weight rows are the first operand, so a lane ends up with 4
//     consecutive N-elements of one output row.
//   * A load in that lane order would touch 64 unrelated 16-byte pieces per instruction, which the address
//     unit handles one by one.  Every wavefront therefore fetches its tiles with LDS-direct loads in memory
//     order (8 neighbouring lanes = the 128 contiguous bytes of a row's chunk; the scales as the 256
//     contiguous bytes that hold a 16-row tile's scale words) into a private ring of DEPTH slots in LDS and
//     reads them back in MFMA lane order; no barrier in the K loop, a wavefront reads only what it loaded.
//   LDS per slot: NT tiles of 16 rows x 128 B (piece p of row r at position p ^ ((r >> 1) & 7): conflict-free
//   reads), then 256 B of scale words per tile.
// -------------------------------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));

// (W = 4, 4 x 4 tiles: 168 VGPRs + 64 AGPRs as compiled, so two workgroups fit a compute unit.  Asking for 2 wavefronts per
// SIMD in the launch bounds moves the accumulators into the VGPRs: 96 x 16384 x 4096 19.1 -> 21.8 us, 512 x 4096 x 7168 28.2 ->
// 26.1, others equal; not done.)
template <int RT, int TT, bool OUT_BF16, int DEPTH, bool RAGGED_K = false, int W = 8>
__global__ __launch_bounds__(W * 64) void mxfp8_skinny_kernel(const Params p) {
  constexpr int NT = RT + TT;
  // activation rows r and r + 32 share their 16-byte scale group, so 32 groups serve any number of tiles
  constexpr int A_SC_BYTES = (TT < 2 ? TT : 2) * 256;
  constexpr int SLOT_BYTES = NT * 2048 + RT * 256 + A_SC_BYTES;
  constexpr int NDMA = 2 * NT + 2;  // loads per chunk and wavefront
  static_assert(DEPTH >= 1 && DEPTH <= 3 && W * DEPTH * SLOT_BYTES <= 160 * 1024 && DEPTH * NDMA <= 63 && RT <= 4 && TT <= 8,
                "ring does not fit");
  extern __shared__ u32x4 lds[];  // ring during the K loop, then [W][tiles][64 lanes] partial sums
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * (16 * RT);
  // activation rows of this workgroup: [m_base, m_base + m_loc); blockIdx.y counts slabs of 16*TT rows
  const int m_base = p.m_base + (int)blockIdx.y * (16 * TT);
  const int m_loc = min(p.m - m_base, 16 * TT);
  const int tt_count = (m_loc + 15) >> 4;
  // K % 128 = 32, 64 or 96: the last chunk is short.  Lanes whose 16 bytes lie past the end of the row write zeros to
  // their LDS unit instead of loading, and the scale bytes of the blocks past K (padding columns of the scale layout,
  // content not defined) are replaced by 2^0, so that the chunk adds exact zeros for them.
  const int chunks = (p.k + 127) >> 7;
  const int k_tail = p.k & 127;
  const int tail_chunk = RAGGED_K ? chunks - 1 : -1;  // (a kernel of its own: K % 128 != 0)
  const int sf_padded = ((p.k >> 5) + 3) & ~3;  // scale columns with the layout's padding

  // ---- load side (memory order).  Payload: tile t, load j (rows 8j..8j+7): lane L = row 8j + L/8, piece
  // (L & 7) ^ ((4j + L/16) & 7).  Scales: lane L = tile L/16, row L%16: the 16 bytes that hold the scale
  // words of rows {row, row+32, row+64, row+96} (mod 128) for the chunk's 4 K-blocks.
  const uint8_t* b_base = p.b + (int64_t)n0 * p.k;
  const uint8_t* bsf_base = p.sfb + (int64_t)(n0 >> 7) * ((int64_t)sf_padded << 7);
  uint32_t b_off[RT][2], a_off[TT][2];
  bool in_tail[2];  // does the lane's piece of load j exist in a short last chunk?
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int row = 8 * j + (lane >> 3);
    const uint32_t piece = (uint32_t)((lane & 7) ^ ((4 * j + (lane >> 4)) & 7)) * 16u;
    in_tail[j] = (int)piece < k_tail;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) b_off[rt][j] = (uint32_t)(rt * 16 + row) * (uint32_t)p.k + piece;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) a_off[tt][j] = (uint32_t)min(tt * 16 + row, m_loc - 1) * (uint32_t)p.k + piece;
  }
  const int st = lane >> 4;  // tile whose scales this lane fetches
  const uint32_t bsf_off = (uint32_t)((((n0 & 127) + min(st, RT - 1) * 16 + r) & 31) * 16);
  const uint8_t* a_base = p.a + (int64_t)m_base * p.k;
  const uint8_t* asf_base = p.sfa + (int64_t)(m_base >> 7) * ((int64_t)sf_padded << 7);
  const uint32_t asf_off = (uint32_t)((lane & 31) * 16);  // scale group of rows {lane, lane + 32, ...} of the 128-row tile
  const uint32_t lds_base = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)lds);
  const uint32_t ring_base = lds_base + (uint32_t)wave * (DEPTH * SLOT_BYTES);
  auto issue_chunk = [&](int c_in, int slot) {  // c_in is wave-uniform
    if (c_in >= chunks) return;
    const uint32_t c = (uint32_t)c_in;
    const uint32_t sb = ring_base + (uint32_t)slot * SLOT_BYTES;
    if (RAGGED_K && c_in == tail_chunk) {
      char* const zp = reinterpret_cast<char*>(lds) + (sb - lds_base) + lane * 16;
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if (in_tail[j]) lds_dma16(sb + t * 2048 + j * 1024, t < RT ? b_base : a_base, (t < RT ? b_off[t][j] : a_off[t - RT][j]) + c * 128u);
          else *reinterpret_cast<u32x4*>(zp + t * 2048 + j * 1024) = u32x4{0, 0, 0, 0};
        }
    } else {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int j = 0; j < 2; ++j) lds_dma16(sb + rt * 2048 + j * 1024, b_base, b_off[rt][j] + c * 128u);
#pragma unroll
      for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int j = 0; j < 2; ++j) lds_dma16(sb + (RT + tt) * 2048 + j * 1024, a_base, a_off[tt][j] + c * 128u);
    }
    // one load each for the scales of all weight tiles / all activation tiles (lanes of tiles that do not
    // exist stay off: a disabled lane writes nothing)
    if (lane < 16 * RT) lds_dma16(sb + NT * 2048, bsf_base, bsf_off + c * 512u);
    if (lane < A_SC_BYTES / 16) lds_dma16(sb + NT * 2048 + RT * 256, asf_base, asf_off + c * 512u);
  };

  // ---- read side (MFMA order)
  const int rd_lo = r * 128 + ((g ^ ((r >> 1) & 7)) * 16);
  const int rd_hi = r * 128 + (((g + 4) ^ ((r >> 1) & 7)) * 16);
  int rd_bsc[RT], rd_asc[TT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) rd_bsc[rt] = NT * 2048 + rt * 256 + r * 16 + ((((n0 & 127) + rt * 16) >> 5) & 3) * 4;
#pragma unroll
  for (int tt = 0; tt < TT; ++tt)
    rd_asc[tt] = NT * 2048 + RT * 256 + ((tt & 1) * 16 + r) * 16 + ((((m_base & 127) + tt * 16) >> 5) & 3) * 4;
  const int sc_shift = g * 8;

  f32x4 acc[RT][TT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) acc[rt][tt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

#pragma unroll
  for (int d = 0; d < DEPTH; ++d) issue_chunk(wave + d * W, d);
  int slot = 0;
  for (int c = wave; c < chunks; c += W) {
    // the oldest chunk in flight has landed when only the loads of the younger ones are pending
    const int younger = min(DEPTH - 1, (chunks - 1 - c) / W);
    if (younger >= 2)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(DEPTH >= 3 ? 2 * NDMA : 0) : "memory");
    else if (younger == 1)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(DEPTH >= 2 ? NDMA : 0) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const char* sp = reinterpret_cast<const char*>(lds) + (wave * DEPTH + slot) * SLOT_BYTES;
    u32x4 lo[NT], hi[NT];
    uint32_t sc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      lo[t] = *reinterpret_cast<const u32x4*>(sp + t * 2048 + rd_lo);
      hi[t] = *reinterpret_cast<const u32x4*>(sp + t * 2048 + rd_hi);
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) sc[rt] = *reinterpret_cast<const uint32_t*>(sp + rd_bsc[rt]) >> sc_shift;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) sc[RT + tt] = *reinterpret_cast<const uint32_t*>(sp + rd_asc[tt]) >> sc_shift;
    if (RAGGED_K && c == tail_chunk && g * 32 >= k_tail) {  // this lane's K-block lies past K
#pragma unroll
      for (int t = 0; t < NT; ++t) sc[t] = 0x7f;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read out: the slot may be refilled
    issue_chunk(c + DEPTH * W, slot);
    slot = (slot + 1 == DEPTH) ? 0 : slot + 1;
    auto frag = [&](int t) {
      return i32x8{(int)lo[t][0], (int)lo[t][1], (int)lo[t][2], (int)lo[t][3], (int)hi[t][0], (int)hi[t][1], (int)hi[t][2], (int)hi[t][3]};
    };
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
      if (tt < tt_count) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
          acc[rt][tt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(frag(rt), frag(RT + tt), acc[rt][tt], 0, 0, 0, (int)sc[rt], 0,
                                                                         (int)sc[RT + tt]);
      }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no LDS-direct load may be pending when the ring is reused
  __syncthreads();

  // ---- sum the wavefronts' partial tiles in wave order and store (RT * TT <= 16 tiles of 1 KiB per wave)
  f32x4* red = reinterpret_cast<f32x4*>(lds);
  const float alpha = p.alpha[0];
  uint16_t* out = static_cast<uint16_t*>(p.out);
  const int tiles = RT * tt_count;  // tile index: rt * tt_count + tt
  const int units = tiles * 64;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
      if (tt < tt_count) red[(wave * tiles + rt * tt_count + tt) * 64 + lane] = acc[rt][tt];
  __syncthreads();
  for (int u = tid; u < units; u += W * 64) {
    const int l = u & 63, tile = u >> 6;
    const int rt = tile / tt_count, tt = tile - rt * tt_count;
    f32x4 s = red[u];
#pragma unroll
    for (int w = 1; w < W; ++w) s += red[w * units + u];
    // element e of lane l: weight row 4*(l/16) + e (output column), activation row l%16 (output row)
    const int tok = tt * 16 + (l & 15);
    if (tok < m_loc) {
      u32x2 v;
      v[0] = pack2(s[0] * alpha, s[1] * alpha, OUT_BF16);
      v[1] = pack2(s[2] * alpha, s[3] * alpha, OUT_BF16);
      *reinterpret_cast<u32x2*>(out + (int64_t)(m_base + tok) * p.out_pitch() + n0 + rt * 16 + 4 * (l >> 4)) = v;
    }
  }
}

template <int RT, int TT, bool OUT_BF16, int W = 8>
int launch_skinny_cfg(const Params& p, hipStream_t stream, int slabs = 1) {
  constexpr int SLOT = (RT + TT) * 2048 + RT * 256 + (TT < 2 ? TT : 2) * 256;
  constexpr int DEPTH = W != 8 ? 1 : 8 * 3 * SLOT <= 160 * 1024 ? 3 : (8 * 2 * SLOT <= 160 * 1024 ? 2 : 1);
  // (4 wavefronts: K % 128 == 0 only, and a ring of one slot, so that two workgroups share a compute unit's LDS)
  if (W != 8 && (p.k & 127) != 0) return fail(NVF_ERR_UNSUPPORTED_SHAPE, "mxfp8_skinny_kernel: 4 wavefronts need K % 128 == 0");
  auto kern = W == 8 && (p.k & 127) != 0 ? mxfp8_skinny_kernel<RT, TT, OUT_BF16, DEPTH, W == 8, W> : mxfp8_skinny_kernel<RT, TT, OUT_BF16, DEPTH, false, W>;
  constexpr int ring = W * DEPTH * SLOT, red = W * RT * TT * 1024;
  constexpr int lds_bytes = ring > red ? ring : red;
  static_assert(lds_bytes <= 160 * 1024, "LDS");
  if (note_launch("mxfp8_skinny_kernel<RT=%d,TT=%d%s> grid=%ux%d m_base=%d", RT, TT, W == 4 ? ",W=4" : "", (unsigned)(p.n / (16 * RT)), slabs, p.m_base)) return NVF_OK;
  static std::atomic<uint64_t> configured[2] = {{0}, {0}};  // per kernel, one bit per device
  if (const int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds_bytes, configured[(p.k & 127) != 0])) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)(p.n / (16 * RT)), (unsigned)slabs), dim3(W * 64), lds_bytes, stream, p);
  return check_launch("mxfp8_skinny_kernel");
}

template <int TT, bool OUT_BF16>
int launch_skinny_rt(const Params& p, int rt, hipStream_t stream, int slabs) {
  if constexpr (TT == 8) return launch_skinny_cfg<1, 8, OUT_BF16>(p, stream, slabs);
  else
    return rt == 4 ? launch_skinny_cfg<4, TT, OUT_BF16>(p, stream, slabs)
         : rt == 2 ? launch_skinny_cfg<2, TT, OUT_BF16>(p, stream, slabs)
                   : launch_skinny_cfg<1, TT, OUT_BF16>(p, stream, slabs);
}

// Estimated duration of the skinny kernel for (slab height, weight tiles per workgroup), in units of about 1 ns: the
// workgroups (one per slab and 16*rt weight rows; one per compute unit at a time, the ring fills its LDS) run in
// rounds over the compute units; a wavefront visits ceil(chunks / 8) chunks, each costing the LDS-direct loads of
// its rt + tt tiles and rt * tt MFMAs, then comes the reduction of rt * tt partial tiles.  A last round that is only
// partly filled costs 70 % of a full one plus its share of the rest; the weight stream bounds the whole from below.
// Constants fitted to a sweep of the seven forms over 140 shapes (M 48..256, N 1024..14336, K 2048..14336): the form
// picked is within 7 % of the best everywhere.
// (duration: the estimate is compared with another kernel's; then a round of workgroups streams the weight rows it
// covers, not all of them - with 28672 weight rows a slab takes two rounds, which made the other floor twice the
// measured time; the choice of the form keeps the floor it was fitted with)
// (w = 4: the form with 4 wavefronts and a ring of one slot, 64-row slabs x 4 weight tiles.  Two of its workgroups share
// a compute unit, so up to twice as many as there are compute units run in one round where the form with 8 wavefronts
// takes two; a wavefront then visits twice the chunks, each 27 % dearer.  Only for that case, and K % 128 == 0.
// Measured, 8 -> 4 wavefronts: 128 x 14336 x 4096 (448 workgroups) 25.4 -> 19.9 us, 64 x 28672 x 4096 26.0 -> 24.1,
// 256 x 7168 x 2048 12.7 -> 10.5, 192 x 7168 x 2048 (336) 11.9 -> 9.8; but with one round either way 256 x 4096 x 4096
// 10.6 -> 12.8 us, 256 x 4096 x 14336 24.9 -> 30.4.  Over the 234 of 2448 shapes (M 33..2048, N 1024..32896, K 512..14336)
// whose launch the form changes, the time falls by 16 % in the geometric mean, by 28-32 % at K <= 1024, where it also
// takes over from the persistent kernel: 160 x 8192 x 1024 10.8 -> 6.5 us.)
int64_t mxfp8_skinny_cost(int64_t m, int64_t n, int64_t k, int slab, int rt, int64_t cus, bool duration = false, int w = 8) {
  if ((slab == 128 && rt != 1) || n % (16 * rt) != 0) return INT64_MAX;
  if (w == 4) {
    const int64_t wgs4 = ceil_div(m, 64) * (n / 64);
    if (slab != 64 || rt != 4 || (n & 63) != 0 || (k & 127) != 0 || m <= 32 || wgs4 <= cus || wgs4 > 2 * cus) return INT64_MAX;
    // (a deep K makes the second, partly filled round of the other form cheap against its first: 96 x 12288 x 14336,
    // 384 workgroups, 51 -> 55 us; and many slabs of few columns gain nothing from K = 7168 on: 1024 x 2048 x 7168 28 -> 30 us)
    if ((k > 8192 && 4 * wgs4 < 7 * cus) || (k > 4096 && m > 8 * 64)) return INT64_MAX;
    const int64_t per_chunk4 = ((4 + 4) * 145 + 4 * 4 * 10 + 100) * 127 / 100;
    return std::max(2 * ceil_div(k >> 7, 8) * per_chunk4 + 4 * 4 * 193 + 2493, n * k / 5400);
  }
  const int64_t slabs = m <= slab ? 1 : ceil_div(m, slab);
  const int tt = m <= slab ? (m <= 16 ? 1 : m <= 32 ? 2 : m <= 64 ? 4 : 8) : slab / 16;
  if (tt == 8 && rt != 1) return INT64_MAX;
  const int64_t wgs = slabs * (n / (16 * rt));
  const int64_t chunks = ceil_div((k + 127) >> 7, 8);
  const int64_t per_chunk = (rt + tt) * 145 + rt * tt * 10 + 100;
  const int64_t wg_time = chunks * per_chunk + rt * tt * 193 + 2493;
  const int64_t full = wgs / cus, rest = wgs - full * cus;
  // every round of workgroups streams the weights again, out of the last-level cache at best: 5.6 TB/s
  // (256 x 14336 x 14336 as 4 slabs in 3.5 rounds: 123 us for 4 x 205 MB)
  const int64_t stream = ceil_div(wgs, cus) * (duration ? std::min<int64_t>(n, cus * 16 * rt) : n) * k / 5400;
  return std::max((full * 100 + (rest ? 70 + 30 * rest / cus : 0)) * wg_time / 100, stream);
}

// best form of the skinny kernel for more than 32 rows: estimated duration, slab height and weight tiles per workgroup
int64_t mxfp8_skinny_best(int64_t m, int64_t n, int64_t k, int64_t cus, int* slab_out, int* rt_out, int* w_out) {
  int slab = 128, rt = 1, w = 8;
  int64_t best = INT64_MAX;
  for (const int s : {32, 64, 128})  // (equal estimates: the lower slab, measured 2-9 % faster)
    for (const int r : {1, 2, 4}) {
      const int64_t c = mxfp8_skinny_cost(m, n, k, s, r, cus);
      if (c < best) best = c, slab = s, rt = r;
    }
  if (const int64_t c = mxfp8_skinny_cost(m, n, k, 64, 4, cus, false, 4); c < best) best = c, slab = 64, rt = 4, w = 4;
  if (slab_out) *slab_out = slab;
  if (rt_out) *rt_out = rt;
  if (w_out) *w_out = w;
  return best;
}
// Estimated duration of the form that mxfp8_skinny_best picks, in ns: what plans and cuts compare with the other kernels.
// From 129 rows on it is scaled to what the kernel takes when the weights change from call to call (150 shapes of 129..3000
// rows; measured / unscaled, median: K <= 1536 0.8, 2048 0.9, 4096 1.0, 7168 1.07, 8192..11008 1.2, 14336 1.2).  Workgroups go
// to the XCDs in turn: with a number of them per slab that is no multiple of 4 the slabs that share weight rows lie in
// different XCDs, each of which reads those rows again (measured / unscaled 1.54 for 256 x 2880 x 8192, 1.30 for
// 192 x 2560 x 8192; 1.31 for 640 x 2880 x 2880, 1.04 for 384 x 2560 x 2880).  With the scaled
// estimate the kernel picked is within 1 % of the fastest in the geometric mean over 336 shapes, 9 % at worst.
int64_t mxfp8_skinny_ns(int64_t m, int64_t n, int64_t k, int64_t cus) {
  int slab, rt, w;
  if (mxfp8_skinny_best(m, n, k, cus, &slab, &rt, &w) == INT64_MAX) return INT64_MAX;
  const int64_t ns = mxfp8_skinny_cost(m, n, k, slab, rt, cus, true, w) * 963 / 1000;
  if (m <= 128) return ns;  // (its constants were fitted there, with weights that stay)
  const int64_t percent = std::min<int64_t>({std::max<int64_t>(77, 50 + 20 * k / 1024), 80 + 5 * k / 1024, 125});
  return ns * percent / 100 * (n / (16 * rt) % 4 ? 5 : 4) / 4;
}

template <bool OUT_BF16>
int launch_skinny(const Params& p, hipStream_t stream) {
  // Up to 32 rows: one slab of 1 or 2 activation tiles (16 x 6144 x 4096: 8.0 us with 1 weight tile per workgroup in 1.5
  // rounds, 6.2 us with 2); more rows: slabs of 128, 64 or 32 rows side by side in one launch (blockIdx.y = slab; the last one may be ragged;
  // the slabs after the first find the weights in the last-level cache) with 1, 2 or 4 weight tiles per workgroup
  // (1 with 128-row slabs, whose 8 activation tiles fill the ring), whichever the estimate above prefers
  // (128 x 4096 x 4096: 10.5 us as one slab of 128 rows, 7.6 us as 4 slabs of 32 rows x 4 weight tiles;
  // 256 x 4096 x 14336: 49.9 -> 26.1 us; 128 x 8192 x 7168: 28.0 -> 16.6 us).
  int slab, rt, w;
  mxfp8_skinny_best(p.m, p.n, p.k, cu_count(), &slab, &rt, &w);
  // Decode sizes against weight rows a multiple of 8 KiB apart: 2 weight tiles per workgroup stream them slower than
  // 1 or 4 do (measured, 8 rows: 8192 x 8192 15.8 us with 2, 14.3 with 1, 12.6 with 4; 7168 x 8192 13.6 / 12.5 / 11.4;
  // other K: as estimated), so 4 where that still leaves 80 workgroups
  if (p.m <= 32 && rt == 2 && (p.k & 8191) == 0 && (p.n & 63) == 0 && p.n / 64 >= 80) rt = 4;
  const int slabs = p.m <= slab ? 1 : (int)ceil_div(p.m, slab);
  const int rows = p.m <= slab ? p.m : slab;
  if (w == 4) return launch_skinny_cfg<4, 4, OUT_BF16, 4>(p, stream, slabs);
  return rows <= 16 ? launch_skinny_rt<1, OUT_BF16>(p, rt, stream, slabs)
       : rows <= 32 ? launch_skinny_rt<2, OUT_BF16>(p, rt, stream, slabs)
       : rows <= 64 ? launch_skinny_rt<4, OUT_BF16>(p, rt, stream, slabs)
                    : launch_skinny_rt<8, OUT_BF16>(p, rt, stream, slabs);
}

template <int BM, int BN, bool OUT_BF16>
int launch_cfg(const Params& p, hipStream_t stream) {
  auto kern = mxfp8_gemm_kernel<BM, BN, OUT_BF16>;
  constexpr int lds_bytes = 2 * (BM + BN) * 128;
  const int64_t tiles = ceil_div(p.m, BM) * ceil_div(p.n, BN);
  if (note_launch("mxfp8_gemm_kernel<%d,%d> grid=%lld", BM, BN, (long long)tiles)) return NVF_OK;
  static std::atomic<uint64_t> configured{0};  // one bit per device
  if (const int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds_bytes, configured)) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3(256), lds_bytes, stream, p);
  return check_launch("mxfp8_gemm_kernel");
}

// Which kernel a shape gets: the weight-streaming kernel, the persistent kernel with one of three tiles, or - too few tiles, a
// shape that neither takes - the tile kernels.
enum class Plan { kStream, kTiles256, kTiles128, kTiles128x128, kOther };
// (ns: the estimated duration, where there is an estimate)
Plan mxfp8_plan(int64_t m, int64_t n, int64_t k, int64_t cus, int64_t* ns = nullptr) {
  if (ns) *ns = INT64_MAX;
  const bool skinny_ok = (k & 31) == 0 && (n & 15) == 0 && k * 64 < (1ll << 31);  // 32-bit lane offsets (a short last chunk is fine)
  // The persistent kernel takes any K % 32 == 0 (its last step may be short), a last row tile with fewer rows (which counts as a
  // whole one: 640 x 14336 x 4096 as 280 tiles of 128 rows in 2 rounds 60 us, 168 of 256 rows 43 us) and, measured from K = 1024
  // on, a last column tile with fewer columns (against a launch of its own for the remaining columns, us: 2048 x 6208 x 1408
  // 22.4 / 36.6, 640 rows of it 10.8 / 27.6, 2048 x 5760 x 2880 41.2 / 49.1, 768 x 2064 x 4096 19.0 / 34.5 streamed, 4096 x 11040
  // x 4096 155 / 159, 8192 x 29568 x 8192 1422 / 1450).
  const bool fast_shape = (k & 31) == 0 && k >= 256 && k * 256 < (1ll << 31) && (n & 15) == 0 && (m > 64 || (m & 127) == 0);
  auto tiles_of = [&](int64_t bm, int64_t bn) { return ceil_div(m, bm) * ceil_div(n, bn); };
  const bool columns_ok = (n & 255) == 0 || (m > 128 && n > 256 && k >= 1024);
  int64_t t256 = tiles_of(256, 256), t128 = tiles_of(128, 256), t128x128 = tiles_of(128, 128);
  if (!fast_shape || t256 < 128 || !columns_ok || !((m & 255) == 0 || m > 128)) t256 = 0;
  // 128x128 tiles: half the work per compute unit in 0.7 of the time, so they win up to a whole round of them, i.e. for half a
  // round of 128x256 tiles (512 x 8192 x 4096 24.1 against 31.3 us, 1024 x 4096 x 4096 23.3 / 29.6, 256 x 14336 x 4096 24.2 / 31.8,
  // 1000 x 4096 x 14336 72.6 / 99.5 and 110 streamed, 160 x 14336 x 4096 22.2 / 30.0 and 36 streamed, 948 x 3840 x 2560 15.4 / 21.5).
  if (!fast_shape || m <= 128 || !columns_ok || k < 512 || t128x128 < 16) t128x128 = 0;
  if (!fast_shape || t128 < 48 || !columns_ok) t128 = 0;
  // Measured with weights that change from call to call, us per 128-deep step of a round (a round of a few tiles, a full one)
  // and per call: 256x256 1.08, 1.48 and 7; 128x256 0.75, 0.95 and 5.2; 128x128 0.53, 0.60 and 2.8, and 0.7 per round besides
  // (300 x 14336 x 512 in two rounds 10.0, as one of 128x256 tiles 9.2; 1280 x 4096 x 768 11.5 / 10.6; but 4096 x 3072 x 512 in
  // three 12.6, as two of 128x256 tiles 13.6).
  auto tile_ns = [&](int64_t tiles, int64_t fixed, int64_t round, int64_t step, int64_t full) {
    if (tiles == 0) return (int64_t)INT64_MAX;
    const int64_t steps = (k + 127) >> 7, rounds = ceil_div(tiles, cus);
    return fixed + rounds * round + steps * (rounds * step + (full - step) * tiles / cus);
  };
  const int64_t ns256 = tile_ns(t256, 7000, 0, 1080, 1480), ns128 = tile_ns(t128, 5200, 0, 750, 950), ns128x128 = tile_ns(t128x128, 2800, 700, 530, 600);
  const int64_t fast_ns = std::min(ns256, std::min(ns128, ns128x128));
  const bool fast = fast_ns != INT64_MAX;
  if (skinny_ok) {
    const int64_t skinny_ns = mxfp8_skinny_ns(m, n, k, cus);
    if (ns) *ns = skinny_ns;
    if (m <= 32) return Plan::kStream;
    if (fast) {
      // Skinny or persistent kernel by estimated duration.  Measured: 512 x 4096 x 7168 36.7 (persistent) against 31.8 us,
      // 700 x 2304 x 5120 22.3 / 23.3, 512 x 4096 x 4096 18.2 / 18.7, 300 x 3072 x 2048 11.4 / 7.1, 1500 x 1408 x 7168 34 / 42.
      if (skinny_ns <= fast_ns) return Plan::kStream;
    } else {
      // No persistent kernel for the shape (ragged M or N, or too few tiles): up to 256 rows, i.e. four passes over
      // the weights, the skinny kernel beats the tile kernels (128 x 4096 x 14336: 20 instead of 117 us); with more
      // rows, a deep K and a small N it fills the chip where they cannot, while its 128-row x 16-column workgroups
      // cover the compute units at most 3 times (measured, K >= 2048).
      const int64_t skinny_rounds = ceil_div(ceil_div(m, 128) * (n / 16), cus);
      if (m <= 256 || (skinny_rounds <= 3 && k >= 2048)) return Plan::kStream;
    }
  }
  if (ns) *ns = fast_ns;
  if (fast) return fast_ns == ns256 ? Plan::kTiles256 : fast_ns == ns128 ? Plan::kTiles128 : Plan::kTiles128x128;
  return Plan::kOther;
}

template <bool OUT_BF16>
int launch_sized(const Params& p, hipStream_t stream) {
  auto tiles = [&](int bm, int bn) { return ceil_div(p.m, bm) * ceil_div(p.n, bn); };
  const int64_t cus = cu_count();
  int64_t whole_ns;
  const Plan whole = mxfp8_plan(p.m, p.n, p.k, cus, &whole_ns);
  // A cut along N or M competes with the kernel the whole shape gets: the tile kernels (no estimate) lose to any cut
  // that works; the weight-streaming kernel loses to a cut whose main part runs on the persistent kernel and is
  // estimated 5 % faster or more (384 x 29568 x 8192: 291 us on tiles, 256 x 29568 x 8192: 169 us streamed), and so do tiles
  // of which the last ones have fewer columns.
  const bool whole_other = whole == Plan::kOther;
  const int64_t bar = whole_other ? INT64_MAX : whole == Plan::kStream || (p.n & 255) != 0 ? whole_ns - whole_ns / 20 : 0;
  auto is_tiles = [](Plan q) { return q == Plan::kTiles256 || q == Plan::kTiles128 || q == Plan::kTiles128x128; };
  // N not a multiple of 256, where the tiles do not take it whole (K < 1024, up to 128 rows) or the last columns would cost
  // them a round (2048 x 4224 x 2048: 256 tiles of 128x256 and 128 columns): the columns up to the last multiple of 256 go to
  // whatever kernel that shape gets, the remaining columns (weight rows) to a launch of their own that writes into the same
  // rows of the result.
  if ((p.n & 255) != 0 && p.n > 256 && (p.n & 15) == 0 && p.m > 64 && (p.k & 31) == 0 && p.k >= 256) {
    int64_t main_ns, rest_ns;
    const Plan main_plan = mxfp8_plan(p.m, p.n & ~255, p.k, cus, &main_ns), rest_plan = mxfp8_plan(p.m, p.n & 255, p.k, cus, &rest_ns);
    if (whole_other && main_plan == Plan::kStream) return launch_skinny<OUT_BF16>(p, stream);  // (takes any N % 16 == 0)
    if (main_plan != Plan::kOther && (whole_other || (is_tiles(main_plan) && rest_plan == Plan::kStream && main_ns != INT64_MAX &&
                                                       rest_ns != INT64_MAX && main_ns + rest_ns < bar))) {
      Params main = p, rest = p;
      main.n = p.n & ~255;
      rest.n = p.n - main.n;
      main.ldc = rest.ldc = p.out_pitch();
      const int64_t sf_padded = ((int64_t)(p.k >> 5) + 3) & ~(int64_t)3;
      rest.b = p.b + (int64_t)main.n * p.k;
      rest.sfb = p.sfb + (int64_t)main.n * sf_padded;
      rest.out = static_cast<uint8_t*>(p.out) + (int64_t)main.n * 2;
      if (const int rc = launch_sized<OUT_BF16>(main, stream)) return rc;
      return launch_sized<OUT_BF16>(rest, stream);
    }
  }
  // M not a multiple of 128 (a prefill of any token count): the rows up to the last multiple of 128 go to whatever kernel
  // that shape gets, the remaining rows (at most 127, a whole number of 128-row scale tiles further on) to the skinny
  // kernel in a launch of their own (4000 x 4096 x 4096: 197 -> 77 us; 8100 x 8192 x 8192: 1475 -> 390 us).
  // The cut is the last multiple of 128 or of 256 (which allows 256x256 tiles), whichever is estimated faster
  // (8100 x 8192 x 8192: 546 us cut at 8064, 128x256 tiles; 390 us cut at 7936).
  if (p.m > 128 && (p.m & 127) != 0 && (p.k & 31) == 0 && (whole_other || whole == Plan::kStream)) {
    int64_t best = bar;
    int cut = 0;
    for (const int c : {p.m & ~127, p.m & ~255}) {
      int64_t ns_main, ns_rest;
      if (c < 128) continue;
      const Plan main_plan = mxfp8_plan(c, p.n, p.k, cus, &ns_main);
      if (main_plan == Plan::kOther || mxfp8_plan(p.m - c, p.n, p.k, cus, &ns_rest) != Plan::kStream) continue;
      if (!whole_other && main_plan == Plan::kStream) continue;  // (the whole shape is on that kernel already)
      if (ns_main == INT64_MAX || ns_rest == INT64_MAX) continue;
      if (ns_main + ns_rest < best) best = ns_main + ns_rest, cut = main_plan == Plan::kStream ? p.m : c;
    }
    if (cut == p.m) return launch_skinny<OUT_BF16>(p, stream);  // (the skinny kernel takes any number of rows)
    if (cut) {
      Params main = p, rest = p;
      main.m = cut;
      rest.m = p.m - cut;
      const int64_t sf_padded = ((int64_t)(p.k >> 5) + 3) & ~(int64_t)3;
      rest.a = p.a + (int64_t)cut * p.k;
      rest.sfa = p.sfa + (int64_t)cut * sf_padded;
      rest.out = static_cast<uint8_t*>(p.out) + (int64_t)cut * p.out_pitch() * 2;
      if (const int rc = launch_sized<OUT_BF16>(main, stream)) return rc;
      return launch_sized<OUT_BF16>(rest, stream);
    }
  }
  switch (whole) {
    case Plan::kStream: return launch_skinny<OUT_BF16>(p, stream);
    case Plan::kTiles256: return launch_tiles<8, 8, OUT_BF16>(p, stream);
    case Plan::kTiles128: return launch_tiles<4, 8, OUT_BF16>(p, stream);
    case Plan::kTiles128x128: return launch_tiles<4, 4, OUT_BF16>(p, stream);
    case Plan::kOther: break;
  }
  if (tiles(256, 256) >= cus) return launch_cfg<256, 256, OUT_BF16>(p, stream);
  if (tiles(128, 128) >= cus) return launch_cfg<128, 128, OUT_BF16>(p, stream);
  return launch_cfg<64, 64, OUT_BF16>(p, stream);
}

}  // namespace

int launch_mxfp8_gemm(const void* a, const void* b, const void* sfa, const void* sfb, const float* alpha, void* out,
                      int64_t m, int64_t n, int64_t k, int out_dtype, hipStream_t stream) {
  if (m > INT32_MAX || n > INT32_MAX || k > INT32_MAX) return fail(NVF_ERR_UNSUPPORTED_SHAPE, "dimension exceeds int32");
  Params p{static_cast<const uint8_t*>(a), static_cast<const uint8_t*>(b), static_cast<const uint8_t*>(sfa),
           static_cast<const uint8_t*>(sfb), alpha, out, (int)m, (int)n, (int)k};
  return out_dtype == NVF_BF16 ? launch_sized<true>(p, stream) : launch_sized<false>(p, stream);
}

}  // namespace nvf
