// GEMMs whose MFMA operands are 16-bit floats, for gfx950:
//   * nvfp4_scaled_mm          (cutlass/nvfp4_scaled_mm.cu:283-312)
//   * nvfp4_scaled_grouped_mm  (cutlass/nvfp4_scaled_group_mm.cu:714-788, pointer rule :83-155)
//   * grouped_mm               (cutlass/group_mm.cu:518-571, pointer rule :76-105)
//
// NVFP4 has one e4m3 scale per 16 elements, which the block-32 / e8m0 scaled MFMA of gfx950 cannot
// express.  An e2m1 value times an e4m3 scale has at most 6 significant bits and an exponent range
// of 2^-10 .. 2^11, so it is exactly representable in fp16: tiles are dequantised to fp16 while
// they are staged into LDS and fed to v_mfma_f32_32x32x16_f16 with fp32 accumulation.  Every
// product is exact; only the fp32 accumulation order differs from any other correct implementation.
//
// The tile kernels (one for 16-bit operands, one for NVFP4) are persistent: a workgroup walks (group,
// m-tile, n-tile) work items whose list is derived on the device from problem_sizes, so no host
// synchronisation is needed and empty groups cost nothing.  The dense op is the one-group case.
// Specialised kernels take the shapes they fit: 256x256 persistent NVFP4 and grouped 16-bit kernels,
// and a weight-streaming NVFP4 kernel for up to 128 activation rows.
//
// Output layout trick: the MFMA is issued with the B fragment as first operand, so that a lane's
// accumulator registers hold 4 consecutive N-elements of one output row and are stored as 8 bytes.
#include "gemm16_device.h"
#include "nvf_internal.h"
#include "tile_loop.h"

#include <algorithm>
#include <mutex>

namespace nvf {
namespace {

// Block-scaled epilogue (cutlass/nvfp4_scaled_mm_blockscale.cu:87-93: the product is quantized to NVFP4 again along
// N before it leaves the kernel).  One 32x32 accumulator tile: lane (li, lg) holds row li, columns 8q + 4lg + e in
// register 4q + e, so each of the row's two 16-column blocks is shared by the lanes (li, 0) and (li, 1): amax over
// the lane's 8 values, one exchange with lane ^ 32, then the block quantizer's arithmetic
// (runtime/block_quantization_kernels.cu:224-263) on alpha * acc.  For block b both lanes get the scale code q8[b];
// h[b] holds this lane's 4 of the block's 8 payload bytes: bits 0..15 = bytes 2lg, 2lg+1, bits 16..31 = bytes
// 4+2lg, 5+2lg.  Must be called by whole wavefronts.
__device__ __forceinline__ void quantize_acc_tile(const f32x16& acc, float alpha, float gs, float decode, bool active, uint32_t h[2],
                                                  uint32_t q8[2]) {
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    float x[8];
    float m = -INFINITY;
    bool nonfinite = false;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x[e] = acc[8 * b + e] * alpha;
      m = fmaxf(m, fabsf(x[e]));  // NaN ignored, as the quantizer does
      nonfinite |= !(fabsf(x[e]) < INFINITY);
    }
    const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    m = fmaxf(m, __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ 32) << 2, __builtin_bit_cast(int, m))));
    float r;
    q8[b] = nvfp4_block_scale(m, true, gs, decode, active, r);
    uint32_t w = 0;
    if (__builtin_amdgcn_ballot_w64(nonfinite) == 0) {
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, x[0] * r, x[1] * r, 1.0f, 0);
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, x[2] * r, x[3] * r, 1.0f, 1);
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, x[4] * r, x[5] * r, 1.0f, 2);
      w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, x[6] * r, x[7] * r, 1.0f, 3);
    } else {  // explicit NaN rule of the narrow cast
#pragma unroll
      for (int t = 0; t < 4; ++t) w |= f32x2_to_e2m1_byte(x[2 * t] * r, x[2 * t + 1] * r) << (8 * t);
    }
    h[b] = w;
  }
}

// fills n bytes with zero (the padding of the block-scaled result's scale buffer for ragged shapes)
__global__ __launch_bounds__(256) void zero_fill_kernel(uint32_t* __restrict__ dst, int64_t words) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < words) dst[i] = 0u;
}

// The kernels, one file each (this translation unit includes them: they share the helpers above and the launchers below)
#include "gemm16_tile_kernels.inl"
#include "nvfp4_streaming_kernel.inl"
#include "nvfp4_group_panel_kernel.inl"
#include "grouped16_kernel.inl"
#include "grouped16_streaming_kernel.inl"

// -------------------------------------------------------------------------------------------------
// Launchers of the tile kernels and the dispatch
// -------------------------------------------------------------------------------------------------
template <bool OUT_BF16, bool GROUPED, int TM = 4, bool OUT_F32 = false, bool OUT_FP4 = false>
int launch_nvfp4_fast(const Params& p, int cus, hipStream_t stream) {
  return launch_nvfp4_persistent(p, OUT_F32 ? Nvfp4Out::kF32 : OUT_FP4 ? Nvfp4Out::kFp4 : OUT_BF16 ? Nvfp4Out::kBf16 : Nvfp4Out::kF16, GROUPED, TM, cus, stream);
}

template <int BM, int BN, bool BF16_MMA, bool OUT_BF16>
int launch_cfg(const Params& p, int grid, hipStream_t stream) {
  auto kern = gemm16_kernel<BM, BN, BF16_MMA, OUT_BF16>;
  constexpr int lds_bytes = 2 * (BM + BN) * 128;
  if (note_launch("gemm16_kernel<%d,%d> grid=%d", BM, BN, grid)) return NVF_OK;
  static std::atomic<uint64_t> configured{0};  // one bit per device
  if (const int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds_bytes, configured)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256), lds_bytes, stream, p);
  return check_launch("gemm16_kernel");
}

template <int BM, int BN, bool OUT_BF16, bool OUT_F32 = false, bool OUT_FP4 = false>
int launch_nvfp4_tile(const Params& p, int grid, hipStream_t stream) {
  auto kern = nvfp4_tile_kernel<BM, BN, OUT_BF16, OUT_F32, false, OUT_FP4>;
  constexpr int lds_bytes = 2 * (BM + BN) * 128;
  if (note_launch("nvfp4_tile_kernel<%d,%d,f32=%d%s> grid=%d skip_whole_256=%d min_rows=%d", BM, BN, (int)OUT_F32, OUT_FP4 ? ",fp4_blockscale" : "", grid,
                  p.skip_whole_256, p.min_rows))
    return NVF_OK;
  static std::atomic<uint64_t> configured{0};  // one bit per device
  if (const int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds_bytes, configured)) return rc;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256), lds_bytes, stream, p);
  return check_launch("nvfp4_tile_kernel");
}

// Dense NVFP4 without a workspace: the weight-streaming kernel, the persistent kernel with 256x256 or 128x256 tiles,
// or the tile kernels?  Costs in units of one round of 256x256 tiles over the compute units = 100 (24 us per 1024 of
// K): a round of 128-row tiles costs 58 (half the flops at 86 % of the rate); the tile kernels run their 128x128 tiles
// two to a compute unit: 68 per such round, 45 for a last round of one tile per compute unit, and 22..47 when there
// is no more than that in all (all measured: M = 128..1024, N = 2048..14336, K = 4096 and 14336).
// The persistent kernel's costs are those of its form with both operands staged in LDS.  The present one takes 0.76..0.9 of
// them from K = 4096 on (768 x 14336 x 4096 77 of 102 us, 512 x 14336 x 4096 51 of 62, 2048 x 14336 x 4096 170 of 198, 1024 x 8192 x
// 14336 177 of 201), as much at K = 1024 (8192 x 8192 106 of 102).  The lines are where they were: near them calls still
// stream that the tiles may do faster.
// the streaming kernel's cost estimate is in ns within 0.8 (K = 2048) .. 1.1 (K = 14336)
// (the form with 4 wavefronts: its discount in the cost holds among the streaming forms; against the tiles it made 26 of
// 91 changed picks slower, at K = 2048 and 7168, and 43 faster, so there only 4 % of it stay, for 3072 <= K < 6144:
// 1536 x 11008 x 4096 162 -> 139 us, 160 x 29568 x 4096 58 -> 46)
int64_t nvfp4_stream_ns(int64_t m, int64_t n, int64_t k, int cus) {
  int slab, rt;
  int64_t cost = nvfp4_skinny_best(m, n, k, cus, &slab, &rt);
  if (slab == 128 && rt == 4 && m > 64 && (k & 127) == 0 && ceil_div(m, 128) * (n / 64) > cus)
    cost = cost * (k >= 3072 && k < 6144 ? 96 : 100) / nvfp4_four_wavefront_percent(k);
  return cost * (k < 3072 ? 82 : k < 6144 ? 96 : k < 10240 ? 103 : 110) / 100;
}
struct DensePlan {
  enum Kernel { kStream, kTiles256, kTiles128, kOther } kernel;
  int64_t ns;  // estimated duration (INT64_MAX: no estimate)
};
DensePlan nvfp4_dense_plan(int64_t m, int64_t n, int64_t k, int cus) {
  const bool stream_ok = (k & 31) == 0 && (n & 15) == 0 && k * 64 < (1ll << 31);  // 32-bit lane offsets (a short last chunk is fine)
  // (a short last span is fine; so is, with whole spans, a last row tile with fewer rows, which counts as a whole one:
  // 384 x 28672 x 4096 as 224 tiles of 256 rows in one round instead of 336 of 128 rows in two.  The kernel would take both at
  // once too: not measured against the cuts that such calls get now)
  const bool persistent_shape = (n & 255) == 0 && (k & 31) == 0 && k >= 256;
  const bool ok256 = persistent_shape && ((m & 255) == 0 || ((k & 127) == 0 && m > 128));
  const bool persistent_ok = persistent_shape && ((m & 127) == 0 || ((k & 127) == 0 && m > 128));
  int64_t cost256 = INT64_MAX, cost128 = INT64_MAX, cost_tile = INT64_MAX;
  if (persistent_ok) {
    const int64_t t256 = ok256 ? ceil_div(m, 256) * (n / 256) : 0, t128 = ceil_div(m, 128) * (n / 256);
    cost256 = t256 ? 100 * ceil_div(t256, cus) : INT64_MAX;
    cost128 = 58 * ceil_div(t128, cus);
    const int64_t small = 2 * t128, full = small / (2 * cus), rest = small - full * 2 * cus;
    cost_tile = full * 68 + (rest == 0 ? 0 : rest > cus ? 68 : full ? 45 : 22 + 25 * rest / cus);
  }
  const int64_t cost_min = std::min(cost256, std::min(cost128, cost_tile));
  const int64_t rest_ns = persistent_ok ? 6000 + cost_min * 240 * ((k + 127) & ~127ll) / 1024 : INT64_MAX;
  if (stream_ok) {
    const int64_t stream_ns = nvfp4_stream_ns(m, n, k, cus);
    bool stream;
    if (m <= 128 || (m <= 256 && !(persistent_ok && k >= 2048))) {
      stream = true;  // at most two passes over the weights (256 x 14336 x 4096: 38 instead of 58 us on tiles)
    } else if (persistent_ok && k >= 2048) {
      // by estimated duration (the tiles' form that the costs were fitted to / streaming kernel, us: 512 x 4096 x 14336 180 / 57, 384 x 8192 x 7168 92 / 53,
      // 640 x 14336 x 14336 295 / 251, 1024 x 8192 x 4096 60 / 66, 384 x 28672 x 4096 91 / 97; over 130 shapes of 160..3000 rows
      // the pick was within 2 % of the fastest in the geometric mean)
      stream = stream_ns <= rest_ns;
    } else {
      // Ragged shapes, which only the tile kernels take otherwise: with a deep K and a small N the streaming kernel
      // fills the chip where they cannot, while its workgroups (one per 128 rows x 16 columns at such N) cover the
      // compute units at most 3 times, 2 times for K < 4096 (measured: 300 x 3072 x 2048 in 18 instead of 16 us,
      // 1000 x 288 x 2560, 2100 x 96 x 4096).
      const int64_t rounds = ceil_div(ceil_div(m, 128) * (n / 16), cus);
      stream = k >= 2048 && rounds <= (k >= 4096 ? 3 : 2);
    }
    if (stream) return {DensePlan::kStream, stream_ns};
  }
  if (persistent_ok) {
    if (cost256 <= cost128 && cost256 <= cost_tile) return {DensePlan::kTiles256, rest_ns};
    if (cost128 <= cost_tile) return {DensePlan::kTiles128, rest_ns};
  }
  return {DensePlan::kOther, rest_ns};
}

// What a dense call does about an N that is no multiple of 256 (29568, 1408): 0 nothing; 1 the whole call goes to the
// weight-streaming kernel (which takes any N % 16 == 0); 2 the columns up to the last multiple of 256 go to whatever
// kernel that shape gets and the remaining columns (weight rows) to a launch of their own that writes into the same rows
// of the result.  A cut competes with the kernel the whole shape gets: the tile kernels (no estimate) lose to any cut;
// the weight-streaming kernel loses to one whose main part runs on the persistent kernel and is estimated 5 % faster.
// (ns: the estimated duration of what is returned, where there is one)
int nvfp4_n_cut(int64_t m, int64_t n, int64_t k, int cus, int64_t* ns = nullptr) {
  if (ns) *ns = INT64_MAX;
  if ((n & 255) == 0 || n <= 256 || m <= 128 || (k & 31) != 0 || k < 256) return 0;
  const DensePlan whole = nvfp4_dense_plan(m, n, k, cus);
  const DensePlan main_plan = nvfp4_dense_plan(m, n & ~255, k, cus), rest_plan = nvfp4_dense_plan(m, n & 255, k, cus);
  const bool whole_other = whole.kernel == DensePlan::kOther;
  if (main_plan.kernel == DensePlan::kOther) return 0;
  const bool have_cut_ns = rest_plan.kernel == DensePlan::kStream && main_plan.ns != INT64_MAX;
  const int64_t cut_ns = have_cut_ns ? main_plan.ns + rest_plan.ns : INT64_MAX;
  if (whole_other) {
    if (main_plan.kernel != DensePlan::kStream) {
      if (ns) *ns = cut_ns;
      return 2;
    }
    // all columns to the streaming kernel, or - a few columns past a whole number of rounds of its workgroups cost a
    // round - those in a launch of their own (512 x 4224 x 8224: 264 workgroups at once, or 256 and then 8)
    const int64_t stream_ns = (k & 31) == 0 && (n & 15) == 0 ? nvfp4_stream_ns(m, n, k, cus) : INT64_MAX;
    const bool cut = have_cut_ns && cut_ns < stream_ns - stream_ns / 20;
    if (ns) *ns = cut ? cut_ns : stream_ns;
    return cut ? 2 : 1;
  }
  if (whole.kernel == DensePlan::kStream && main_plan.kernel != DensePlan::kStream && have_cut_ns && cut_ns < whole.ns - whole.ns / 20) {
    if (ns) *ns = cut_ns;
    return 2;
  }
  return 0;
}

// Dense shapes whose M is not a multiple of 128 and that only the tile kernels would take whole: the number of rows
// (the last multiple of 128) that go to a launch of their own, if that shape gets a better kernel; else 0.  If that
// kernel is the weight-streaming one, which takes any number of rows, the answer is m: no cut, all rows to it.
int64_t nvfp4_rows_before_remainder(int64_t m, int64_t n, int64_t k, int cus) {
  if (m <= 128 || (m & 127) == 0 || (k & 15) != 0) return 0;
  // Against the kernel the whole shape gets: the tile kernels (no estimate) lose to any cut; the weight-streaming kernel
  // loses to a cut whose first part runs on the persistent kernel and is estimated 5 % faster or more (192 rows against
  // 28672 weight rows: 128 of them on 128x256 tiles).
  const DensePlan whole = nvfp4_dense_plan(m, n, k, cus);
  const bool whole_other = whole.kernel == DensePlan::kOther;
  if (!whole_other && whole.kernel != DensePlan::kStream) return 0;
  // the cut is the last multiple of 128 or of 256 (which allows 256x256 tiles), whichever is estimated faster
  int64_t best = whole_other ? INT64_MAX : whole.ns - whole.ns / 20, cut = 0;
  for (const int64_t c : {m & ~(int64_t)127, m & ~(int64_t)255}) {
    if (c < 128) continue;
    const DensePlan main = nvfp4_dense_plan(c, n, k, cus), rest = nvfp4_dense_plan(m - c, n, k, cus);
    if (main.kernel == DensePlan::kOther || rest.kernel != DensePlan::kStream || main.ns == INT64_MAX) continue;
    if (!whole_other && main.kernel == DensePlan::kStream) continue;  // (the whole shape is on that kernel already)
    if (main.ns + rest.ns < best) best = main.ns + rest.ns, cut = main.kernel == DensePlan::kStream ? m : c;
  }
  return cut;
}

// Split of K for dense NVFP4 shapes with fewer 128x128 tiles than compute units and a deep K (decode and
// small prefill batches against a down projection): about two work items per compute unit, at least eight
// 128-deep spans each.  Every split writes and the reduction re-reads an fp32 copy of the output, so for
// K below 8192 the split costs more than it gains (measured) and 1 is returned.
int nvfp4_splits(int64_t m, int64_t n, int64_t k, int cus) {
  const int64_t tiles = ceil_div(m, 128) * ceil_div(n, 128), nspans = ceil_div(k, 128);
  if (m <= 64 || tiles >= cus || nspans < 64) return 1;
  // not where the weight-streaming kernel runs, which splits K over the wavefronts of a workgroup (256 x 2048 x 8192:
  // 14 us against 28 us for this split; 512 x 4096 x 14336: 56 against 78 us)
  if (nvfp4_dense_plan(m, n, k, cus).kernel == DensePlan::kStream) return 1;
  int64_t s = (2 * (int64_t)cus) / tiles;
  if (s > nspans / 8) s = nspans / 8;
  if (s > 32) s = 32;
  if (s < 2) return 1;
  // N no multiple of 256: the split has to be estimated faster (25 us + 2 us per span of an item, two items to a compute
  // unit) than what the call does otherwise - all columns, or those up to the last multiple of 256, on another kernel
  // (384 x 4224 x 8224 50 us against 42 us streamed, 384 x 6176 x 14368 100 against 122 us)
  int64_t other_ns;
  if (nvfp4_n_cut(m, n, k, cus, &other_ns) != 0 && other_ns < 25000 + 2000 * ceil_div(nspans, s) * ceil_div(tiles * s, 2 * (int64_t)cus)) return 1;
  return (int)s;
}

// Split of K over workgroups for the weight-streaming kernel with one slab of 65..96 activation rows: every
// workgroup converts all activation rows of its K range next to its weight rows, so 64 weight rows per workgroup
// (4 tiles against 8 activation tiles: 12 conversions for 32 MFMA tiles) halve the conversion work of 16 (1 against
// 8: 9 for 8), and where N / 64 workgroups leave compute units idle, K is split over as many workgroups as fit.
int nvfp4_skinny_splits(int64_t m, int64_t n, int64_t k, int cus) {
  // (measured against the forms without a split: 65 x 4096 x 14336 18.7 against 21.7 us, 96 x 8192 x 14336 30.9
  // against 33.2, 65 x 6144 x 8192 17.7 against 19.1; from 97 rows on, or with a weight matrix of less than 48 Mi
  // elements, the second launch costs more than the split gains: 128 x 8192 x 14336 38.1 against 35.3, 65 x 4096 x 8192
  // 16.3 against 13.9, 65 x 2048 x 14336 15.5 against 14.0)
  if (m <= 64 || m > 96 || (k & 127) != 0 || (n & 63) != 0 || k * 64 >= (1ll << 31) || n * k < (48ll << 20)) return 1;
  const int64_t wgs = n / 64, chunks = k >> 7;
  int64_t s = cus / wgs;
  if (s > chunks / 28) s = chunks / 28;
  if (s > 8) s = 8;
  if (wgs * s * 2 < cus) return 1;  // would leave most compute units idle: the tile kernel's split has more items
  return s < 2 ? 1 : (int)s;
}

template <bool OUT_BF16>
int launch_nvfp4_splitk(const Params& p0, int splits, float* workspace, hipStream_t stream) {
  Params p = p0;
  const int nspans = (p.k + 127) >> 7;
  p.spans_per_split = (nspans + splits - 1) / splits;
  p.splits = (nspans + p.spans_per_split - 1) / p.spans_per_split;  // no empty split
  p.partial = workspace;
  auto kern = nvfp4_tile_kernel<128, 128, OUT_BF16, false, true>;
  constexpr int lds_bytes = 2 * (128 + 128) * 128;
  const int64_t items = ceil_div(p.m, 128) * ceil_div(p.n, 128) * p.splits;
  if (note_launch("nvfp4_tile_kernel<128,128,split_k> grid=%lld splits=%d + splitk_reduce_kernel", (long long)items, p.splits)) return NVF_OK;
  static std::atomic<uint64_t> configured{0};  // one bit per device
  if (const int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds_bytes, configured)) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)items), dim3(256), lds_bytes, stream, p);
  int rc = check_launch("nvfp4_tile_kernel (split K)");
  if (rc != NVF_OK) return rc;
  const int64_t mn = (int64_t)p.m * p.n;
  hipLaunchKernelGGL(splitk_reduce_kernel<OUT_BF16>, dim3((unsigned)ceil_div(mn / 4, 256)), dim3(256), 0, stream, workspace, p.splits,
                     mn, p.alpha, static_cast<uint16_t*>(p.out));
  return check_launch("splitk_reduce_kernel");
}

// tile kernel of the operand type: NVFP4 or 16-bit
template <int BM, int BN, bool NVFP4, bool BF16_MMA, bool OUT_BF16>
int launch_tile(const Params& p, int grid, hipStream_t stream) {
  if constexpr (NVFP4) return launch_nvfp4_tile<BM, BN, OUT_BF16>(p, grid, stream);
  else return launch_cfg<BM, BN, BF16_MMA, OUT_BF16>(p, grid, stream);
}

// Grouped NVFP4: rows in all from which a call counts as a prefill, whose large groups get launches of their own on the
// persistent kernel.  Below, those launches find a handful of tiles each and run one after the other at a tile's
// latency (256 experts, Zipf loads, K=7168: 2048 rows 732 -> 576 us, 4096 rows 769 -> 608 us without them; 8192 rows
// 807 with against 753 without, but evenly loaded experts 639 against 771).
constexpr int64_t kPrefillRows = 6144;

// Grouped NVFP4, the groups of 129 rows and more: in slabs of 32 rows on the persistent streaming kernel, in calls of at most
// 1024 rows whose 128x128 tiles (256x256 from 512 rows per group on) would leave compute units idle, each walking all of K on
// one of them: 1024 rows over 8 experts, K = 7168, N = 2048 118 -> 56 us, 512 rows with Zipf loads 123 -> 38.  Every slab reads
// the weights again and adds partial sums, so the fuller the chip is with tiles and the shallower K is, the more the tiles
// gain.  Slabs / tiles, us, 256 rows per group, tiles for 1/2, 3/4, 7/8 and all of the compute units: K = 512 15 / 16, 20 / 17,
// 23 / 17, 25 / 17; K = 1024 17 / 21, 22 / 22, 25 / 22, 28 / 23; K = 2048 23 / 33, 33 / 34, 37 / 34, 41 / 34; K = 4096 35 / 55,
// 49 / 56, 56 / 56, 63 / 57; K = 7168 51 / 88, 73 / 89, 84 / 90, 91 / 90.
// Below 129 rows per group only some groups are that large, and from 512 on the tiles are 256x256: twice as many tiles' worth
// (8 experts with Zipf loads, 1024 rows, as many tiles as compute units: K = 512 24 / 23, K = 1024 29 / 31; two experts of 512
// rows: K = 256 25 / 26).  Where two tiles for every group of fewer than 256 rows need a second round, slabs from K = 1024 on
// (6 groups of 160 rows, N = 4096: K = 512 25 / 21, K = 1024 28 / 29, K = 4096 61 / 77; 3 groups, N = 6144, K = 1024 22 / 28).
bool nvfp4_large_groups_stream(int64_t groups, int64_t m, int64_t n, int64_t k, int cus) {
  const int64_t tiles = ceil_div(m, 128) * ceil_div(n, 128);
  if (m < 129 || m > 1024 || tiles > cus) return false;
  const bool few_or_large = m < 129 * groups || m >= 512 * groups;
  if (m >= 129 * groups && m < 256 * groups && k >= 1024 && 2 * groups * ceil_div(n, 128) > cus) return true;
  const int64_t share = k < 256 ? 4 : k < 512 ? 6 : k < 1024 ? 8 : k < 2048 ? 10 : k < 4096 ? 12 : k < 7168 ? 14 : 16;
  return 16 * tiles <= (few_or_large ? 2 : 1) * share * cus;
}

// Grouped NVFP4, the groups of 1..32 rows: on the streaming kernel whose 8 wavefronts own 64 (N % 512 = 0) or 32 weight rows
// each and walk K alone, instead of the persistent kernel, whose wavefronts split K.  With a shallow K the latter has a step
// or two per item next to a sum and its barriers; up to K < 4096 it is behind where the other's workgroups are one round of
// the compute units.  Persistent kernel against this one, us: 256 experts of 4096 x 128, 512 rows with Zipf loads 51 / 23, x 512
// 53 / 43; 24 rows each: 32 experts of 4096 x 1024 1.26 times as slow, x 2048 equal, 16 of 8192 x 2560 1.27 (32 of 8192 1.07),
// x 3584 1.12 (1.00), 64 of 2048 x 3584 1.16; for half as many workgroups as compute units 8 of 8192 x 512 1.10, x 1024 1.00,
// x 2048 0.99, 4096 x 512 (a quarter) 0.84.  From 128 rows per group on such groups are few, and the two are within 7 %.
// `with_large`: the persistent kernel would take the groups of 129 rows and more along; a launch of it for them alone costs
// 5-20 % of a call with Zipf loads, which K < 512 outweighs, and up to K = 2048 (where even loads gain 8-20 %) a full round.
// Below three times 129 rows in all there is hardly such a group.
bool nvfp4_wavefronts_own_rows(int64_t groups, int64_t m, int64_t n, int64_t k, int cus, bool with_large) {
  const bool large = with_large && m >= 3 * 129;
  const int64_t rows = (n & 511) == 0 ? 512 : 256;
  if ((k & 127) != 0 || n % rows != 0 || m >= 128 * groups) return false;
  const int64_t wgs = std::min(groups, m) * (n / rows);
  if (k < 512 || (k < 2048 && !large)) return 2 * wgs >= cus;
  if (k < 2048) return wgs >= cus && (k < 1024 || wgs < 8 * (int64_t)cus);
  return k > 2048 && k < 4096 && !large && 8 * wgs >= 7 * (int64_t)cus && wgs <= cus;
}

// Grouped NVFP4, calls of at most 1024 rows (as many slabs as that kernel's list holds): the groups of 33..128 rows in slabs of 32
// rows on the persistent streaming kernel, which takes the groups of 1..32 rows, and no launch of their own.  That one takes 2 us with no such group, and with any as long as a
// workgroup walks all of K; every slab reads the weights again.  Decided by the call's sizes alone, for what its groups could
// be at worst (two slabs for every 33 rows): were it decided by the groups' sizes, where both kernels can see them, a group's
// bits would depend on the others' (they sum K in different orders).
// Few rows per group: up to four items (slab x 64 weight rows) per compute unit.  Own launch / slabs, us, Zipf loads: 512 rows
// over 256 experts, N = 2048, K = 7168 221 / 190, over 64 125 / 94, 128 experts, N = 1024, K = 4096, 1024 rows 78 / 60, 16 of
// 4096 x 4096, 256 rows 46 / 36; even ones, where no group is so large: 256 of 2048 x 7168, 512 rows 288 / 285, 16 of 2048 x 2048, 384
// rows 17 / 15.  Beyond four Zipf loads gain 2 % (512 rows, N = 7168, K = 2048 203 / 199).  What it costs where all rows are in
// groups of 36: up to three items 1.5 times (108 rows over 64, N = 4096, K = 14336 30 / 44), at four 1.7.
// From 24 rows per group on most groups may be such ones: up to one item.  Even loads, one item: 4 groups of 34 rows, N = 2048,
// K = 7168 18.0 / 15.4, 2 of 64, 4096 x 4096 14.9 / 10.0, 16 of 34, N = 512, K = 4096 13.3 / 13.6; two items: 8 of 34, N = 2048,
// K = 7168 21.7 / 26.3, 4 of 40, 4096 x 4096 15.6 / 18.6, 2 of 34, N = 7168, K = 2048 10.4 / 11.9.
bool nvfp4_mid_groups_as_slabs(int64_t groups, int64_t m, int64_t n, int cus) {
  return m > 32 && m <= 1024 && 2 * (m / 33) * (n / 64) <= (m <= 24 * groups ? 4 : 1) * (int64_t)cus;
}

template <bool NVFP4, bool BF16_MMA, bool OUT_BF16>
int launch_sized(const Params& p, int64_t m_hint, int cus, void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  // Pick the largest tile that still yields about one work item per compute unit.
  auto tiles = [&](int bm, int bn) { return ceil_div(m_hint, bm) * ceil_div(p.n, bn); };
  const bool dense = p.problem_sizes == nullptr;
  // grouped NVFP4: does the call count as a prefill (see kPrefillRows)?  Also with fewer rows where the large groups'
  // launches find (nearly) a round of 256x256 tiles - with 128 rows per group on average, or two rounds whatever the groups
  // (8 experts, 1536 rows, N=14336, K=4096: 320 -> 223 us; 16 experts, 3072 rows: 540 -> 394; 128 experts, 5632 rows,
  // N=7168, K=2048: 460 -> 336; at 96 rows per group and one round the other launches stay faster: 125 against 167 us)
  const int64_t tiles256 = (m_hint / 256) * (p.n / 256);
  const bool is_prefill = m_hint >= kPrefillRows || (8 * tiles256 >= 7 * (int64_t)cus && m_hint >= 128 * (int64_t)p.groups) || tiles256 >= 2 * (int64_t)cus;
  if constexpr (NVFP4) {
    if (dense && workspace != nullptr) {
      const int skinny_splits = nvfp4_skinny_splits(p.m, p.n, p.k, cus);
      if (skinny_splits > 1 && workspace_bytes >= (int64_t)skinny_splits * p.m * p.n * 4) {
        Params q = p;
        const int chunks = p.k >> 7;
        q.partial = static_cast<float*>(workspace);
        q.spans_per_split = (chunks + skinny_splits - 1) / skinny_splits;
        q.splits = (chunks + q.spans_per_split - 1) / q.spans_per_split;  // no empty split
        return launch_nvfp4_skinny_ring_cfg<4, 8, OUT_BF16>(q, stream, 1);
      }
      const int splits = nvfp4_splits(p.m, p.n, p.k, cus);
      if (splits > 1 && workspace_bytes >= (int64_t)splits * p.m * p.n * 4)
        return launch_nvfp4_splitk<OUT_BF16>(p, splits, static_cast<float*>(workspace), stream);
    }
    if (dense) {
      const DensePlan plan = nvfp4_dense_plan(p.m, p.n, p.k, cus);
      if (plan.kernel == DensePlan::kStream) return launch_nvfp4_skinny<OUT_BF16>(p, cus, stream);
      if (plan.kernel == DensePlan::kTiles256) return launch_nvfp4_fast<OUT_BF16, false, 4>(p, cus, stream);
      if (plan.kernel == DensePlan::kTiles128) return launch_nvfp4_fast<OUT_BF16, false, 2>(p, cus, stream);
    }
  }
  if constexpr (!NVFP4) {
    // grouped_mm with groups of 128 rows or more on average and tiles for half the compute units: persistent LDS-direct
    // kernel with 256x256 tiles (at 128..255 rows per group the 128x128 tile kernel used to run: 8 experts, 1536 rows, N=14336,
    // K=4096 373 -> 272 us; 64 experts, 8192 rows, N=7168, K=2048 571 -> 449 us)
    const bool lds_direct = !dense && (p.n & 7) == 0 && (p.k & 63) == 0 && (int64_t)p.k * 2 * 256 < (1ll << 31);
    if (lds_direct && m_hint >= 128 * (int64_t)p.groups && tiles(256, 256) >= cus / 2 && p.k >= ((p.n & 255) == 0 ? 128 : 256))
      return launch_grouped16_fast<BF16_MMA, OUT_BF16>(p, cus, stream);
    // A decode step: few rows per group on average.  The streaming kernel's partial sums cost more per item the shallower K
    // and the more rows there are; the 128x128 tiles lose most where they leave compute units idle.  128x128 tiles (the kernel
    // below; where K % 64 != 0, the tile kernel) against streaming kernel, even and Zipf loads, us: 8 experts of 1024 x 1024, 48
    // rows each 10.9 / 8.4 and 11.2 / 13.2; 4096 x 4096, 48 rows 65 / 64 and 80 / 70; 64 of 2048 x 7168, 16 rows 296 / 286 and
    // 343 / 316, 24 rows 303 / 312 and 350 / 360; 8 of 14336 x 4096, 24 rows 194 / 171 and 182 / 182; 8 of 4096 x 14336, 24 rows
    // 152 / 161 and 168 / 207, 48 rows 178 / 177 and 271 / 240; 32 of 2880 x 2880, 16 rows 90 / 96 and 104 / 101, 24 rows 91 / 114
    // and 105 / 119; 16 of 4096 x 2048, 16 rows 63 / 58 and 64 / 60; 8 of 3000 x 1288, 16 rows 25 / 19 and 25 / 20, 48 rows
    // 26 / 27; 64 of 1024 x 1024, 8 rows 28 / 33 and 28 / 36.
    const int64_t first_tiles = p.groups * ceil_div(p.n, 128);
    int rows_on_average = 0;
    if (p.k >= 1024 && 4 * first_tiles <= cus) rows_on_average = 48;
    else if (p.k >= 4096) rows_on_average = first_tiles <= cus ? 48 : 24;
    else if (p.k >= 2048 || (p.k >= 1024 && 4 * first_tiles <= 3 * (int64_t)cus)) rows_on_average = 16;
    if (!dense && m_hint <= rows_on_average * (int64_t)p.groups && (m_hint / kStream16Rows + p.groups) * ceil_div(p.n, 32) < (1ll << 31))
      return launch_grouped16_streaming<BF16_MMA>(p, cus, stream);
    // ... else the same kernel with 128x128 tiles, with two exceptions.  A shallow K with more tiles than compute units and so
    // few rows that there is one tile per weight panel and group: the tile kernel runs two workgroups per compute unit (tile
    // kernel / this one, us: 64 experts of 1024 x 1024, 8 rows each 27.3 / 29.5, of 1024 x 512 17.4 / 19.0; 16 of 4096 x 512 17.1 /
    // 18.3; 32 of 4096 x 256, 32 rows 20.6 / 22.5, 64 rows 23.7 / 24.1; 64 of 1024 x 1024, 16 rows: even loads 27.9 / 30.3, Zipf,
    // where some groups have two tiles, 47 / 39).  And a wide N with N / 128 no multiple of 8: each XCD then owns a piece of the
    // list instead of the same share of every group, and skewed groups make the pieces uneven (Zipf, 32 experts of 13824 x 2112, 57
    // rows 457 / 488, 16 of them, 24 rows 197 / 214, 64 of 11840 x 2560, 57 rows 943 / 1039; even loads 190 / 165 for 16 of 13824 x
    // 2112, 32 rows; narrower ones, Zipf: 64 of 8000 x 2048, 20 rows 461 / 406, 57 rows 543 / 529; dealt lists, Zipf: 8 of 14336 x
    // 2048, 100 rows 144 / 129, 32 of 12288 x 2880 538 / 484, 64 of 14336 x 1024 484 / 436).
    const bool two_per_cu = first_tiles > cus && (p.k < 512 ? m_hint <= 32 * (int64_t)p.groups
                                                            : p.k <= 1024 && first_tiles <= 2 * (int64_t)cus && m_hint <= 8 * (int64_t)p.groups);
    const bool uneven = (ceil_div(p.n, 128) & 7) != 0 && p.n > 10240 && p.k < 3072;
    if (lds_direct && p.k >= 256 && !two_per_cu && !uneven)
      return launch_grouped16_small_tiles<BF16_MMA, OUT_BF16>(p, cus, stream);
  }
  if constexpr (NVFP4) {
    // Grouped NVFP4: the groups of 1..32 rows and those of 33..128 rows (MoE decode, the small experts of a prefill) have
    // launches of their own, which stream their experts' weights; the launches below then skip them.  The group sizes live
    // on the device, so every kernel is always launched; workgroups without work return at once.
    if (!dense && p.min_rows == 0) {
      const bool with_large = nvfp4_large_groups_stream(p.groups, m_hint, p.n, p.k, cus) && !is_prefill;
      const bool own_rows = nvfp4_wavefronts_own_rows(p.groups, m_hint, p.n, p.k, cus, with_large);
      Gemm16Args small{};
      small.a = p.a, small.b = p.b, small.sfa = p.sfa, small.sfb = p.sfb, small.alpha = p.alpha, small.out = p.out;
      small.problem_sizes = p.problem_sizes, small.expert_offsets = p.expert_offsets, small.sf_offsets = p.sf_offsets;
      small.groups = p.groups, small.m = p.m, small.n = p.n, small.k = p.k, small.dtype = OUT_BF16 ? NVF_BF16 : NVF_F16;
      const bool mid_along = !own_rows && nvfp4_mid_groups_as_slabs(p.groups, m_hint, p.n, cus);
      int rc = NVF_OK, tail_done = 0;
      if (own_rows) rc = (p.n & 511) == 0 ? launch_nvfp4_skinny_grouped<4, 2, OUT_BF16, true>(p, 1, 32, stream)
                                          : launch_nvfp4_skinny_grouped<2, 2, OUT_BF16, true>(p, 1, 32, stream);
      if (rc == NVF_OK && (!own_rows || with_large)) rc = launch_nvfp4_decode(small, own_rows ? 0 : mid_along ? 128 : 32, with_large, stream);
      if (rc != NVF_OK || m_hint <= 32) return rc;
      // Below the prefill size the groups of 33..128 rows are few: they stream their weights like the smaller ones,
      // found by rank among the groups of their size (a launch with few workgroups when there are few rows in all), unless the
      // launch above has taken them along.  A
      // 128x256 tile of the persistent kernel walks all of K on one compute unit: with 64 or 256 experts, 512..5600
      // rows and K = 4096..14336 the call is 5-40 % slower that way wherever such groups exist and 0-3 % faster where
      // none does; with K < 4096 the tiles win from about 2048 rows on.
      if ((p.k & 127) != 0 || m_hint <= 1024 || (p.k >= 4096 && !is_prefill)) {
        // (also where K % 128 = 64: the form with a short last chunk)
        if (!mid_along) rc = launch_nvfp4_skinny_grouped<4, 8, OUT_BF16, false>(p, 33, 128, stream);
        if (with_large || m_hint <= 128) return rc;
      } else if ((p.k < 4096 || !is_prefill) && (p.n & 255) == 0 && p.k >= 256) {
        // shallow K: one 128x256 tile of the persistent kernel per weight panel converts a group's rows once per 256
        // weight rows; the streaming kernel whose wavefronts own rows converts them once per wavefront.
        Params mid = p;
        mid.rows_lo = 33;
        mid.rows_hi = 128;
        if (is_prefill) mid.min_rows = 129;  // the 256x256 kernel follows: take the ends of its groups along
        tail_done = mid.min_rows != 0;
        if (is_prefill && (p.n & 511) == 0 && p.k >= 1024) {
          // a prefill: the groups of up to 80 rows on the panel kernel, which multiplies row tiles of 16 (config 5,
          // K=2048: 5376 tiles of 128x256 in 680 us -> 325 us + 1792 tiles in 227 us)
          rc = launch_nvfp4_group_panel<4, 5, 2, OUT_BF16>(p, 33, 80, stream);
          if (rc != NVF_OK) return rc;
          mid.rows_lo = 81;
        }
        rc = launch_nvfp4_fast<OUT_BF16, true, 2>(mid, cus, stream);
      } else if (p.k < 4096 && (p.n & 255) == 0) {
        rc = launch_nvfp4_skinny_grouped<2, 8, OUT_BF16, true>(p, 33, 128, stream);
      } else if ((p.n & 511) == 0) {
        rc = launch_nvfp4_group_panel<4, 5, 2, OUT_BF16>(p, 33, 80, stream);
        if (rc == NVF_OK) {
          // groups of 81..128 rows and the ends of the groups that the 256x256 kernel takes: 128x256 tiles of the
          // persistent kernel, at 1.2 times the rate of the 128x128 tile kernel
          Params ends = p;
          ends.rows_lo = 81;
          ends.rows_hi = 128;
          ends.min_rows = 129;
          tail_done = 1;
          rc = launch_nvfp4_fast<OUT_BF16, true, 2>(ends, cus, stream);
        }
      } else {
        rc = launch_nvfp4_skinny_grouped<4, 8, OUT_BF16, false>(p, 33, 128, stream);
      }
      if (rc != NVF_OK) return rc;
      Params rest = p;
      rest.min_rows = 129;
      rest.tail_done = tail_done;
      return launch_sized<NVFP4, BF16_MMA, OUT_BF16>(rest, m_hint, cus, workspace, workspace_bytes, stream);
    }
    // Grouped NVFP4 with room for whole 256-row tiles: those go to the 256x256 kernel (about 1.4 times as
    // fast per flop), the ends of the groups to the 128x128 tile kernel.  The group sizes live on the
    // device, so both kernels are always launched; one that finds no work returns at once.
    if (!dense && (p.n & 255) == 0 && (p.k & 31) == 0 && p.k >= 256 && is_prefill) {
      const int rc = launch_nvfp4_fast<OUT_BF16, true>(p, cus, stream);
      if (rc != NVF_OK || p.tail_done) return rc;
      Params rest = p;
      rest.skip_whole_256 = 1;
      const int64_t upper = 2 * (int64_t)p.groups * ceil_div(p.n, 128), cap = 2 * (int64_t)cus;
      return launch_nvfp4_tile<128, 128, OUT_BF16>(rest, (int)(upper < cap ? upper : cap), stream);
    }
  }
  // grouped: the tile height follows the average group (a 256-row tile on a 77-row group is mostly padding)
  if (dense ? tiles(256, 256) >= cus : m_hint >= 512 * (int64_t)p.groups) {
    const int64_t upper = dense ? tiles(256, 256) : (ceil_div(p.m, 256) + p.groups) * ceil_div(p.n, 256);
    return launch_tile<256, 256, NVFP4, BF16_MMA, OUT_BF16>(p, (int)(upper < cus ? upper : cus), stream);
  }
  if (tiles(128, 128) >= cus || !dense) {
    const int64_t upper = dense ? tiles(128, 128) : (ceil_div(p.m, 128) + p.groups) * ceil_div(p.n, 128);
    const int64_t cap = 2 * (int64_t)cus;
    return launch_tile<128, 128, NVFP4, BF16_MMA, OUT_BF16>(p, (int)(upper < cap ? upper : cap), stream);
  }
  const int64_t upper = tiles(64, 64);
  const int64_t cap = 4 * (int64_t)cus;
  return launch_tile<64, 64, NVFP4, BF16_MMA, OUT_BF16>(p, (int)(upper < cap ? upper : cap), stream);
}

// Dense NVFP4 whose result leaves the kernel re-quantized to NVFP4 (FP4: nvfp4_scaled_mm_blockscale) or as the fp32
// product itself (that op's optional dump of what it quantized).  Both take the same kernel for a shape, so that
// the dump holds exactly the accumulators the quantized result was made from.
template <bool FP4>
int launch_nvfp4_wide_part(const Params& p, int cus, hipStream_t stream);

template <bool FP4>
int launch_nvfp4_wide(const Params& p, int cus, hipStream_t stream) {
  // A call that one launch of the weight-streaming kernel or of the persistent kernel (whose last row tile may hold
  // fewer rows) takes whole leaves that padding zero itself: no launch for it.
  const DensePlan::Kernel like16 = (p.k & 127) == 0 ? nvfp4_dense_plan(p.m, p.n, p.k, cus).kernel : DensePlan::kOther;
  const bool one_launch = like16 == DensePlan::kStream || like16 == DensePlan::kTiles256 || like16 == DensePlan::kTiles128;
  const bool cut_m = !one_launch && (p.n & 255) == 0 && (p.k & 127) == 0 && p.k >= 256 && p.m > 256 && (p.m & 127) != 0 &&
                     ceil_div(p.m / 128 * 128, 128) * (p.n / 256) >= cus / 2;
  const bool streams_whole = like16 == DensePlan::kStream;
  if (FP4 && !one_launch && ((p.m & 127) != 0 || ((p.n >> 4) & 3) != 0)) {
    // ragged: the padding rows / columns of the scale buffer's last 128x4 tiles are written as zero first
    const int64_t words = round_up(p.m, 128) * round_up(p.n >> 4, 4) / 4;
    if (!note_launch("zero_fill_kernel grid=%lld", (long long)ceil_div(words, 256))) {
      hipLaunchKernelGGL(zero_fill_kernel, dim3((unsigned)ceil_div(words, 256)), dim3(256), 0, stream, reinterpret_cast<uint32_t*>(p.out_sf), words);
      if (const int rc = check_launch("zero_fill_kernel")) return rc;
    }
  }
  if (cut_m) {
    // M not a multiple of 128 and enough rows for the persistent kernel: the rows up to the last multiple of 128 go
    // there, the rest to the tile kernels (their part of the result and of its scale tiles starts a whole number of
    // 128-row tiles further on)
    Params main = p, rest = p;
    main.m = p.m & ~127;
    rest.m = p.m - main.m;
    rest.a = p.a + (int64_t)main.m * (p.k >> 1);
    rest.sfa = p.sfa + (int64_t)main.m * round_up(p.k >> 4, 4);
    rest.out = static_cast<uint8_t*>(p.out) + (FP4 ? (int64_t)main.m * (p.n >> 1) : (int64_t)main.m * p.n * 4);
    if (FP4) rest.out_sf = p.out_sf + (int64_t)main.m * round_up(p.n >> 4, 4);
    if (const int rc = launch_nvfp4_wide_part<FP4>(main, cus, stream)) return rc;
    return launch_nvfp4_wide_part<FP4>(rest, cus, stream);
  }
  if (FP4 && streams_whole) {
    Params q = p;
    q.stream_zero_pad = 1;
    return launch_nvfp4_wide_part<FP4>(q, cus, stream);
  }
  return launch_nvfp4_wide_part<FP4>(p, cus, stream);
}

template <bool FP4>
int launch_nvfp4_wide_part(const Params& p, int cus, hipStream_t stream) {
  auto tiles = [&](int bm, int bn) { return ceil_div(p.m, bm) * ceil_div(p.n, bn); };
  // Decode-sized and other shapes that the 16-bit op streams: the same kernel, whose last stage then quantizes the
  // summed product (or stores it as it is) instead of rounding it to 16 bits (16 x 4096 x 4096: 28 -> 6 us, 128 x 4096 x
  // 14336: 85 -> 24 us on the tile kernels before).
  if ((p.k & 127) == 0 && nvfp4_dense_plan(p.m, p.n, p.k, cus).kernel == DensePlan::kStream) {
    Params q = p;
    q.stream_result = FP4 ? 1 : 2;
    return launch_nvfp4_skinny<true>(q, cus, stream);
  }
  if ((p.n & 255) == 0 && (p.k & 127) == 0 && p.k >= 256) {
    // as for the 16-bit results: persistent 256x256 or 128x256 tiles where they fill the compute units
    const DensePlan::Kernel like16 = nvfp4_dense_plan(p.m, p.n, p.k, cus).kernel;
    if (like16 == DensePlan::kTiles256) return launch_nvfp4_fast<false, false, 4, !FP4, FP4>(p, cus, stream);
    if (like16 == DensePlan::kTiles128) return launch_nvfp4_fast<false, false, 2, !FP4, FP4>(p, cus, stream);
    const int64_t t256 = (p.m & 255) == 0 ? tiles(256, 256) : 0, t128 = (p.m & 127) == 0 ? tiles(128, 256) : 0;
    const int64_t cost256 = t256 ? 100 * ceil_div(t256, cus) : INT64_MAX;
    const int64_t cost128 = t128 ? 58 * ceil_div(t128, cus) : INT64_MAX;
    const int64_t cost_tile = 144 * tiles(128, 256) / (2 * cus);
    if (t256 && cost256 <= cost128 && cost256 <= cost_tile) return launch_nvfp4_fast<false, false, 4, !FP4, FP4>(p, cus, stream);
    if (t128 && cost128 <= cost_tile) return launch_nvfp4_fast<false, false, 2, !FP4, FP4>(p, cus, stream);
  }
  if (tiles(256, 256) >= cus) return launch_nvfp4_tile<256, 256, false, !FP4, FP4>(p, cus, stream);
  if (tiles(128, 128) >= cus) {
    const int64_t t = tiles(128, 128);
    return launch_nvfp4_tile<128, 128, false, !FP4, FP4>(p, (int)(t < 2 * cus ? t : 2 * cus), stream);
  }
  const int64_t t = tiles(64, 64);
  return launch_nvfp4_tile<64, 64, false, !FP4, FP4>(p, (int)(t < 4 * cus ? t : 4 * cus), stream);
}

}  // namespace

int launch_gemm16(int op, const Gemm16Args& a, hipStream_t stream) {
  if (a.groups > kMaxGroups) return fail(NVF_ERR_UNSUPPORTED_SHAPE, "at most %d groups are supported, got %d", kMaxGroups, a.groups);
  if (a.m > INT32_MAX || a.n > INT32_MAX || a.k > INT32_MAX) return fail(NVF_ERR_UNSUPPORTED_SHAPE, "dimension exceeds int32");
  // (the kernels address a tile's 256 rows with 32-bit byte offsets)
  if (a.k >= (1 << 22)) return fail(NVF_ERR_UNSUPPORTED_SHAPE, "K = %lld: at most 4194303 is supported", (long long)a.k);
  Params p;
  p.a = static_cast<const uint8_t*>(a.a);
  p.b = static_cast<const uint8_t*>(a.b);
  p.sfa = static_cast<const uint8_t*>(a.sfa);
  p.sfb = static_cast<const uint8_t*>(a.sfb);
  p.alpha = a.alpha;
  p.out = a.out;
  p.problem_sizes = a.problem_sizes;
  p.expert_offsets = a.expert_offsets;
  p.sf_offsets = a.sf_offsets;
  p.groups = op == 0 ? 1 : a.groups;
  p.m = (int)a.m;
  p.n = (int)a.n;
  p.k = (int)a.k;
  p.ldc = (int)a.ldc;
  const int cus = cu_count();
  const bool bf16 = a.dtype == NVF_BF16;
  if (op == 0 && a.dtype == NVF_F32) return launch_nvfp4_wide<false>(p, cus, stream);
  if (op == 0 && a.dtype == kDtypeFp4BlockScaled) {
    p.out_sf = static_cast<uint8_t*>(a.out_sf);
    p.gnorm = a.gnorm;
    return launch_nvfp4_wide<true>(p, cus, stream);
  }
  if (op == 0 || op == 1) {
    auto launch = [&](const Params& q, void* workspace, int64_t workspace_bytes) {
      return bf16 ? launch_sized<true, false, true>(q, q.m, cus, workspace, workspace_bytes, stream)
                  : launch_sized<true, false, false>(q, q.m, cus, workspace, workspace_bytes, stream);
    };
    // Dense with M not a multiple of 128 (a prefill of any token count), which leaves the whole call to the tile
    // kernels: the rows up to the last multiple of 128 go to whatever kernel that shape gets, the remaining rows
    // (at most 127, a whole number of 128-row scale tiles further on) to the weight-streaming kernel in a launch of
    // their own (4000 x 4096 x 4096: 145 -> 116 us; 8100 x 8192 x 8192: 1002 -> 850 us).
    // Dense with N not a multiple of 256 (29568, 1408) and enough rows for the persistent kernel: the columns up to the
    // last multiple of 256 go to whatever kernel that shape gets, the remaining columns (weight rows) to a launch of
    // their own that writes into the same rows of the result.
    const bool split_wins = op == 0 && a.workspace != nullptr && nvfp4_splits(p.m, p.n, p.k, cus) > 1 &&
                            a.workspace_bytes >= (int64_t)nvfp4_splits(p.m, p.n, p.k, cus) * p.m * p.n * 4;
    if (const int n_cut = op == 0 && !split_wins ? nvfp4_n_cut(p.m, p.n, p.k, cus) : 0) {
      if (n_cut == 1) return bf16 ? launch_nvfp4_skinny<true>(p, cus, stream) : launch_nvfp4_skinny<false>(p, cus, stream);
      {
        Gemm16Args main = a, rest = a;
        main.n = p.n & ~255;
        rest.n = p.n - main.n;
        main.ldc = rest.ldc = a.ldc ? a.ldc : a.n;
        main.workspace = rest.workspace = nullptr;  // (a split of K keeps partial results at the pitch of its own N)
        main.workspace_bytes = rest.workspace_bytes = 0;
        const int64_t sf_padded = ((int64_t)(p.k >> 4) + 3) & ~(int64_t)3;
        rest.b = static_cast<const uint8_t*>(a.b) + main.n * (p.k >> 1);
        rest.sfb = static_cast<const uint8_t*>(a.sfb) + main.n * sf_padded;
        rest.out = static_cast<uint8_t*>(a.out) + main.n * 2;
        if (const int rc = launch_gemm16(op, main, stream)) return rc;
        return launch_gemm16(op, rest, stream);
      }
    }
    const int64_t main_rows = op == 0 ? nvfp4_rows_before_remainder(p.m, p.n, p.k, cus) : 0;
    if (main_rows == p.m) return bf16 ? launch_nvfp4_skinny<true>(p, cus, stream) : launch_nvfp4_skinny<false>(p, cus, stream);
    if (main_rows) {
      Params main = p, rest = p;
      main.m = (int)main_rows;
      rest.m = p.m - main.m;
      const int64_t sf_padded = ((int64_t)(p.k >> 4) + 3) & ~(int64_t)3;
      rest.a = p.a + (int64_t)main.m * (p.k >> 1);
      rest.sfa = p.sfa + (int64_t)main.m * sf_padded;
      rest.out = static_cast<uint8_t*>(p.out) + (int64_t)main.m * p.out_pitch() * 2;
      if (const int rc = launch(main, a.workspace, a.workspace_bytes)) return rc;
      return launch(rest, nullptr, 0);
    }
    return launch(p, a.workspace, a.workspace_bytes);
  }
  return bf16 ? launch_sized<false, true, true>(p, a.m, cus, nullptr, 0, stream)
              : launch_sized<false, false, false>(p, a.m, cus, nullptr, 0, stream);
}

// -------------------------------------------------------------------------------------------------
// Scratch memory that needs no allocation: the fp32 partial tiles of the split of K, for callers that cannot
// allocate (code under HIP graph capture, tight serving loops).  One array per device, held until the process
// ends; it keeps the contents of the last call, and the split-K kernels need no clearing because every partial
// tile the reduction reads has been written by the launch before it.  Calls that overlap on one device race.
// -------------------------------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

// Device address of this device's copy of the array.  The array's name is only a host-side stand-in; the address
// comes from hipGetSymbolAddress, asked once per device with that device current.
int static_scratch(void** ptr) {
  static std::mutex mu;
  static void* addr[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return fail(NVF_ERR_NO_DEVICE, "hipGetDevice failed");
  if (dev < 0 || dev >= 64) return fail(NVF_ERR_NO_DEVICE, "device id %d is out of range", dev);
  std::lock_guard<std::mutex> lock(mu);
  if (addr[dev] == nullptr) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) return fail(NVF_ERR_LAUNCH, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
    addr[dev] = p;
  }
  *ptr = addr[dev];
  return NVF_OK;
}

int64_t nvfp4_gemm_workspace_bytes(int64_t m, int64_t n, int64_t k) {
  if (m <= 0 || n <= 0 || k <= 0 || m > INT32_MAX || n > INT32_MAX || k > INT32_MAX) return 0;
  if (const int64_t main_rows = nvfp4_rows_before_remainder(m, n, k, cu_count())) {
    if (main_rows == m) return 0;  // all rows to the weight-streaming kernel
    m = main_rows;                 // the launch that may split K
  }
  const int skinny_splits = nvfp4_skinny_splits(m, n, k, cu_count());
  const int splits = skinny_splits > 1 ? skinny_splits : nvfp4_splits(m, n, k, cu_count());
  return splits > 1 ? (int64_t)splits * m * n * 4 : 0;
}

}  // namespace nvf
