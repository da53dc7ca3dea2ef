// bevpool.hip -- gfx950 (MI355X, CDNA4) kernels and C ABI for the LSS
// camera-to-BEV pooling path of ziyangyeh/bevfusion-triton.
//
// Pipeline (all stream-ordered on the caller's stream, no host sync):
//
//   index stage
//     quantize_geom_kernel / coord_ranks_kernel  point -> int32 rank (-1 dropped)
//       / quantize_frustum_kernel                + radix pass-0 block histogram
//                                                (frustum: geometry computed from
//                                                the camera matrices in-kernel)
//     radix_scan_kernel                          per-digit exclusive scan of the
//                                                block histograms (+ zero cell ranges)
//     radix_scatter_kernel<from_rank>            stable wave-ballot ranked scatter;
//                                                pass 0 also compacts kept points
//     radix_hist_kernel                          block histograms of passes >= 1
//     cell_ranges_kernel                         dense [start, end) per cell
//     bucket_sort_kernel                         ranks of 11..20 bits: after one
//                                                global pass by the high digit,
//                                                one block per group sorts the low
//                                                digit and writes its cell ranges
//                                                (replaces the passes >= 1 and
//                                                cell_ranges_kernel)
//     count_starts_kernel + scan_counts_kernel
//       + interval_write_kernel                  compacted interval starts/lengths
//   forward
//     accum_pipe_kernel<T,..>   ranges of 256 sorted points (snapped to cell
//                               boundaries); loader waves gather 16-byte row
//                               pieces through a register ring into LDS, one
//                               summing wave keeps a sequential fp32
//                               accumulator per channel
//     accum_group_kernel<T>     small inputs, wide or unaligned rows and the
//                               depth-weighted rows: groups of lanes walk
//                               their own cells, no LDS staging, no barriers
//     accum_rows_kernel<T>      rows of fewer than 16 bytes
//     rows_to_bev_kernel<T>     cell-major rows -> channel-first tile via LDS
//                               transpose; empty cells written as zero
//   backward
//     bev_to_rows_kernel<T>     channel-first grad tile -> cell-major rows
//                               (occupied cells only) via LDS transpose
//     gather_rows_kernel<V>     leading blocks read the ranks (per XCD) and the
//                               occupied rows once so the rest find them
//                               cached; then a point-order streaming copy of
//                               each point's cell row (zero rows for dropped
//                               points)
//   planar (channel-first) operands
//     planar_tile_kernel        (BN, C, S) -> channel-last rows (context, or
//                               channel-first camera features)
//     gather_planar_kernel      backward straight into a (BN, C, S) gradient
//   depth-weighted pooling (fused depth x context)
//     accum_group_kernel        forward sums of depth[p] * ctx[pix(p)]
//     depth_grad_kernel         grad_depth (dot products) and grad_context
//                               (depth-weighted sums along each ray)
//
// Numerics: the quantisation is IEEE fp32 subtraction followed by a correctly
// rounded fp32 division (built without fast-math, with
// -fhip-fp32-correctly-rounded-divide-sqrt and -ffp-contract=off), exactly as
// torch evaluates ((g - (bx - dx/2)) / dx) on the CPU.  Forward sums start at
// +0.0 and add the cell's points in increasing point index order, which is
// the order torch's CPU index_add_ uses, so fp32 results are bit-identical.

#include <hip/hip_runtime.h>

#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>

#include <mutex>
#include <type_traits>
#include <string>
#include <unordered_map>
#include <vector>

#include "bevpool.h"
#include "channel_blocks.h"

namespace {

using channel_blocks::kTileChannels;
using channel_blocks::first_channel;
using channel_blocks::planar_blocks;
using channel_blocks::planar_channels;
using channel_blocks::tile_channels;

// ---------------------------------------------------------------------------
// constants
// ---------------------------------------------------------------------------
constexpr int kThreads = 256;              // threads per block, every kernel
constexpr int kWaves = kThreads / 64;      // wave64 waves per block
// Keys per thread of the sort's tile kernels (quantise / coord ranks, radix
// histogram and scatter): 8 (tiles of 2048 keys) up to kLargeSortPoints
// points, 16 (4096) above.  Larger tiles halve the [digit][tile] histogram
// that every pass writes, scans and reads: at 4 x 360 x 360 and 2 x 720 x 720
// the forward took 7 and 16 us less on MI355X; at 1 x 360 x 360, whose tiles
// fill the chip in one round, 3-5 us more.
constexpr int kItemsSmall = 8, kItemsLarge = 16;
constexpr int64_t kLargeSortPoints = int64_t(4) << 20;
inline int sort_items(int64_t n_points) {
  return n_points > kLargeSortPoints ? kItemsLarge : kItemsSmall;
}
constexpr int kMaxDigitBits = 10;
constexpr int kMaxRadix = 1 << kMaxDigitBits;
constexpr int kCellTile = 64;              // cells per transpose tile

// 16- and 8-byte integer vectors.  HIP's uint4 struct blocks register
// promotion.  Float vectors are avoided on purpose: with packed fp32 ops
// disabled, hipcc 7.2 lowered a <2 x float> add of a 64-bit LDS load into two
// scalar adds that both read the low half.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
#ifndef BEVPOOL_RANGE_POINTS
#define BEVPOOL_RANGE_POINTS 256
#endif
constexpr int64_t kRangePoints = BEVPOOL_RANGE_POINTS;  // nominal sorted points per forward range
#ifndef BEVPOOL_XCD_MAP
#define BEVPOOL_XCD_MAP 1
#endif
constexpr int kXcds = 8;                   // MI355X: 8 XCDs, one L2 each

// Workgroup i of a launch runs on XCD i % 8.  xcd_chunk maps it to chunk
// (i % 8) * (n / 8) + i / 8 of a grid of n workgroups (n a multiple of 8,
// padded by xcd_grid), so each XCD walks one contiguous eighth of the
// chunks and neighbouring chunks share that XCD's L2.  A bijection on [0, n).
__device__ __forceinline__ int64_t xcd_chunk(int64_t i, int64_t n) {
#if BEVPOOL_XCD_MAP
  return (i % kXcds) * (n / kXcds) + i / kXcds;
#else
  (void)n;
  return i;
#endif
}

inline unsigned xcd_grid(int64_t blocks) {
#if BEVPOOL_XCD_MAP
  return unsigned((blocks + kXcds - 1) / kXcds * kXcds);
#else
  return unsigned(blocks);
#endif
}

// Grid of a kernel that walks the tiles of the sort (at least one
// block: block 0 also resets meta).  Such kernels take tile
// xcd_chunk(blockIdx.x, gridDim.x), so the 32 tiles that share a 128-byte
// line of a digit's histogram row are written from one XCD's L2.
inline unsigned sort_grid(int64_t tiles) { return tiles > 0 ? xcd_grid(tiles) : 1u; }

// ---------------------------------------------------------------------------
// error reporting
// ---------------------------------------------------------------------------
thread_local std::string g_last_error;

int fail(int code, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

// An AQL dispatch carries the grid size in work-items as 32 bits: a launch of
// more blocks * threads than that is rejected here instead of being
// truncated (which would leave part of the output unwritten).
int check_grid(int64_t blocks, int threads, const char *what) {
  if (blocks < 0 || blocks * int64_t(threads) > int64_t(UINT32_MAX))
    return fail(BEVPOOL_EINVAL, "%s: %lld blocks of %d threads exceed the 2^32 work-item grid",
                what, static_cast<long long>(blocks), threads);
  return BEVPOOL_OK;
}

int check_launch(const char *what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(BEVPOOL_EHIP, "%s: %s", what, hipGetErrorString(e));
  return BEVPOOL_OK;
}

// ---------------------------------------------------------------------------
// optional per-kernel timing (benchmark instrumentation)
// ---------------------------------------------------------------------------
struct TimingRecord {
  const char *name;
  hipEvent_t start, stop;
};
struct TimingTotal {
  double ms = 0.0;
  int64_t launches = 0;
};
std::mutex g_timing_mu;
bool g_timing_enabled = false;
// Set while an allocation-free entry point runs on this thread: its launches
// are never bracketed by timing events (creating one may allocate).
thread_local bool g_no_alloc_call = false;
std::vector<TimingRecord> g_timing_pending;
std::vector<hipEvent_t> g_event_pool;
std::vector<std::pair<std::string, TimingTotal>> g_timing_totals;

hipEvent_t take_event() {
  if (!g_event_pool.empty()) {
    hipEvent_t e = g_event_pool.back();
    g_event_pool.pop_back();
    return e;
  }
  hipEvent_t e = nullptr;
  if (hipEventCreate(&e) != hipSuccess) return nullptr;
  return e;
}

// Brackets one kernel launch with events when timing is enabled.
struct LaunchTimer {
  const char *name;
  hipStream_t stream;
  hipEvent_t start = nullptr, stop = nullptr;
  LaunchTimer(const char *n, hipStream_t s) : name(n), stream(s) {
    if (g_no_alloc_call) return;
    std::lock_guard<std::mutex> lk(g_timing_mu);
    if (!g_timing_enabled) return;
    start = take_event();
    stop = take_event();
    if (start && stop) (void)hipEventRecord(start, stream);
  }
  ~LaunchTimer() {
    if (!start || !stop) return;
    (void)hipEventRecord(stop, stream);
    std::lock_guard<std::mutex> lk(g_timing_mu);
    g_timing_pending.push_back({name, start, stop});
  }
};

// ---------------------------------------------------------------------------
// device helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

__device__ __forceinline__ uint64_t lanes_below() {
  return (uint64_t(1) << lane_id()) - 1;
}

__device__ __forceinline__ int key_rank(uint64_t k) { return int(uint32_t(k >> 32)); }
__device__ __forceinline__ uint32_t key_index(uint64_t k) { return uint32_t(k); }

__device__ __forceinline__ unsigned key_digit(uint64_t k, int shift, unsigned mask) {
  return unsigned(k >> (32 + shift)) & mask;
}

// Counts the digits held by the 64 lanes of a wave into cnt with one LDS
// atomic per run of equal digits in consecutive lanes (its first lane adds
// the run length).  Sorted keys hold long runs of one digit, which a
// per-lane atomic would serialise on one LDS address.  Lanes with valid ==
// false count nothing and end any run.  All 64 lanes must be active.
__device__ __forceinline__ void count_digit_runs(int *cnt, unsigned digit, bool valid) {
  const unsigned d = valid ? digit : 0xffffffffu;
  // digit of the lane below (wave shift right by one); lane 0 gets ~d
  const unsigned below = unsigned(__builtin_amdgcn_update_dpp(int(~d), int(d), 0x138, 0xf, 0xf,
                                                              false));
  const bool head = d != below;
  const uint64_t heads = __ballot(head);
  const int lane = lane_id();
  const uint64_t after = heads & ~((uint64_t(2) << lane) - 1);  // heads above this lane
  const int next = after ? __builtin_ctzll(after) : 64;
  if (valid && head) atomicAdd(&cnt[d], next - lane);
}

// OR of v over the 64 lanes (all active), in every lane's SGPR: DPP row
// shifts, row broadcasts 15 / 31, lane 63.
__device__ __forceinline__ unsigned wave_or(unsigned v) {
  int x = int(v);
  x |= __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
  x |= __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
  x |= __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
  x |= __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
  x |= __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
  x |= __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return unsigned(__builtin_amdgcn_readlane(x, 63));
}

// The valid lanes of the wave whose digit equals this lane's (a stable
// in-wave rank is the count of them below this lane).  Only the digit bits
// that differ between valid lanes can split them: one wave OR finds those,
// and each costs a ballot and a per-lane 64-bit combine (the VALU cost of
// the rank).  Sorted and clustered keys leave most bits uniform in a wave.
// All 64 lanes must be active.
__device__ __forceinline__ uint64_t peer_mask(unsigned dg, bool valid) {
  const uint64_t vm = __ballot(valid);
  if (vm == 0) return 0;
  const unsigned d0 = unsigned(__builtin_amdgcn_readlane(int(dg), int(__builtin_ctzll(vm))));
  uint64_t peers = vm;
  for (unsigned m = wave_or(valid ? dg ^ d0 : 0u); m; m &= m - 1) {
    const bool bit = (dg >> __builtin_ctz(m)) & 1u;
    const uint64_t bal = __ballot(bit);
    peers &= bit ? bal : ~bal;
  }
  return peers;
}

// Stable rank of this lane's key among the valid lanes of its wave with the
// same digit (`below`: how many come before it) and their number (`same`).
// When every lane is valid and the digits are monotone across the lanes (as
// keys in point order often are), each digit forms one run of lanes and both
// follow from the run starts: a DPP shift, four ballots and a few bit scans.
// Otherwise from the peer mask.  Either way the same numbers.  All 64 lanes
// must be active.
__device__ __forceinline__ void digit_rank(unsigned dg, bool valid, int &below, int &same) {
  const int lane = lane_id();
  const uint64_t le = (uint64_t(2) << lane) - 1;  // lanes <= this one
  if (__ballot(valid) == ~uint64_t(0)) {
    // digit of the lane below (lane 0 keeps its own)
    const unsigned prev =
        unsigned(__builtin_amdgcn_update_dpp(int(dg), int(dg), 0x138, 0xf, 0xf, false));
    if (__ballot(dg < prev) == 0 || __ballot(dg > prev) == 0) {
      const uint64_t heads = __ballot(dg != prev) | uint64_t(1);
      const int start = 63 - __builtin_clzll(heads & le);
      const uint64_t after = heads & ~le;
      below = lane - start;
      same = (after ? __builtin_ctzll(after) : 64) - start;
      return;
    }
  }
  const uint64_t peers = peer_mask(dg, valid);
  below = __popcll(peers & (le >> 1));
  same = __popcll(peers);
}

// Exclusive scan of one int per thread across a block of kW waves (256
// threads by default).  `scratch` holds kW ints.  Every thread must call it.
template <int kW = kWaves>
__device__ int block_exclusive_scan(int v, int *scratch, int *total) {
  const int lane = lane_id(), w = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) scratch[w] = x;
  __syncthreads();
  int before = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < kW; ++i) {
    int s = scratch[i];
    before += (i < w) ? s : 0;
    tot += s;
  }
  __syncthreads();
  *total = tot;
  return before + x - v;
}

// 16 and 8 bytes at element alignment: gfx950 loads and stores them in one
// instruction at any address, so rows need no vector alignment.
struct __attribute__((packed, aligned(2))) Bytes16 {
  u32x4 v;
};
struct __attribute__((packed, aligned(2))) Bytes8 {
  u32x2 v;
};
typedef u32x4 __attribute__((aligned(2))) u32x4_any;
typedef u32x2 __attribute__((aligned(2))) u32x2_any;

// fp32 / fp16 / bf16 element conversion.
struct F32 {
  using raw = uint32_t;
  __device__ static float load(const uint32_t *p) { return __builtin_bit_cast(float, *p); }
  __device__ static void store(uint32_t *p, float v) { *p = __builtin_bit_cast(uint32_t, v); }
  __device__ static uint32_t to_raw(float v) { return __builtin_bit_cast(uint32_t, v); }
};
struct F16 {
  using raw = uint16_t;
  __device__ static float load(const uint16_t *p) {
    return float(__builtin_bit_cast(_Float16, *p));
  }
  __device__ static void store(uint16_t *p, float v) {
    *p = __builtin_bit_cast(uint16_t, _Float16(v));
  }
  __device__ static uint16_t to_raw(float v) { return __builtin_bit_cast(uint16_t, _Float16(v)); }
  __device__ static float from_raw(uint32_t r) {
    return float(__builtin_bit_cast(_Float16, uint16_t(r)));
  }
};
struct BF16 {
  using raw = uint16_t;
  __device__ static float load(const uint16_t *p) {
    return __builtin_bit_cast(float, uint32_t(*p) << 16);
  }
  // round to nearest even; NaN -> canonical quiet NaN (torch's c10::BFloat16)
  __device__ static uint16_t to_raw(float v) {
    uint32_t u = __builtin_bit_cast(uint32_t, v);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;
    u += 0x7fffu + ((u >> 16) & 1u);
    return uint16_t(u >> 16);
  }
  __device__ static void store(uint16_t *p, float v) { *p = to_raw(v); }
  __device__ static float from_raw(uint32_t r) { return __builtin_bit_cast(float, r << 16); }
};

// ---------------------------------------------------------------------------
// index stage kernels
// ---------------------------------------------------------------------------

// n / d for n < 2^31 by multiply-high and shift (Granlund & Montgomery,
// "Division by invariant integers using multiplication", 1994): with
// s = ceil(log2 d) and m = floor(2^32 (2^s - d) / d) + 1 (host side),
// q = (mulhi(n, m) + n) >> s; mulhi(n, m) <= n keeps the sum in 32 bits.
struct FastDiv {
  uint32_t d, m, s;
  __device__ __forceinline__ uint32_t div(uint32_t n) const {
    return (__umulhi(n, m) + n) >> s;
  }
};

inline FastDiv make_fast_div(uint32_t d) {
  uint32_t s = 0;
  while ((uint64_t(1) << s) < d) ++s;
  const uint64_t m = ((uint64_t(1) << 32) * ((uint64_t(1) << s) - d)) / d + 1;
  return FastDiv{d, uint32_t(m), s};
}

// models/vtransforms/base.py:139-158: q = ((g - (bx - dx/2)) / dx).long(),
// kept iff 0 <= q_k < nx[k].  In fp32, trunc(q) in [0, n) <=> q > -1 && q < n
// (NaN fails both), which avoids converting out-of-range floats.
// Rank: ops/bev_pool/src/bev_pool_triton.py:34-39 with (D, H, W) = (nz, nx, ny).
__device__ __forceinline__ int quantize_point(float gx, float gy, float gz, int b, float o0,
                                              float o1, float o2, float d0, float d1, float d2,
                                              int n0, int n1, int n2) {
  const float q0 = (gx - o0) / d0;
  const float q1 = (gy - o1) / d1;
  const float q2 = (gz - o2) / d2;
  const bool kept = (q0 > -1.0f) & (q0 < float(n0)) & (q1 > -1.0f) & (q1 < float(n1)) &
                    (q2 > -1.0f) & (q2 < float(n2));
  if (!kept) return -1;
  const int x = int(q0), y = int(q1), z = int(q2);
  return ((b * n2 + z) * n0 + x) * n1 + y;
}

// Each thread handles groups of 4 consecutive points (group g of the block:
// points base + 4 * (g * kThreads + tid) + 0..3); with kVec (row stride 3
// floats, 16-byte aligned base) a group is three 16-byte loads and one
// 16-byte rank store.  All groups' loads are issued before any is used.
template <bool kVec, int kIt>
__global__ __launch_bounds__(kThreads) void quantize_geom_kernel(
    const float *__restrict__ geom, int64_t n_points, int64_t gstride, FastDiv ppb, float o0,
    float o1, float o2, float d0, float d1, float d2, int n0, int n1, int n2,
    int32_t *__restrict__ rank, int32_t *__restrict__ hist, int nblocks, int shift, int bits,
    int32_t *__restrict__ meta) {
  constexpr int kGroups = kIt / 4;
  __shared__ int cnt[kMaxRadix];
  if (blockIdx.x == 0 && threadIdx.x < BEVPOOL_META_LEN)  // nothing else touches meta here
    meta[threadIdx.x] = threadIdx.x == BEVPOOL_META_FIRST_BAD ? 0x7fffffff : 0;
  const int tile = int(xcd_chunk(blockIdx.x, gridDim.x));
  if (tile >= nblocks) return;  // grid padding, or the one block of an empty launch
  const int R = 1 << bits;
  const unsigned mask = unsigned(R - 1);
  for (int d = threadIdx.x; d < R; d += kThreads) cnt[d] = 0;
  const uint32_t base = uint32_t(tile) * (kThreads * kIt);  // n_points < 2^31
  const uint32_t n = uint32_t(n_points);
  // raw fp32 bits: lanes of a 16-byte load are never bit cast to float
  // while still in vector form (hipcc 7.2 folded such casts of lanes y/z/w
  // into lane x)
  uint32_t g[kGroups][12];
  const uint32_t *gb = reinterpret_cast<const uint32_t *>(geom);
#pragma unroll
  for (int k = 0; k < kGroups; ++k) {
    const uint32_t p0 = base + 4u * (uint32_t(k) * kThreads + threadIdx.x);
    if (kVec) {
      // groups past the last whole one read that one (in bounds, n >= 4);
      // a partial group is reloaded point by point below
      const uint32_t last = (n - 4) & ~3u;
      const uint32_t q0 = p0 + 3 < n ? p0 : last;
      const u32x4 *src = reinterpret_cast<const u32x4 *>(gb + int64_t(q0) * 3);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const u32x4 v = src[j];
        g[k][4 * j + 0] = v.x;
        g[k][4 * j + 1] = v.y;
        g[k][4 * j + 2] = v.z;
        g[k][4 * j + 3] = v.w;
      }
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t p = p0 + u < n ? p0 + u : n - 1;
        const uint32_t *gp = gb + int64_t(p) * gstride;
        g[k][3 * u + 0] = gp[0];
        g[k][3 * u + 1] = gp[1];
        g[k][3 * u + 2] = gp[2];
      }
    }
  }
  __syncthreads();  // cnt zeroed
#pragma unroll
  for (int k = 0; k < kGroups; ++k) {
    const uint32_t p0 = base + 4u * (uint32_t(k) * kThreads + threadIdx.x);
    if (kVec && p0 < n && p0 + 3 >= n) {
#pragma unroll
      for (int u = 0; u < 3; ++u) {
        if (p0 + u < n) {
          const uint32_t *gp = gb + int64_t(p0 + u) * 3;
          g[k][3 * u + 0] = gp[0];
          g[k][3 * u + 1] = gp[1];
          g[k][3 * u + 2] = gp[2];
        }
      }
    }
    int r[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      r[u] = quantize_point(__builtin_bit_cast(float, g[k][3 * u]),
                            __builtin_bit_cast(float, g[k][3 * u + 1]),
                            __builtin_bit_cast(float, g[k][3 * u + 2]), int(ppb.div(p0 + u)),
                            o0, o1, o2, d0, d1, d2, n0, n1, n2);
      count_digit_runs(cnt, (unsigned(r[u]) >> shift) & mask, r[u] >= 0 && p0 + u < n);
    }
    if (kVec && p0 + 3 < n) {
      u32x4 w;
      w.x = uint32_t(r[0]);
      w.y = uint32_t(r[1]);
      w.z = uint32_t(r[2]);
      w.w = uint32_t(r[3]);
      *reinterpret_cast<u32x4 *>(rank + p0) = w;
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (p0 + u < n) rank[p0 + u] = r[u];
    }
  }
  __syncthreads();
  for (int d = threadIdx.x; d < R; d += kThreads) hist[int64_t(d) * nblocks + tile] = cnt[d];
}

// ---- geometry from camera matrices, fused with the quantisation -----------
//
// models/vtransforms/base.py:82-126 (get_geometry) per point, in fp32 with
// every product and sum rounded separately (no contraction), each 3x3
// product summed left to right:
//   a = frustum[d, h, w] - post_trans          (base.py:95)
//   b = post_rots^T a                           (:96-98)
//   c = (b0 b2, b1 b2, b2)                      (:100-106)
//   g = combine c + camera2lidar_trans          (:107-112)
//   g = extra_rots g + extra_trans              (:114-123, when given)
// then quantize_point as for a geometry tensor.  combine = rots inv(intrins)
// (the reference's linalg.solve) is formed in double from the adjugate of
// intrins and rounded to fp32 once.  Per camera the kernel works from a
// 24-float table: post_rots^T (9, row-major), post_trans (3), combine (9),
// camera2lidar_trans (3); per batch a 12-float table: extra_rots (9),
// extra_trans (3).
constexpr int kCamFloats = 24;
constexpr int kBatchFloats = 12;
constexpr int kCamSlots = 16;  // cameras a block stages in LDS

struct CameraMats {  // fp32, row-major, contiguous per camera / batch
  const float *rots, *trans, *intrins, *post_rots, *post_trans;  // [B*N][9|3]
  const float *extra_rots, *extra_trans;                         // [B][9|3] or null
  int n_per_batch;                                               // N
  __device__ __forceinline__ bool has_extra() const { return extra_rots || extra_trans; }
};

// One camera's inputs, all loaded before any is used (one round trip).
struct CamIn {
  float pr[9], pt[3], k[9], r[9], tr[3];
};

__device__ __forceinline__ void load_camera(const CameraMats &m, uint32_t cam, CamIn &c) {
  const int64_t o9 = int64_t(cam) * 9, o3 = int64_t(cam) * 3;
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    c.pr[i] = m.post_rots[o9 + i];
    c.k[i] = m.intrins[o9 + i];
    c.r[i] = m.rots[o9 + i];
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    c.pt[i] = m.post_trans[o3 + i];
    c.tr[i] = m.trans[o3 + i];
  }
}

__device__ void build_camera_table(const CamIn &c, float *__restrict__ t) {
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) t[3 * i + j] = c.pr[3 * j + i];  // post_rots^T
  for (int i = 0; i < 3; ++i) t[9 + i] = c.pt[i];
  double k[9];
  for (int i = 0; i < 9; ++i) k[i] = double(c.k[i]);
  const double c00 = k[4] * k[8] - k[5] * k[7], c01 = k[5] * k[6] - k[3] * k[8];
  const double c02 = k[3] * k[7] - k[4] * k[6];
  const double det = k[0] * c00 + k[1] * c01 + k[2] * c02;
  double inv[9] = {c00, k[2] * k[7] - k[1] * k[8], k[1] * k[5] - k[2] * k[4],
                   c01, k[0] * k[8] - k[2] * k[6], k[2] * k[3] - k[0] * k[5],
                   c02, k[1] * k[6] - k[0] * k[7], k[0] * k[4] - k[1] * k[3]};
  for (int i = 0; i < 9; ++i) inv[i] /= det;
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) {
      double v = 0.0;
      for (int q = 0; q < 3; ++q) v += double(c.r[3 * i + q]) * inv[3 * q + j];
      t[12 + 3 * i + j] = float(v);
    }
  for (int i = 0; i < 3; ++i) t[21 + i] = c.tr[i];
}

__device__ void camera_table(const CameraMats &m, uint32_t cam, float *__restrict__ t) {
  CamIn c;
  load_camera(m, cam, c);
  build_camera_table(c, t);
}

// The lidar-augmentation table of batch b (identity when absent), with one
// branch per pointer so that its loads are issued together.
__device__ __forceinline__ void batch_table(const CameraMats &m, uint32_t b,
                                            float *__restrict__ t) {
  if (m.extra_rots) {
#pragma unroll
    for (int i = 0; i < 9; ++i) t[i] = m.extra_rots[int64_t(b) * 9 + i];
  } else {
#pragma unroll
    for (int i = 0; i < 9; ++i) t[i] = i % 4 == 0 ? 1.0f : 0.0f;
  }
  if (m.extra_trans) {
#pragma unroll
    for (int i = 0; i < 3; ++i) t[9 + i] = m.extra_trans[int64_t(b) * 3 + i];
  } else {
#pragma unroll
    for (int i = 0; i < 3; ++i) t[9 + i] = 0.0f;
  }
}

__device__ __forceinline__ void frustum_point(const float *__restrict__ c,
                                              const float *__restrict__ e, float fx, float fy,
                                              float fz, float &gx, float &gy, float &gz) {
  const float a0 = fx - c[9], a1 = fy - c[10], a2 = fz - c[11];
  const float b0 = (c[0] * a0 + c[1] * a1) + c[2] * a2;
  const float b1 = (c[3] * a0 + c[4] * a1) + c[5] * a2;
  const float b2 = (c[6] * a0 + c[7] * a1) + c[8] * a2;
  const float c0 = b0 * b2, c1 = b1 * b2;
  gx = ((c[12] * c0 + c[13] * c1) + c[14] * b2) + c[21];
  gy = ((c[15] * c0 + c[16] * c1) + c[17] * b2) + c[22];
  gz = ((c[18] * c0 + c[19] * c1) + c[20] * b2) + c[23];
  if (e) {
    const float h0 = ((e[0] * gx + e[1] * gy) + e[2] * gz) + e[9];
    const float h1 = ((e[3] * gx + e[4] * gy) + e[5] * gz) + e[10];
    const float h2 = ((e[6] * gx + e[7] * gy) + e[8] * gz) + e[11];
    gx = h0;
    gy = h1;
    gz = h2;
  }
}

// Point p = cam * DHW + f (cam = b*N + n, f = (d*fH + h)*fW + w); frustum
// fp32 (D, fH, fW, 3) contiguous.  A block takes kThreads * kIt consecutive points
// (as quantize_geom_kernel, so the pass-0 histograms line up); its first
// threads build the tables of the cameras it spans in LDS.  A block spanning
// more than kCamSlots cameras (frustums under ~140 points) builds each
// point's table in registers instead.
template <int kIt>
__global__ __launch_bounds__(kThreads) void quantize_frustum_kernel(
    const float *__restrict__ frustum, int64_t n_points, FastDiv dhw, FastDiv npb, CameraMats cm,
    float o0,
    float o1, float o2, float d0, float d1, float d2, int n0, int n1, int n2,
    int32_t *__restrict__ rank, int32_t *__restrict__ hist, int nblocks, int shift, int bits,
    int32_t *__restrict__ meta) {
  __shared__ int cnt[kMaxRadix];
  __shared__ float lcam[kCamSlots][kCamFloats];
  __shared__ float lbat[kCamSlots][kBatchFloats];
  if (blockIdx.x == 0 && threadIdx.x < BEVPOOL_META_LEN)
    meta[threadIdx.x] = threadIdx.x == BEVPOOL_META_FIRST_BAD ? 0x7fffffff : 0;
  const int tile = int(xcd_chunk(blockIdx.x, gridDim.x));
  if (tile >= nblocks) return;
  const int R = 1 << bits;
  const unsigned mask = unsigned(R - 1);
  for (int d = threadIdx.x; d < R; d += kThreads) cnt[d] = 0;
  const uint32_t n = uint32_t(n_points);
  const uint32_t base = uint32_t(tile) * (kThreads * kIt);
  const uint32_t last = (base + (kThreads * kIt) < n ? base + (kThreads * kIt) : n) - 1;
  const uint32_t cam_lo = dhw.div(base), cam_hi = dhw.div(last);
  const bool staged = cam_hi - cam_lo < uint32_t(kCamSlots);
  const bool extra = cm.has_extra();
  // all frustum loads first (points past n reload point n - 1), issued
  // before the camera tables are built so that their latencies overlap
  float fx[kIt], fy[kIt], fz[kIt];
  uint32_t camv[kIt];
  if (staged) {
#pragma unroll
    for (int k = 0; k < kIt; ++k) {
      const uint32_t p = base + uint32_t(k) * kThreads + threadIdx.x;
      const uint32_t pc = p < n ? p : n - 1;
      const uint32_t cam = dhw.div(pc), f = pc - cam * dhw.d;
      camv[k] = cam;
      fx[k] = frustum[int64_t(f) * 3];
      fy[k] = frustum[int64_t(f) * 3 + 1];
      fz[k] = frustum[int64_t(f) * 3 + 2];
    }
  }
  if (staged && threadIdx.x <= cam_hi - cam_lo) {
    // the camera's and its batch's inputs loaded together, then the tables
    const uint32_t cam = cam_lo + threadIdx.x;
    CamIn c;
    load_camera(cm, cam, c);
    float e[kBatchFloats];
    if (extra) batch_table(cm, npb.div(cam), e);
    build_camera_table(c, lcam[threadIdx.x]);
    if (extra)
#pragma unroll
      for (int i = 0; i < kBatchFloats; ++i) lbat[threadIdx.x][i] = e[i];
  }
  __syncthreads();
  if (staged) {
    // then the products; digit counts by runs (every lane active)
#pragma unroll
    for (int k = 0; k < kIt; ++k) {
      const uint32_t p = base + uint32_t(k) * kThreads + threadIdx.x;
      const uint32_t c = camv[k] - cam_lo;
      float gx, gy, gz;
      frustum_point(lcam[c], extra ? lbat[c] : nullptr, fx[k], fy[k], fz[k], gx, gy, gz);
      const int r = quantize_point(gx, gy, gz, int(npb.div(camv[k])), o0, o1, o2, d0, d1, d2, n0,
                                   n1, n2);
      count_digit_runs(cnt, (unsigned(r) >> shift) & mask, p < n && r >= 0);
      if (p < n) rank[p] = r;
    }
  } else {
    // more cameras than LDS slots: each point's tables in registers
    for (int k = 0; k < kIt; ++k) {
      const uint32_t p = base + uint32_t(k) * kThreads + threadIdx.x;
      int r = -1;
      if (p < n) {
        const uint32_t cam = dhw.div(p), f = p - cam * dhw.d;
        const float *fr = frustum + int64_t(f) * 3;
        float gx, gy, gz;
        float ct[kCamFloats], bt[kBatchFloats];
        camera_table(cm, cam, ct);
        if (extra) batch_table(cm, npb.div(cam), bt);
        frustum_point(ct, extra ? bt : nullptr, fr[0], fr[1], fr[2], gx, gy, gz);
        r = quantize_point(gx, gy, gz, int(npb.div(cam)), o0, o1, o2, d0, d1, d2, n0, n1, n2);
        if (r >= 0) atomicAdd(&cnt[(unsigned(r) >> shift) & mask], 1);
        rank[p] = r;
      }
    }
  }
  __syncthreads();
  for (int d = threadIdx.x; d < R; d += kThreads) hist[int64_t(d) * nblocks + tile] = cnt[d];
}

// ops/bev_pool/src/bev_pool_triton.py:34-39 in int64 (wrapping) arithmetic.
// Invalid ranks are counted into meta with atomics (meta initialised by an
// earlier launch) or, with kTileBad, per tile into tile_bad[tile] (count) and
// tile_bad[nblocks + tile] (smallest point index, INT32_MAX if none), which
// the first scatter reduces into meta -- so the op level needs no separate
// launch to initialise meta.
template <typename TC, int kIt, bool kTileBad>
__global__ __launch_bounds__(kThreads) void coord_ranks_kernel(
    const TC *__restrict__ coords, int64_t n_points, int64_t cstride, int64_t B, int64_t D,
    int64_t H, int64_t W, int32_t *__restrict__ rank, int32_t *__restrict__ meta,
    int32_t *__restrict__ hist, int nblocks, int shift, int bits,
    int32_t *__restrict__ tile_bad) {
  __shared__ int cnt[kMaxRadix];
  __shared__ int s_bad[2];
  const int R = 1 << bits;
  const unsigned mask = unsigned(R - 1);
  const int tile = int(xcd_chunk(blockIdx.x, gridDim.x));
  if (tile >= nblocks) return;  // grid padding
  for (int d = threadIdx.x; d < R; d += kThreads) cnt[d] = 0;
  if (kTileBad && threadIdx.x == 0) {
    s_bad[0] = 0;
    s_bad[1] = INT32_MAX;
  }
  __syncthreads();
  const int64_t base = int64_t(tile) * (kThreads * kIt);
  const uint64_t cells = uint64_t(B * D * H * W);
  // the coordinates of kBatch points per thread are loaded before any is
  // used (clamped to the last point, so the loads need no branch); the
  // digits are counted one atomic per run of equal digits
  constexpr int kBatch = sizeof(TC) == 4 ? 8 : 4;  // 32 VGPRs of coordinates
  static_assert(kIt % kBatch == 0, "whole batches per thread");
  for (int k0 = 0; k0 < kIt; k0 += kBatch) {
    TC cv[kBatch][4];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int64_t p = base + int64_t(k0 + u) * kThreads + threadIdx.x;
      const TC *c = coords + (p < n_points ? p : n_points - 1) * cstride;
#pragma unroll
      for (int j = 0; j < 4; ++j) cv[u][j] = c[j];
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int64_t p = base + int64_t(k0 + u) * kThreads + threadIdx.x;
      const uint64_t x = uint64_t(int64_t(cv[u][0])), y = uint64_t(int64_t(cv[u][1]));
      const uint64_t z = uint64_t(int64_t(cv[u][2])), b = uint64_t(int64_t(cv[u][3]));
      const uint64_t r64 = ((b * uint64_t(D) + z) * uint64_t(H) + x) * uint64_t(W) + y;
      const bool ok = p < n_points && r64 < cells;  // unsigned: negative ranks fail too
      const int r = ok ? int(r64) : -1;
      count_digit_runs(cnt, (unsigned(r) >> shift) & mask, ok);  // every lane takes part
      if (p < n_points) {
        if (!ok) {
          if (kTileBad) {
            atomicAdd(&s_bad[0], 1);
            atomicMin(&s_bad[1], int(p));
          } else {
            atomicAdd(&meta[BEVPOOL_META_N_BAD], 1);
            atomicMin(&meta[BEVPOOL_META_FIRST_BAD], int(p));
          }
        }
        rank[p] = r;
      }
    }
  }
  __syncthreads();
  for (int d = threadIdx.x; d < R; d += kThreads) hist[int64_t(d) * nblocks + tile] = cnt[d];
  if (kTileBad && threadIdx.x == 0) {
    tile_bad[tile] = s_bad[0];
    tile_bad[nblocks + tile] = s_bad[1];
  }
}

__global__ void init_meta_kernel(int32_t *meta) {
  if (threadIdx.x < BEVPOOL_META_LEN)
    meta[threadIdx.x] = threadIdx.x == BEVPOOL_META_FIRST_BAD ? 0x7fffffff : 0;
}


// One block per digit: exclusive scan over the blocks of hist[d][*] in place,
// totals[d] = row sum.  Optionally zeroes the dense cell ranges (grid-stride).
__global__ __launch_bounds__(kThreads) void radix_scan_kernel(
    int32_t *__restrict__ hist, int nblocks, int32_t *__restrict__ totals,
    int32_t *__restrict__ cstart, int32_t *__restrict__ cend, int64_t zero_cells) {
  __shared__ int scratch[kWaves];
  int32_t *row = hist + int64_t(blockIdx.x) * nblocks;
  int carry = 0;
  for (int t0 = 0; t0 < nblocks; t0 += kThreads * 4) {
    int v[4], s = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int j = t0 + threadIdx.x * 4 + i;
      v[i] = j < nblocks ? row[j] : 0;
      s += v[i];
    }
    int tot;
    int ex = block_exclusive_scan(s, scratch, &tot) + carry;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int j = t0 + threadIdx.x * 4 + i;
      if (j < nblocks) row[j] = ex;
      ex += v[i];
    }
    carry += tot;
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
  for (int64_t c = int64_t(blockIdx.x) * kThreads + threadIdx.x; c < zero_cells;
       c += int64_t(gridDim.x) * kThreads) {
    cstart[c] = 0;
    cend[c] = 0;
  }
}

// Block histogram of one digit over the sorted keys of the previous pass.
template <int kIt>
__global__ __launch_bounds__(kThreads) void radix_hist_kernel(
    const uint64_t *__restrict__ keys, const int32_t *__restrict__ meta,
    int32_t *__restrict__ hist, int nblocks, int shift, int bits) {
  __shared__ int cnt[kMaxRadix];
  const int R = 1 << bits;
  const unsigned mask = unsigned(R - 1);
  const int tile = int(xcd_chunk(blockIdx.x, gridDim.x));
  if (tile >= nblocks) return;  // grid padding
  for (int d = threadIdx.x; d < R; d += kThreads) cnt[d] = 0;
  __syncthreads();
  const int64_t n = meta[BEVPOOL_META_N_KEPT];
  const int64_t base = int64_t(tile) * (kThreads * kIt);
  // all loads first (in bounds: past n they read key 0), then the counts
  uint64_t key[kIt];
#pragma unroll
  for (int k = 0; k < kIt; ++k) {
    const int64_t e = base + int64_t(k) * kThreads + threadIdx.x;
    key[k] = keys[e < n ? e : 0];
  }
#pragma unroll
  for (int k = 0; k < kIt; ++k)
    count_digit_runs(cnt, key_digit(key[k], shift, mask),
                     base + int64_t(k) * kThreads + threadIdx.x < n);
  __syncthreads();
  for (int d = threadIdx.x; d < R; d += kThreads) hist[int64_t(d) * nblocks + tile] = cnt[d];
}

// Stable scatter of one LSD radix pass.  Wave w of block b owns the 64 * kIt
// consecutive keys [(b*4 + w) * 64 * kIt, +64 * kIt) and walks them 64 at a
// time in order; a key's destination is
//   (keys of smaller digits overall) + (same digit in earlier blocks)
//   + (same digit in earlier waves of this block) + (same digit earlier in
//   this wave),
// the last term from a ballot-built peer mask, so equal digits keep their
// input order.  Pass 0 (kFromRank) reads int32 ranks in point order, skips
// dropped points (compaction) and builds the (rank << 32 | point) keys.
template <bool kFromRank, int kIt>
__global__ __launch_bounds__(kThreads) void radix_scatter_kernel(
    const int32_t *__restrict__ rank_in, const uint64_t *__restrict__ keys_in,
    int64_t n_points, int32_t *__restrict__ meta, uint64_t *__restrict__ keys_out,
    const int32_t *__restrict__ hist, const int32_t *__restrict__ totals, int nblocks,
    int shift, int bits, const int32_t *__restrict__ tile_bad, int32_t *__restrict__ gstart) {
  __shared__ int s_base[kMaxRadix];
  __shared__ int s_cnt[kWaves * kMaxRadix];
  __shared__ int s_scan[kWaves];
  const int R = 1 << bits;
  const unsigned mask = unsigned(R - 1);
  const int tid = threadIdx.x, lane = lane_id(), w = tid >> 6;
  const int64_t n = kFromRank ? n_points : int64_t(meta[BEVPOOL_META_N_KEPT]);
  // XCD-contiguous tiles: a digit's runs from neighbouring tiles are adjacent
  // in the output, so writing them from one XCD lets its L2 merge them into
  // whole lines
  const int tile = int(xcd_chunk(blockIdx.x, gridDim.x));
  const int64_t blk0 = int64_t(tile) * (kThreads * kIt);
  if (tile >= nblocks || blk0 >= n) return;  // whole block leaves before any barrier

  // this wave's keys, in order (loads issued first so that their latency
  // overlaps the digit-base computation below)
  uint64_t key[kIt];
  bool valid[kIt];
  const int64_t wbase = blk0 + int64_t(w) * (64 * kIt);
#pragma unroll
  for (int k = 0; k < kIt; ++k) {
    const int64_t e = wbase + k * 64 + lane;
    if (kFromRank) {
      const int r = rank_in[e < n ? e : n - 1];
      valid[k] = e < n && r >= 0;
      key[k] = (uint64_t(uint32_t(r)) << 32) | uint64_t(uint32_t(e));
    } else {
      valid[k] = e < n;
      key[k] = keys_in[e < n ? e : n - 1];
    }
  }

  // digit bases: exclusive scan of the digit totals + this block's prefix
  // (both loaded before the scan, so their latencies overlap); tile 0's bases
  // are the digit starts, kept in gstart for the per-group sort
  constexpr int kPer = kMaxRadix / kThreads;  // digits per thread (4)
  int loc[kPer], pre[kPer], tsum = 0;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int d = tid * kPer + i;
    loc[i] = d < R ? totals[d] : 0;
    pre[i] = d < R ? hist[int64_t(d) * nblocks + tile] : 0;
  }
#pragma unroll
  for (int i = 0; i < kPer; ++i) tsum += loc[i];
  for (int d = tid; d < kWaves * R; d += kThreads) s_cnt[d] = 0;
  int total;
  int ex = block_exclusive_scan(tsum, s_scan, &total);
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int d = tid * kPer + i;
    if (d < R) {
      s_base[d] = ex + pre[i];
      if (gstart && tile == 0) gstart[d] = ex;
    }
    ex += loc[i];
  }
  if (kFromRank && tile == 0) {
    if (tile_bad) {
      // ranks from coord_ranks_kernel<..., true>: meta was never initialised;
      // write all of it (kept count, the reduced invalid-rank counters, zeros)
      int nbad = 0, first = INT32_MAX;
      for (int t = tid; t < nblocks; t += kThreads) {
        nbad += tile_bad[t];
        first = min(first, tile_bad[nblocks + t]);
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        nbad += __shfl_xor(nbad, o, 64);
        first = min(first, __shfl_xor(first, o, 64));
      }
      __shared__ int s_red[2 * kWaves];
      if (lane == 0) {
        s_red[w] = nbad;
        s_red[kWaves + w] = first;
      }
      __syncthreads();
      if (tid < BEVPOOL_META_LEN) {
        int v = 0;
        if (tid == BEVPOOL_META_N_KEPT) {
          v = total;
        } else if (tid == BEVPOOL_META_N_BAD) {
#pragma unroll
          for (int i = 0; i < kWaves; ++i) v += s_red[i];
        } else if (tid == BEVPOOL_META_FIRST_BAD) {
          v = INT32_MAX;
#pragma unroll
          for (int i = 0; i < kWaves; ++i) v = min(v, s_red[kWaves + i]);
        }
        meta[tid] = v;
      }
    } else if (tid == 0) {
      meta[BEVPOOL_META_N_KEPT] = total;
    }
  }
  __syncthreads();

  // per-wave digit counts
  int *cnt = s_cnt + w * R;
#pragma unroll
  for (int k = 0; k < kIt; ++k) count_digit_runs(cnt, key_digit(key[k], shift, mask), valid[k]);
  __syncthreads();
  for (int d = tid; d < R; d += kThreads) {
    int run = s_base[d];
#pragma unroll
    for (int ww = 0; ww < kWaves; ++ww) {
      const int c = s_cnt[ww * R + d];
      s_cnt[ww * R + d] = run;
      run += c;
    }
  }
  __syncthreads();

#pragma unroll
  for (int k = 0; k < kIt; ++k) {
    const unsigned dg = key_digit(key[k], shift, mask);
    int below, same;
    digit_rank(dg, valid[k], below, same);
    if (valid[k]) {
      const int pos = cnt[dg] + below;
      keys_out[pos] = key[k];
      if (below == 0) cnt[dg] = pos + same;
    }
  }
}

// Second half of the sort when the ranks need 11..20 bits.  One global pass
// (radix_scatter_kernel<true> by the high digit rank >> lbits) has grouped
// the kept keys by high digit, each group in point order.  The keys of group
// b are sorted stably by the low lbits bits, so the keys end sorted by rank
// with ties in point order, as two LSD passes would leave them, and the dense
// [start, end) of the group's 2^lbits cells is written (0, 0 when empty),
// which replaces cell_ranges_kernel and the zeroing of the cell ranges.
// A group of gn keys is cut into P = min(parts_max, ceil(gn / part_keys))
// consecutive parts, one block each, so that a large group (the cells near
// the cameras) is not ranked by one block alone.  The block of part p first
// counts the digits of the group's other keys (those before its part apart),
// then walks its own part as one block walks a whole group:
// Wave w of kBucketWaves owns the w-th slice of the part (a multiple of 64
// keys) and walks it 64 keys at a time, in order, twice: the first walk
// counts its digits, the second puts each key at
//   (group start) + (smaller digits in the group) + (same digit in earlier
//   parts) + (same digit in earlier waves) + (same digit earlier in this
//   wave),
// the last term from a ballot-built peer mask as in radix_scatter_kernel.
// No block waits for another.  Block i takes part parts_max - 1 - i / n of
// group i % n (n groups): the blocks of the later parts, of which only the
// large groups' do any work, come first, so that those start at once.  The
// block of part 0 writes the cell ranges.  Keys are loaded kBucketBatch
// sub-batches (of 64) at a time; a wave whose slice fits in one batch keeps
// it in registers for the second walk.  Otherwise the second walk drains
// each batch's loads before its first key store: vmcnt counts loads and
// stores together, so a wait for a load issued after a store would also wait
// for the store.  Dynamic LDS: (kBucketWaves + 2) * 2^lbits ints (16 waves,
// up to 512 digits: at most 36 KB per block).  Groups of 1024 cells take the
// sliced form below instead.
template <int kBucketWaves>
__global__ __launch_bounds__(64 * kBucketWaves, 8) void bucket_sort_kernel(
    const uint64_t *__restrict__ keys_in, const int32_t *__restrict__ totals,
    const int32_t *__restrict__ gstart, int n_buckets, int64_t n_cells,
    uint64_t *__restrict__ keys_out, int32_t *__restrict__ cstart, int32_t *__restrict__ cend,
    int lbits, int parts_max, int part_keys) {
  constexpr int kBucketThreads = 64 * kBucketWaves;
  // sub-batches per load batch: 12 keeps the 16-wave kernel within 64 VGPRs
  // (56; two blocks per CU) and a wave's part of any group up to 12,288 keys
  // in registers between its two walks (16 spills)
  constexpr int kBucketBatch = 12;
  extern __shared__ int s_cnt[];  // [kBucketWaves][R] own part, then [R] other parts, [R] before
  __shared__ int s_scan[kBucketWaves];
  const int bkt = int(blockIdx.x) % n_buckets;
  const int part = parts_max - 1 - int(blockIdx.x) / n_buckets;
  const int tid = threadIdx.x, lane = lane_id(), w = tid >> 6;
  const int R = 1 << lbits;
  const unsigned mask = unsigned(R - 1);

  // group start (keys of smaller high digits, from the global pass) and size
  const int gs = gstart[bkt];
  const int gn = totals[bkt];
  const int np = gn > part_keys ? (gn + part_keys - 1) / part_keys : 1;
  const int P = np < parts_max ? np : parts_max;
  if (part >= P) return;
  // this part: [ps, pe), a multiple of 64 keys but the last
  const int L = ((gn + P - 1) / P + 63) & ~63;
  const int64_t ge = int64_t(gs) + gn;
  const int ps = int(gs + int64_t(part) * L < ge ? gs + int64_t(part) * L : ge);
  const int pe = int(gs + int64_t(part + 1) * L < ge ? gs + int64_t(part + 1) * L : ge);
  int *s_out = s_cnt + kBucketWaves * R;  // digits of the group's other parts
  int *s_before = s_out + R;              // digits of the parts before this one
  for (int d = tid; d < (kBucketWaves + 2) * R; d += kBucketThreads) s_cnt[d] = 0;
  const int64_t q = (int64_t(pe - ps) + kBucketThreads - 1) / kBucketThreads * 64;  // keys per wave
  const int wb = int(ps + w * q < pe ? ps + w * q : pe);
  const int we = int(ps + (w + 1) * q < pe ? ps + (w + 1) * q : pe);
  __syncthreads();

  uint64_t key[kBucketBatch];
  if (P > 1) {
    // the other parts' keys: [gs, ps) (counted as before this part too) and
    // [pe, ge), each range cut into wave slices
#pragma unroll 1
    for (int r = 0; r < 2; ++r) {
      const int a = r == 0 ? gs : pe, e = r == 0 ? ps : int(ge);
      const int64_t qo = (int64_t(e - a) + kBucketThreads - 1) / kBucketThreads * 64;
      const int ob = int(a + w * qo < e ? a + w * qo : e);
      const int oe = int(a + (w + 1) * qo < e ? a + (w + 1) * qo : e);
      for (int e0 = ob; e0 < oe; e0 += 64 * kBucketBatch) {
#pragma unroll
        for (int j = 0; j < kBucketBatch; ++j) {
          const int i = e0 + 64 * j + lane;
          if (e0 + 64 * j < oe) key[j] = keys_in[i < oe ? i : ob];
        }
#pragma unroll
        for (int j = 0; j < kBucketBatch; ++j)
          if (e0 + 64 * j < oe) {
            const unsigned dg = key_digit(key[j], 0, mask);
            const bool valid = e0 + 64 * j + lane < oe;
            count_digit_runs(s_out, dg, valid);
            if (r == 0) count_digit_runs(s_before, dg, valid);
          }
      }
    }
  }

  int *cnt = s_cnt + w * R;
  const bool resident = we - wb <= 64 * kBucketBatch;  // wave-uniform
  for (int e0 = wb; e0 < we; e0 += 64 * kBucketBatch) {
    // sub-batches past the slice end are skipped (wave-uniform tests)
#pragma unroll
    for (int j = 0; j < kBucketBatch; ++j) {
      const int e = e0 + 64 * j + lane;
      if (e0 + 64 * j < we) key[j] = keys_in[e < we ? e : wb];
    }
#pragma unroll
    for (int j = 0; j < kBucketBatch; ++j)
      if (e0 + 64 * j < we)
        count_digit_runs(cnt, key_digit(key[j], 0, mask), e0 + 64 * j + lane < we);
  }
  __syncthreads();

  // digit starts within the group (digits kPer * tid + i), the cells'
  // ranges (part 0), per-wave bases of this part
  constexpr int kPer = kMaxRadix / kBucketThreads;  // digits per thread (1 or 2)
  int tot[kPer], tsum = 0;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int d = kPer * tid + i;
    tot[i] = 0;
    if (d < R) {
#pragma unroll
      for (int ww = 0; ww < kBucketWaves; ++ww) tot[i] += s_cnt[ww * R + d];
      tot[i] += s_out[d];
    }
    tsum += tot[i];
  }
  int gtotal;
  int ex = gs + block_exclusive_scan<kBucketWaves>(tsum, s_scan, &gtotal);
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int d = kPer * tid + i;
    if (d < R) {
      const int64_t cell = int64_t(bkt) * R + d;
      if (part == 0 && cell < n_cells) {
        cstart[cell] = tot[i] ? ex : 0;
        cend[cell] = tot[i] ? ex + tot[i] : 0;
      }
      int run = ex + s_before[d];
#pragma unroll
      for (int ww = 0; ww < kBucketWaves; ++ww) {
        const int c = s_cnt[ww * R + d];
        s_cnt[ww * R + d] = run;
        run += c;
      }
    }
    ex += tot[i];
  }
  __syncthreads();

  for (int e0 = wb; e0 < we; e0 += 64 * kBucketBatch) {
    if (!resident) {
#pragma unroll
      for (int j = 0; j < kBucketBatch; ++j) {
        const int e = e0 + 64 * j + lane;
        if (e0 + 64 * j < we) key[j] = keys_in[e < we ? e : wb];
      }
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the batch is in registers
    }
#pragma unroll
    for (int j = 0; j < kBucketBatch; ++j) {
      if (e0 + 64 * j >= we) break;
      const bool valid = e0 + 64 * j + lane < we;
      const unsigned dg = key_digit(key[j], 0, mask);
      int below, same;
      digit_rank(dg, valid, below, same);
      if (valid) {
        const int pos = cnt[dg] + below;
        keys_out[pos] = key[j];
        if (below == 0) cnt[dg] = pos + same;
      }
    }
  }
}

// Sliced form of the second half of the sort (same result as
// bucket_sort_kernel).  Each group of equal high digit, in point order after
// the global pass, is cut into slices of kSliceKeys consecutive keys, so that
// a large group (the cells near the cameras: up to ~65 K keys at 2 x 720 x
// 720) is spread over several blocks instead of being walked by one:
//   bucket_count_kernel   one block per slice: the slice's low-digit counts;
//   bucket_scan_kernel    one block per group: each slice's first sorted
//                         position per digit (in place of its counts) and
//                         the group's dense cell ranges;
//   bucket_place_kernel   one block per slice: each key to its position
//                         (the ranking of bucket_sort_kernel within a slice).
// Slices are numbered group by group; a block finds its slice from the group
// sizes (exclusive scans over the <= 1024 groups), so no kernel waits on
// another block.
constexpr int kSliceKeys = 8192;
// Groups of 2^kSlicedBits cells take the sliced form.  Smaller groups (at
// most ~35 K keys measured) take bucket_sort_kernel, whose one launch is
// faster there (MI355X: 21.6 against 41 us at 1 x 360 x 360, 51 against 74
// at 4 x 360 x 360; sorting one-slice groups in their place block and
// counting only the others still lost: 30.5 and 63 us); at 2^10 cells per
// group the sliced form takes 103 against 148 us (2 x 720 x 720).
constexpr int kSlicedBits = 10;
constexpr int kSliceWaves = 8;  // 8 waves x 2^10 per-wave digit counts: 32 KB of LDS

template <int kW>
struct SliceShape {
  static constexpr int kT = 64 * kW;
  static constexpr int kBatch = kSliceKeys / kT;  // 64-key sub-batches per wave
  static_assert(kBatch * kT == kSliceKeys && kBatch <= 16, "slice shape");
};

__host__ __device__ inline int slices_of(int keys) {
  return (keys + kSliceKeys - 1) / kSliceKeys;
}

// This block's slice: group g, slice id (== blockIdx.x; slices are numbered
// group by group), sorted positions [first, end).  False (for the whole
// block) past the last slice.  (Dealing the slices to the XCDs in 8
// contiguous ranges, so that a group's interleaved writes share one L2, was
// measured slower on MI355X.)
struct SliceLoc {
  int g, id, first, end;
};

template <int kW>
__device__ bool find_slice(const int32_t *__restrict__ totals, int n_groups, SliceLoc *loc) {
  constexpr int kT = 64 * kW;
  constexpr int kG = (kMaxRadix + kT - 1) / kT;  // groups per thread
  __shared__ int s_scan[kW];
  __shared__ int s_loc[4];
  const int tid = threadIdx.x;
  int gn[kG], tk = 0, ts = 0;
#pragma unroll
  for (int i = 0; i < kG; ++i) {
    const int g = tid * kG + i;
    gn[i] = g < n_groups ? totals[g] : 0;
    tk += gn[i];
    ts += slices_of(gn[i]);
  }
  if (tid == 0) s_loc[0] = -1;  // ordered before the writes below by the scans' barriers
  int unused, n_slices;
  int kb = block_exclusive_scan<kW>(tk, s_scan, &unused);
  int sb = block_exclusive_scan<kW>(ts, s_scan, &n_slices);
  const int b = int(blockIdx.x);
  if (b >= n_slices) return false;  // block-uniform
#pragma unroll
  for (int i = 0; i < kG; ++i) {
    const int ns = slices_of(gn[i]);
    if (b >= sb && b < sb + ns) {
      const int first = kb + (b - sb) * kSliceKeys;
      s_loc[0] = tid * kG + i;
      s_loc[1] = b;
      s_loc[2] = first;
      s_loc[3] = gn[i] - (b - sb) * kSliceKeys < kSliceKeys ? kb + gn[i] : first + kSliceKeys;
    }
    sb += ns;
    kb += gn[i];
  }
  __syncthreads();
  loc->g = s_loc[0];
  loc->id = s_loc[1];
  loc->first = s_loc[2];
  loc->end = s_loc[3];
  return true;
}

// The keys of this wave's part of the slice (kBatch sub-batches of 64; past
// the slice end they read its first key).
template <int kW>
__device__ __forceinline__ void load_slice_keys(const uint64_t *__restrict__ keys_in,
                                                const SliceLoc &L, int w, int lane,
                                                uint64_t (&key)[SliceShape<kW>::kBatch]) {
  constexpr int kB = SliceShape<kW>::kBatch;
  const int wb = L.first + w * 64 * kB;
#pragma unroll
  for (int j = 0; j < kB; ++j) {
    const int e = wb + 64 * j + lane;
    key[j] = keys_in[e < L.end ? e : L.first];
  }
}

template <int kW>
__global__ __launch_bounds__(64 * kW) void bucket_count_kernel(
    const uint64_t *__restrict__ keys_in, const int32_t *__restrict__ totals, int n_groups,
    int lbits, int32_t *__restrict__ slice_cnt) {
  constexpr int kT = SliceShape<kW>::kT, kB = SliceShape<kW>::kBatch;
  extern __shared__ int s_cnt[];  // [R]
  SliceLoc L;
  if (!find_slice<kW>(totals, n_groups, &L)) return;
  const int tid = threadIdx.x, lane = lane_id(), w = tid >> 6;
  const int R = 1 << lbits;
  const unsigned mask = unsigned(R - 1);
  uint64_t key[kB];
  load_slice_keys<kW>(keys_in, L, w, lane, key);
  for (int d = tid; d < R; d += kT) s_cnt[d] = 0;
  __syncthreads();
  const int wb = L.first + w * 64 * kB;
#pragma unroll
  for (int j = 0; j < kB; ++j)
    if (wb + 64 * j < L.end)  // wave-uniform
      count_digit_runs(s_cnt, key_digit(key[j], 0, mask), wb + 64 * j + lane < L.end);
  __syncthreads();
  int32_t *out = slice_cnt + int64_t(L.id) * R;
  for (int d = tid; d < R; d += kT) out[d] = s_cnt[d];
}

__global__ __launch_bounds__(kThreads) void bucket_scan_kernel(
    const int32_t *__restrict__ totals, int n_groups, int64_t n_cells, int lbits,
    int32_t *__restrict__ slice_cnt, int32_t *__restrict__ cstart, int32_t *__restrict__ cend) {
  __shared__ int s_scan[kWaves];
  const int g = int(blockIdx.x);
  if (g >= n_groups) return;
  const int tid = threadIdx.x;
  const int R = 1 << lbits;
  // group start and first slice: sums over the groups before g
  int pk = 0, ps = 0;
  for (int d = tid; d < g; d += kThreads) {
    const int t = totals[d];
    pk += t;
    ps += slices_of(t);
  }
  int gs, sb;
  block_exclusive_scan(pk, s_scan, &gs);
  block_exclusive_scan(ps, s_scan, &sb);
  const int ns = slices_of(totals[g]);
  int32_t *sc = slice_cnt + int64_t(sb) * R;
  // thread t owns digits 4t .. 4t+3 (R is a multiple of 4, >= 32): the
  // group's totals per digit, then the digit starts
  constexpr int kU = 8;  // slices whose counts are loaded together
  const int d0 = 4 * tid;
  const bool mine = d0 < R;
  u32x4 tot = {0u, 0u, 0u, 0u};
  if (mine) {
    for (int k0 = 0; k0 < ns; k0 += kU) {
      u32x4 v[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u)
        v[u] = k0 + u < ns ? *reinterpret_cast<const u32x4 *>(sc + int64_t(k0 + u) * R + d0)
                           : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int u = 0; u < kU; ++u) tot += v[u];
    }
  }
  int unused;
  int ex = gs + block_exclusive_scan(int(tot.x + tot.y + tot.z + tot.w), s_scan, &unused);
  if (!mine) return;
  // first sorted position of each of the four digits in slice 0
  u32x4 run;
  run.x = uint32_t(ex);
  run.y = run.x + tot.x;
  run.z = run.y + tot.y;
  run.w = run.z + tot.z;
  const int64_t cell0 = int64_t(g) * R + d0;
  const uint32_t t4[4] = {tot.x, tot.y, tot.z, tot.w};
  const uint32_t r4[4] = {run.x, run.y, run.z, run.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (cell0 + i < n_cells) {
      cstart[cell0 + i] = t4[i] ? int(r4[i]) : 0;
      cend[cell0 + i] = t4[i] ? int(r4[i] + t4[i]) : 0;
    }
  }
  for (int k0 = 0; k0 < ns; k0 += kU) {
    u32x4 v[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u)
      v[u] = k0 + u < ns ? *reinterpret_cast<const u32x4 *>(sc + int64_t(k0 + u) * R + d0)
                         : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      if (k0 + u < ns) *reinterpret_cast<u32x4 *>(sc + int64_t(k0 + u) * R + d0) = run;
      run += v[u];
    }
  }
}

template <int kW>
__global__ __launch_bounds__(64 * kW) void bucket_place_kernel(
    const uint64_t *__restrict__ keys_in, const int32_t *__restrict__ totals, int n_groups,
    int lbits, const int32_t *__restrict__ slice_cnt, uint64_t *__restrict__ keys_out) {
  constexpr int kT = SliceShape<kW>::kT, kB = SliceShape<kW>::kBatch;
  extern __shared__ int s_cnt[];  // [kW][R]
  SliceLoc L;
  if (!find_slice<kW>(totals, n_groups, &L)) return;
  const int tid = threadIdx.x, lane = lane_id(), w = tid >> 6;
  const int R = 1 << lbits;
  const unsigned mask = unsigned(R - 1);
  uint64_t key[kB];
  load_slice_keys<kW>(keys_in, L, w, lane, key);
  for (int d = tid; d < kW * R; d += kT) s_cnt[d] = 0;
  __syncthreads();
  int *cnt = s_cnt + w * R;
  const int wb = L.first + w * 64 * kB;
#pragma unroll
  for (int j = 0; j < kB; ++j)
    if (wb + 64 * j < L.end)
      count_digit_runs(cnt, key_digit(key[j], 0, mask), wb + 64 * j + lane < L.end);
  __syncthreads();
  // per-wave bases: the slice's first position of the digit + earlier waves
  const int32_t *base = slice_cnt + int64_t(L.id) * R;
  for (int d = tid; d < R; d += kT) {
    int run = base[d];
#pragma unroll
    for (int ww = 0; ww < kW; ++ww) {
      const int c = s_cnt[ww * R + d];
      s_cnt[ww * R + d] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kB; ++j) {
    if (wb + 64 * j >= L.end) break;
    const bool valid = wb + 64 * j + lane < L.end;
    const unsigned dg = key_digit(key[j], 0, mask);
    int below, same;
    digit_rank(dg, valid, below, same);
    if (valid) {
      const int pos = cnt[dg] + below;
      keys_out[pos] = key[j];
      if (below == 0) cnt[dg] = pos + same;
    }
  }
}

// bev_pool_legacy.py:56-61 boundary flags on the sorted ranks: writes the
// dense [start, end) of every occupied cell.  Thread t handles sorted
// positions 4t .. 4t+3 (two 16-byte loads when kVec: keys 16-byte aligned).
template <bool kVec>
__global__ __launch_bounds__(kThreads) void cell_ranges_kernel(
    const uint64_t *__restrict__ keys, const int32_t *__restrict__ meta,
    int32_t *__restrict__ cstart, int32_t *__restrict__ cend) {
  const int64_t n = meta[BEVPOOL_META_N_KEPT];
  const int64_t i0 = (int64_t(blockIdx.x) * kThreads + threadIdx.x) * 4;
  if (i0 >= n) return;
  const uint32_t *kw = reinterpret_cast<const uint32_t *>(keys);  // rank = odd words
  int r[6];  // ranks of positions i0-1 .. i0+4 (-1 outside [0, n))
  r[0] = i0 > 0 ? int(kw[2 * (i0 - 1) + 1]) : -1;
  if (kVec && i0 + 3 < n) {
    const u32x4 a = *reinterpret_cast<const u32x4 *>(kw + 2 * i0);
    const u32x4 b = *reinterpret_cast<const u32x4 *>(kw + 2 * i0 + 4);
    r[1] = int(a.y);
    r[2] = int(a.w);
    r[3] = int(b.y);
    r[4] = int(b.w);
  } else {
#pragma unroll
    for (int u = 0; u < 4; ++u) r[1 + u] = i0 + u < n ? int(kw[2 * (i0 + u) + 1]) : -1;
  }
  r[5] = i0 + 4 < n ? int(kw[2 * (i0 + 4) + 1]) : -1;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int64_t i = i0 + u;
    if (i < n) {
      if (r[u] != r[u + 1]) cstart[r[u + 1]] = int(i);
      if (r[u + 2] != r[u + 1]) cend[r[u + 1]] = int(i + 1);
    }
  }
}

// Interval starts (r[i] != r[i-1]) per block of 256 sorted keys: wave ballot
// + popcount, summed over the block's waves.
__global__ __launch_bounds__(kThreads) void count_starts_kernel(
    const uint64_t *__restrict__ keys, const int32_t *__restrict__ meta,
    int32_t *__restrict__ bcount) {
  __shared__ int s_w[kWaves];
  const int64_t n = meta[BEVPOOL_META_N_KEPT];
  const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  bool is_start = false;
  if (i < n) is_start = (i == 0) || key_rank(keys[i - 1]) != key_rank(keys[i]);
  const uint64_t b = __ballot(is_start);
  if (lane_id() == 0) s_w[threadIdx.x >> 6] = __popcll(b);
  __syncthreads();
  if (threadIdx.x == 0) {
    int s = 0;
    for (int j = 0; j < kWaves; ++j) s += s_w[j];
    bcount[blockIdx.x] = s;
  }
}

// Single-block exclusive scan of counts[0..n) in place; *total_out = sum.
__global__ __launch_bounds__(kThreads) void scan_counts_kernel(int32_t *__restrict__ counts,
                                                               int64_t n,
                                                               int32_t *__restrict__ total_out) {
  __shared__ int scratch[kWaves];
  int carry = 0;
  for (int64_t t0 = 0; t0 < n; t0 += kThreads * 4) {
    int v[4], s = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t j = t0 + threadIdx.x * 4 + i;
      v[i] = j < n ? counts[j] : 0;
      s += v[i];
    }
    int tot;
    int ex = block_exclusive_scan(s, scratch, &tot) + carry;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t j = t0 + threadIdx.x * 4 + i;
      if (j < n) counts[j] = ex;
      ex += v[i];
    }
    carry += tot;
  }
  if (threadIdx.x == 0) *total_out = carry;
}

// Compacted interval j (the j-th start in sorted order): starts[j], lengths[j]
// (= end - start, the legacy "difference of starts"), cells[j] = rank.
__global__ __launch_bounds__(kThreads) void interval_write_kernel(
    const uint64_t *__restrict__ keys, const int32_t *__restrict__ meta,
    const int32_t *__restrict__ cend, const int32_t *__restrict__ boff,
    int32_t *__restrict__ starts, int32_t *__restrict__ lengths, int32_t *__restrict__ cells) {
  __shared__ int s_w[kWaves];
  const int64_t n = meta[BEVPOOL_META_N_KEPT];
  const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  const int w = threadIdx.x >> 6;
  bool is_start = false;
  int r = 0;
  if (i < n) {
    r = key_rank(keys[i]);
    is_start = (i == 0) || key_rank(keys[i - 1]) != r;
  }
  const uint64_t b = __ballot(is_start);
  if (lane_id() == 0) s_w[w] = __popcll(b);
  __syncthreads();
  if (is_start) {
    int off = boff[blockIdx.x] + __popcll(b & lanes_below());
    for (int j = 0; j < w; ++j) off += s_w[j];
    starts[off] = int(i);
    lengths[off] = cend[r] - int(i);
    cells[off] = r;
  }
}

// ---------------------------------------------------------------------------
// forward kernels
// ---------------------------------------------------------------------------

// First sorted position >= i that starts a cell (n if none).
__device__ __forceinline__ int64_t snap_to_cell(int64_t i, int64_t n,
                                                const uint64_t *__restrict__ keys,
                                                const int32_t *__restrict__ cend) {
  if (i <= 0) return 0;
  if (i >= n) return n;
  const int r = key_rank(keys[i]);
  if (key_rank(keys[i - 1]) != r) return i;
  return cend[r];
}

// Rows of fewer than 16 bytes.  Block b owns the sorted positions
// [snap(b*P), snap((b+1)*P)): whole cells only, so every cell's sum is one
// sequential chain.  Rows (feats[point]) of R sorted points at a time are
// gathered into LDS by all threads; thread c then adds column c of the R rows
// in order into its fp32 accumulator and stores it to acc[cell*C + c] when
// the cell ends.
template <typename T>
__global__ __launch_bounds__(kThreads) void accum_rows_kernel(
    const typename T::raw *__restrict__ x, int64_t ld, int C, int R,
    const uint64_t *__restrict__ keys, const int32_t *__restrict__ meta,
    const int32_t *__restrict__ cend, float *__restrict__ acc, int64_t P) {
  extern __shared__ float smem[];
  float *buf = smem;                                // R * C floats
  int *rk = reinterpret_cast<int *>(smem + R * C);  // R + 1 ints
  const int tid = threadIdx.x;
  const int64_t n = meta[BEVPOOL_META_N_KEPT];
  const int64_t r0 = int64_t(blockIdx.x) * P;
  if (r0 >= n) return;
  const int64_t s = snap_to_cell(r0, n, keys, cend);
  const int64_t e = snap_to_cell(r0 + P < n ? r0 + P : n, n, keys, cend);
  if (s >= e) return;
  float a = 0.0f;
  for (int64_t base = s; base < e; base += R) {
    const int rows = int(e - base < R ? e - base : R);
    __syncthreads();
    for (int j = tid; j <= rows; j += kThreads)
      rk[j] = (base + j < e) ? key_rank(keys[base + j]) : -1;
    for (int slot = tid; slot < rows * C; slot += kThreads) {
      const int j = slot / C, c = slot - j * C;
      const int64_t idx = key_index(keys[base + j]);
      buf[slot] = T::load(x + idx * ld + c);
    }
    __syncthreads();
    if (tid < C) {
      for (int j = 0; j < rows; ++j) {
        a += buf[j * C + tid];
        const int r = rk[j];
        if (rk[j + 1] != r) {
          acc[int64_t(r) * C + tid] = a;
          a = 0.0f;
        }
      }
    }
  }
}

// ---- software-pipelined forward accumulation (16-byte rows) ---------------
//
// Same ownership as accum_rows_kernel (block b owns the sorted positions
// [snap(b*P), snap((b+1)*P)), whole cells only), restructured so memory
// latency is hidden inside the block.  Roles:
//   * loader waves (1..4, 256 threads) gather the rows of each stage of
//     kStageRows sorted points with 16-byte loads (loader slot i of thread t
//     covers row (t + 256 i) / rowq, 16-byte column (t + 256 i) % rowq) into
//     a ring of kDepth register stages, and move the oldest arrived stage to
//     LDS once per step;
//   * wave 0 sums the stage in LDS, one channel per lane (channels l + 64 j),
//     each lane adding its column in row order into one fp32 accumulator; a
//     cell's sum is stored to acc when the next cell starts (start flags from
//     a ballot over the stage's ranks) or the range ends, so a cell spanning
//     stages keeps one sequential chain.
// Step k: wave 0 sums stage k from LDS buffer k&1 while the loaders issue the
// rows of stage k+kDepth and the point indices of stage k+2*kDepth, then store
// stage k+1 (issued kDepth-1 steps earlier) into buffer (k+1)&1; one barrier.
// The loaders issue loads only and always fetch a stage's indices kDepth steps
// before its rows, so every wait they need (indices of stage k+kDepth, rows of
// stage k+1) leaves all younger row loads in flight (vmcnt retires in issue
// order).  The summing wave issues no loads, so its stores never hold up a
// wait.  Loads of stages past the range end are pointed at the range's first
// row (a single line) so the code stays straight-line.
#ifndef BEVPOOL_STAGE_ROWS
#define BEVPOOL_STAGE_ROWS 32
#endif
#ifndef BEVPOOL_DEPTH
#define BEVPOOL_DEPTH 2
#endif
constexpr int kStageRows = BEVPOOL_STAGE_ROWS;  // sorted points per stage
constexpr int kDepth = BEVPOOL_DEPTH;           // row stages in flight per loader thread
#ifndef BEVPOOL_SUMMERS
#define BEVPOOL_SUMMERS 1
#endif
#ifndef BEVPOOL_LOADER_WAVES
#define BEVPOOL_LOADER_WAVES 2
#endif
constexpr int kSummers = BEVPOOL_SUMMERS;       // summing waves (waves 0..kSummers-1)
constexpr int kLoaders = 64 * BEVPOOL_LOADER_WAVES;  // loader threads (the other waves)
constexpr int kPipeThreads = 64 * kSummers + kLoaders;
// Only 32-row stages are built and tested.  A 64-row variant built with
// -DBEVPOOL_STAGE_ROWS=64 failed one camera-index parity case on MI355X and
// passed it on the next run, without a cause found; 16-row stages were only
// ever timed.  Other values are therefore refused at compile time.
static_assert(kStageRows == 32, "only 32-row accumulation stages are supported");

// native 16-byte vector (register-promotable, unlike the HIP uint4 wrapper)

// How the accumulations load their rows:
//   kRowsPlain   feature rows, ordinary loads;
//   kRowsStream  feature rows, non-temporal loads: the rows are read once,
//                and keeping them out of the caches keeps the index (ranks,
//                keys) and the cell rows there for the transposes and the
//                backward gather.  Measured on MI355X at 1 x 360 x 360
//                (638 MB of feature rows): forward -3.5 us, backward -5 us per
//                step.  With 2.6-5.1 GB of rows (4 x 360 x 360, 2 x 720 x 720)
//                the accumulation itself got 4-6% slower and nothing else
//                faster, so inputs of more than kStreamRowBytes of rows keep
//                ordinary loads.  accum_group_kernel takes the same rule:
//                level for rows of whole lines (128 fp32 channels, 1.6 M points:
//                accumulation 176 us, 173 with ordinary loads, the step 385 and
//                391), slower for rows that share lines with their neighbours
//                (90 fp16 channels, 1.06 M points: 80 and 65, the step 179 and
//                172; 50 bf16 channels, 4.8 M: 254 and 177, 504 and 434).
//   kRowsDepth   depth-weighted context rows (DepthRows), ordinary loads:
//                a context row is read for every depth bin
//                (accum_group_kernel only).
//   kRowsRun     consecutive rows: position p of a cell is row p
//                (legacy_sum_kernel only).
constexpr int kRowsPlain = 0, kRowsDepth = 1, kRowsStream = 2, kRowsRun = 3;
constexpr int64_t kStreamRowBytes = int64_t(1) << 30;

struct PipeRange {
  int64_t s, e;  // sorted positions [s, e)
  int rowq;      // 16-byte pieces per row
  __device__ __forceinline__ int rows(int k) const {
    const int64_t b = s + int64_t(k) * kStageRows;
    return b >= e ? 0 : int(e - b < kStageRows ? e - b : kStageRows);
  }
};

// Register ring of one loader thread.
template <int kSlots>
struct LoaderRing {
  u32x4 d[kDepth][kSlots];       // gathered 16-byte pieces of a stage
  uint32_t idx[kDepth][kSlots];  // point indices of a later stage
  int rk[kDepth];                // rank of row (lt % kStageRows) of a stage
  int srow[kSlots];              // row of slot i within a stage (unclamped)
  int sq[kSlots];                // 16-byte column of slot i
};

// Point indices of stage k into ring slot j.  Slots past the stage's rows
// repeat its last row; a stage past the range end reads the range's first row.
template <int kSlots, int j>
__device__ __forceinline__ void ring_index(LoaderRing<kSlots> &R,
                                           const uint32_t *__restrict__ kw, const PipeRange &pr,
                                           int k) {
  const int rows = pr.rows(k);
  const int64_t base = pr.s + int64_t(k) * kStageRows;
#pragma unroll
  for (int i = 0; i < kSlots; ++i) {
    const int r = R.srow[i] < rows - 1 ? R.srow[i] : rows - 1;
    R.idx[j][i] = kw[2 * (rows > 0 ? base + r : pr.s)];  // low word: point index
  }
}

// Rows of stage k into ring slot j (its indices are in R.idx[j]), plus the rank
// of row lt % kStageRows.
template <int kSlots, int j, int kRows>
__device__ __forceinline__ void ring_rows(LoaderRing<kSlots> &R, int lt,
                                          const uint32_t *__restrict__ kw,
                                          const char *__restrict__ xb, int64_t ld_bytes,
                                          const PipeRange &pr, int k) {
  const bool live = pr.rows(k) > 0;
#pragma unroll
  for (int i = 0; i < kSlots; ++i) {
    const int q = live ? R.sq[i] : 0;
    const u32x4 *src =
        reinterpret_cast<const u32x4 *>(xb + int64_t(R.idx[j][i]) * ld_bytes + q * 16);
    if constexpr (kRows == kRowsStream)
      R.d[j][i] = __builtin_nontemporal_load(src);
    else
      R.d[j][i] = *src;
  }
  const int64_t b = pr.s + int64_t(k) * kStageRows;
  int64_t p = b + (lt & (kStageRows - 1));
  p = b >= pr.e ? pr.s : (p < pr.e ? p : pr.e - 1);
  R.rk[j] = kw[2 * p + 1];  // high word: rank
}

// Ring slot j (stage k) into an LDS buffer.
template <int kSlots, int j>
__device__ __forceinline__ void ring_store(const LoaderRing<kSlots> &R, int lt,
                                           const PipeRange &pr, int k, u32x4 *__restrict__ lbuf,
                                           int *__restrict__ lrk) {
  const int n = pr.rows(k) * pr.rowq;
#pragma unroll
  for (int i = 0; i < kSlots; ++i) {
    const int slot = lt + kLoaders * i;
    if (slot < n) lbuf[slot] = R.d[j][i];
  }
  if (lt < kStageRows) lrk[lt] = R.rk[j];
}

// One loader step k with ring slot r = k % kDepth (a template constant).
template <int kSlots, int r, int kRows>
__device__ __forceinline__ void loader_step(LoaderRing<kSlots> &R, int lt,
                                            const uint32_t *__restrict__ kw,
                                            const char *__restrict__ xb, int64_t ld_bytes,
                                            const PipeRange &pr, int k, int nst,
                                            u32x4 *__restrict__ buf0, u32x4 *__restrict__ buf1,
                                            int *__restrict__ rk0s, int *__restrict__ rk1s) {
  ring_rows<kSlots, r, kRows>(R, lt, kw, xb, ld_bytes, pr, k + kDepth);
  ring_index<kSlots, r>(R, kw, pr, k + 2 * kDepth);
  if (k + 1 < nst) {
    if ((k + 1) & 1)
      ring_store<kSlots, (r + 1) % kDepth>(R, lt, pr, k + 1, buf1, rk1s);
    else
      ring_store<kSlots, (r + 1) % kDepth>(R, lt, pr, k + 1, buf0, rk0s);
  }
  __syncthreads();
}

// Sequential per-channel sums of one stage by one summing wave: lane l owns
// channels c0 + l + 64 i (i < kCPL, c0 the wave's first channel).  Rows are
// read from LDS 16 at a time before they are added (one LDS latency per 16
// dependent adds).  A 16-row chunk without a cell start is 16 straight adds;
// a chunk with exactly one start at row b jumps (16-way switch) to
// straight-line code for that b: add rows [0, b), store the finished cell,
// restart from +0.0, add rows [b, 16); other chunks go row by row.
// A finished cell row is stored in the output's element type: fp32 for fp32
// input; for 16-bit input the fp32 sum rounded once (T::to_raw), the value
// the output gets, so the transpose that follows moves half the bytes.
// With 16-bit input a lane owns channel pairs instead (pair l + 64 i =
// channels 2(l + 64 i), +1): one 4-byte LDS read per row and one packed
// 4-byte store per finished cell; kCPL then counts pairs per lane.
template <typename T, int kCPL>
struct RowSum {
  using TO = typename std::conditional<sizeof(typename T::raw) == 2, typename T::raw, float>::type;
  static constexpr bool kPair = sizeof(typename T::raw) == 2;
  static constexpr int kA = kPair ? 2 * kCPL : kCPL;  // fp32 accumulators per lane
  float a[kA];
  int cur = -1;    // rank of the current cell
  int carry = -1;  // rank of the previous stage's last row

  __device__ __forceinline__ void flush(int nch, TO *__restrict__ out, int64_t row_elems) {
    if (cur >= 0) {
      TO *o = out + int64_t(cur) * row_elems;
      const int lane = lane_id();
      if constexpr (kPair) {
        uint32_t *o32 = reinterpret_cast<uint32_t *>(o);  // row and channel offsets even
#pragma unroll
        for (int i = 0; i < kCPL; ++i)
          if (2 * (lane + 64 * i) < nch)
            o32[lane + 64 * i] =
                uint32_t(T::to_raw(a[2 * i])) | (uint32_t(T::to_raw(a[2 * i + 1])) << 16);
      } else {
#pragma unroll
        for (int i = 0; i < kCPL; ++i)
          if (lane + 64 * i < nch) o[lane + 64 * i] = a[i];
      }
    }
  }

  template <int kB, int kStart>
  __device__ __forceinline__ void split_chunk(const float (&v)[kB][kA], int rkl, int j0, int nch,
                                              TO *__restrict__ out, int64_t row_elems) {
#pragma unroll
    for (int u = 0; u < kStart; ++u)
#pragma unroll
      for (int i = 0; i < kA; ++i) a[i] += v[u][i];
    flush(nch, out, row_elems);
#pragma unroll
    for (int i = 0; i < kA; ++i) a[i] = 0.0f;
    cur = __builtin_amdgcn_readlane(rkl, j0 + kStart);
#pragma unroll
    for (int u = kStart; u < kB; ++u)
#pragma unroll
      for (int i = 0; i < kA; ++i) a[i] += v[u][i];
  }

  // lb: the stage's rows in LDS (row stride cb elements), col: this lane's
  // columns; nch: channels of this wave (stores of lanes past nch are skipped).
  __device__ __forceinline__ void add_stage(const typename T::raw *__restrict__ lb,
                                            const int *__restrict__ lrk, int rows, int cb,
                                            const int (&col)[kCPL], int nch,
                                            TO *__restrict__ out, int64_t row_elems) {
    const int lane = lane_id();
    const int rkl = lane < rows ? lrk[lane] : -1;
    int prev = __shfl_up(rkl, 1, 64);
    if (lane == 0) prev = carry;
    const uint64_t starts = __ballot(lane < rows && rkl != prev);
    if (rows > 0) carry = __builtin_amdgcn_readlane(rkl, rows - 1);
    constexpr int kB = kStageRows < 16 ? kStageRows : 16;
    for (int j0 = 0; j0 < rows; j0 += kB) {
      float v[kB][kA];
      if constexpr (kPair) {  // col[i]: pair index; cb even
        const uint32_t *lb32 = reinterpret_cast<const uint32_t *>(lb);
#pragma unroll
        for (int u = 0; u < kB; ++u)
#pragma unroll
          for (int i = 0; i < kCPL; ++i) {
            const uint32_t w = lb32[(j0 + u) * (cb >> 1) + col[i]];
            v[u][2 * i] = T::from_raw(w & 0xffffu);
            v[u][2 * i + 1] = T::from_raw(w >> 16);
          }
      } else {
#pragma unroll
        for (int u = 0; u < kB; ++u)
#pragma unroll
          for (int i = 0; i < kCPL; ++i) v[u][i] = T::load(lb + (j0 + u) * cb + col[i]);
      }
      const uint32_t chunk = uint32_t(starts >> j0) & uint32_t((uint64_t(1) << kB) - 1);
      const bool full = j0 + kB <= rows;
      if (full && chunk == 0) {
#pragma unroll
        for (int u = 0; u < kB; ++u)
#pragma unroll
          for (int i = 0; i < kA; ++i) a[i] += v[u][i];
      } else if (full && (chunk & (chunk - 1)) == 0) {
        switch (__builtin_ctz(chunk)) {
#define BEVPOOL_SPLIT(B)                                                                       \
  case B:                                                                                     \
    if constexpr ((B) < kB) split_chunk<kB, ((B) < kB ? (B) : 0)>(v, rkl, j0, nch, out, row_elems); \
    break;
          BEVPOOL_SPLIT(0) BEVPOOL_SPLIT(1) BEVPOOL_SPLIT(2) BEVPOOL_SPLIT(3)
          BEVPOOL_SPLIT(4) BEVPOOL_SPLIT(5) BEVPOOL_SPLIT(6) BEVPOOL_SPLIT(7)
          BEVPOOL_SPLIT(8) BEVPOOL_SPLIT(9) BEVPOOL_SPLIT(10) BEVPOOL_SPLIT(11)
          BEVPOOL_SPLIT(12) BEVPOOL_SPLIT(13) BEVPOOL_SPLIT(14) BEVPOOL_SPLIT(15)
#undef BEVPOOL_SPLIT
          default:
            break;
        }
      } else {
#pragma unroll
        for (int u = 0; u < kB; ++u) {
          const int j = j0 + u;
          if (j < rows) {
            if ((chunk >> u) & 1) {
              flush(nch, out, row_elems);
#pragma unroll
              for (int i = 0; i < kA; ++i) a[i] = 0.0f;
              cur = __builtin_amdgcn_readlane(rkl, j);
            }
#pragma unroll
            for (int i = 0; i < kA; ++i) a[i] += v[u][i];
          }
        }
      }
    }
  }
};

template <typename T, int kSlots, int kCPL, int kRows>
__global__ __launch_bounds__(kPipeThreads) void accum_pipe_kernel(
    const char *__restrict__ xb, int64_t ld_bytes, int C, const uint64_t *__restrict__ keys,
    const int32_t *__restrict__ meta, const int32_t *__restrict__ cend, float *__restrict__ acc,
    int64_t P) {
  using raw = typename T::raw;
  extern __shared__ u32x4 smem4[];
  PipeRange pr;
  pr.rowq = C * int(sizeof(raw)) / 16;
  u32x4 *buf0 = smem4;
  u32x4 *buf1 = smem4 + kStageRows * pr.rowq;
  int *rk0s = reinterpret_cast<int *>(smem4 + 2 * kStageRows * pr.rowq);
  int *rk1s = rk0s + kStageRows;
  const uint32_t *kw = reinterpret_cast<const uint32_t *>(keys);

  const int64_t n = meta[BEVPOOL_META_N_KEPT];
  const int64_t r0 = int64_t(blockIdx.x) * P;
  if (r0 >= n) return;
  pr.s = snap_to_cell(r0, n, keys, cend);
  pr.e = snap_to_cell(r0 + P < n ? r0 + P : n, n, keys, cend);
  if (pr.s >= pr.e) return;
  const int nst = int((pr.e - pr.s + kStageRows - 1) / kStageRows);
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const bool summer = wave < kSummers;
  const int lt = int(threadIdx.x) - 64 * kSummers;  // loader thread index (loader waves only)

  if (summer) {
    // summing wave `wave` owns channels [wch, wch + nch)
    // (an even count with 16-bit input, whose lanes take channel pairs)
    constexpr bool kPair = RowSum<T, kCPL>::kPair;
    int cps = (C + kSummers - 1) / kSummers;
    if (kPair) cps += cps & 1;
    const int wch = wave * cps;
    const int nch = C - wch < cps ? (C - wch > 0 ? C - wch : 0) : cps;
    int col[kCPL];
#pragma unroll
    for (int i = 0; i < kCPL; ++i) {
      const int c = lane_id() + 64 * i;
      if (kPair) {  // pair index within the stage row
        const int np = nch >> 1;
        const int pc = (wch >> 1) + (c < np ? c : (np > 0 ? np - 1 : 0));
        col[i] = pc < (C >> 1) ? pc : (C >> 1) - 1;
      } else {
        const int cc = wch + (c < nch ? c : (nch > 0 ? nch - 1 : 0));
        col[i] = cc < C ? cc : C - 1;  // idle lanes read a valid column
      }
    }
    using TO = typename RowSum<T, kCPL>::TO;  // 16-bit rows for 16-bit input
    TO *out = reinterpret_cast<TO *>(acc) + wch;
    RowSum<T, kCPL> st;
    __syncthreads();  // stage 0 is in buffer 0
    for (int k = 0; k < nst; k += kDepth) {  // barriers match the loaders'
#pragma unroll
      for (int r = 0; r < kDepth; ++r) {
        const int kk = k + r;
        st.add_stage(reinterpret_cast<const raw *>((kk & 1) ? buf1 : buf0),
                     (kk & 1) ? rk1s : rk0s, pr.rows(kk), C, col, nch, out, C);
        __syncthreads();
      }
    }
    st.flush(nch, out, C);
  } else {
    LoaderRing<kSlots> R;
#pragma unroll
    for (int i = 0; i < kSlots; ++i) {
      const int slot = lt + kLoaders * i;
      R.srow[i] = slot / pr.rowq;
      R.sq[i] = slot - R.srow[i] * pr.rowq;
    }
    // prologue: indices of stages 0..D-1, rows of 0..D-1 each followed by the
    // indices of stage j+D; then stage 0 into LDS
#define BEVPOOL_RING_PRO(J)                                                                    \
  if constexpr ((J) < kDepth) ring_index<kSlots, (J)>(R, kw, pr, (J));
    BEVPOOL_RING_PRO(0) BEVPOOL_RING_PRO(1) BEVPOOL_RING_PRO(2) BEVPOOL_RING_PRO(3)
    BEVPOOL_RING_PRO(4) BEVPOOL_RING_PRO(5) BEVPOOL_RING_PRO(6) BEVPOOL_RING_PRO(7)
#undef BEVPOOL_RING_PRO
#define BEVPOOL_RING_PRO(J)                                                                    \
  if constexpr ((J) < kDepth) {                                                               \
    ring_rows<kSlots, (J), kRows>(R, lt, kw, xb, ld_bytes, pr, (J));                           \
    ring_index<kSlots, (J)>(R, kw, pr, (J) + kDepth);                                          \
  }
    BEVPOOL_RING_PRO(0) BEVPOOL_RING_PRO(1) BEVPOOL_RING_PRO(2) BEVPOOL_RING_PRO(3)
    BEVPOOL_RING_PRO(4) BEVPOOL_RING_PRO(5) BEVPOOL_RING_PRO(6) BEVPOOL_RING_PRO(7)
#undef BEVPOOL_RING_PRO
    ring_store<kSlots, 0>(R, lt, pr, 0, buf0, rk0s);
    __syncthreads();
    for (int k = 0; k < nst; k += kDepth) {
#define BEVPOOL_RING_STEP(J)                                                                   \
  if constexpr ((J) < kDepth)                                                                 \
    loader_step<kSlots, (J), kRows>(R, lt, kw, xb, ld_bytes, pr, k + (J), nst, buf0, buf1,     \
                                    rk0s, rk1s);
      BEVPOOL_RING_STEP(0) BEVPOOL_RING_STEP(1) BEVPOOL_RING_STEP(2) BEVPOOL_RING_STEP(3)
      BEVPOOL_RING_STEP(4) BEVPOOL_RING_STEP(5) BEVPOOL_RING_STEP(6) BEVPOOL_RING_STEP(7)
#undef BEVPOOL_RING_STEP
    }
  }
}

// ---- grouped forward accumulation ------------------------------------------
//
// Used for depth-weighted context rows, for rows that are no run of aligned
// 16-byte pieces, for rows of more than kPipeRowBytes and for small inputs
// (group_plan).  A row is cut into q 16-byte pieces (the last one ends at the
// row's end and overlaps the piece before it where the row is no multiple of
// 16 bytes: both lanes then hold and store the same sums), a wave into ng =
// 64 / q groups of q lanes.  Each group owns the cells that start in its P
// nominal sorted positions and walks their points in order, lane j keeping
// the sums of piece j in registers and storing them when the rank changes: no
// barrier, and one load, 4 (8) products and sums per lane for ng rows at a
// time, where accum_pipe_kernel spends loader and summer instructions on
// every row.
//   * Row addresses, ranks and depth weights of kK points per group are
//     worked out once, by one lane per point, and read back from the wave's
//     64 LDS entries; the keys of the batch after next and the weights of the
//     next one are in flight meanwhile.
//   * Rows are in flight kK at a time in two register halves: one is added
//     while the other loads.
// What bounds it with context rows (counters at C = 80, 7.1 M points on 4 x 360 x
// 360, 190 us, and 1.8 M on 1 x 360 x 360, 55 us): no unit by itself.  L2 takes
// 157 and 123 G requests/s, about half of one per channel and clock, 77 and 80%
// of them hits; an L1 miss returns after 274 and 252 clocks; the L1s make 0.7 and
// 0.6 accesses per clock; the vector units issue 45 and 38% of the time, with 2.5
// and 2.2 waves per SIMD resident.  (accum_pipe_kernel took 339 and 88 us.)
// Feature rows come from HBM.  There 16-byte aligned rows of one channel block
// stay with accum_pipe_kernel, whose blocks keep more rows of few cells in
// flight (131 against 147 us at 1 x 360 x 360).  Rows of 128 fp32 channels, two
// channel blocks to that kernel, take 189 against 215 us; 180-byte fp16 rows at
// 1.06 M points 80 against 457 us for accum_rows_kernel's element-wise loads.
// Walking the ranges in XCD-contiguous eighths cost 5-10%, rings of 4 + 4 rows
// 3-10%, and a register limit for 4 waves per SIMD spilled.
//
// Long cells.  One group would walk a cell of L points as a chain of L / kK
// round trips, so cells of at least lcell points go to the launch's first
// blocks instead: a cell of lcell or more sorted points covers a multiple of
// lcell, so lane l of such a block tests the cell at one multiple and takes
// it if that is the cell's first.  A long cell is summed by one wave per 64
// bytes of the row: 16 rows per load, 64 in flight and 64 more being added,
// transposed through LDS so that lane c adds element c of the rows in order.
// Every element is still one sequential chain from +0.0 in point order.
// The slowest of these blocks sets the kernel's time where cells are long, so
// a block takes kLongPieces pieces of its cells, one 64-byte slice per wave,
// and rows of more are dealt to several blocks (with all slices of a cell in
// one block, 5 or 8 of them on 4 waves: 1.43 M depth-weighted points on 2 x 127
// x 127 cells, C = 92, 144 us; one per wave 73, accum_pipe_kernel 160).

// Rows of the depth-weighted forward (fused depth x context pooling): the row
// of point p = (bn*D + d)*HW + hw is context row pix = bn*HW + hw, weighted by
// depth[p] (the reference materialises depth[p] * context[pix, c],
// models/vtransforms/depth_lss.py:91-94).
struct DepthRows {
  const float *depth;  // (BN, D, HW) contiguous: depth[p]
  FastDiv hw, nd;      // HW and D
  // p = (bn*D + d)*HW + hw -> bn*HW + hw, with e = p / HW = bn*D + d
  __device__ __forceinline__ uint32_t pix(uint32_t p) const {
    const uint32_t e = hw.div(p);
    return nd.div(e) * hw.d + (p - e * hw.d);
  }
};

// The running sums of one lane's 16-byte piece of a row.
template <typename T>
struct PieceSum {
  static constexpr int kE = 16 / int(sizeof(typename T::raw));  // elements per piece
  float a[kE];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < kE; ++i) a[i] = 0.0f;
  }
  template <bool kMul>
  __device__ __forceinline__ void add(u32x4 v, float w) {
    const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (kE == 4) {
        // one fp32 product, then the sum (the reference's product and sum)
        const float x = __uint_as_float(d[i]);
        a[i] += kMul ? x * w : x;
      } else {
        a[2 * i] += T::from_raw(d[i] & 0xffffu);
        a[2 * i + 1] += T::from_raw(d[i] >> 16);
      }
    }
  }
  // the sums in the output's element type (16-bit: rounded once)
  __device__ __forceinline__ u32x4 bits() const {
    uint32_t d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (kE == 4)
        d[i] = __float_as_uint(a[i]);
      else
        d[i] = uint32_t(T::to_raw(a[2 * i])) | (uint32_t(T::to_raw(a[2 * i + 1])) << 16);
    }
    return u32x4{d[0], d[1], d[2], d[3]};
  }
};

template <int kRows>
__device__ __forceinline__ u32x4 load_piece(const char *p) {
  if constexpr (kRows == kRowsStream) {
    return __builtin_nontemporal_load(reinterpret_cast<const u32x4_any *>(p));
  } else {
    return reinterpret_cast<const Bytes16 *>(p)->v;
  }
}

// Orders this wave's LDS accesses (its lanes exchange data through LDS; one
// wave's LDS operations complete in order, so no wait is needed).
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// kH rows of a group: this lane's pieces, and each row's rank and weight.
template <int kH>
struct GroupRing {
  u32x4 v[kH];
  int rk[kH];
  float w[kH];
};

// Loads the rows of kH entries (ent: row offset, rank, weight).
template <int kH, int kRows>
__device__ __forceinline__ void group_load(GroupRing<kH> &R, const u32x4 *ent, const char *xp) {
#pragma unroll
  for (int u = 0; u < kH; ++u) {
    const u32x4 e = ent[u];
    R.rk[u] = int(e.z);
    if constexpr (kRows == kRowsDepth) R.w[u] = __uint_as_float(e.w);
    R.v[u] = load_piece<kRows>(xp + (uint64_t(e.x) | (uint64_t(e.y) << 32)));
  }
}

// Adds kH rows; where the rank changes, the finished cell's piece is stored.
template <typename T, int kH, int kRows>
__device__ __forceinline__ void group_add(const GroupRing<kH> &R, PieceSum<T> &sum, int &cur,
                                          bool own, char *op, int64_t out_row_bytes) {
#pragma unroll
  for (int u = 0; u < kH; ++u) {
    if (R.rk[u] != cur) {
      if (cur >= 0 && own)
        reinterpret_cast<Bytes16 *>(op + int64_t(cur) * out_row_bytes)->v = sum.bits();
      sum.clear();
      cur = R.rk[u];
    }
    sum.template add<kRows == kRowsDepth>(R.v[u], kRows == kRowsDepth ? R.w[u] : 0.0f);
  }
}

// One wave's share of a long cell: elements of pieces [j0, j0 + 4) of the row
// (pieces from jend on repeat the last one and are not stored) summed over
// sorted positions [b0, b1).  The loads run up to 192 positions ahead of the
// sum, and b1 may be 2^31 - 1: positions are counted from the cell's last.
// tile: the wave's 64 16-byte LDS entries.
template <typename T, int kRows>
__device__ __forceinline__ void sum_long_cell(const char *__restrict__ xb, int64_t ld_bytes,
                                              int row_bytes, int j0, int jend,
                                              const uint32_t *__restrict__ kw, int b0, int b1,
                                              char *__restrict__ out_row, u32x4 *tile,
                                              const DepthRows &dr) {
  using raw = typename T::raw;
  constexpr bool kMul = kRows == kRowsDepth;
  constexpr int kPe = 16 / int(sizeof(raw));  // elements per piece
  constexpr int kEl = 4 * kPe;                // elements of the four pieces
  constexpr int kT = 4;                       // 16-row loads in flight
  const int lane = lane_id(), slot = lane >> 2;
  const int j = j0 + (lane & 3) < jend ? j0 + (lane & 3) : jend - 1;
  const char *xp = xb + (16 * j < row_bytes - 16 ? 16 * j : row_bytes - 16);
  float a = 0.0f, w[kT];
  u32x4 v[kT];
  uint32_t idx[kT];
  auto indices = [&](int rest) {  // from `rest` before the last point; past that: itself
#pragma unroll
    for (int t = 0; t < kT; ++t) {
      const int back = rest - (16 * t + slot);
      const int p = b1 - 1 - (back > 0 ? back : 0);
      idx[t] = kRows == kRowsRun ? uint32_t(p) : kw[2 * int64_t(p)];
    }
  };
  auto rows = [&]() {
#pragma unroll
    for (int t = 0; t < kT; ++t) {
      const uint32_t row = kMul ? dr.pix(idx[t]) : idx[t];
      if constexpr (kMul) w[t] = dr.depth[idx[t]];
      v[t] = load_piece<kRows>(xp + int64_t(row) * ld_bytes);
    }
  };
  indices(b1 - 1 - b0);
  rows();
  indices(b1 - 1 - b0 - 16 * kT);
  for (int rest = b1 - 1 - b0; rest >= 0; rest -= 16 * kT) {
    u32x4 c[kT];
#pragma unroll
    for (int t = 0; t < kT; ++t) {
      c[t] = v[t];
      if constexpr (kMul) {
        const float x0 = __uint_as_float(v[t].x) * w[t];
        const float x1 = __uint_as_float(v[t].y) * w[t];
        const float x2 = __uint_as_float(v[t].z) * w[t];
        const float x3 = __uint_as_float(v[t].w) * w[t];
        c[t] = u32x4{__float_as_uint(x0), __float_as_uint(x1), __float_as_uint(x2),
                     __float_as_uint(x3)};
      }
    }
    rows();  // of the next 64 positions, whose indices have arrived
    indices(rest - 32 * kT);
#pragma unroll
    for (int t = 0; t < kT; ++t) {
      const int left = rest + 1 - 16 * t;
      if (left <= 0) break;
      wave_lds_order();
      tile[lane] = c[t];
      wave_lds_order();
      const raw *col = reinterpret_cast<const raw *>(tile) + (lane < kEl ? lane : kEl - 1);
      float x[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) x[u] = T::load(col + u * kEl);
      if (left >= 16) {
#pragma unroll
        for (int u = 0; u < 16; ++u) a += x[u];
      } else {
#pragma unroll
        for (int u = 0; u < 16; ++u)
          if (u < left) a += x[u];
      }
    }
  }
  const int jo = j0 + lane / kPe;
  if (lane < kEl && jo < jend) {
    const int pb = 16 * jo < row_bytes - 16 ? 16 * jo : row_bytes - 16;
    reinterpret_cast<raw *>(out_row + pb)[lane % kPe] = T::to_raw(a);
  }
}

constexpr int kLongPieces = 4 * kWaves;  // row pieces per block of long cells

// blockIdx.y: block of at most qmax (<= 64) row pieces.  The first
// long_blocks blocks of x take the long cells (long_sets sets of long_lanes
// candidates, each set once per kLongPieces pieces), the others the ranges.
// Feature rows in batches of 4 keep to 80 VGPRs, 6 waves per SIMD (82: 5, and 90
// -> 113 us at 1.6 M rows of 27 fp32 channels); with context rows that spills.
template <typename T, int kK, int kRows>
__global__ __launch_bounds__(kThreads, kK == 4 && kRows != kRowsDepth ? 6 : 1) void
accum_group_kernel(
    const char *__restrict__ xb, int64_t ld_bytes, int C, int qmax,
    const uint64_t *__restrict__ keys, const int32_t *__restrict__ meta,
    const int32_t *__restrict__ cstart, const int32_t *__restrict__ cend, char *__restrict__ acc,
    int P, int lcell, int long_blocks, int long_sets, int long_lanes, DepthRows dr) {
  constexpr bool kMul = kRows == kRowsDepth;
  constexpr int kH = kK / 2;
  __shared__ u32x4 s_ent[kWaves][64];
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  u32x4 *ent = s_ent[wave];
  const uint32_t *kw = reinterpret_cast<const uint32_t *>(keys);  // low word: point index
  const int n = meta[BEVPOOL_META_N_KEPT];
  if (n <= 0) return;
  const int row_bytes = C * int(sizeof(typename T::raw));
  const int q0 = int(blockIdx.y) * qmax;
  const int qt = (row_bytes + 15) >> 4;
  const int q = qt - q0 < qmax ? qt - q0 : qmax;

  if (int(blockIdx.x) < long_blocks) {
    const int part = int(blockIdx.x) / long_sets, set = int(blockIdx.x) - part * long_sets;
    const int js = q0 + kLongPieces * part;
    const int je = q0 + q < js + kLongPieces ? q0 + q : js + kLongPieces;
    const int64_t pos = (int64_t(lane) * long_sets + set) * lcell;
    int cs = 0, ce = 0, r = 0;
    bool found = false;
    if (lane < long_lanes && pos < n) {
      r = key_rank(keys[pos]);
      cs = cstart[r];
      ce = cend[r];
      found = ce - cs >= lcell && int64_t(cs) > pos - lcell;
    }
    int task = 0;  // the block's waves take its (cell, four pieces) tasks in turn
    for (uint64_t m = __ballot(found); m; m &= m - 1) {
      const int src = __builtin_ctzll(m);
      const int b0 = __builtin_amdgcn_readlane(cs, src), b1 = __builtin_amdgcn_readlane(ce, src);
      const int cell = __builtin_amdgcn_readlane(r, src);
      for (int j0 = js; j0 < je; j0 += 4)
        if ((task++ & (kWaves - 1)) == wave)
          sum_long_cell<T, kRows>(xb, ld_bytes, row_bytes, j0, je, kw, b0, b1,
                                  acc + int64_t(cell) * row_bytes, ent, dr);
    }
    return;
  }

  const int ng = 64 / q < 64 / kK ? 64 / q : 64 / kK;
  const int64_t gw = (int64_t(blockIdx.x) - long_blocks) * kWaves + wave;
  if (gw * ng * P >= n) return;  // no barriers below
  // lanes past the last group repeat its last piece and store nothing
  const bool own = lane / q < ng;
  const int g = own ? lane / q : ng - 1;
  const int li = lane - g * q < q ? lane - g * q : q - 1;
  const int pb = 16 * (q0 + li) < row_bytes - 16 ? 16 * (q0 + li) : row_bytes - 16;
  const char *xp = xb + pb;
  char *op = acc + pb;

  // this group's whole cells: sorted positions [s, e).  A long cell that
  // starts in the range is its last cell (P < lcell) and ends it.
  int s, e;
  {
    const int64_t p0 = (gw * ng + g) * P, p1 = p0 + P;
    const int64_t a0 = p0 < n ? p0 : n - 1, a1 = p1 < n ? p1 : n - 1;
    const int r0 = key_rank(keys[a0]), r0b = key_rank(keys[a0 > 0 ? a0 - 1 : 0]);
    const int r1 = key_rank(keys[a1]), r1b = key_rank(keys[a1 > 0 ? a1 - 1 : 0]);
    const int e0 = cend[r0], s1 = cstart[r1], e1 = cend[r1];
    s = p0 >= n ? n : (p0 == 0 || r0b != r0 ? int(p0) : e0);
    e = p1 >= n ? n : (r1b != r1 ? int(p1) : (e1 - s1 >= lcell ? s1 : e1));
  }
  const int len = e > s ? e - s : 0;
  int most = len;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_xor(most, o, 64);
    most = most > y ? most : y;
  }
  const int nb = __builtin_amdgcn_readfirstlane((most + kK - 1) / kK);
  if (nb == 0) return;
  // this lane's LDS entry: point lane % kK of each batch of group lane / kK
  const int eg = lane / kK < ng ? lane / kK : ng - 1;
  const int es = __shfl(s, eg * q, 64), el = __shfl(len, eg * q, 64);
  const int er = lane % kK;

  auto fetch = [&](int b) -> uint64_t {  // past the group's points: its first key
    const int i = b * kK + er;
    return keys[i < el ? es + i : (el > 0 ? es : 0)];
  };
  // Entries of batch b.  Past the group's points: rank -2, which ends the
  // last cell; what is added then is never stored.
  auto put = [&](int b, uint64_t key, float w) {
    const uint32_t row = kMul ? dr.pix(key_index(key)) : key_index(key);
    const uint64_t off = uint64_t(row) * uint64_t(ld_bytes);
    const int rk = b * kK + er < el ? key_rank(key) : -2;
    wave_lds_order();
    ent[lane] = u32x4{uint32_t(off), uint32_t(off >> 32), uint32_t(rk), __float_as_uint(w)};
    wave_lds_order();
  };

  PieceSum<T> sum;
  sum.clear();
  int cur = -1;
  GroupRing<kH> A, B;
  const u32x4 *ge = ent + g * kK;
  uint64_t k0 = fetch(0), k1 = fetch(1);
  float w = 0.0f;
  if constexpr (kMul) w = dr.depth[key_index(k0)];
  put(0, k0, w);
  k0 = k1;
  if constexpr (kMul) w = dr.depth[key_index(k0)];
  k1 = fetch(2);
  group_load<kH, kRows>(A, ge, xp);
  for (int b = 0; b < nb; ++b) {
    // k0, w: keys and weights of batch b + 1; k1: keys of batch b + 2
    group_load<kH, kRows>(B, ge + kH, xp);
    put(b + 1, k0, w);
    k0 = k1;
    if constexpr (kMul) w = dr.depth[key_index(k0)];
    k1 = fetch(b + 3);
    group_add<T, kH, kRows>(A, sum, cur, own, op, row_bytes);
    group_load<kH, kRows>(A, ge, xp);
    group_add<T, kH, kRows>(B, sum, cur, own, op, row_bytes);
  }
  if (cur >= 0 && own)
    reinterpret_cast<Bytes16 *>(op + int64_t(cur) * row_bytes)->v = sum.bits();
}

// ---------------------------------------------------------------------------
// transposes between cell-major rows and the channel-first BEV
// ---------------------------------------------------------------------------
// A tile is 64 consecutive cells (ranks); rows are staged in LDS as
// [cell][channel] with a pitch of CT + 1 elements, CT = channels per pass.
// On the channel-first side each thread moves 4 consecutive cells of one
// channel with one 16-byte (fp32) or 8-byte (16-bit) access.  With kVecBev
// (n_xy, the b/z/c strides and the base are multiples of 4 elements) 4 cells
// starting at a multiple of 4 always share a (b, z) plane and the access is
// aligned (and the output's stores non-temporal: it is not read again here);
// otherwise it is an access at element alignment, and the few groups
// of 4 cells that a plane's end cuts go cell by cell.  On the row side
// kVecRow (rows of 16 bytes or more) moves 16-byte pieces of a row; where the
// row is no multiple of 16 bytes the last piece ends at the row's end and
// overlaps the one before it.  Measured (MI355X, 3 x 201 x 199 cells of 90
// fp16 channels, which no vector width divides): rows_to_bev 32.6 -> 19.2,
// bev_to_rows 21.8 -> 14.3 us against element-wise loads and stores.

// Offset of cell `cell` (< 2^31) in a channel-first (b, c, z, xy) tensor
// without the channel term.  The divisions by n_xy and n_z are multiplies:
// every thread of bev_to_rows divides twice, which was half that kernel's time
// on a sparse grid (6 x 685 x 685 cells, 16 channels: 87 -> 70 us).
struct CellMap {
  FastDiv xy, z;
  int64_t sb, sz;
  __device__ __forceinline__ int64_t operator()(uint32_t cell) const {
    const uint32_t plane = xy.div(cell), b = z.div(plane);
    return int64_t(b) * sb + int64_t(plane - b * z.d) * sz + int64_t(cell - plane * xy.d);
  }
  // Are 4 cells, the first a multiple of 4, at offsets first .. last
  // consecutive elements?  They lie in two planes at most, each a run of its
  // own, so the ends tell; planes of one cell, of which there are 4, can lie in
  // any order between them.
  __device__ __forceinline__ bool run_of_4(int64_t first, int64_t last) const {
    return xy.d > 1 && last == first + 3;
  }
};

// acc rows (cell-major fp32, written for occupied cells only) -> out
// (channel-first, dtype T); empty cells are written as 0.  The tile holds the
// raw fp32 bits, and a staged 16-byte piece is never converted lane by lane
// to float (hipcc 7.2 with packed fp32 ops disabled folded bit casts of lanes
// y/z/w of such a vector into lane x).  With kVecRow each wave first reads
// the tile's 64 cell ends as a ballot mask, then loads every row piece of the
// occupied cells up front (kTileSlots per thread, clamped in-bounds
// addresses), so a block pays two memory latencies before its stores and
// reads no row of an empty cell (measured on MI355X: 53 -> 43 us at B = 4,
// 360 x 360, unchanged at B = 1).  Occupancy: cell_end != 0 (cell ranges are
// zeroed before the sort writes the occupied ones).
constexpr int kTileSlots = kCellTile * (kTileChannels / 4) / kThreads;  // 8
// bev_to_rows on grids of at least this many cells reads the occupancy of a
// thread's 4 cells before its gradient loads (one more memory latency per
// block, no loads for 4 empty cells); smaller grids issue every load up
// front.  Measured on MI355X: 3-10% faster from 518,400 cells (B = 4 at
// 360 x 360) up, slower at 129,600.  The same per-thread scheme for
// rows_to_bev was slower (it uses the wave-wide mask above instead).
constexpr int64_t kOccFirstCells = 200000;

// Optional copy of the meta counters into memory the host reads (pinned host
// memory through its device address), made by a kernel that runs anyway.
// One thread writes the counters as system-scope stores and then sets the
// done flag dst[BEVPOOL_META_LEN] with a system-scope release store, so a
// host that sees the flag sees the counters (the release orders the
// thread's earlier stores before the flag; no event is involved).
struct MetaReport {
  const int32_t *meta = nullptr;
  int32_t *dst = nullptr;
};

__device__ __forceinline__ void store_meta_report(const int32_t *__restrict__ meta,
                                                  int32_t *__restrict__ dst) {
  if (threadIdx.x == 0) {
    int32_t v[BEVPOOL_META_LEN];
#pragma unroll
    for (int i = 0; i < BEVPOOL_META_LEN; ++i) v[i] = meta[i];
#pragma unroll
    for (int i = 0; i < BEVPOOL_META_LEN; ++i)
      __hip_atomic_store(dst + i, v[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(dst + BEVPOOL_META_LEN, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

__device__ __forceinline__ void write_meta_report(const MetaReport &rep) {
  if (rep.dst && blockIdx.x == 0) store_meta_report(rep.meta, rep.dst);
}

// bevpool_meta_report: the counters and the done flag, one block of 64 (its
// first thread does the work).
__global__ void meta_report_kernel(const int32_t *__restrict__ meta, int32_t *__restrict__ dst) {
  store_meta_report(meta, dst);
}

// kRaw16: the cell rows already hold the output's 16-bit values (the
// pipelined accumulation stores them rounded once), moved without conversion;
// otherwise they are fp32 sums converted on the way out.
template <typename T, bool kVecRow, bool kVecBev, bool kRaw16 = false>
__global__ __launch_bounds__(kThreads) void rows_to_bev_kernel(
    const float *__restrict__ acc, int C, int CT, const int32_t *__restrict__ cend,
    int64_t n_cells, CellMap cell_offset, int64_t sc,
    typename T::raw *__restrict__ out, MetaReport report) {
  using raw = typename T::raw;
  static_assert(!kRaw16 || sizeof(raw) == 2, "16-bit rows for 16-bit output only");
  write_meta_report(report);
  extern __shared__ uint32_t tile_bits[];  // kCellTile * (CT + 1)
  __shared__ int occ[kCellTile];
  __shared__ int64_t off[kCellTile];
  const int tid = threadIdx.x;
  const int64_t cell0 = int64_t(blockIdx.x) * kCellTile;
  const uint32_t *accb = reinterpret_cast<const uint32_t *>(acc);
  const int pitch = CT + 1;
  // occupancy of the tile's 64 cells as a mask in every wave (lane j loads
  // cell j's end), so that only occupied cells' rows are loaded: one more
  // dependent load, and no row bytes for empty cells (most cells of the
  // sparser grids); wave 0's mask also gives each cell's own flag, so the
  // ends are loaded once
  uint64_t occm = 0;
  if (kVecRow) {
    const int64_t cj = cell0 + lane_id();
    occm = __ballot(cj < n_cells && cend[cj] != 0);
    if (occm == 0) {
      // an empty tile: zeros, no rows, no LDS
      const int j = (tid & 15) * 4;
      if (cell0 + j >= n_cells) return;
      int64_t o[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        o[u] = cell0 + j + u < n_cells ? cell_offset(uint32_t(cell0 + j + u)) : -1;
      const bool run = kVecBev || cell_offset.run_of_4(o[0], o[3]);
      for (int c = tid >> 4; c < C; c += kThreads / 16) {
        if (run) {
          using V = typename std::conditional<sizeof(raw) == 4, u32x4, u32x2>::type;
          using VA = typename std::conditional<sizeof(raw) == 4, u32x4_any, u32x2_any>::type;
          raw *dst = out + o[0] + int64_t(c) * sc;
          if constexpr (kVecBev)
            __builtin_nontemporal_store(V{}, reinterpret_cast<V *>(dst));
          else
            *reinterpret_cast<VA *>(dst) = V{};
        } else {
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (o[u] >= 0) out[o[u] + int64_t(c) * sc] = raw(0);
        }
      }
      return;
    }
  }
  int occ_mine = 0;
  int64_t off_mine = -1;
  if (tid < kCellTile && cell0 + tid < n_cells) {
    occ_mine = kVecRow ? int((occm >> tid) & 1u) : (cend[cell0 + tid] != 0 ? 1 : 0);
    off_mine = cell_offset(uint32_t(cell0 + tid));
  }
  if (!kVecRow) {
    if (tid < kCellTile) {
      occ[tid] = occ_mine;
      off[tid] = off_mine;
    }
    __syncthreads();
  }
  const uint16_t *acch = reinterpret_cast<const uint16_t *>(acc);
  constexpr uint32_t kPer = kRaw16 ? 8 : 4;  // channels per 16-byte piece
  for (int cn = 0; cn < C; cn += CT) {
    const int c0 = first_channel(C, kVecRow ? int(kPer) : 1, cn);
    const int cb = C - c0 < CT ? C - c0 : CT;
    if (kVecRow) {
      const uint32_t q = (uint32_t(cb) + kPer - 1) / kPer;  // 16-byte pieces per row
      const uint32_t last = uint32_t(cb) - kPer;            // first channel of the last one
      const uint32_t n_items = kCellTile * q;
      u32x4 v[kTileSlots];
#pragma unroll
      for (int it = 0; it < kTileSlots; ++it) {
        if (uint32_t(it * kThreads) >= n_items) break;  // block-uniform: no pieces left
        const uint32_t i = tid + it * kThreads;
        uint32_t t = i / q, k = i - t * q;
        if (i >= n_items || cell0 + t >= n_cells) t = k = 0;
        const uint32_t c = kPer * k < last ? kPer * k : last;
        const void *src = kRaw16 ? static_cast<const void *>(acch + (cell0 + t) * C + c0 + c)
                                 : static_cast<const void *>(accb + (cell0 + t) * C + c0 + c);
        v[it] = ((occm >> t) & 1) ? reinterpret_cast<const Bytes16 *>(src)->v
                                  : u32x4{0u, 0u, 0u, 0u};
      }
      if (cn == 0 && tid < kCellTile) {
        occ[tid] = occ_mine;
        off[tid] = off_mine;
      }
#pragma unroll
      for (int it = 0; it < kTileSlots; ++it) {
        const uint32_t i = tid + it * kThreads;
        if (i < n_items) {
          const uint32_t t = i / q, k = i - t * q;
          uint32_t *d = tile_bits + t * pitch + (kPer * k < last ? kPer * k : last);
          if constexpr (kRaw16) {  // 8 values, low half first
            d[0] = v[it].x & 0xffffu;
            d[1] = v[it].x >> 16;
            d[2] = v[it].y & 0xffffu;
            d[3] = v[it].y >> 16;
            d[4] = v[it].z & 0xffffu;
            d[5] = v[it].z >> 16;
            d[6] = v[it].w & 0xffffu;
            d[7] = v[it].w >> 16;
          } else {
            d[0] = v[it].x;
            d[1] = v[it].y;
            d[2] = v[it].z;
            d[3] = v[it].w;
          }
        }
      }
    } else {
      for (uint32_t i = tid; i < uint32_t(kCellTile * cb); i += kThreads) {
        const uint32_t t = i / uint32_t(cb), c = i - t * uint32_t(cb);
        if (occ[t])
          tile_bits[t * pitch + c] = kRaw16 ? uint32_t(acch[(cell0 + t) * C + c0 + c])
                                            : accb[(cell0 + t) * C + c0 + c];
      }
    }
    __syncthreads();
    for (int i = tid; i < cb * (kCellTile / 4); i += kThreads) {
      const int c = i >> 4, j = (i & 15) * 4;
      raw r[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t b = occ[j + u] ? tile_bits[(j + u) * pitch + c] : 0u;
        if constexpr (kRaw16)
          r[u] = raw(b);
        else
          r[u] = T::to_raw(__builtin_bit_cast(float, b));
      }
      if (kVecBev && off[j] < 0) continue;
      if (kVecBev || (off[j] >= 0 && cell_offset.run_of_4(off[j], off[j + 3]))) {
        raw *dst = out + off[j] + int64_t(c0 + c) * sc;
        if constexpr (sizeof(raw) == 4) {
          u32x4 w;
          w.x = r[0];
          w.y = r[1];
          w.z = r[2];
          w.w = r[3];
          if constexpr (kVecBev)
            __builtin_nontemporal_store(w, reinterpret_cast<u32x4 *>(dst));
          else
            reinterpret_cast<Bytes16 *>(dst)->v = w;
        } else {
          u32x2 w;
          w.x = uint32_t(r[0]) | (uint32_t(r[1]) << 16);
          w.y = uint32_t(r[2]) | (uint32_t(r[3]) << 16);
          if constexpr (kVecBev)
            __builtin_nontemporal_store(w, reinterpret_cast<u32x2 *>(dst));
          else
            reinterpret_cast<Bytes8 *>(dst)->v = w;
        }
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (off[j + u] >= 0) out[off[j + u] + int64_t(c0 + c) * sc] = r[u];
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// backward kernels
// ---------------------------------------------------------------------------

// grad (channel-first, any b/c/z strides, xy contiguous) -> cell-major rows of
// the occupied cells (raw bits copied).  Each thread always handles the same
// 4 cells (j = 4 * (tid % 16)) of channels tid / 16 + 16 it; all its tile
// loads are issued up front (clamped in-bounds addresses, empty cells
// included) together with the occupancy loads, or, with occ_first, after
// reading its 4 cells' occupancy (none when all 4 are empty).
template <typename TR, bool kVecRow, bool kVecBev>
__global__ __launch_bounds__(kThreads) void bev_to_rows_kernel(
    const TR *__restrict__ grad, int C, int CT, const int32_t *__restrict__ cend,
    int64_t n_cells, CellMap cell_offset, int64_t sc, bool occ_first,
    TR *__restrict__ rows) {
  extern __shared__ u32x4 smem_b2r[];
  TR *tile = reinterpret_cast<TR *>(smem_b2r);  // kCellTile * (CT + 1)
  __shared__ int occ[kCellTile];
  const int tid = threadIdx.x;
  const int64_t cell0 = int64_t(blockIdx.x) * kCellTile;
  const int pitch = CT + 1;
  constexpr int kPer = 16 / int(sizeof(TR));  // elements per 16-byte row piece
  const int j = (tid & 15) * 4;
  // with kVecBev a live thread's 4 cells all exist (n_cells % 4 == 0)
  const bool live = cell0 + j < n_cells;
  // sparse grids: the 4 cells' occupancy first, no gradient loads when all are
  // empty, nothing more for a tile without an occupied cell
  bool need = kVecBev || live;
  if (occ_first) {
    int o[4] = {0, 0, 0, 0};
    if (kVecBev || cell0 + j + 3 < n_cells) {
      if (live) {
        const u32x4 v = reinterpret_cast<const Bytes16 *>(cend + cell0 + j)->v;
        o[0] = v.x != 0;
        o[1] = v.y != 0;
        o[2] = v.z != 0;
        o[3] = v.w != 0;
      }
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) o[u] = cell0 + j + u < n_cells && cend[cell0 + j + u] != 0;
    }
    need = o[0] | o[1] | o[2] | o[3];
    if (__syncthreads_or(need ? 1 : 0) == 0) return;
    if (tid < 16)
#pragma unroll
      for (int u = 0; u < 4; ++u) occ[j + u] = o[u];
  }
  const int64_t offj = cell_offset(uint32_t(live ? cell0 + j : cell0));
  // are they 4 consecutive elements of a channel?
  const bool run =
      kVecBev || (cell0 + j + 3 < n_cells &&
                  cell_offset.run_of_4(offj, cell_offset(uint32_t(cell0 + j + 3))));
  for (int cn = 0; cn < C; cn += CT) {
    const int c0 = first_channel(C, kVecRow ? kPer : 1, cn);
    const int cb = C - c0 < CT ? C - c0 : CT;
    using V = typename std::conditional<sizeof(TR) == 4, u32x4, u32x2>::type;
    using VA = typename std::conditional<sizeof(TR) == 4, Bytes16, Bytes8>::type;
    V v[kTileSlots];
    if (run) {
#pragma unroll
      for (int it = 0; it < kTileSlots; ++it) {
        if (16 * it >= cb) break;  // block-uniform: no channels left
        int c = (tid >> 4) + 16 * it;
        c = c < cb ? c : 0;
        const TR *src = grad + offj + int64_t(c0 + c) * sc;
        if constexpr (kVecBev)
          v[it] = need ? *reinterpret_cast<const V *>(src) : V{};
        else
          v[it] = need ? reinterpret_cast<const VA *>(src)->v : V{};
      }
    } else {
      // a plane or the grid ends among the 4 cells
      int64_t ou[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        ou[u] = cell0 + j + u < n_cells ? cell_offset(uint32_t(cell0 + j + u)) : offj;
#pragma unroll
      for (int it = 0; it < kTileSlots; ++it) {
        if (16 * it >= cb) break;
        int c = (tid >> 4) + 16 * it;
        c = c < cb ? c : 0;
        uint32_t e[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) e[u] = need ? grad[ou[u] + int64_t(c0 + c) * sc] : 0u;
        if constexpr (sizeof(TR) == 4)
          v[it] = u32x4{e[0], e[1], e[2], e[3]};
        else
          v[it] = u32x2{e[0] | (e[1] << 16), e[2] | (e[3] << 16)};
      }
    }
    // the cells' occupancy, loaded after the gradient loads so that one
    // round trip brings both
    if (!occ_first && cn == 0 && tid < kCellTile)
      occ[tid] = cell0 + tid < n_cells && cend[cell0 + tid] != 0 ? 1 : 0;
#pragma unroll
    for (int it = 0; it < kTileSlots; ++it) {
      const int c = (tid >> 4) + 16 * it;
      if (c < cb) {
        TR e[4];
        if constexpr (sizeof(TR) == 4) {
          e[0] = v[it].x;
          e[1] = v[it].y;
          e[2] = v[it].z;
          e[3] = v[it].w;
        } else {
          e[0] = TR(v[it].x);
          e[1] = TR(v[it].x >> 16);
          e[2] = TR(v[it].y);
          e[3] = TR(v[it].y >> 16);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) tile[(j + u) * pitch + c] = e[u];
      }
    }
    __syncthreads();
    if (kVecRow) {
      const uint32_t q = (uint32_t(cb) + kPer - 1) / kPer;  // 16-byte pieces per row
      const uint32_t last = uint32_t(cb) - kPer;
      for (uint32_t i = tid; i < kCellTile * q; i += kThreads) {
        const uint32_t t = i / q, k = i - t * q;
        if (!occ[t]) continue;
        const uint32_t c = kPer * k < last ? kPer * k : last;
        const TR *srow = tile + t * pitch + c;
        u32x4 w;
        if constexpr (sizeof(TR) == 4) {
          w.x = srow[0];
          w.y = srow[1];
          w.z = srow[2];
          w.w = srow[3];
        } else {
          w.x = uint32_t(srow[0]) | (uint32_t(srow[1]) << 16);
          w.y = uint32_t(srow[2]) | (uint32_t(srow[3]) << 16);
          w.z = uint32_t(srow[4]) | (uint32_t(srow[5]) << 16);
          w.w = uint32_t(srow[6]) | (uint32_t(srow[7]) << 16);
        }
        reinterpret_cast<Bytes16 *>(rows + (cell0 + t) * C + c0 + c)->v = w;
      }
    } else {
      for (uint32_t i = tid; i < uint32_t(kCellTile * cb); i += kThreads) {
        const uint32_t t = i / uint32_t(cb), c = i - t * uint32_t(cb);
        if (occ[t]) rows[(cell0 + t) * C + c0 + c] = tile[t * pitch + c];
      }
    }
    __syncthreads();
  }
}

// Cache warm-up for gather_rows_kernel (its leading blocks).  Each gather piece is a dependent
// chain rank -> row -> store; with the rank array and the gradient rows
// fetched from HBM while the gather's write stream saturates it, the chains
// take about twice as long (measured 92 us vs 155-185 us at the det shape).
// Rows written by bev_to_rows_kernel are not reliably kept by the caches, rows
// that were read are, so this kernel reads both once:
//   * blocks [0, 8 * per_xcd): block wb runs on XCD wb % 8 and reads a share
//     of the ranks that XCD's gather blocks will need (the gather walks
//     XCD-contiguous eighths of its pieces, xcd_span pieces each), so they are
//     in that XCD's L2;
//   * the other blocks read the rows of the occupied cells of kWarmCells
//     consecutive cells each (16-byte pieces).
// Nothing is written: the only store is guarded by `never`, a launch argument
// that is always 0, which keeps the loads from being optimised away.
#ifndef BEVPOOL_WARM_CELLS
#define BEVPOOL_WARM_CELLS 512
#endif
constexpr int kWarmCells = BEVPOOL_WARM_CELLS;  // cells per row-warming block
constexpr int kWarmBatch = 8;                   // loads in flight per thread

struct GatherWarm {
  const u32x4 *rank16;   // rank array as 16-byte pieces (null: skip)
  int64_t n16;           // whole pieces in the array
  int64_t xcd_span;      // gather pieces (vectors of xg) per XCD
  int vpr;               // gather pieces per point
  int per_xcd;           // rank blocks per XCD
  const char *rows;      // gradient rows, 16 bytes or more each (null: skip)
  int rowq;              // 16-byte pieces per row (as gather_rows_kernel's)
  int row_bytes;
};

// Warm-up work of block wb (< warm_blocks(w, tiles)); returns nothing, reads only.
__device__ __forceinline__ void gather_warm_block(const GatherWarm &w, int wb, int64_t n_points,
                                                  const int32_t *__restrict__ cstart,
                                                  const int32_t *__restrict__ cend,
                                                  int64_t n_cells, int never,
                                                  uint32_t *__restrict__ sink) {
  __shared__ int occ[kWarmCells];
  const int rank_blocks = w.rank16 ? kXcds * w.per_xcd : 0;
  uint32_t m = 0;
  if (wb < rank_blocks) {
    const int x = wb % kXcds, j = wb / kXcds;
    // points [p0, p1) are gathered by XCD x; their ranks are pieces [q0, q1)
    const int64_t p0 = int64_t(x) * w.xcd_span / w.vpr;
    int64_t p1 = (int64_t(x + 1) * w.xcd_span + w.vpr - 1) / w.vpr;
    p1 = p1 < n_points ? p1 : n_points;
    const int64_t q0 = p0 / 4;
    int64_t q1 = (p1 + 3) / 4;
    q1 = q1 < w.n16 ? q1 : w.n16;
    const int64_t share = (q1 - q0 + w.per_xcd - 1) / w.per_xcd;
    const int64_t b0 = q0 + int64_t(j) * share;
    int64_t b1 = b0 + share;
    b1 = b1 < q1 ? b1 : q1;
    for (int64_t i = b0 + threadIdx.x; i < b1; i += kThreads) {
      const u32x4 v = w.rank16[i];
      m ^= v.x ^ v.y ^ v.z ^ v.w;
    }
  } else if (w.rows) {
    // kWarmCells consecutive cells per block: occupancy, then the occupied
    // rows' pieces, kWarmBatch loads in flight per thread
    const int64_t cell0 = int64_t(wb - rank_blocks) * kWarmCells;
    for (int t = threadIdx.x; t < kWarmCells; t += kThreads) {
      const int64_t cell = cell0 + t;
      occ[t] = (cell < n_cells && cend[cell] > cstart[cell]) ? 1 : 0;
    }
    __syncthreads();
    const uint32_t q = uint32_t(w.rowq);
    const uint32_t n = kWarmCells * q;
    for (uint32_t i0 = threadIdx.x; i0 < n; i0 += kThreads * kWarmBatch) {
      u32x4 v[kWarmBatch];
#pragma unroll
      for (int b = 0; b < kWarmBatch; ++b) {
        const uint32_t i = i0 + uint32_t(b) * kThreads < n ? i0 + uint32_t(b) * kThreads : n - 1;
        const uint32_t t = i / q, k = i - t * q;
        const int o = int(16 * k) < w.row_bytes - 16 ? int(16 * k) : w.row_bytes - 16;
        v[b] = occ[t] ? reinterpret_cast<const Bytes16 *>(w.rows + (cell0 + t) * w.row_bytes + o)->v
                      : u32x4{0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int b = 0; b < kWarmBatch; ++b) m ^= v[b].x ^ v[b].y ^ v[b].z ^ v[b].w;
    }
  }
  if (never) sink[threadIdx.x] = m;
}

// x_grad[p, :] = rows[rank[p], :] (kept) or 0 (dropped); point order, so the
// writes stream.  A row is moved as vpr vectors V: 16-byte ones for rows of
// 16 bytes or more (kAny: at element alignment, the last one ending at the
// row's end and overlapping the one before it with the same bytes), else
// elements.  Each thread copies one vector, blocks walk XCD-contiguous chunks
// (an XCD's points map to a compact set of cells, whose rows then stay in its
// L2), and the destination is written with non-temporal stores (it is not
// read again here, and keeping it out of L2 leaves room for the gradient
// rows).  Each piece is a dependent chain rank -> row -> store, so the leading
// warm_blocks blocks first pull the ranks and the rows into the caches
// (gather_warm_block).  kNarrow: indices fit in 32 bits.  What bounds it is
// the write stream (6.6 TB/s at 1 x 360 x 360, C = 80; a fill reaches 6.9).
// Rows of 90 fp16 values (1.06 M points, 191 MB written) take 38 us with
// unaligned 16-byte vectors, 147 element by element.
template <typename V, bool kNarrow, bool kAny>
__global__ __launch_bounds__(kThreads) void gather_rows_kernel(
    const char *__restrict__ rows, int vpr, int row_bytes, const int32_t *__restrict__ rank,
    int64_t n_points, char *__restrict__ xg, int64_t xg_ld, int warm_blocks, GatherWarm w,
    const int32_t *__restrict__ cstart, const int32_t *__restrict__ cend, int64_t n_cells,
    int never, int zero_dropped) {
  // the first warm_blocks blocks (a multiple of 8, so XCD parity is kept)
  // only pull ranks and rows into the caches ahead of the others
  if (int(blockIdx.x) < warm_blocks) {
    gather_warm_block(w, int(blockIdx.x), n_points, cstart, cend, n_cells, never,
                      reinterpret_cast<uint32_t *>(xg));
    return;
  }
  const int64_t total = n_points * vpr;
  const int64_t gb = int64_t(blockIdx.x) - warm_blocks;
  const int64_t i = xcd_chunk(gb, int64_t(gridDim.x) - warm_blocks) * kThreads + threadIdx.x;
  if (i >= total) return;
  int64_t p;
  int q;
  if (kNarrow) {
    const uint32_t ui = uint32_t(i), up = ui / uint32_t(vpr);
    p = up;
    q = int(ui - up * uint32_t(vpr));
  } else {
    p = i / vpr;
    q = int(i - p * vpr);
  }
  int o = q * int(sizeof(V));
  if (kAny) o = o < row_bytes - 16 ? o : row_bytes - 16;
  const int r = rank[p];
  if (r < 0 && !zero_dropped) return;  // the caller keeps dropped rows as they are
  char *dst = xg + p * xg_ld + o;
  if constexpr (kAny) {
    u32x4 v = u32x4{0u, 0u, 0u, 0u};
    if (r >= 0) v = reinterpret_cast<const Bytes16 *>(rows + int64_t(r) * row_bytes + o)->v;
    __builtin_nontemporal_store(v, reinterpret_cast<u32x4_any *>(dst));
  } else {
    V v = V{};
    if (r >= 0) v = *reinterpret_cast<const V *>(rows + int64_t(r) * row_bytes + o);
    __builtin_nontemporal_store(v, reinterpret_cast<V *>(dst));
  }
}

// ---------------------------------------------------------------------------
// legacy native interface (caller-provided intervals)
// ---------------------------------------------------------------------------

// Zero bytes [0, n16 * 16) as 16-byte vectors plus a 4-byte tail (n4 words
// from `tail`), grid-stride; with `when`, only if *when != 0.  A kernel
// rather than a memset so that a graph capture records no memset node.
__global__ __launch_bounds__(kThreads) void zero_fill_kernel(u32x4 *__restrict__ p, int64_t n16,
                                                             uint32_t *__restrict__ tail,
                                                             int64_t n4,
                                                             const int32_t *__restrict__ when) {
  if (when && *when == 0) return;
  const int64_t stride = int64_t(gridDim.x) * kThreads;
  for (int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x; i < n16; i += stride)
    p[i] = u32x4{0u, 0u, 0u, 0u};
  for (int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x; i < n4; i += stride) tail[i] = 0u;
}

// Validates interval j and returns its cell ((b*D + z)*H + x)*W + y from the
// coordinates of its first row, geom[s] = (x, y, z, b) (the cell of
// ops/bev_pool/csrc/bev_pool_cuda.cu:33-35), or -1 when its rows [s, s+len)
// or its cell lie outside the arrays (the reference reads and writes out of
// bounds there).
__device__ __forceinline__ int64_t legacy_cell(const int32_t *__restrict__ geom, int64_t n,
                                               int64_t s, int64_t len, int nb, int nd, int nh,
                                               int nw) {
  if (s < 0 || len < 0 || s >= n || s + len > n) return -1;
  const int gx = geom[4 * s], gy = geom[4 * s + 1], gz = geom[4 * s + 2], gb = geom[4 * s + 3];
  if (gx < 0 || gx >= nh || gy < 0 || gy >= nw || gz < 0 || gz >= nd || gb < 0 || gb >= nb)
    return -1;
  return ((int64_t(gb) * nd + gz) * nh + gx) * nw + gy;
}

// Interval count: the caller's host count, or min(capacity, device count).
__device__ __forceinline__ int64_t legacy_count(int64_t cap, const int32_t *__restrict__ dev) {
  if (!dev) return cap;
  const int64_t c = *dev;
  return c < cap ? (c > 0 ? c : 0) : cap;
}

// ops/bev_pool/csrc/bev_pool_cuda.cu:20-42: interval j sums rows [s, s + len)
// of x (n, C) -- fp32 from +0.0, rows in order -- and stores the sum to
// out[cell, :] (channels last).  Invalid intervals are skipped and counted in
// meta[BEVPOOL_META_N_BAD] (meta may be null).
//
// Rows of 4 channels or more are cut into 16-byte pieces (the last one ends
// at the row's end), a wave into 64 / q groups of q lanes, one interval per
// group, 8 rows in flight while 8 are added.  Intervals of kLegacyLong rows or
// more are left to the block's waves together afterwards, one per 64 bytes of
// the row (sum_long_cell), so that no chain of loads outlasts the rest.
// Neighbouring intervals go to different blocks: the long ones, the cells
// near the cameras, are neighbours.  The rows are read once, so HBM bounds it:
// 1.54 M rows of 80 channels (494 MB, 514 fetched) in 39 K intervals 118 us, 4.5
// TB/s with the sums written (a copy makes 5.2), against 230 with one wave per
// interval and 4 bytes per lane.
constexpr int kLegacyLong = 256;
// Blocks of a legacy launch; more intervals loop (2048 and 16384 blocks: forward
// 129 and 133 us, backward 110 and 108).
constexpr int kLegacyBlocks = 4096;

__global__ __launch_bounds__(kThreads) void legacy_sum_kernel(
    const char *__restrict__ x, int64_t n, int C, int qmax, const int32_t *__restrict__ geom,
    const int32_t *__restrict__ starts, const int32_t *__restrict__ lengths, int64_t cap,
    const int32_t *__restrict__ count_dev, int nb, int nd, int nh, int nw,
    char *__restrict__ out, int32_t *__restrict__ meta) {
  constexpr int kU = 8;
  __shared__ u32x4 s_tile[kWaves][64];
  __shared__ int s_long[kThreads], s_n;  // this pass's long intervals
  const int64_t n_int = legacy_count(cap, count_dev);
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int row_bytes = C * 4;
  const int q0 = int(blockIdx.y) * qmax, qt = (row_bytes + 15) >> 4;
  const int q = qt - q0 < qmax ? qt - q0 : qmax;
  const int ng = 64 / q;
  const bool own = lane / q < ng;  // lanes past the last group repeat its last piece
  const int g = own ? lane / q : ng - 1;
  const int li = lane - g * q < q ? lane - g * q : q - 1;
  const int pb = 16 * (q0 + li) < row_bytes - 16 ? 16 * (q0 + li) : row_bytes - 16;
  if (threadIdx.x == 0) s_n = 0;
  __syncthreads();
  const int64_t per_pass = int64_t(kWaves) * ng * gridDim.x;
  for (int64_t j0 = 0; j0 < n_int; j0 += per_pass) {
    const int64_t j = j0 + int64_t(wave * ng + g) * gridDim.x + blockIdx.x;
    int64_t s = 0, cell = -1;
    int len = 0;
    if (j < n_int) {
      s = starts[j];
      len = lengths[j];
      cell = legacy_cell(geom, n, s, len, nb, nd, nh, nw);
    }
    const bool lead = own && li == 0 && j < n_int;
    if (cell < 0) {
      if (meta && lead && blockIdx.y == 0) atomicAdd(meta + BEVPOOL_META_N_BAD, 1);
      s = len = 0;
    } else if (len >= kLegacyLong) {
      if (lead) s_long[atomicAdd(&s_n, 1)] = int(j);
      s = len = 0;
      cell = -1;
    }
    int most = len;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_xor(most, o, 64);
      most = most > y ? most : y;
    }
    most = __builtin_amdgcn_readfirstlane(most);
    PieceSum<F32> sum;
    sum.clear();
    if (most > 0) {
      const char *xp = x + s * row_bytes + pb;
      u32x4 a[kU], b[kU];
      auto load = [&](u32x4(&v)[kU], int i0) {  // past the interval: its last row
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          const int r = i0 + u < len ? i0 + u : (len > 0 ? len - 1 : 0);
          v[u] = reinterpret_cast<const Bytes16 *>(xp + int64_t(r) * row_bytes)->v;
        }
      };
      // rows past the interval add +0.0, which changes no sum that started
      // at +0.0 (it is never -0.0)
      auto add = [&](const u32x4(&v)[kU], int i0) {
#pragma unroll
        for (int u = 0; u < kU; ++u)
          sum.add<false>(i0 + u < len ? v[u] : u32x4{0u, 0u, 0u, 0u}, 0.0f);
      };
      load(a, 0);
      for (int i = 0; i < most; i += 2 * kU) {
        load(b, i + kU);
        add(a, i);
        load(a, i + 2 * kU);
        add(b, i + kU);
      }
    }
    if (cell >= 0 && own)
      reinterpret_cast<Bytes16 *>(out + cell * row_bytes + pb)->v = sum.bits();
    __syncthreads();
    const int slices = (q + 3) >> 2, tasks = s_n * slices;
    for (int t = wave; t < tasks; t += kWaves) {
      const int64_t jl = s_long[t / slices];
      const int64_t sl = starts[jl];
      const int ll = lengths[jl];
      const int64_t cl = legacy_cell(geom, n, sl, ll, nb, nd, nh, nw);
      const int b0 = __builtin_amdgcn_readfirstlane(int(sl));
      const int b1 = b0 + __builtin_amdgcn_readfirstlane(ll);
      sum_long_cell<F32, kRowsRun>(x, row_bytes, row_bytes, q0 + 4 * (t % slices), q0 + q, nullptr,
                                   b0, b1, out + cl * row_bytes, s_tile[wave], DepthRows{});
    }
    __syncthreads();
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
  }
}

// The same for rows of fewer than 4 channels: one wave per interval, lane l
// owns channel l, 8 rows at a time.
__global__ __launch_bounds__(kThreads) void legacy_sum_narrow_kernel(
    const float *__restrict__ x, int64_t n, int C, const int32_t *__restrict__ geom,
    const int32_t *__restrict__ starts, const int32_t *__restrict__ lengths, int64_t cap,
    const int32_t *__restrict__ count_dev, int nb, int nd, int nh, int nw,
    float *__restrict__ out, int32_t *__restrict__ meta) {
  constexpr int kU = 8;
  const int64_t n_int = legacy_count(cap, count_dev);
  const int lane = lane_id();
  const int64_t nwaves = (int64_t(gridDim.x) * kThreads) >> 6;
  for (int64_t j = (int64_t(blockIdx.x) * kThreads + threadIdx.x) >> 6; j < n_int; j += nwaves) {
    const int64_t s = starts[j], len = lengths[j];
    const int64_t cell = legacy_cell(geom, n, s, len, nb, nd, nh, nw);
    if (cell < 0) {
      if (meta && lane == 0) atomicAdd(meta + BEVPOOL_META_N_BAD, 1);
      continue;
    }
    const int col = lane < C ? lane : C - 1;  // lanes past C store nothing
    float acc = 0.0f;
    for (int64_t r0 = 0; r0 < len; r0 += kU) {
      float v[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) v[u] = x[(s + (r0 + u < len ? r0 + u : 0)) * C + col];
#pragma unroll
      for (int u = 0; u < kU; ++u)
        if (r0 + u < len) acc += v[u];
    }
    if (lane < C) out[cell * C + lane] = acc;
  }
}

// Longest gap (rows between two intervals) that legacy_spread_kernel writes.
// One wave writes it, so a few very long ones would outlast the launch: 100
// intervals 15,000 rows apart (1.5 M rows of 80 channels) 149 us, 116 with the
// fill; 2,000 intervals 750 rows apart 108, 119 with the fill.
constexpr int64_t kLegacyGap = 4096;

// Sets *unordered unless the intervals lie within the n rows, in order,
// without overlap and without gaps of more than kLegacyGap rows, and there is
// at least one.  Then legacy_spread_kernel writes every row itself (rows
// between the intervals as zeros) and the gradient needs no zero fill before
// it.
__global__ __launch_bounds__(kThreads) void legacy_order_kernel(
    const int32_t *__restrict__ starts, const int32_t *__restrict__ lengths, int64_t cap,
    const int32_t *__restrict__ count_dev, int64_t n, int32_t *__restrict__ unordered) {
  const int64_t n_int = legacy_count(cap, count_dev);
  if (n_int == 0 && blockIdx.x == 0 && threadIdx.x == 0) *unordered = 1;
  bool bad = false;
  for (int64_t j = int64_t(blockIdx.x) * kThreads + threadIdx.x; j < n_int;
       j += int64_t(gridDim.x) * kThreads) {
    const int64_t s = starts[j], len = lengths[j];
    const int64_t next = j + 1 < n_int ? int64_t(starts[j + 1]) : n;
    bad |= s < 0 || len < 0 || s + len > next || next - (s + len) > kLegacyGap;
    if (j == 0) bad |= s > kLegacyGap;
  }
  if (bad) *unordered = 1;  // every writer writes the same
}

// ops/bev_pool/csrc/bev_pool_cuda.cu:61-84: every row of interval j gets the
// gradient row of its cell, x_grad[r, :] = g[cell, :] (g channels last).  One
// wave per interval; V (16-byte pieces at element alignment, or elements for
// rows of fewer than 4 channels) of ng rows per store, non-temporal.
// unordered: null or *unordered != 0: x_grad is zero already and invalid
// intervals are skipped; else the wave also writes its interval's gap up to
// the next one (and up to the first one) as zeros, and an invalid cell's rows.
// The write stream bounds it: 1.54 M rows of 80 channels (494 MB, 500 written) in
// 104 us, 4.8 TB/s where a fill makes 6.9 (and 6 + 3 us for the order check and
// the skipped fill), against 78 us of zero fill and 154 us with 4 bytes per lane.
// Temporal stores took 94 us and the forward that follows 36 us more.
template <bool kWide>
__global__ __launch_bounds__(kThreads) void legacy_spread_kernel(
    const char *__restrict__ g, int64_t n, int C, int qmax, const int32_t *__restrict__ geom,
    const int32_t *__restrict__ starts, const int32_t *__restrict__ lengths, int64_t cap,
    const int32_t *__restrict__ count_dev, int nb, int nd, int nh, int nw,
    char *__restrict__ xg, int32_t *__restrict__ meta, const int32_t *__restrict__ unordered) {
  constexpr int kV = kWide ? 16 : 4;
  const int64_t n_int = legacy_count(cap, count_dev);
  const bool ordered = unordered && *unordered == 0;
  const int lane = lane_id(), wave = int(threadIdx.x) >> 6;
  const int row_bytes = C * 4;
  const int q0 = int(blockIdx.y) * qmax, qt = (row_bytes + kV - 1) / kV;
  const int q = qt - q0 < qmax ? qt - q0 : qmax;
  const int ng = 64 / q, gi = lane / q, li = lane - gi * q;
  const int pb = kV * (q0 + li) < row_bytes - kV ? kV * (q0 + li) : row_bytes - kV;
  const int64_t stride = int64_t(gridDim.x) * kWaves;
  for (int64_t j = int64_t(blockIdx.x) * kWaves + wave; j < n_int; j += stride) {
    const int64_t s = starts[j], len = lengths[j];
    const int64_t cell = legacy_cell(geom, n, s, len, nb, nd, nh, nw);
    if (cell < 0) {
      if (meta && lane == 0 && blockIdx.y == 0) atomicAdd(meta + BEVPOOL_META_N_BAD, 1);
      if (!ordered) continue;
    }
    u32x4 v = u32x4{0u, 0u, 0u, 0u};
    if (cell >= 0) {
      if constexpr (kWide)
        v = reinterpret_cast<const Bytes16 *>(g + cell * row_bytes + pb)->v;
      else
        v.x = *reinterpret_cast<const uint32_t *>(g + cell * row_bytes + pb);
    }
    auto fill = [&](int64_t a, int64_t b, u32x4 w) {
      for (int64_t r = a + gi; r < b; r += ng) {
        char *dst = xg + r * row_bytes + pb;
        if constexpr (kWide)
          __builtin_nontemporal_store(w, reinterpret_cast<u32x4_any *>(dst));
        else
          __builtin_nontemporal_store(uint32_t(w.x), reinterpret_cast<uint32_t *>(dst));
      }
    };
    if (gi < ng) {
      if (ordered && j == 0) fill(0, s, u32x4{0u, 0u, 0u, 0u});
      fill(s, s + len, v);
      if (ordered)
        fill(s + len, j + 1 < n_int ? int64_t(starts[j + 1]) : n, u32x4{0u, 0u, 0u, 0u});
    }
  }
}

// Run boundaries of a rank array (ops/bev_pool/bev_pool_legacy.py:56-61:
// flag[0] = 1, flag[i] = rank[i] != rank[i-1]).  A block takes kRunTile
// consecutive positions, a wave kRunIt batches of 64 of them in order.
constexpr int kRunIt = 4;
constexpr int kRunTile = kThreads * kRunIt;

// The start flags of this wave's batches, as one mask per batch.
template <typename TR>
__device__ __forceinline__ void run_flags(const TR *__restrict__ ranks, int64_t n, int64_t base,
                                          uint64_t (&flags)[kRunIt]) {
  TR r[kRunIt], before[kRunIt];
#pragma unroll
  for (int k = 0; k < kRunIt; ++k) {  // all loads first
    const int64_t i = base + 64 * k + lane_id(), c = i < n ? i : n - 1;
    r[k] = ranks[c];
    before[k] = ranks[c > 0 ? c - 1 : 0];
  }
#pragma unroll
  for (int k = 0; k < kRunIt; ++k) {
    const int64_t i = base + 64 * k + lane_id();
    flags[k] = __ballot(i < n && (i == 0 || r[k] != before[k]));
  }
}

// Per block: the number of run starts.  Block 0 also resets meta.
template <typename TR>
__global__ __launch_bounds__(kThreads) void run_count_kernel(const TR *__restrict__ ranks,
                                                             int64_t n,
                                                             int32_t *__restrict__ bcount,
                                                             int32_t *__restrict__ meta) {
  __shared__ int s_w[kWaves];
  if (blockIdx.x == 0 && threadIdx.x < BEVPOOL_META_LEN)
    meta[threadIdx.x] = threadIdx.x == BEVPOOL_META_FIRST_BAD ? 0x7fffffff : 0;
  const int w = threadIdx.x >> 6;
  uint64_t flags[kRunIt];
  run_flags(ranks, n, int64_t(blockIdx.x) * kRunTile + int64_t(w) * 64 * kRunIt, flags);
  int c = 0;
#pragma unroll
  for (int k = 0; k < kRunIt; ++k) c += __popcll(flags[k]);
  if (lane_id() == 0) s_w[w] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    int s = 0;
    for (int j = 0; j < kWaves; ++j) s += s_w[j];
    bcount[blockIdx.x] = s;
  }
}

// Run starts in order, at the block offsets scanned from run_count_kernel.
template <typename TR>
__global__ __launch_bounds__(kThreads) void run_write_kernel(const TR *__restrict__ ranks,
                                                             int64_t n,
                                                             const int32_t *__restrict__ boff,
                                                             int32_t *__restrict__ starts) {
  __shared__ int s_w[kWaves];
  const int w = threadIdx.x >> 6;
  const int64_t base = int64_t(blockIdx.x) * kRunTile + int64_t(w) * 64 * kRunIt;
  uint64_t flags[kRunIt];
  run_flags(ranks, n, base, flags);
  int c = 0;
#pragma unroll
  for (int k = 0; k < kRunIt; ++k) c += __popcll(flags[k]);
  if (lane_id() == 0) s_w[w] = c;
  __syncthreads();
  int off = boff[blockIdx.x];
  for (int j = 0; j < w; ++j) off += s_w[j];
#pragma unroll
  for (int k = 0; k < kRunIt; ++k) {
    if ((flags[k] >> lane_id()) & 1)
      starts[off + __popcll(flags[k] & lanes_below())] = int(base + 64 * k + lane_id());
    off += __popcll(flags[k]);
  }
}

// lengths[j] = starts[j + 1] - starts[j], the last one n - starts[j]
// (bev_pool_legacy.py:58-61), for the count(meta) runs.
__global__ __launch_bounds__(kThreads) void run_length_kernel(const int32_t *__restrict__ starts,
                                                              int64_t n,
                                                              const int32_t *__restrict__ count,
                                                              int32_t *__restrict__ lengths) {
  const int64_t m = *count;
  const int64_t j = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  if (j < m) lengths[j] = int((j + 1 < m ? int64_t(starts[j + 1]) : n) - starts[j]);
}

// ---------------------------------------------------------------------------
// depth-weighted (fused depth x context) pooling helpers
// ---------------------------------------------------------------------------

// ---- planar (channel-first) <-> rows ---------------------------------------
//
// A planar tensor (BN, C, S) has element (bn, c, s) at bn*sbn + c*sc + s (s
// contiguous): the depth-net context (S = fH*fW) and channel-first camera
// features (S = D*fH*fW, the storage behind the reference's rearrange view,
// depth_lss.py:94).  Point p = bn*S + s.

__device__ __forceinline__ void store16(float *p, u32x4 v) {
  __builtin_nontemporal_store(v, reinterpret_cast<u32x4_any *>(p));
}

// planar -> rows (BN*S, C), fp32, for C >= 4 and S >= 4 of any alignment: a
// block moves kPlanarTile consecutive s of one bn and a block of channels
// (planar_channels) through an LDS tile [s][channel] (<= 66 KB).  Each group of
// kPlanarTile / 4 lanes loads kPlanarTile * 4 contiguous bytes of one channel
// (kPer 16-byte loads per thread, all issued before the tile is written);
// after one barrier the block writes its rows, 16 bytes per thread,
// consecutive threads at consecutive addresses.  Ragged sizes keep to 16-byte
// accesses by overlap: a camera's last tile is shifted back to end at S, a
// row's last piece to end at its last channel; what is moved twice is the
// same.  Non-temporal stores, which are level with ordinary ones: the transpose
// is slower, the accumulation that gathers the rows faster (us, 550 MB of rows at
// 1 x 256 x 256 219 + 128 against 207 + 136, whole passes 538 and 533; 359 MB
// 122 + 81 and 114 + 87, 346 and 341; 159 MB 57 + 43 and 52 + 44, 186 and 181;
// 200 MB of 64 channels 72 + 49 and 70 + 54, 231 and 236).  With `rank`, rows of
// dropped points (rank -1), which nothing reads, are not written.
// HBM traffic bounds it (1.28 GB at 1 x 360 x 360: 235 us; 64-point tiles 6 us
// more, a register transpose whose stores scatter 16-byte pieces 288 us).
// Without the dropped points' rows, 14% of them at 1 x 256 x 256, it takes 219
// us, and with four height bins, where 46% are dropped, 183 us.  Maps that 4
// does not divide (2 x 6 x 45 x 29 x 51 points, C = 64): 80 us, 244 one element
// per thread (and the planar gradient 42 us, 155).
constexpr int kPlanarTile = 128;
template <int kPer>
__global__ __launch_bounds__(kThreads) void planar_tile_kernel(
    const float *__restrict__ src, int C, int cmax, int64_t S, int64_t tiles_s, int64_t sbn,
    int64_t sc, const int32_t *__restrict__ rank, float *__restrict__ rows) {
  constexpr int kQ = kPlanarTile / 4;  // 16-byte pieces per channel of a tile
  extern __shared__ float tile[];  // [kPlanarTile][cb + 1]
  __shared__ int s_rank[kPlanarTile];
  const int tid = threadIdx.x;
  const int c0 = first_channel(C, 4, int(blockIdx.y) * cmax);
  const int cb = C - c0 < cmax ? C - c0 : cmax;
  const int pitch = cb + 1;
  const int64_t bn = int64_t(blockIdx.x) / tiles_s;
  const int np = S < kPlanarTile ? int(S) : kPlanarTile;
  int64_t s0 = (int64_t(blockIdx.x) - bn * tiles_s) * kPlanarTile;
  s0 = s0 < S - np ? s0 : S - np;
  const float *in = src + bn * sbn + int64_t(c0) * sc + s0;
  u32x4 v[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    // piece e: channel e / kQ, points 4 (e % kQ) + [0, 4), or the last 4;
    // pieces past the channels reload the last one and are not written
    const int e = tid + kThreads * i;
    const int c = e / kQ < cb ? e / kQ : cb - 1;
    const int p = 4 * (e % kQ) < np - 4 ? 4 * (e % kQ) : np - 4;
    v[i] = reinterpret_cast<const Bytes16 *>(in + int64_t(c) * sc + p)->v;
  }
  if (rank && tid < np) s_rank[tid] = rank[bn * S + s0 + tid];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int e = tid + kThreads * i;
    const int c = e / kQ, p = 4 * (e % kQ) < np - 4 ? 4 * (e % kQ) : np - 4;
    if (c < cb) {
      float *t = tile + p * pitch + c;
      t[0] = __uint_as_float(v[i].x);
      t[pitch] = __uint_as_float(v[i].y);
      t[2 * pitch] = __uint_as_float(v[i].z);
      t[3 * pitch] = __uint_as_float(v[i].w);
    }
  }
  __syncthreads();
  const int q = (cb + 3) >> 2, n = np * q;
  float *out = rows + (bn * S + s0) * C + c0;
  for (int e = tid; e < n; e += kThreads) {
    const int p = e / q;  // row p, its piece e % q
    const int c = 4 * (e - p * q) < cb - 4 ? 4 * (e - p * q) : cb - 4;
    if (rank && s_rank[p] < 0) continue;
    const float *t = tile + p * pitch + c;
    store16(out + int64_t(p) * C + c, u32x4{__float_as_uint(t[0]), __float_as_uint(t[1]),
                                            __float_as_uint(t[2]), __float_as_uint(t[3])});
  }
}

// The same one element per thread, for fewer than 4 channels or few points.
__global__ __launch_bounds__(kThreads) void planar_rows_kernel(
    const float *__restrict__ src, int C, int64_t S, int64_t n_rows, int64_t sbn, int64_t sc,
    float *__restrict__ rows) {
  const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  if (i >= n_rows * C) return;
  const int64_t r = i / C;
  const int c = int(i - r * C);
  const int64_t bn = r / S, sp = r - bn * S;
  rows[i] = src[bn * sbn + int64_t(c) * sc + sp];
}

// Backward of the op-level pooling into a planar gradient:
// x_grad[bn, c, s] = g[rank[bn*S + s], c] (0 for dropped points), g the
// cell-major rows of bev_to_rows_kernel.  Vector form (C >= 4, S >= 4, any
// alignment; what does not divide by 4 overlaps as in planar_tile_kernel): a
// thread takes 4 consecutive points of one bn and walks the channels 4 at a
// time, kIt such groups in flight: four 16-byte row loads (cache-resident
// rows), a register transpose, four 16-byte stores along s (a wave writes 1 KB
// contiguous per channel).  Blocks map XCD-contiguously.  The write stream
// bounds it: 638 MB at 1 x 360 x 360 in 130-140 us.  Aligned stores are
// non-temporal (kStream; temporal ones took 148 us there and the next forward
// 50 more, and gained nothing over whole steps on new inputs where the
// memory-side cache holds the gradient); stores at other addresses are
// temporal, so that the caches merge the lines that two of them share.
template <bool kVec, bool kStream>
__global__ __launch_bounds__(kThreads) void gather_planar_kernel(
    const float *__restrict__ g, int C, const int32_t *__restrict__ rank, int64_t n_points,
    int64_t S, FastDiv groups, int64_t n_groups, int64_t sbn, int64_t sc,
    float *__restrict__ x_grad) {
  if constexpr (kVec) {
    constexpr int kIt = 2;
    const int64_t gi = xcd_chunk(blockIdx.x, gridDim.x) * kThreads + threadIdx.x;
    if (gi >= n_groups) return;
    // groups of 4 points per bn, the last one shifted back to end at S
    const uint32_t bn = groups.div(uint32_t(gi));
    int64_t sp = 4 * int64_t(uint32_t(gi) - bn * groups.d);
    sp = sp < S - 4 ? sp : S - 4;
    const u32x4 rk = reinterpret_cast<const Bytes16 *>(rank + bn * S + sp)->v;
    const int r0 = int(rk.x), r1 = int(rk.y), r2 = int(rk.z), r3 = int(rk.w);
    const float *g0 = g + int64_t(r0 >= 0 ? r0 : 0) * C;
    const float *g1 = g + int64_t(r1 >= 0 ? r1 : 0) * C;
    const float *g2 = g + int64_t(r2 >= 0 ? r2 : 0) * C;
    const float *g3 = g + int64_t(r3 >= 0 ? r3 : 0) * C;
    const uint32_t m0 = r0 >= 0 ? 0xFFFFFFFFu : 0u, m1 = r1 >= 0 ? 0xFFFFFFFFu : 0u;
    const uint32_t m2 = r2 >= 0 ? 0xFFFFFFFFu : 0u, m3 = r3 >= 0 ? 0xFFFFFFFFu : 0u;
    float *out = x_grad + int64_t(bn) * sbn + sp;
    auto put = [](float *p, u32x4 v) {
      if constexpr (kStream)
        store16(p, v);
      else
        reinterpret_cast<Bytes16 *>(p)->v = v;
    };
    auto piece = [](const float *p) { return reinterpret_cast<const Bytes16 *>(p)->v; };
    for (int cb = 0; cb < C; cb += 4 * kIt) {
      u32x4 a[kIt][4];
#pragma unroll
      for (int i = 0; i < kIt; ++i) {  // every row piece of kIt groups, then the stores
        const int c = cb + 4 * i < C - 4 ? cb + 4 * i : C - 4;
        a[i][0] = piece(g0 + c) & m0;
        a[i][1] = piece(g1 + c) & m1;
        a[i][2] = piece(g2 + c) & m2;
        a[i][3] = piece(g3 + c) & m3;
      }
#pragma unroll
      for (int i = 0; i < kIt; ++i) {
        if (cb + 4 * i < C) {
          float *o = out + int64_t(cb + 4 * i < C - 4 ? cb + 4 * i : C - 4) * sc;
          put(o, u32x4{a[i][0].x, a[i][1].x, a[i][2].x, a[i][3].x});
          put(o + sc, u32x4{a[i][0].y, a[i][1].y, a[i][2].y, a[i][3].y});
          put(o + 2 * sc, u32x4{a[i][0].z, a[i][1].z, a[i][2].z, a[i][3].z});
          put(o + 3 * sc, u32x4{a[i][0].w, a[i][1].w, a[i][2].w, a[i][3].w});
        }
      }
    }
  } else {
    const int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= n_points * C) return;
    const int c = int(i / n_points);
    const int64_t p = i - int64_t(c) * n_points;
    const int r = rank[p];
    const int64_t bn = p / S, sp = p - bn * S;
    x_grad[bn * sbn + int64_t(c) * sc + sp] = r >= 0 ? g[int64_t(r) * C + c] : 0.0f;
  }
}

// Sum over the 16 lanes of a DPP row (lanes 16r..16r+15) in a fixed order:
// xor 1, xor 2 (quad permutes), then the half-row and row mirrors.  Each
// step adds two equal-order partial sums, so every lane of the row ends with
// the same value.
__device__ __forceinline__ float row_sum16(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                                             0xB1, 0xF, 0xF, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                                             0x4E, 0xF, 0xF, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                                             0x141, 0xF, 0xF, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                                             0x140, 0xF, 0xF, false));
  return v;
}

constexpr int kDgPix = 16;  // pixels per depth_grad block (4 per wave)

// Backward of out[cell] = sum_{p in cell} depth[p] * ctx[pix(p)] (the
// reference's autograd through depth_lss.py:91-94 and the pooling):
//   grad_depth[p]        = sum_c g[rank[p], c] * ctx[pix(p), c]  (0 if dropped)
//   grad_ctx[bn, c, hw]  = sum_d g[rank[p_d], c] * depth[p_d]
// with p_d = (bn*D + d)*HW + hw.
// A block takes a patch of kDgPix pixels: 4 rows of 4 columns of the image
// (pw = 4), or 16 in a row (pw = 16, fH = 1) where patches do not fit.  Their ranks and depths are staged in LDS ([d][pixel]); each wave
// then takes 4 pixels, one per 16-lane row of the wave: of a 4 x 4 patch a
// column of 4, which lie above each other and so, bin by bin, mostly hit one
// cell: the wave's four row loads are then one row's lines.  Lane j of a row
// holds channels 64 q + 4 j + 0..3 (q < kX = C / 64, one 16-byte load each) and
// 64 kX + 16 k + j (k < kR, the rest).  Per bin a row gathers its cell's
// gradient row, reduces the dot product with row_sum16 and adds depth * row to
// its context sums, bins d = 4 i + u in chain u; the chains are added in order
// at the end.  The dot products replace the ranks in LDS and, like the context
// sums, are written out from there.  g: cell-major fp32 rows of the occupied
// cells; ctx: channel-last rows (planar_tile_kernel).  Blocks map
// XCD-contiguously, so the cells of neighbouring pixels' rays meet in one L2.
// Vector instructions bound it: at 4 x 360 x 360, C = 80, 162 us, a SIMD issues
// 98 K of them (50 per bin and wave), 4 clocks each, with 5.9 waves resident; L2
// takes 80 G requests/s, 73% hits.  One bin per row of the wave and 4-byte loads
// took 216 us, 16-byte loads 184, the columns 162.
template <int kX, int kR>
__global__ __launch_bounds__(kThreads) void depth_grad_kernel(
    const float *__restrict__ g, int C, const int32_t *__restrict__ rank,
    const float *__restrict__ depth, const float *__restrict__ ctx, int D, int fH, int fW, int pw,
    int h_tiles, int w_tiles, int64_t n_tiles, uint32_t *__restrict__ grad_depth,
    float *__restrict__ grad_ctx, int64_t gsbn, int64_t gsc) {
  constexpr int kK = 4 * kX + kR;
  constexpr int kU = 4;  // bins in flight (2, 3, 6, 8: 210, 194, 183, 198 against 184 us)
  extern __shared__ int dg_smem[];
  int *lr = dg_smem;                                             // [D][kDgPix]
  float *ldp = reinterpret_cast<float *>(dg_smem + D * kDgPix);  // [D][kDgPix]
  float *lgc = ldp + D * kDgPix;                                 // [C][kDgPix]
  const int tid = threadIdx.x;
  const int64_t tile = xcd_chunk(blockIdx.x, gridDim.x);
  if (tile >= n_tiles) return;  // XCD padding blocks
  const int64_t bn = tile / (h_tiles * w_tiles);
  const int tr = int(tile - bn * (h_tiles * w_tiles));
  const int h0 = tr / w_tiles * (kDgPix / pw), w0 = tr % w_tiles * pw;
  const int64_t plane = int64_t(fH) * fW;
  // pixel t of the patch
  auto pixel = [&](int t, int &h, int &w) {
    h = h0 + t / pw;
    w = w0 + t % pw;
    return h < fH && w < fW;
  };
  {
    int h, w;  // kThreads is a multiple of kDgPix: a thread stays with one pixel
    const bool ok = pixel(tid % kDgPix, h, w);
    const int64_t p0 = bn * D * plane + int64_t(h) * fW + w;
    for (int i = tid; i < D * kDgPix; i += kThreads) {
      const int64_t p = p0 + (i / kDgPix) * plane;
      lr[i] = ok ? rank[p] : -1;
      ldp[i] = ok ? depth[p] : 0.0f;
    }
  }
  __syncthreads();
  const int lane = lane_id(), j = lane & 15;
  const int t = (lane >> 4) * 4 + (tid >> 6);  // this row's pixel
  // channels past C (possible in the last of the single ones only) are read
  // clamped and masked
  const int c1 = 64 * kX + 16 * (kR - 1) + j;
  const bool last_ok = kR == 0 || c1 < C;
  const int c1c = last_ok ? c1 : C - 1;
  // a row's values for this lane, as raw bits
  auto load_row = [&](const uint32_t *row, uint32_t(&v)[kK]) {
#pragma unroll
    for (int q = 0; q < kX; ++q) {
      const u32x4 p = reinterpret_cast<const Bytes16 *>(row + 64 * q + 4 * j)->v;
      v[4 * q] = p.x;
      v[4 * q + 1] = p.y;
      v[4 * q + 2] = p.z;
      v[4 * q + 3] = p.w;
    }
#pragma unroll
    for (int k = 0; k < kR; ++k)
      v[4 * kX + k] = row[k + 1 < kR ? 64 * kX + 16 * k + j : c1c];
  };
  float xc[kK], gc[kU][kK];
  {
    int h, w;
    const bool ok = pixel(t, h, w);
    const int64_t pix = ok ? bn * plane + int64_t(h) * fW + w : 0;
    uint32_t v[kK];
    load_row(reinterpret_cast<const uint32_t *>(ctx + pix * C), v);
#pragma unroll
    for (int k = 0; k < kK; ++k) {
      xc[k] = kR > 0 && k == kK - 1 && !last_ok ? 0.0f : __uint_as_float(v[k]);
#pragma unroll
      for (int u = 0; u < kU; ++u) gc[u][k] = 0.0f;
    }
  }
  const uint32_t *gb = reinterpret_cast<const uint32_t *>(g);
  for (int d0 = 0; d0 < D; d0 += kU) {
    int rr[kU];
    float dp[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int d = d0 + u, dc = d < D ? d : D - 1;
      const int r = lr[dc * kDgPix + t];
      const float w = ldp[dc * kDgPix + t];
      rr[u] = d < D ? r : -1;
      dp[u] = d < D ? w : 0.0f;
    }
    // every load is issued (clamped rows/columns) and masked by a bitwise
    // AND afterwards: a select would let the compiler sink each load into
    // a branch of its own and wait for it there
    float gv[kU][kK];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      uint32_t v[kK];
      load_row(gb + int64_t(rr[u] >= 0 ? rr[u] : 0) * C, v);
      const uint32_t m = rr[u] >= 0 ? 0xFFFFFFFFu : 0u, ml = last_ok ? m : 0u;
#pragma unroll
      for (int k = 0; k < kK; ++k)
        gv[u][k] = __uint_as_float(v[k] & (kR > 0 && k == kK - 1 ? ml : m));
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      float part = 0.0f;
#pragma unroll
      for (int k = 0; k < kK; ++k) part += gv[u][k] * xc[k];
      const float dot = row_sum16(part);
      if (j == 0 && d0 + u < D)
        lr[(d0 + u) * kDgPix + t] = __builtin_bit_cast(int, rr[u] >= 0 ? dot : 0.0f);
#pragma unroll
      for (int k = 0; k < kK; ++k) gc[u][k] += gv[u][k] * dp[u];
    }
  }
#pragma unroll
  for (int k = 0; k < kK; ++k) {
    const float tot = ((gc[0][k] + gc[1][k]) + gc[2][k]) + gc[3][k];
    const int c = k < 4 * kX ? 64 * (k >> 2) + 4 * j + (k & 3) : 64 * kX + 16 * (k - 4 * kX) + j;
    if (c < C) lgc[c * kDgPix + t] = tot;
  }
  __syncthreads();
  {
    int h, w;
    if (!pixel(tid % kDgPix, h, w)) return;
    const int64_t hw = int64_t(h) * fW + w;
    for (int i = tid; i < D * kDgPix; i += kThreads)
      grad_depth[(bn * D + i / kDgPix) * plane + hw] = uint32_t(lr[i]);
    for (int i = tid; i < C * kDgPix; i += kThreads)
      grad_ctx[bn * gsbn + int64_t(i / kDgPix) * gsc + hw] = lgc[i];
  }
}

// ---------------------------------------------------------------------------
// host helpers
// ---------------------------------------------------------------------------
inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
inline size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

// LSD passes of at most kMaxDigitBits bits each; or, for ranks of 11..20
// bits (local_bits > 0), one global pass by the high digit (shift[0] =
// local_bits) and bucket_sort_kernel for the low local_bits bits.
#ifndef BEVPOOL_BUCKET_SORT
#define BEVPOOL_BUCKET_SORT 1
#endif
// Per-group sort: a group of more than kBucketPartKeys keys is ranked by up to
// kBucketParts blocks.  Each part's block also counts the rest of its group,
// so more parts cost more counting: at 1 x 360 x 360 the per-group sort took
// 21.6 us with one block per group, 19.0 with 2 parts above 8192 keys, 20.0
// with 4, 20.7 with 4 above 6144 keys and 22.6 with 4 above 4096 (MI355X).
#ifndef BEVPOOL_BUCKET_PARTS
#define BEVPOOL_BUCKET_PARTS 2
#endif
#ifndef BEVPOOL_BUCKET_PART_KEYS
#define BEVPOOL_BUCKET_PART_KEYS 8192
#endif
constexpr int kBucketParts = BEVPOOL_BUCKET_PARTS;
constexpr int kBucketPartKeys = BEVPOOL_BUCKET_PART_KEYS;
struct DigitPlan {
  int passes = 1;
  int bits[4] = {1, 0, 0, 0};
  int shift[4] = {0, 0, 0, 0};
  int local_bits = 0;
};

DigitPlan plan_digits(int64_t n_cells) {
  int total_bits = 0;
  for (uint64_t v = uint64_t(n_cells > 1 ? n_cells - 1 : 0); v; v >>= 1) ++total_bits;
  if (total_bits < 1) total_bits = 1;
  DigitPlan p;
  if (BEVPOOL_BUCKET_SORT && total_bits > kMaxDigitBits && total_bits <= 2 * kMaxDigitBits) {
    p.bits[0] = (total_bits + 1) / 2;  // high digit: global pass
    // Narrower groups shorten the per-group sort, whose largest group sets
    // its length; tile histograms of up to 2^9 digits cost the global pass
    // no more than 2^8, 2^10 cost it ~5 us at 1 x 360 x 360 (MI355X).  So a
    // 16-bit rank space takes 9 + 7 bits (256 x 256: per-group sort 25.0 ->
    // 16.9 us), while 17 bits keep 9 + 8.
    if (total_bits - p.bits[0] > 7 && p.bits[0] < 9)
      p.bits[0] = total_bits - 7 < 9 ? total_bits - 7 : 9;
    p.local_bits = total_bits - p.bits[0];
    p.shift[0] = p.local_bits;
    return p;
  }
  p.passes = int((total_bits + kMaxDigitBits - 1) / kMaxDigitBits);
  const int per = (total_bits + p.passes - 1) / p.passes;
  int shift = 0;
  for (int i = 0; i < p.passes; ++i) {
    p.shift[i] = shift;
    p.bits[i] = total_bits - shift < per ? total_bits - shift : per;
    shift += p.bits[i];
  }
  return p;
}

struct IndexLayout {
  size_t keys_tmp, hist, totals, gstart, bcount, tile_bad, slices, total;
  int64_t sort_blocks, cell_blocks;
  int items;  // keys per thread of the tile kernels (sort_items)
};

// Slices of the sliced bucket sort (an upper bound: every group may end in a
// partial slice) and the bytes of their low-digit counts.
int64_t slice_bound(int64_t n_points, int64_t n_cells, int lbits) {
  return ceil_div(n_cells, int64_t(1) << lbits) + ceil_div(n_points, int64_t(kSliceKeys));
}

size_t slice_count_bytes(int64_t n_points, int64_t n_cells) {
  const DigitPlan plan = plan_digits(n_cells);
  if (plan.local_bits < kSlicedBits) return 0;
  return size_t(slice_bound(n_points, n_cells, plan.local_bits)) << plan.local_bits << 2;
}

// Index-stage workspace.  The slice counts at the end depend on n_cells; a
// caller that only uses the other regions may pass n_cells = 1.
IndexLayout index_layout(int64_t n_points, int64_t n_cells) {
  IndexLayout L;
  L.items = sort_items(n_points);
  L.sort_blocks = ceil_div(n_points, int64_t(kThreads) * L.items);
  L.cell_blocks = ceil_div(n_points, kThreads);
  size_t o = 0;
  L.keys_tmp = o;
  o = align256(o + size_t(n_points) * sizeof(uint64_t));
  L.hist = o;
  o = align256(o + size_t(kMaxRadix) * size_t(L.sort_blocks) * sizeof(int32_t));
  L.totals = o;
  o = align256(o + size_t(kMaxRadix) * sizeof(int32_t));
  L.gstart = o;  // start of each group of the global pass (per-group sort)
  o = align256(o + size_t(kMaxRadix) * sizeof(int32_t));
  L.bcount = o;
  o = align256(o + size_t(L.cell_blocks) * sizeof(int32_t));
  L.tile_bad = o;  // op level: invalid-rank count and first index per tile
  o = align256(o + size_t(2) * size_t(L.sort_blocks) * sizeof(int32_t));
  L.slices = o;
  o = align256(o + slice_count_bytes(n_points, n_cells));
  L.total = o;
  return L;
}

template <typename P>
P *at(void *base, size_t off) {
  return reinterpret_cast<P *>(static_cast<char *>(base) + off);
}

int check_index_args(int64_t n_points, int64_t n_cells, const void *rank, const void *meta,
                     void *ws, size_t ws_bytes) {
  if (n_points < 0 || n_points > int64_t(INT32_MAX))
    return fail(BEVPOOL_EINVAL, "n_points=%lld out of range [0, 2^31)", (long long)n_points);
  if (n_cells < 1 || n_cells > int64_t(INT32_MAX))
    return fail(BEVPOOL_EINVAL, "B*D*H*W=%lld out of range [1, 2^31)", (long long)n_cells);
  if (!meta || !ws) return fail(BEVPOOL_EINVAL, "null meta or workspace");
  if (n_points > 0 && !rank) return fail(BEVPOOL_EINVAL, "null rank");
  const size_t need = index_layout(n_points, n_cells).total;
  if (ws_bytes < need)
    return fail(BEVPOOL_ESPACE, "index workspace %zu bytes < required %zu", ws_bytes, need);
  return BEVPOOL_OK;
}

size_t dtype_size(int32_t dtype) { return dtype == BEVPOOL_F32 ? 4 : 2; }

// 4 consecutive cells of one channel of a channel-first tensor form one
// aligned 4-element vector when n_xy and the b/c/z strides are multiples of
// 4 and the base is aligned to 4 elements (tiles start at multiples of 64).
bool bev_vec_ok(const void *base, size_t es, int64_t n_xy, int64_t sb, int64_t sc,
                int64_t sz) {
  return n_xy % 4 == 0 && sb % 4 == 0 && sc % 4 == 0 && sz % 4 == 0 &&
         reinterpret_cast<uintptr_t>(base) % (4 * es) == 0;
}

template <typename T, int kCPL>
int launch_accum_pipe_t(int slots, unsigned grid, size_t smem, hipStream_t s, const char *x,
                        int64_t ld_bytes, int C, const uint64_t *keys, const int32_t *meta,
                        const int32_t *cend, float *acc, bool stream_rows) {
#define BEVPOOL_PIPE_CASE(K)                                                                   \
  case K:                                                                                      \
    if (stream_rows)                                                                           \
      hipLaunchKernelGGL((accum_pipe_kernel<T, K, kCPL, kRowsStream>), dim3(grid),             \
                         dim3(kPipeThreads), smem, s, x, ld_bytes, C, keys, meta, cend, acc,   \
                         kRangePoints);                                                        \
    else                                                                                       \
      hipLaunchKernelGGL((accum_pipe_kernel<T, K, kCPL, kRowsPlain>), dim3(grid),              \
                         dim3(kPipeThreads), smem, s, x, ld_bytes, C, keys, meta, cend, acc,   \
                         kRangePoints);                                                        \
    break;
  switch (slots) {
    BEVPOOL_PIPE_CASE(1)
    BEVPOOL_PIPE_CASE(2)
    BEVPOOL_PIPE_CASE(3)
    BEVPOOL_PIPE_CASE(4)
    BEVPOOL_PIPE_CASE(5)
    BEVPOOL_PIPE_CASE(6)
    default:
      return fail(BEVPOOL_EINVAL, "internal: %d slots per thread", slots);
  }
#undef BEVPOOL_PIPE_CASE
  return check_launch("accum_pipe");
}

// Widest row of the pipelined accumulation: 6 16-byte slots per loader thread
// and stage, two stages and their ranks in 24.3 KB of LDS.  Wider rows took
// it several passes; the grouped kernel takes them in one (128 fp32 channels
// at 1 x 360 x 360: 215 -> 189 us).
constexpr int kPipeRowBytes = 384;

// Pipelined forward accumulation into cell-major rows, for rows of at most
// kPipeRowBytes that are runs of aligned 16-byte pieces.
int launch_accum_pipe(int32_t dtype, const char *x, int64_t ld_bytes, int C, int64_t n_points,
                      const uint64_t *keys, const int32_t *meta, const int32_t *cend, float *acc,
                      bool stream_rows, hipStream_t s) {
  const size_t es = dtype_size(dtype);
  // plain block order: ranges that run at the same time then read rows from
  // one window of the feature tensor (an XCD-contiguous order measured slower)
  const unsigned grid = unsigned(ceil_div(n_points, kRangePoints));
  const int rowq = int(size_t(C) * es / 16);
  const int slots = (kStageRows * rowq + kLoaders - 1) / kLoaders;
  const size_t smem = size_t(2) * kStageRows * rowq * 16 + size_t(2) * kStageRows * sizeof(int);
  // channels (pairs with 16-bit rows) per lane of a summing wave
  const int lanes = es == 4 ? C : (C + 1) / 2;
  const bool wide = (lanes + kSummers - 1) / kSummers > 64;
#define BEVPOOL_PIPE_DTYPE(T)                                                                  \
  return wide ? launch_accum_pipe_t<T, 2>(slots, grid, smem, s, x, ld_bytes, C, keys, meta,    \
                                          cend, acc, stream_rows)                              \
              : launch_accum_pipe_t<T, 1>(slots, grid, smem, s, x, ld_bytes, C, keys, meta,    \
                                          cend, acc, stream_rows);
  switch (dtype) {
    case BEVPOOL_F32:
      BEVPOOL_PIPE_DTYPE(F32)
    case BEVPOOL_F16:
      BEVPOOL_PIPE_DTYPE(F16)
    default:
      BEVPOOL_PIPE_DTYPE(BF16)
  }
#undef BEVPOOL_PIPE_DTYPE
}

// Shape of a grouped accumulation (accum_group_kernel) of n_points rows.
struct GroupPlan {
  int qmax, nblk;   // 16-byte pieces per channel block, channel blocks
  int kk, ng;       // points per batch and groups per wave
  int P, lcell;     // nominal points per group, points of a long cell (P < lcell)
  int long_parts, long_sets, long_lanes;  // blocks of the long cells
  int64_t waves64;  // waves at 64 points per group
  bool small;       // faster than accum_pipe_kernel where that takes the rows
};

// Points per group: 16 where 64 would leave the chip without waves, since a
// group's chain of loads is the whole kernel there (MI355X: 31 K points, C = 80,
// 11-13 us with 16 points a group, 14-15 with 64; 467 K, C = 20, 14 against 22).
// Batches of fewer than 16 points make the chain longer, and on sparse grids few
// cells are long at 16 points a group, hence three lines (170 K points, C = 52: on
// 393 x 393 cells 12-13 us with 16, 15-16 with 64, on 128 x 128 17 and 16; C = 80,
// 885 waves of 64: on 128 x 128 20-21 and 16-17, on 360 x 360 16-17 and 14-15).
//
// Points per batch: as many as the groups' LDS entries hold.  Context rows of 4
// to 7 pieces would leave 9 to 16 groups 4 rows each; with enough waves fewer
// groups of 8 are faster (2 M points, C = 16, 51 -> 36 us, accum_pipe_kernel 48;
// C = 24 48 -> 41, 51), of 16 on grids with few points a cell (2.35 M on 7 x
// 330 x 330, C = 24, 74, 66 and 54 us with 4, 8 and 16, accum_pipe_kernel 60).
//
// Points of a long cell: a group's chain of lcell / kk round trips must not
// outlast the rest of the launch (lcell <= kk * waves64 / 96: 0.75 us per round
// trip against the time that the rows of all waves take), but the groups move
// rows faster than the long cells' waves do, so cells that are ordinary for the
// grid, up to 6 times its mean (kk / 4 times at kk = 4 and 8: 25.5 M points, C =
// 28, 268 a cell, 457 us, 485 with 3 times), stay with them; cells of fewer than
// 64 to 256 points always do.  Depth-weighted forwards of 6 cameras, C = 80, us
// with 256 for every grid, with this rule and with accum_pipe_kernel: 64 x 176 x
// 118 points on 360 x 360 cells 302, 273, 309; on 128 x 128 772, 355, 532; on
// 90 x 90 861, 487, 647; 32 x 88 x 118 on 90 x 90 190, 117, 167.
//
// Blocks of the long cells: about kLongBlocks, so that the candidates are
// spread over the chip (60 K points in cells of 100: 45 us with 16 candidates
// a block, 20 so), up to kLongLanes candidates for each part where more blocks
// would only wait for their keys to learn that they have nothing to do (7.1 M
// points on 4 x 360 x 360: 192 us with 16, 189 with 32).
//
// Aligned rows of at most kPipeRowBytes: from 4 waves per CU on (C = 80: 197 K
// points) the pipelined blocks are as fast or faster (25 against 25-31 us at 249
// K points, 131 against 147 at 2 M), below them the groups' shorter chain is:
// 23.5 -> 21-22.5 us at 188 K points, C = 80, 22 -> 18 at 121 K, 23 -> 10-12 at
// 31 K and 18 -> 11 at C = 16.
constexpr int64_t kGroupFewWaves = 2 * 256, kPipeWaves = 4 * 256, kGroupManyWaves = 16 * 256;
constexpr int kLongBlocks = 384, kLongLanes = 16;

GroupPlan group_plan(int32_t dtype, int C, int64_t n_points, int64_t n_cells, bool depth_rows) {
  GroupPlan g;
  const int qt = int((size_t(C) * dtype_size(dtype) + 15) / 16);
  g.nblk = (qt + 63) / 64;
  g.qmax = (qt + g.nblk - 1) / g.nblk;
  const int per = 64 / g.qmax;  // groups a wave's lanes allow
  g.kk = per <= 4 ? 16 : (per <= 8 ? 8 : 4);
  g.ng = per < 64 / g.kk ? per : 64 / g.kk;
  g.waves64 = ceil_div(ceil_div(n_points, int64_t(64)), int64_t(g.ng));
  const bool sparse = n_points < n_cells + n_cells / 4;
  const int few_halves = g.kk == 16 ? (sparse ? 3 : 2) : 4;
  const bool few = g.waves64 < few_halves * (kGroupFewWaves / 2);
  if (depth_rows && g.kk == 4 && g.qmax >= 4 && !few) {
    g.kk = n_points < 8 * n_cells ? 16 : 8;
    g.ng = 64 / g.kk;
    g.waves64 = ceil_div(ceil_div(n_points, int64_t(64)), int64_t(g.ng));
  }
  g.small = g.waves64 < kPipeWaves;
  g.P = few ? 16 : 64;
  const int64_t least = few ? 64 : (g.waves64 < kGroupManyWaves ? 128 : 256);
  const int64_t mean = (g.kk == 16 ? 6 : g.kk / 4) * n_points / n_cells;
  const int64_t chain = g.kk * g.waves64 / 96;
  const int64_t lcell = mean < chain ? mean : chain;
  g.lcell = int(lcell > least ? lcell : least);
  g.long_parts = int(ceil_div(g.qmax, kLongPieces));
  const int64_t candidates = ceil_div(n_points, int64_t(g.lcell));
  const int64_t lanes = ceil_div(candidates * g.long_parts, int64_t(kLongBlocks));
  const int64_t most = kLongLanes * g.long_parts;  // <= 64 lanes
  g.long_lanes = int(lanes < most ? lanes : most);
  g.long_sets = int(ceil_div(candidates, int64_t(g.long_lanes)));
  return g;
}

// Grouped forward accumulation into cell-major rows (rows of 16 bytes or
// more, any element alignment).  dr.depth: context rows, else feature rows.
int launch_accum_group(int32_t dtype, const GroupPlan &g, const char *x, int64_t ld_bytes, int C,
                       int64_t n_points, const uint64_t *keys, const int32_t *meta,
                       const int32_t *cstart, const int32_t *cend, void *acc, const DepthRows &dr,
                       bool stream_rows, hipStream_t s) {
  const int long_blocks = g.long_sets * g.long_parts;
  const int64_t waves = ceil_div(ceil_div(n_points, int64_t(g.P)), int64_t(g.ng));
  const int64_t blocks = long_blocks + ceil_div(waves, kWaves);
  if (int st = check_grid(blocks, kThreads, "accum_group")) return st;
  const dim3 grid{unsigned(blocks), unsigned(g.nblk), 1};
#define BEVPOOL_AG(T, K, M)                                                                    \
  hipLaunchKernelGGL((accum_group_kernel<T, K, M>), grid, dim3(kThreads), 0, s, x, ld_bytes, C, \
                     g.qmax, keys, meta, cstart, cend, static_cast<char *>(acc), g.P, g.lcell, \
                     long_blocks, g.long_sets, g.long_lanes, dr)
#define BEVPOOL_AG_K(T, M)                                                                     \
  {                                                                                            \
    if (g.kk == 16) BEVPOOL_AG(T, 16, M);                                                     \
    else if (g.kk == 8) BEVPOOL_AG(T, 8, M);                                                  \
    else BEVPOOL_AG(T, 4, M);                                                                 \
  }
#define BEVPOOL_AG_T(T)                                                                        \
  {                                                                                            \
    if (stream_rows) BEVPOOL_AG_K(T, kRowsStream) else BEVPOOL_AG_K(T, kRowsPlain)            \
  }
  if (dr.depth) BEVPOOL_AG_K(F32, kRowsDepth)
  else if (dtype == BEVPOOL_F32) BEVPOOL_AG_T(F32)
  else if (dtype == BEVPOOL_F16) BEVPOOL_AG_T(F16)
  else BEVPOOL_AG_T(BF16)
#undef BEVPOOL_AG_T
#undef BEVPOOL_AG_K
#undef BEVPOOL_AG
  return check_launch("accum_group");
}

// cell-major fp32 rows -> channel-first output (zeros for empty cells).
int launch_rows_to_bev(const float *acc, int32_t dtype, int C, const int32_t *cell_end,
                       int64_t n_cells, int n_z, int64_t n_xy, int64_t out_stride_b,
                       int64_t out_stride_c, int64_t out_stride_z, void *out,
                       hipStream_t s, MetaReport report = {}, bool raw16 = false) {
  if (int st = check_grid(ceil_div(n_cells, kCellTile), kThreads, "cell tiles")) return st;
  const unsigned tiles = unsigned(ceil_div(n_cells, kCellTile));
  const int CT = tile_channels(C);
  const size_t es = dtype_size(dtype);
  const size_t smem = size_t(kCellTile) * size_t(CT + 1) * sizeof(uint32_t);
  if (raw16 && es != 2) return fail(BEVPOOL_EINVAL, "internal: 16-bit rows for a 32-bit output");
  // 16-byte row pieces: 4 fp32 or 8 16-bit channels
  const bool vrow = C >= (raw16 ? 8 : 4);
  const bool vbev = bev_vec_ok(out, es, n_xy, out_stride_b, out_stride_c, out_stride_z);
  const CellMap cells{make_fast_div(uint32_t(n_xy)), make_fast_div(uint32_t(n_z)), out_stride_b,
                      out_stride_z};
  LaunchTimer t("rows_to_bev", s);
#define BEVPOOL_R2B(T, VR, VB, R16)                                                            \
  hipLaunchKernelGGL((rows_to_bev_kernel<T, VR, VB, R16>), dim3(tiles), dim3(kThreads), smem,  \
                     s, acc, C, CT, cell_end, n_cells, cells, out_stride_c,                     \
                     static_cast<T::raw *>(out), report)
#define BEVPOOL_R2B_T(T, R16)                                                                  \
  if (vrow && vbev) BEVPOOL_R2B(T, true, true, R16);                                          \
  else if (vrow) BEVPOOL_R2B(T, true, false, R16);                                            \
  else if (vbev) BEVPOOL_R2B(T, false, true, R16);                                            \
  else BEVPOOL_R2B(T, false, false, R16);
  switch (dtype) {
    case BEVPOOL_F32:
      BEVPOOL_R2B_T(F32, false)
      break;
    case BEVPOOL_F16:
      if (raw16) {
        BEVPOOL_R2B_T(F16, true)
      } else {
        BEVPOOL_R2B_T(F16, false)
      }
      break;
    default:
      if (raw16) {
        BEVPOOL_R2B_T(BF16, true)
      } else {
        BEVPOOL_R2B_T(BF16, false)
      }
      break;
  }
#undef BEVPOOL_R2B_T
#undef BEVPOOL_R2B
  return check_launch("rows_to_bev");
}

// channel-first gradient -> cell-major rows of the occupied cells (raw bits).
int launch_bev_to_rows(const void *grad, size_t es, int64_t gsb, int64_t gsc, int64_t gsz, int C,
                       const int32_t *cell_end, int64_t n_cells, int n_z, int64_t n_xy,
                       void *rows, hipStream_t s) {
  if (int st = check_grid(ceil_div(n_cells, kCellTile), kThreads, "cell tiles")) return st;
  const unsigned tiles = unsigned(ceil_div(n_cells, kCellTile));
  const int CT = tile_channels(C);
  const size_t smem = size_t(kCellTile) * size_t(CT + 1) * es;
  const bool vrow = size_t(C) * es >= 16;
  const bool vbev = bev_vec_ok(grad, es, n_xy, gsb, gsc, gsz);
  const bool occ_first = n_cells >= kOccFirstCells;
  const CellMap cells{make_fast_div(uint32_t(n_xy)), make_fast_div(uint32_t(n_z)), gsb, gsz};
  LaunchTimer t("bev_to_rows", s);
#define BEVPOOL_B2R(TR, VR, VB)                                                                \
  hipLaunchKernelGGL((bev_to_rows_kernel<TR, VR, VB>), dim3(tiles), dim3(kThreads), smem, s,   \
                     static_cast<const TR *>(grad), C, CT, cell_end, n_cells, cells, gsc,       \
                     occ_first, static_cast<TR *>(rows))
#define BEVPOOL_B2R_T(TR)                                                                      \
  if (vrow && vbev) BEVPOOL_B2R(TR, true, true);                                              \
  else if (vrow) BEVPOOL_B2R(TR, true, false);                                                \
  else if (vbev) BEVPOOL_B2R(TR, false, true);                                                \
  else BEVPOOL_B2R(TR, false, false);
  if (es == 4) {
    BEVPOOL_B2R_T(uint32_t)
  } else {
    BEVPOOL_B2R_T(uint16_t)
  }
#undef BEVPOOL_B2R_T
#undef BEVPOOL_B2R
  return check_launch("bev_to_rows");
}

// Zero `bytes` bytes at p (4-byte aligned, a multiple of 4 bytes) with
// zero_fill_kernel; with `when` (device memory), only if *when != 0.
int launch_zero_fill(void *p, size_t bytes, hipStream_t s, const int32_t *when = nullptr) {
  if (bytes == 0) return BEVPOOL_OK;
  const bool vec = reinterpret_cast<uintptr_t>(p) % 16 == 0;
  const int64_t n16 = vec ? int64_t(bytes / 16) : 0;
  const int64_t n4 = int64_t((bytes - size_t(n16) * 16) / 4);
  const int64_t items = n16 > n4 ? n16 : n4;
  const int64_t blocks = ceil_div(items, kThreads) < 4096 ? ceil_div(items, kThreads) : 4096;
  LaunchTimer t("zero_fill", s);
  hipLaunchKernelGGL(zero_fill_kernel, dim3(unsigned(blocks)), dim3(kThreads), 0, s,
                     static_cast<u32x4 *>(p), n16,
                     reinterpret_cast<uint32_t *>(static_cast<char *>(p) + n16 * 16), n4, when);
  return check_launch("zero_fill");
}

// Launch shape of the legacy kernels for rows cut into pieces of `piece`
// bytes: at most 64 pieces per channel block (grid.y), `per_wave` intervals
// per wave of at most kLegacyBlocks blocks (grid.x; more intervals loop).
struct LegacyShape {
  int qmax;
  dim3 grid;
};
LegacyShape legacy_shape(int C, int piece, int64_t cap, bool groups) {
  const int qt = (C * 4 + piece - 1) / piece, nblk = (qt + 63) / 64;
  const int qmax = (qt + nblk - 1) / nblk;
  const int64_t blocks = ceil_div(cap, int64_t(kWaves) * (groups ? 64 / qmax : 1));
  return {qmax, dim3(unsigned(blocks < 1 ? 1 : (blocks < kLegacyBlocks ? blocks : kLegacyBlocks)),
                     unsigned(nblk))};
}

int check_legacy_args(int64_t n, int32_t C, const void *geom, const void *starts,
                      const void *lengths, int64_t n_intervals, int32_t b, int32_t d, int32_t h,
                      int32_t w, const void *out) {
  if (n < 0 || n > int64_t(INT32_MAX)) return fail(BEVPOOL_EINVAL, "n=%lld out of range", (long long)n);
  if (C < 1) return fail(BEVPOOL_EINVAL, "C must be positive");
  if (b < 1 || d < 1 || h < 1 || w < 1)
    return fail(BEVPOOL_EINVAL, "b, d, h, w must be positive");
  if (int64_t(b) * d * h * w > int64_t(INT32_MAX))
    return fail(BEVPOOL_EINVAL, "b*d*h*w exceeds 2^31-1");
  if (n_intervals < 0 || n_intervals > int64_t(INT32_MAX))
    return fail(BEVPOOL_EINVAL, "n_intervals out of range");
  if (!out) return fail(BEVPOOL_EINVAL, "null output");
  if (n_intervals > 0 && (!geom || !starts || !lengths))
    return fail(BEVPOOL_EINVAL, "null geom_feats / interval arrays");
  return BEVPOOL_OK;
}

// Layout of the op-level buffers (bevpool_op_forward / bevpool_op_backward).
// The index buffer keeps what the backward needs: meta, ranks, sorted keys and
// cell ranges.  The scratch buffer holds the index-stage workspace and the
// cell rows; it is needed only during a call.
struct OpIndexLayout {
  size_t meta, rank, keys, cstart, cend, total;
};

OpIndexLayout op_index_layout(int64_t n, int64_t cells) {
  OpIndexLayout L;
  size_t o = 0;
  L.meta = o;
  o = align256(o + BEVPOOL_META_LEN * sizeof(int32_t));
  L.rank = o;
  o = align256(o + size_t(n) * sizeof(int32_t));
  L.keys = o;
  o = align256(o + size_t(n) * sizeof(uint64_t));
  L.cstart = o;
  o = align256(o + size_t(cells) * sizeof(int32_t));
  L.cend = o;
  o = align256(o + size_t(cells) * sizeof(int32_t));
  L.total = o;
  return L;
}

struct OpScratchLayout {
  size_t index_ws, rows, total;
};

OpScratchLayout op_scratch_layout(int64_t n, int64_t cells, int32_t C) {
  OpScratchLayout L;
  size_t o = 0;
  L.index_ws = o;
  o = align256(o + index_layout(n, cells).total);
  L.rows = o;
  o = align256(o + size_t(cells) * size_t(C) * sizeof(float));
  L.total = o;
  return L;
}

// Scratch of the allocation-free op-level forward: the index buffer
// (op_index_layout) and the scratch (op_scratch_layout) of one call live in
// this array, one copy per GPU, held until
// the process ends.  Host code never passes `scratch` itself to a kernel or
// a copy (in host code the name is a host-side stand-in, not a device
// address): it uses the device address hipGetSymbolAddress returns for the
// current device, cached per device by noalloc_scratch().
constexpr size_t kNoAllocScratchBytes = BEVPOOL_NOALLOC_MAX_BYTES;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

// legacy backward: the counter slot that holds its order check
constexpr int kMetaUnordered = 4;

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device (resolved once per
// device, with that device current), or nullptr with the error recorded.
void *noalloc_scratch() {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    fail(BEVPOOL_EHIP, "hipGetDevice: %s", hipGetErrorString(e));
    return nullptr;
  }
  if (dev < 0 || dev >= kMaxDevices) {
    fail(BEVPOOL_EINVAL, "device %d beyond the %d devices the scratch table holds", dev,
         kMaxDevices);
    return nullptr;
  }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      fail(BEVPOOL_EHIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev,
           hipGetErrorString(e));
      return nullptr;
    }
    g_scratch_ptr[dev] = p;
  }
  return g_scratch_ptr[dev];
}

}  // namespace

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
extern "C" {

int bevpool_abi_version(void) { return BEVPOOL_ABI_VERSION; }

const char *bevpool_last_error(void) { return g_last_error.c_str(); }

size_t bevpool_index_workspace_bytes(int64_t n_points, int64_t n_cells) {
  if (n_points < 0) return 0;
  return index_layout(n_points, n_cells < 1 ? 1 : n_cells).total;
}

int bevpool_quantize_geom(const float *geom, int64_t n_points, int64_t geom_row_stride,
                          int64_t points_per_batch, int32_t n_batch, const float offset[3],
                          const float dx[3], const int32_t nx[3], int32_t *rank, int32_t *meta,
                          void *workspace, size_t workspace_bytes, void *stream) {
  g_last_error.clear();
  if (!offset || !dx || !nx) return fail(BEVPOOL_EINVAL, "null offset/dx/nx");
  if (n_batch < 1 || nx[0] < 1 || nx[1] < 1 || nx[2] < 1)
    return fail(BEVPOOL_EINVAL, "grid sizes must be positive (B=%d nx=%d,%d,%d)", n_batch, nx[0],
                nx[1], nx[2]);
  const int64_t n_cells = int64_t(n_batch) * nx[0] * nx[1] * nx[2];
  int st = check_index_args(n_points, n_cells, rank, meta, workspace, workspace_bytes);
  if (st) return st;
  if (n_points > 0 && (!geom || geom_row_stride < 3 || points_per_batch < 1 ||
                       ceil_div(n_points, points_per_batch) > n_batch))
    return fail(BEVPOOL_EINVAL, "bad geometry layout (row stride %lld, points/batch %lld)",
                (long long)geom_row_stride, (long long)points_per_batch);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const IndexLayout L = index_layout(n_points, n_cells);
  const DigitPlan plan = plan_digits(n_cells);
  {
    // also resets meta (block 0); an empty input still launches that block
    LaunchTimer t("quantize_geom", s);
    const unsigned grid = sort_grid(L.sort_blocks);
    // batch index = point / points_per_batch (every point index is < 2^31)
    const FastDiv ppb = make_fast_div(uint32_t(
        points_per_batch < 1 ? 1 : (points_per_batch > (int64_t(1) << 31) ? (int64_t(1) << 31)
                                                                          : points_per_batch)));
    const bool vec = geom_row_stride == 3 && n_points >= 4 &&
                     reinterpret_cast<uintptr_t>(geom) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(rank) % 16 == 0;
#define BEVPOOL_QUANT(V, IT)                                                                   \
  hipLaunchKernelGGL((quantize_geom_kernel<V, IT>), dim3(grid), dim3(kThreads), 0, s, geom,     \
                     n_points, geom_row_stride, ppb, offset[0], offset[1], offset[2], dx[0],     \
                     dx[1], dx[2], nx[0], nx[1], nx[2], rank, at<int32_t>(workspace, L.hist),   \
                     int(L.sort_blocks), plan.shift[0], plan.bits[0], meta)
    if (L.items == kItemsLarge) {
      if (vec) BEVPOOL_QUANT(true, kItemsLarge); else BEVPOOL_QUANT(false, kItemsLarge);
    } else {
      if (vec) BEVPOOL_QUANT(true, kItemsSmall); else BEVPOOL_QUANT(false, kItemsSmall);
    }
#undef BEVPOOL_QUANT
  }
  return check_launch("quantize_geom");
}

int bevpool_quantize_cameras(const float *frustum, int32_t D, int32_t fH, int32_t fW,
                             const float *rots, const float *trans, const float *intrins,
                             const float *post_rots, const float *post_trans,
                             const float *extra_rots, const float *extra_trans,
                             int32_t n_cams_per_batch, int32_t n_batch, const float offset[3],
                             const float dx[3], const int32_t nx[3], int32_t *rank,
                             int32_t *meta, void *workspace, size_t workspace_bytes,
                             void *stream) {
  g_last_error.clear();
  if (!offset || !dx || !nx) return fail(BEVPOOL_EINVAL, "null offset/dx/nx");
  if (n_batch < 1 || n_cams_per_batch < 1 || D < 1 || fH < 1 || fW < 1)
    return fail(BEVPOOL_EINVAL, "bad frustum/camera sizes");
  if (nx[0] < 1 || nx[1] < 1 || nx[2] < 1) return fail(BEVPOOL_EINVAL, "bad grid");
  const int64_t dhw = int64_t(D) * fH * fW;
  const int64_t n_points = dhw * n_cams_per_batch * n_batch;
  const int64_t n_cells = int64_t(n_batch) * nx[0] * nx[1] * nx[2];
  int st = check_index_args(n_points, n_cells, rank, meta, workspace, workspace_bytes);
  if (st) return st;
  if (!frustum || !rots || !trans || !intrins || !post_rots || !post_trans)
    return fail(BEVPOOL_EINVAL, "null frustum/camera matrices");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const IndexLayout L = index_layout(n_points, n_cells);
  const DigitPlan plan = plan_digits(n_cells);
  const CameraMats cm{rots, trans, intrins, post_rots, post_trans, extra_rots, extra_trans,
                      n_cams_per_batch};
  LaunchTimer t("quantize_cameras", s);
#define BEVPOOL_QCAM(IT)                                                                       \
  hipLaunchKernelGGL((quantize_frustum_kernel<IT>), dim3(sort_grid(L.sort_blocks)),           \
                     dim3(kThreads), 0, s, frustum, n_points, make_fast_div(uint32_t(dhw)),    \
                     make_fast_div(uint32_t(n_cams_per_batch)), cm, offset[0], offset[1],      \
                     offset[2], dx[0], dx[1], dx[2], nx[0], nx[1], nx[2], rank,                \
                     at<int32_t>(workspace, L.hist), int(L.sort_blocks), plan.shift[0],        \
                     plan.bits[0], meta)
  if (L.items == kItemsLarge) BEVPOOL_QCAM(kItemsLarge); else BEVPOOL_QCAM(kItemsSmall);
#undef BEVPOOL_QCAM
  return check_launch("quantize_cameras");
}

// tile_bad: count invalid ranks per tile in the index workspace (for
// sort_impl's first scatter to reduce into meta) instead of initialising meta
// here and counting into it with atomics.
static int coord_ranks_impl(const void *coords, int32_t coord_bytes, int64_t n_points,
                            int64_t coords_row_stride, int32_t B, int32_t D, int32_t H,
                            int32_t W, int32_t *rank, int32_t *meta, void *workspace,
                            size_t workspace_bytes, void *stream, bool tile_bad) {
  if (B < 1 || D < 1 || H < 1 || W < 1)
    return fail(BEVPOOL_EINVAL, "B, D, H, W must be positive");
  if (coord_bytes != 4 && coord_bytes != 8)
    return fail(BEVPOOL_EINVAL, "coord_bytes must be 4 or 8, got %d", coord_bytes);
  const int64_t n_cells = int64_t(B) * D * H * W;
  int st = check_index_args(n_points, n_cells, rank, meta, workspace, workspace_bytes);
  if (st) return st;
  if (n_points > 0 && (!coords || coords_row_stride < 4))
    return fail(BEVPOOL_EINVAL, "bad coords layout");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (!tile_bad || n_points == 0) {  // no points: no scatter writes meta
    {
      LaunchTimer t("init_meta", s);
      hipLaunchKernelGGL(init_meta_kernel, dim3(1), dim3(64), 0, s, meta);
    }
    if ((st = check_launch("init_meta"))) return st;
  }
  if (n_points == 0) return BEVPOOL_OK;
  const IndexLayout L = index_layout(n_points, n_cells);
  const DigitPlan plan = plan_digits(n_cells);
  int32_t *bad = at<int32_t>(workspace, L.tile_bad);
  LaunchTimer t("coord_ranks", s);
#define BEVPOOL_CRANKS(TC, IT, TB)                                                             \
  hipLaunchKernelGGL((coord_ranks_kernel<TC, IT, TB>), dim3(sort_grid(L.sort_blocks)),         \
                     dim3(kThreads), 0, s, static_cast<const TC *>(coords), n_points,          \
                     coords_row_stride, int64_t(B), int64_t(D), int64_t(H), int64_t(W), rank,  \
                     meta, at<int32_t>(workspace, L.hist), int(L.sort_blocks), plan.shift[0],  \
                     plan.bits[0], bad)
#define BEVPOOL_CRANKS_T(TC, IT)                                                               \
  if (tile_bad) BEVPOOL_CRANKS(TC, IT, true); else BEVPOOL_CRANKS(TC, IT, false);
  if (coord_bytes == 4) {
    if (L.items == kItemsLarge) { BEVPOOL_CRANKS_T(int32_t, kItemsLarge) }
    else { BEVPOOL_CRANKS_T(int32_t, kItemsSmall) }
  } else {
    if (L.items == kItemsLarge) { BEVPOOL_CRANKS_T(int64_t, kItemsLarge) }
    else { BEVPOOL_CRANKS_T(int64_t, kItemsSmall) }
  }
#undef BEVPOOL_CRANKS_T
#undef BEVPOOL_CRANKS
  return check_launch("coord_ranks");
}

int bevpool_coord_ranks(const void *coords, int32_t coord_bytes, int64_t n_points,
                        int64_t coords_row_stride, int32_t B, int32_t D, int32_t H, int32_t W,
                        int32_t *rank, int32_t *meta, void *workspace, size_t workspace_bytes,
                        void *stream) {
  g_last_error.clear();
  return coord_ranks_impl(coords, coord_bytes, n_points, coords_row_stride, B, D, H, W, rank,
                          meta, workspace, workspace_bytes, stream, false);
}

// tile_bad: the per-tile invalid-rank counts of coord_ranks_impl(...,
// tile_bad = true) in this workspace; the first scatter then writes all of
// meta.  nullptr: meta was initialised by the rank kernel's call.
static int sort_impl(const int32_t *rank, int64_t n_points, int64_t n_cells, uint64_t *keys,
                     int32_t *cell_start, int32_t *cell_end, int32_t *meta, void *workspace,
                     size_t workspace_bytes, void *stream, bool tile_bad) {
  int st = check_index_args(n_points, n_cells, rank, meta, workspace, workspace_bytes);
  if (st) return st;
  if (!cell_start || !cell_end) return fail(BEVPOOL_EINVAL, "null cell_start/cell_end");
  if (n_points > 0 && !keys) return fail(BEVPOOL_EINVAL, "null keys");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const IndexLayout L = index_layout(n_points, n_cells);
  const DigitPlan plan = plan_digits(n_cells);
  int32_t *hist = at<int32_t>(workspace, L.hist);
  int32_t *totals = at<int32_t>(workspace, L.totals);
  int32_t *gstart = at<int32_t>(workspace, L.gstart);
  uint64_t *tmp = at<uint64_t>(workspace, L.keys_tmp);
  if (n_points == 0) {
    // no points: only the dense cell ranges need clearing
    LaunchTimer t("radix_scan", s);
    hipLaunchKernelGGL(radix_scan_kernel, dim3(64), dim3(kThreads), 0, s, hist, 0, totals,
                       cell_start, cell_end, n_cells);
    return check_launch("radix_scan");
  }
  const int nb = int(L.sort_blocks);
  const uint64_t *src = nullptr;
  const bool bucketed = plan.local_bits > 0;
  for (int pass = 0; pass < plan.passes; ++pass) {
    uint64_t *dst = bucketed ? tmp : (((plan.passes - 1 - pass) % 2 == 0) ? keys : tmp);
    const bool large = L.items == kItemsLarge;
    if (pass > 0) {
      LaunchTimer t("radix_hist", s);
#define BEVPOOL_RHIST(IT)                                                                      \
  hipLaunchKernelGGL((radix_hist_kernel<IT>), dim3(sort_grid(nb)), dim3(kThreads), 0, s, src,   \
                     meta, hist, nb, plan.shift[pass], plan.bits[pass])
      if (large) BEVPOOL_RHIST(kItemsLarge); else BEVPOOL_RHIST(kItemsSmall);
#undef BEVPOOL_RHIST
      if ((st = check_launch("radix_hist"))) return st;
    }
    {
      LaunchTimer t("radix_scan", s);
      hipLaunchKernelGGL(radix_scan_kernel, dim3(1u << plan.bits[pass]), dim3(kThreads), 0, s,
                         hist, nb, totals, cell_start, cell_end,
                         pass == 0 && !bucketed ? n_cells : 0);
      if ((st = check_launch("radix_scan"))) return st;
    }
    {
      LaunchTimer t("radix_scatter", s);
#define BEVPOOL_RSCAT(FROM_RANK, IT)                                                           \
  hipLaunchKernelGGL((radix_scatter_kernel<FROM_RANK, IT>), dim3(xcd_grid(nb)), dim3(kThreads), \
                     0, s, FROM_RANK ? rank : nullptr, FROM_RANK ? nullptr : src, n_points,    \
                     meta, dst, hist, totals, nb, plan.shift[pass], plan.bits[pass],           \
                     FROM_RANK && tile_bad ? at<int32_t>(workspace, L.tile_bad) : nullptr,     \
                     bucketed ? gstart : nullptr)
      if (pass == 0) {
        if (large) BEVPOOL_RSCAT(true, kItemsLarge); else BEVPOOL_RSCAT(true, kItemsSmall);
      } else {
        if (large) BEVPOOL_RSCAT(false, kItemsLarge); else BEVPOOL_RSCAT(false, kItemsSmall);
      }
#undef BEVPOOL_RSCAT
      if ((st = check_launch("radix_scatter"))) return st;
    }
    src = dst;
  }
  if (bucketed && plan.local_bits >= kSlicedBits) {
    // groups of 2^10 cells (up to ~65 K keys at 2 x 720 x 720), cut into
    // slices -> sorted keys and the dense cell ranges
    const int lb = plan.local_bits;
    const int n_groups = int(ceil_div(n_cells, int64_t(1) << lb));
    const int64_t n_slices = slice_bound(n_points, n_cells, lb);
    if ((st = check_grid(n_slices, kThreads, "bucket slices"))) return st;
    int32_t *scnt = at<int32_t>(workspace, L.slices);
    const size_t R4 = size_t(4) << lb;
    {
      LaunchTimer t("bucket_count", s);
      hipLaunchKernelGGL(bucket_count_kernel<kSliceWaves>, dim3(unsigned(n_slices)),
                         dim3(64 * kSliceWaves), R4, s, src, totals, n_groups, lb, scnt);
      if ((st = check_launch("bucket_count"))) return st;
    }
    {
      LaunchTimer t("bucket_scan", s);
      hipLaunchKernelGGL(bucket_scan_kernel, dim3(unsigned(n_groups)), dim3(kThreads), 0, s,
                         totals, n_groups, n_cells, lb, scnt, cell_start, cell_end);
      if ((st = check_launch("bucket_scan"))) return st;
    }
    LaunchTimer t("bucket_place", s);
    hipLaunchKernelGGL(bucket_place_kernel<kSliceWaves>, dim3(unsigned(n_slices)),
                       dim3(64 * kSliceWaves), kSliceWaves * R4, s, src, totals, n_groups, lb,
                       scnt, keys);
    return check_launch("bucket_place");
  }
  if (bucketed) {
    // groups of at most 2^9 cells -> sorted keys and the dense cell ranges
    LaunchTimer t("bucket_sort", s);
    const int64_t n_buckets = ceil_div(n_cells, int64_t(1) << plan.local_bits);
    hipLaunchKernelGGL(bucket_sort_kernel<16>, dim3(unsigned(n_buckets * kBucketParts)),
                       dim3(16 * 64), size_t(16 + 2) << plan.local_bits << 2, s, src, totals,
                       gstart, int(n_buckets), n_cells, keys, cell_start, cell_end,
                       plan.local_bits, kBucketParts, kBucketPartKeys);
    return check_launch("bucket_sort");
  }
  {
    LaunchTimer t("cell_ranges", s);
    const unsigned g = unsigned(ceil_div(n_points, int64_t(kThreads) * 4));
    if (reinterpret_cast<uintptr_t>(keys) % 16 == 0)
      hipLaunchKernelGGL(cell_ranges_kernel<true>, dim3(g), dim3(kThreads), 0, s, keys, meta,
                         cell_start, cell_end);
    else
      hipLaunchKernelGGL(cell_ranges_kernel<false>, dim3(g), dim3(kThreads), 0, s, keys, meta,
                         cell_start, cell_end);
  }
  return check_launch("cell_ranges");
}

int bevpool_sort(const int32_t *rank, int64_t n_points, int64_t n_cells, uint64_t *keys,
                 int32_t *cell_start, int32_t *cell_end, int32_t *meta, void *workspace,
                 size_t workspace_bytes, void *stream) {
  g_last_error.clear();
  return sort_impl(rank, n_points, n_cells, keys, cell_start, cell_end, meta, workspace,
                   workspace_bytes, stream, false);
}

// Device address for writing to `dst`: pinned host memory through its device
// address, device memory of the current device as is; anything else
// (pageable host memory the GPU cannot reach) is refused.
static int report_address(int32_t *dst, int32_t **dev_dst) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, dst) != hipSuccess) {
    (void)hipGetLastError();  // unknown pointer: clear the lookup's error
    return fail(BEVPOOL_EINVAL, "report destination is neither pinned host nor device memory");
  }
  if (a.type == hipMemoryTypeHost) {
    void *d = nullptr;
    if (hipHostGetDevicePointer(&d, dst, 0) != hipSuccess || !d) {
      (void)hipGetLastError();
      return fail(BEVPOOL_EHIP, "hipHostGetDevicePointer failed for the report destination");
    }
    *dev_dst = static_cast<int32_t *>(d);
    return BEVPOOL_OK;
  }
  if (a.type == hipMemoryTypeDevice) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev != a.device)
      return fail(BEVPOOL_EINVAL, "report destination on device %d, current device %d",
                  a.device, dev);
    *dev_dst = dst;
    return BEVPOOL_OK;
  }
  return fail(BEVPOOL_EINVAL, "report destination is neither pinned host nor device memory");
}

int bevpool_meta_report(const int32_t *meta, int32_t *dst, void *stream) {
  g_last_error.clear();
  if (!meta || !dst) return fail(BEVPOOL_EINVAL, "null meta or destination");
  int32_t *dev_dst = nullptr;
  if (int st = report_address(dst, &dev_dst)) return st;
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(meta_report_kernel, dim3(1), dim3(64), 0, s, meta, dev_dst);
  return check_launch("meta_report");
}

int bevpool_intervals(const uint64_t *keys, int64_t n_points, const int32_t *cell_end,
                      int32_t *starts, int32_t *lengths, int32_t *cells, int32_t *meta,
                      void *workspace, size_t workspace_bytes, void *stream) {
  g_last_error.clear();
  if (n_points < 0 || n_points > int64_t(INT32_MAX))
    return fail(BEVPOOL_EINVAL, "n_points out of range");
  if (!meta) return fail(BEVPOOL_EINVAL, "meta is null");
  const IndexLayout L = index_layout(n_points, 1);
  if (workspace_bytes < L.total) return fail(BEVPOOL_ESPACE, "index workspace too small");
  hipStream_t s = static_cast<hipStream_t>(stream);
  int32_t *bcount = at<int32_t>(workspace, L.bcount);
  if (n_points == 0) {
    // meta[N_INTERVALS] was zeroed by the rank stage
    return BEVPOOL_OK;
  }
  if (!keys || !cell_end || !starts || !lengths || !cells)
    return fail(BEVPOOL_EINVAL, "null interval argument");
  int st;
  {
    LaunchTimer t("count_starts", s);
    hipLaunchKernelGGL(count_starts_kernel, dim3(unsigned(L.cell_blocks)), dim3(kThreads), 0, s,
                       keys, meta, bcount);
    if ((st = check_launch("count_starts"))) return st;
  }
  {
    LaunchTimer t("scan_counts", s);
    hipLaunchKernelGGL(scan_counts_kernel, dim3(1), dim3(kThreads), 0, s, bcount, L.cell_blocks,
                       meta + BEVPOOL_META_N_INTERVALS);
    if ((st = check_launch("scan_counts"))) return st;
  }
  LaunchTimer t("interval_write", s);
  hipLaunchKernelGGL(interval_write_kernel, dim3(unsigned(L.cell_blocks)), dim3(kThreads), 0, s,
                     keys, meta, cell_end, bcount, starts, lengths, cells);
  return check_launch("interval_write");
}

size_t bevpool_forward_scratch_bytes(int64_t n_cells, int32_t C) {
  if (n_cells < 0 || C < 0) return 0;
  return size_t(n_cells) * size_t(C) * sizeof(float);
}

// bevpool_forward; `report` (optional) is written by the transpose's first
// block.
static int forward_impl(const void *feats, int32_t dtype, int64_t feats_row_stride, int32_t C,
                        int64_t n_points, const uint64_t *keys, const int32_t *cell_start,
                        const int32_t *cell_end, const int32_t *meta, int32_t n_batch,
                        int32_t n_z, int64_t n_xy, int64_t out_stride_b, int64_t out_stride_c,
                        int64_t out_stride_z, void *out, void *scratch, size_t scratch_bytes,
                        void *stream, MetaReport report) {
  if (dtype != BEVPOOL_F32 && dtype != BEVPOOL_F16 && dtype != BEVPOOL_BF16)
    return fail(BEVPOOL_EINVAL, "unsupported dtype code %d", dtype);
  if (C < 1) return fail(BEVPOOL_EINVAL, "C must be positive");
  if (n_batch < 1 || n_z < 1 || n_xy < 1) return fail(BEVPOOL_EINVAL, "bad grid");
  const int64_t n_cells = int64_t(n_batch) * n_z * n_xy;
  if (n_cells > int64_t(INT32_MAX)) return fail(BEVPOOL_EINVAL, "too many cells");
  if (n_points < 0 || n_points > int64_t(INT32_MAX))
    return fail(BEVPOOL_EINVAL, "n_points out of range");
  if (!out || !cell_start || !cell_end || !meta) return fail(BEVPOOL_EINVAL, "null argument");
  if (n_points > 0 && (!feats || !keys || feats_row_stride < C))
    return fail(BEVPOOL_EINVAL, "bad feats layout");
  if (scratch_bytes < bevpool_forward_scratch_bytes(n_cells, C) || !scratch)
    return fail(BEVPOOL_ESPACE, "forward scratch too small");
  hipStream_t s = static_cast<hipStream_t>(stream);
  float *acc = static_cast<float *>(scratch);
  int st;
  bool raw16 = false;  // cell rows hold 16-bit output values (rows of 16 bytes or more)
  if (n_points > 0) {
    const size_t es = dtype_size(dtype);
    const size_t row_bytes = size_t(C) * es;
    const int64_t ld_bytes = int64_t(size_t(feats_row_stride) * es);
    const char *x = static_cast<const char *>(feats);
    const bool vec16 = row_bytes % 16 == 0 && ld_bytes % 16 == 0 &&
                       reinterpret_cast<uintptr_t>(feats) % 16 == 0;
    // rows of every point (an upper bound of the kept rows read)
    const bool stream_rows = n_points * int64_t(row_bytes) <= kStreamRowBytes;
    const GroupPlan plan = group_plan(dtype, C, n_points, n_cells, false);
    LaunchTimer t("accum_rows", s);
    if (vec16 && row_bytes <= size_t(kPipeRowBytes) && !plan.small) {
      st = launch_accum_pipe(dtype, x, ld_bytes, C, n_points, keys, meta, cell_end, acc,
                             stream_rows, s);
    } else if (row_bytes >= 16) {
      st = launch_accum_group(dtype, plan, x, ld_bytes, C, n_points, keys, meta, cell_start,
                              cell_end, acc, DepthRows{nullptr, {}, {}}, stream_rows, s);
    } else {
      // rows of fewer than 16 bytes: element by element
      const unsigned grid = unsigned(ceil_div(n_points, kRangePoints));
      const int R = 64;
      const size_t smem = size_t(R) * C * sizeof(float) + size_t(R + 1) * sizeof(int);
#define BEVPOOL_ROWS(T)                                                                        \
  hipLaunchKernelGGL(accum_rows_kernel<T>, dim3(grid), dim3(kThreads), smem, s,                \
                     static_cast<const T::raw *>(feats), feats_row_stride, C, R, keys, meta,   \
                     cell_end, acc, kRangePoints)
      if (dtype == BEVPOOL_F32) BEVPOOL_ROWS(F32);
      else if (dtype == BEVPOOL_F16) BEVPOOL_ROWS(F16);
      else BEVPOOL_ROWS(BF16);
#undef BEVPOOL_ROWS
      st = check_launch("accum_rows");
    }
    if (st) return st;
    raw16 = es == 2 && row_bytes >= 16;
  }
  return launch_rows_to_bev(acc, dtype, C, cell_end, n_cells, n_z, n_xy,
                            out_stride_b, out_stride_c, out_stride_z, out, s, report, raw16);
}

int bevpool_forward(const void *feats, int32_t dtype, int64_t feats_row_stride, int32_t C,
                    int64_t n_points, const uint64_t *keys, const int32_t *cell_start,
                    const int32_t *cell_end, const int32_t *meta, int32_t n_batch, int32_t n_z,
                    int64_t n_xy, int64_t out_stride_b, int64_t out_stride_c,
                    int64_t out_stride_z, void *out, void *scratch, size_t scratch_bytes,
                    void *stream) {
  g_last_error.clear();
  return forward_impl(feats, dtype, feats_row_stride, C, n_points, keys, cell_start, cell_end,
                      meta, n_batch, n_z, n_xy, out_stride_b, out_stride_c, out_stride_z, out,
                      scratch, scratch_bytes, stream, MetaReport{});
}

// rank: null, or the points' ranks: rows of dropped points need not be written.
static int planar_rows_impl(const float *src, int64_t stride_bn, int64_t stride_c, int32_t BN,
                            int32_t C, int64_t S, const int32_t *rank, float *rows,
                            void *stream) {
  if (BN < 0 || C < 1 || S < 0) return fail(BEVPOOL_EINVAL, "bad planar shape");
  const int64_t n_rows = int64_t(BN) * S;
  if (n_rows == 0) return BEVPOOL_OK;
  if (!src || !rows) return fail(BEVPOOL_EINVAL, "null argument");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t tiles_s = ceil_div(S, kPlanarTile);
  const int64_t tiles = BN * tiles_s, elements = ceil_div(n_rows * C, kThreads);  // blocks
  // the launch limit is the tiles' where 4 divides every size, else that of one
  // element per thread (within which the tiles' grid always fits)
  const bool even = C % 4 == 0 && S % 4 == 0 && stride_bn % 4 == 0 && stride_c % 4 == 0;
  if (int st = check_grid(even ? tiles : elements, kThreads, "planar_rows")) return st;
  // A tile of a few points costs what a larger one does: with fewer than 12
  // points or 400 elements one element per thread is faster (tiles against
  // elements, us, 1 M rows: C = 80, S = 5 647 and 254, S = 15 271 and 321; C =
  // 16, S = 15 55 and 39, S = 31 33 and 41).
  const bool small = S < 12 || S * C < 400;
  const bool vec = C >= 4 && S >= 4 && !(small && elements * kThreads <= int64_t(UINT32_MAX));
  LaunchTimer t("planar_rows", s);
  if (vec) {
    const int cmax = planar_channels(C);
    const size_t smem = size_t(kPlanarTile) * size_t(cmax + 1) * sizeof(float);
    const dim3 grid(unsigned(tiles), unsigned(planar_blocks(C)));
#define BEVPOOL_PT(K)                                                                          \
  case K:                                                                                      \
    hipLaunchKernelGGL((planar_tile_kernel<K>), grid, dim3(kThreads), smem, s, src, C, cmax, S, \
                       tiles_s, stride_bn, stride_c, rank, rows);                              \
    break;
    switch (ceil_div(int64_t(cmax) * (kPlanarTile / 4), kThreads)) {
      BEVPOOL_PT(1) BEVPOOL_PT(2) BEVPOOL_PT(3) BEVPOOL_PT(4)
      BEVPOOL_PT(5) BEVPOOL_PT(6) BEVPOOL_PT(7) BEVPOOL_PT(8)
      BEVPOOL_PT(9) BEVPOOL_PT(10) BEVPOOL_PT(11) BEVPOOL_PT(12)
      BEVPOOL_PT(13) BEVPOOL_PT(14) BEVPOOL_PT(15) BEVPOOL_PT(16)
      default:
        return fail(BEVPOOL_EINVAL, "internal: %d channels per planar tile", cmax);
    }
#undef BEVPOOL_PT
  } else {
    hipLaunchKernelGGL(planar_rows_kernel, dim3(unsigned(elements)), dim3(kThreads), 0, s, src, C,
                       S, n_rows, stride_bn, stride_c, rows);
  }
  return check_launch("planar_rows");
}

int bevpool_planar_rows(const float *src, int64_t stride_bn, int64_t stride_c, int32_t BN,
                        int32_t C, int64_t S, float *rows, void *stream) {
  g_last_error.clear();
  return planar_rows_impl(src, stride_bn, stride_c, BN, C, S, nullptr, rows, stream);
}

int bevpool_planar_kept_rows(const float *src, int64_t stride_bn, int64_t stride_c, int32_t BN,
                             int32_t C, int64_t S, const int32_t *rank, float *rows,
                             void *stream) {
  g_last_error.clear();
  if (BN > 0 && S > 0 && !rank) return fail(BEVPOOL_EINVAL, "null rank");
  return planar_rows_impl(src, stride_bn, stride_c, BN, C, S, rank, rows, stream);
}

int bevpool_context_rows(const float *context, int64_t stride_bn, int64_t stride_c, int32_t BN,
                         int32_t C, int64_t HW, float *rows, void *stream) {
  return bevpool_planar_rows(context, stride_bn, stride_c, BN, C, HW, rows, stream);
}

int bevpool_backward_planar(const float *grad, int64_t grad_stride_b, int64_t grad_stride_c,
                            int64_t grad_stride_z, int32_t C, const int32_t *rank,
                            int64_t n_points, const int32_t *cell_start,
                            const int32_t *cell_end, int32_t n_batch, int32_t n_z, int64_t n_xy,
                            int64_t S, float *x_grad, int64_t x_stride_bn, int64_t x_stride_c,
                            void *scratch, size_t scratch_bytes, void *stream) {
  g_last_error.clear();
  if (C < 1) return fail(BEVPOOL_EINVAL, "C must be positive");
  if (n_batch < 1 || n_z < 1 || n_xy < 1) return fail(BEVPOOL_EINVAL, "bad grid");
  const int64_t n_cells = int64_t(n_batch) * n_z * n_xy;
  if (n_cells > int64_t(INT32_MAX)) return fail(BEVPOOL_EINVAL, "too many cells");
  if (S < 1 || n_points < 0 || n_points > int64_t(INT32_MAX) || n_points % S != 0)
    return fail(BEVPOOL_EINVAL, "n_points must be a multiple of S");
  if (n_points == 0) return BEVPOOL_OK;
  if (!grad || !rank || !cell_start || !cell_end || !x_grad)
    return fail(BEVPOOL_EINVAL, "null argument");
  if (!scratch || scratch_bytes < bevpool_backward_scratch_bytes(n_cells, C, BEVPOOL_F32))
    return fail(BEVPOOL_ESPACE, "backward scratch too small");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool vec = C >= 4 && S >= 4;
  const int64_t per_bn = ceil_div(S, 4), n_groups = n_points / S * per_bn;  // groups of 4 points
  // (sizes that do not divide by 4 keep the limit of one element per thread)
  const bool even = C % 4 == 0 && S % 4 == 0 && x_stride_bn % 4 == 0 && x_stride_c % 4 == 0;
  int st;
  if ((st = check_grid(vec && even ? ceil_div(n_groups, kThreads) + kXcds
                           : ceil_div(n_points * C, kThreads),
                       kThreads, "gather_planar")))
    return st;
  if ((st = launch_bev_to_rows(grad, 4, grad_stride_b, grad_stride_c, grad_stride_z, C,
                               cell_end, n_cells, n_z, n_xy, scratch, s)))
    return st;
  const float *g = static_cast<const float *>(scratch);
  LaunchTimer t("gather_planar", s);
  const FastDiv groups = make_fast_div(uint32_t(per_bn));
  const bool past_caches = even && reinterpret_cast<uintptr_t>(x_grad) % 16 == 0;
#define BEVPOOL_GP(VEC, STREAM, BLOCKS)                                                        \
  hipLaunchKernelGGL((gather_planar_kernel<VEC, STREAM>), dim3(BLOCKS), dim3(kThreads), 0, s, g, \
                     C, rank, n_points, S, groups, n_groups, x_stride_bn, x_stride_c, x_grad)
  const unsigned group_blocks = xcd_grid(ceil_div(n_groups, kThreads));
  if (vec && past_caches) BEVPOOL_GP(true, true, group_blocks);
  else if (vec) BEVPOOL_GP(true, false, group_blocks);
  else BEVPOOL_GP(false, false, unsigned(ceil_div(n_points * C, kThreads)));
#undef BEVPOOL_GP
  return check_launch("gather_planar");
}

int bevpool_forward_depth(const float *depth, const float *context_rows, int32_t C,
                          int64_t n_points, int32_t D, int64_t HW, const uint64_t *keys,
                          const int32_t *cell_start, const int32_t *cell_end,
                          const int32_t *meta, int32_t n_batch, int32_t n_z, int64_t n_xy,
                          int64_t out_stride_b, int64_t out_stride_c, int64_t out_stride_z,
                          float *out, void *scratch, size_t scratch_bytes, void *stream) {
  g_last_error.clear();
  if (C < 1 || C % 4 != 0) return fail(BEVPOOL_EINVAL, "C must be a positive multiple of 4");
  if (D < 1 || HW < 1) return fail(BEVPOOL_EINVAL, "bad depth layout (D=%d, HW=%lld)", D,
                                   (long long)HW);
  if (n_batch < 1 || n_z < 1 || n_xy < 1) return fail(BEVPOOL_EINVAL, "bad grid");
  const int64_t n_cells = int64_t(n_batch) * n_z * n_xy;
  if (n_cells > int64_t(INT32_MAX)) return fail(BEVPOOL_EINVAL, "too many cells");
  if (n_points < 0 || n_points > int64_t(INT32_MAX) || n_points % (int64_t(D) * HW) != 0)
    return fail(BEVPOOL_EINVAL, "n_points must be a multiple of D*HW");
  if (!out || !cell_start || !cell_end || !meta) return fail(BEVPOOL_EINVAL, "null argument");
  if (n_points > 0 && (!depth || !context_rows || !keys))
    return fail(BEVPOOL_EINVAL, "null depth/context/keys");
  if (reinterpret_cast<uintptr_t>(context_rows) % 16 != 0)
    return fail(BEVPOOL_EINVAL, "context rows must be 16-byte aligned");
  if (scratch_bytes < bevpool_forward_scratch_bytes(n_cells, C) || !scratch)
    return fail(BEVPOOL_ESPACE, "forward scratch too small");
  hipStream_t s = static_cast<hipStream_t>(stream);
  float *acc = static_cast<float *>(scratch);
  int st;
  if (n_points > 0) {
    const DepthRows dr{depth, make_fast_div(uint32_t(HW)), make_fast_div(uint32_t(D))};
    LaunchTimer t("accum_rows", s);
    st = launch_accum_group(BEVPOOL_F32, group_plan(BEVPOOL_F32, C, n_points, n_cells, true),
                            reinterpret_cast<const char *>(context_rows), int64_t(C) * 4, C,
                            n_points, keys, meta, cell_start, cell_end, acc, dr, false, s);
    if (st) return st;
  }
  return launch_rows_to_bev(acc, BEVPOOL_F32, C, cell_end, n_cells, n_z, n_xy,
                            out_stride_b, out_stride_c, out_stride_z, out, s);
}

// fH, fW: the image plane (HW = fH * fW); fH = 1 if its width is not known.
static int backward_depth_impl(const float *grad, int64_t grad_stride_b, int64_t grad_stride_c,
                               int64_t grad_stride_z, int32_t C, const int32_t *rank,
                               int64_t n_points, int32_t D, int64_t HW, int32_t fH,
                               const float *depth,
                               const float *context_rows, const int32_t *cell_start,
                               const int32_t *cell_end, int32_t n_batch, int32_t n_z, int64_t n_xy,
                               float *grad_depth, float *grad_context, int64_t gctx_stride_bn,
                               int64_t gctx_stride_c, void *scratch, size_t scratch_bytes,
                               void *stream) {
  if (C < 1 || C > 256) return fail(BEVPOOL_EINVAL, "C must be in [1, 256]");
  if (D < 1 || HW < 1) return fail(BEVPOOL_EINVAL, "bad depth layout");
  if (n_batch < 1 || n_z < 1 || n_xy < 1) return fail(BEVPOOL_EINVAL, "bad grid");
  const int64_t n_cells = int64_t(n_batch) * n_z * n_xy;
  if (n_cells > int64_t(INT32_MAX)) return fail(BEVPOOL_EINVAL, "too many cells");
  if (n_points < 0 || n_points > int64_t(INT32_MAX) || n_points % (int64_t(D) * HW) != 0)
    return fail(BEVPOOL_EINVAL, "n_points must be a multiple of D*HW");
  if (n_points == 0) return BEVPOOL_OK;
  if (!grad || !rank || !depth || !context_rows || !cell_start || !cell_end || !grad_depth ||
      !grad_context)
    return fail(BEVPOOL_EINVAL, "null argument");
  if (!scratch || scratch_bytes < bevpool_backward_scratch_bytes(n_cells, C, BEVPOOL_F32))
    return fail(BEVPOOL_ESPACE, "backward scratch too small");
  const int64_t n_pix = n_points / D;
  const size_t smem = size_t(2 * int64_t(D) + C) * kDgPix * sizeof(float);
  if (smem > 65536)
    return fail(BEVPOOL_EINVAL, "depth bins and channels too many (2*D + C = %lld > 1024)",
                (long long)(2 * int64_t(D) + C));
  if (HW > INT32_MAX) return fail(BEVPOOL_EINVAL, "bad depth layout");
  hipStream_t s = static_cast<hipStream_t>(stream);
  int fW = int(HW / fH);
  int pw = 4, h_tiles = int(ceil_div(fH, 4)), w_tiles = int(ceil_div(fW, 4));
  // 4 x 4 pixels per block, or 16 in a row of all HW where the image plane is
  // not known or cuts into more than 1.1 times as many patches, some of them
  // partial: a patch is at most that much faster than 16 pixels in a row.  Both
  // in us, C = 80: 24 maps of 32 x 88 (1408 blocks each) 162 and 184, 24 of 25 x
  // 41 (1848 and 1560) 82 and 68, 6 of 704 x 2 (1056 and 528) 73 and 21, 3000 of
  // 5 x 5 (12,000 and 6000) 190 and 117.
  if (int64_t(h_tiles) * w_tiles * 10 > ceil_div(HW, kDgPix) * 11) {
    pw = kDgPix;
    fH = h_tiles = 1;
    fW = int(HW);
    w_tiles = int(ceil_div(HW, kDgPix));
  }
  const int64_t n_tiles = n_pix / HW * h_tiles * w_tiles;
  int st;
  if ((st = check_grid(n_tiles + kXcds, kThreads, "depth_grad"))) return st;
  if ((st = launch_bev_to_rows(grad, 4, grad_stride_b, grad_stride_c, grad_stride_z, C,
                               cell_end, n_cells, n_z, n_xy, scratch, s)))
    return st;
  const unsigned grid = xcd_grid(n_tiles);
  LaunchTimer t("depth_grad", s);
  const float *g = static_cast<const float *>(scratch);
  uint32_t *gd = reinterpret_cast<uint32_t *>(grad_depth);
#define BEVPOOL_DG(X, R)                                                                       \
  case 5 * X + R:                                                                              \
    hipLaunchKernelGGL((depth_grad_kernel<X, R>), dim3(grid), dim3(kThreads), smem, s, g, C,    \
                       rank, depth, context_rows, D, fH, fW, pw, h_tiles, w_tiles, n_tiles,    \
                       gd, grad_context, gctx_stride_bn, gctx_stride_c);                       \
    break;
  // a lane's channels: 4 for each 64, then one for each 16 of the rest
  switch (5 * (C / 64) + (C % 64 + 15) / 16) {
    BEVPOOL_DG(0, 1) BEVPOOL_DG(0, 2) BEVPOOL_DG(0, 3) BEVPOOL_DG(0, 4)
    BEVPOOL_DG(1, 0) BEVPOOL_DG(1, 1) BEVPOOL_DG(1, 2) BEVPOOL_DG(1, 3) BEVPOOL_DG(1, 4)
    BEVPOOL_DG(2, 0) BEVPOOL_DG(2, 1) BEVPOOL_DG(2, 2) BEVPOOL_DG(2, 3) BEVPOOL_DG(2, 4)
    BEVPOOL_DG(3, 0) BEVPOOL_DG(3, 1) BEVPOOL_DG(3, 2) BEVPOOL_DG(3, 3) BEVPOOL_DG(3, 4)
    BEVPOOL_DG(4, 0)
  }
#undef BEVPOOL_DG
  return check_launch("depth_grad");
}

int bevpool_backward_depth(const float *grad, int64_t grad_stride_b, int64_t grad_stride_c,
                           int64_t grad_stride_z, int32_t C, const int32_t *rank,
                           int64_t n_points, int32_t D, int64_t HW, const float *depth,
                           const float *context_rows, const int32_t *cell_start,
                           const int32_t *cell_end, int32_t n_batch, int32_t n_z, int64_t n_xy,
                           float *grad_depth, float *grad_context, int64_t gctx_stride_bn,
                           int64_t gctx_stride_c, void *scratch, size_t scratch_bytes,
                           void *stream) {
  g_last_error.clear();
  return backward_depth_impl(grad, grad_stride_b, grad_stride_c, grad_stride_z, C, rank, n_points,
                             D, HW, 1, depth, context_rows, cell_start, cell_end, n_batch, n_z,
                             n_xy, grad_depth, grad_context, gctx_stride_bn, gctx_stride_c,
                             scratch, scratch_bytes, stream);
}

int bevpool_backward_depth_image(const float *grad, int64_t grad_stride_b, int64_t grad_stride_c,
                                 int64_t grad_stride_z, int32_t C, const int32_t *rank,
                                 int64_t n_points, int32_t D, int32_t fH, int32_t fW,
                                 const float *depth, const float *context_rows,
                                 const int32_t *cell_start, const int32_t *cell_end,
                                 int32_t n_batch, int32_t n_z, int64_t n_xy, float *grad_depth,
                                 float *grad_context, int64_t gctx_stride_bn,
                                 int64_t gctx_stride_c, void *scratch, size_t scratch_bytes,
                                 void *stream) {
  g_last_error.clear();
  if (fH < 1 || fW < 1) return fail(BEVPOOL_EINVAL, "bad feature map (%d x %d)", fH, fW);
  return backward_depth_impl(grad, grad_stride_b, grad_stride_c, grad_stride_z, C, rank, n_points,
                             D, int64_t(fH) * fW, fH, depth, context_rows, cell_start, cell_end,
                             n_batch, n_z, n_xy, grad_depth, grad_context, gctx_stride_bn,
                             gctx_stride_c, scratch, scratch_bytes, stream);
}

size_t bevpool_backward_scratch_bytes(int64_t n_cells, int32_t C, int32_t dtype) {
  if (n_cells < 0 || C < 0) return 0;
  return size_t(n_cells) * size_t(C) * dtype_size(dtype);
}

int bevpool_backward(const void *grad, int32_t dtype, int64_t grad_stride_b,
                     int64_t grad_stride_c, int64_t grad_stride_z, int32_t C,
                     const int32_t *rank, int64_t n_points, const int32_t *cell_start,
                     const int32_t *cell_end, int32_t n_batch, int32_t n_z, int64_t n_xy,
                     void *x_grad, int64_t x_grad_row_stride, int32_t zero_dropped,
                     void *scratch, size_t scratch_bytes, void *stream) {
  g_last_error.clear();
  if (dtype != BEVPOOL_F32 && dtype != BEVPOOL_F16 && dtype != BEVPOOL_BF16)
    return fail(BEVPOOL_EINVAL, "unsupported dtype code %d", dtype);
  if (C < 1) return fail(BEVPOOL_EINVAL, "C must be positive");
  if (n_batch < 1 || n_z < 1 || n_xy < 1) return fail(BEVPOOL_EINVAL, "bad grid");
  const int64_t n_cells = int64_t(n_batch) * n_z * n_xy;
  if (n_cells > int64_t(INT32_MAX)) return fail(BEVPOOL_EINVAL, "too many cells");
  if (n_points < 0 || n_points > int64_t(INT32_MAX))
    return fail(BEVPOOL_EINVAL, "n_points out of range");
  if (n_points == 0) return BEVPOOL_OK;
  if (!grad || !rank || !cell_start || !cell_end || !x_grad)
    return fail(BEVPOOL_EINVAL, "null argument");
  if (x_grad_row_stride < C) return fail(BEVPOOL_EINVAL, "bad x_grad row stride");
  if (!scratch || scratch_bytes < bevpool_backward_scratch_bytes(n_cells, C, dtype))
    return fail(BEVPOOL_ESPACE, "backward scratch too small");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const size_t es = dtype_size(dtype);
  // gather layout (decided first: the warm-up blocks mirror it)
  const size_t row_bytes = size_t(C) * es;
  const int64_t ld_bytes = int64_t(size_t(x_grad_row_stride) * es);
  const bool wide = row_bytes >= 16;  // 16-byte pieces, else elements
  const bool aligned = row_bytes % 16 == 0 && ld_bytes % 16 == 0 &&
                       reinterpret_cast<uintptr_t>(x_grad) % 16 == 0 &&
                       reinterpret_cast<uintptr_t>(scratch) % 16 == 0;
  const int vpr = wide ? int((row_bytes + 15) / 16) : int(C);
  const int64_t total = n_points * vpr;
  const int64_t gather_blocks = ceil_div(total, int64_t(kThreads));
  int st;
  // (rows that are no run of aligned pieces keep the limit of one element per thread)
  if ((st = check_grid((aligned ? gather_blocks : ceil_div(n_points * C, kThreads)) + kXcds,
                       kThreads, "gather_rows")))
    return st;
  const unsigned grid = xcd_grid(gather_blocks);
  const bool narrow = total < (int64_t(1) << 32);
  // cache warm-up (gather_warm_block): ranks per XCD + occupied rows
  GatherWarm w{};
  int rank_blocks = 0;
  if (BEVPOOL_XCD_MAP && reinterpret_cast<uintptr_t>(rank) % 16 == 0 && n_points >= 4) {
    w.rank16 = reinterpret_cast<const u32x4 *>(rank);
    w.n16 = n_points / 4;
    w.xcd_span = int64_t(grid / kXcds) * kThreads;
    w.vpr = vpr;
    const int64_t pts = ceil_div(w.xcd_span, int64_t(vpr)) + 1;
    w.per_xcd = int(ceil_div(ceil_div(pts, 4), int64_t(kThreads) * 16));  // <= 16 pieces/thread
    rank_blocks = kXcds * w.per_xcd;
  }
  int row_blocks = 0;
  if (BEVPOOL_XCD_MAP && wide) {
    w.rows = static_cast<const char *>(scratch);
    w.rowq = vpr;
    w.row_bytes = int(row_bytes);
    row_blocks = int(ceil_div(n_cells, kWarmCells));
  }
  int warm_blocks = rank_blocks + row_blocks;
  warm_blocks = int(ceil_div(warm_blocks, kXcds) * kXcds);  // keep XCD parity
  if ((st = check_grid(int64_t(grid) + warm_blocks, kThreads, "gather_rows"))) return st;
  if ((st = launch_bev_to_rows(grad, es, grad_stride_b, grad_stride_c, grad_stride_z, C,
                               cell_end, n_cells, n_z, n_xy, scratch, s)))
    return st;
  LaunchTimer t("gather_rows", s);
#define BEVPOOL_GATHER(V, NARROW, ANY)                                                         \
  hipLaunchKernelGGL((gather_rows_kernel<V, NARROW, ANY>), dim3(grid + unsigned(warm_blocks)), \
                     dim3(kThreads), 0, s, static_cast<const char *>(scratch), vpr,            \
                     int(row_bytes), rank, n_points, static_cast<char *>(x_grad), ld_bytes,    \
                     warm_blocks, w, cell_start, cell_end, n_cells, 0, zero_dropped ? 1 : 0)
#define BEVPOOL_GATHER_V(V, ANY)                                                               \
  {                                                                                            \
    if (narrow) BEVPOOL_GATHER(V, true, ANY); else BEVPOOL_GATHER(V, false, ANY);             \
  }
  if (wide && aligned) BEVPOOL_GATHER_V(u32x4, false)
  else if (wide) BEVPOOL_GATHER_V(u32x4, true)
  else if (es == 4) BEVPOOL_GATHER_V(uint32_t, false)
  else BEVPOOL_GATHER_V(uint16_t, false)
#undef BEVPOOL_GATHER_V
#undef BEVPOOL_GATHER
  return check_launch("gather_rows");
}

int bevpool_legacy_forward(const float *x, int64_t n, int32_t C, const int32_t *geom_feats,
                           const int32_t *interval_starts, const int32_t *interval_lengths,
                           int64_t n_intervals, const int32_t *n_intervals_dev, int32_t b,
                           int32_t d, int32_t h, int32_t w, float *out, int32_t *meta,
                           void *stream) {
  g_last_error.clear();
  int st = check_legacy_args(n, C, geom_feats, interval_starts, interval_lengths, n_intervals, b,
                             d, h, w, out);
  if (st) return st;
  if (n_intervals > 0 && n > 0 && !x) return fail(BEVPOOL_EINVAL, "null x");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t cells = int64_t(b) * d * h * w;
  if ((st = launch_zero_fill(out, size_t(cells) * size_t(C) * sizeof(float), s))) return st;
  if (n_intervals == 0) return BEVPOOL_OK;
  LaunchTimer t("legacy_forward", s);
  if (C >= 4) {
    const LegacyShape L = legacy_shape(C, 16, n_intervals, true);
    hipLaunchKernelGGL(legacy_sum_kernel, L.grid, dim3(kThreads), 0, s,
                       reinterpret_cast<const char *>(x), n, C, L.qmax, geom_feats,
                       interval_starts, interval_lengths, n_intervals, n_intervals_dev, b, d, h,
                       w, reinterpret_cast<char *>(out), meta);
  } else {
    hipLaunchKernelGGL(legacy_sum_narrow_kernel, legacy_shape(C, 4, n_intervals, false).grid,
                       dim3(kThreads), 0, s, x, n, C, geom_feats, interval_starts,
                       interval_lengths, n_intervals, n_intervals_dev, b, d, h, w, out, meta);
  }
  return check_launch("legacy_forward");
}

int bevpool_legacy_backward(const float *out_grad, int64_t n, int32_t C,
                            const int32_t *geom_feats, const int32_t *interval_starts,
                            const int32_t *interval_lengths, int64_t n_intervals,
                            const int32_t *n_intervals_dev, int32_t b, int32_t d, int32_t h,
                            int32_t w, float *x_grad, int32_t *meta, void *stream) {
  g_last_error.clear();
  int st = check_legacy_args(n, C, geom_feats, interval_starts, interval_lengths, n_intervals, b,
                             d, h, w, n > 0 ? x_grad : reinterpret_cast<float *>(1));
  if (st) return st;
  if (n_intervals > 0 && !out_grad) return fail(BEVPOOL_EINVAL, "null out_grad");
  hipStream_t s = static_cast<hipStream_t>(stream);
  // Intervals in order and without overlap, the usual case, write every row
  // themselves: the device decides (meta[4] holds the answer during the call;
  // a caller's leftover there only costs the fill).
  int32_t *unordered = nullptr;
  if (meta && n_intervals > 0 && n > 0) {
    unordered = meta + kMetaUnordered;
    LaunchTimer t("legacy_order", s);
    const int64_t blocks = ceil_div(n_intervals, int64_t(kThreads));
    hipLaunchKernelGGL(legacy_order_kernel, dim3(unsigned(blocks < 512 ? blocks : 512)),
                       dim3(kThreads), 0, s, interval_starts, interval_lengths, n_intervals,
                       n_intervals_dev, n, unordered);
    if ((st = check_launch("legacy_order"))) return st;
  }
  if ((st = launch_zero_fill(x_grad, size_t(n) * size_t(C) * sizeof(float), s, unordered)))
    return st;
  if (n_intervals == 0 || n == 0) return BEVPOOL_OK;
  LaunchTimer t("legacy_backward", s);
  const LegacyShape L = legacy_shape(C, C >= 4 ? 16 : 4, n_intervals, false);
#define BEVPOOL_LS(WIDE)                                                                       \
  hipLaunchKernelGGL(legacy_spread_kernel<WIDE>, L.grid, dim3(kThreads), 0, s,                 \
                     reinterpret_cast<const char *>(out_grad), n, C, L.qmax, geom_feats,        \
                     interval_starts, interval_lengths, n_intervals, n_intervals_dev, b, d, h, \
                     w, reinterpret_cast<char *>(x_grad), meta, unordered)
  if (C >= 4) BEVPOOL_LS(true); else BEVPOOL_LS(false);
#undef BEVPOOL_LS
  return check_launch("legacy_backward");
}

size_t bevpool_runs_workspace_bytes(int64_t n) {
  if (n < 0) return 0;
  return align256(size_t(ceil_div(n, kThreads) + 1) * sizeof(int32_t));
}

int bevpool_runs(const void *ranks, int32_t rank_bytes, int64_t n, int32_t *starts,
                 int32_t *lengths, int32_t *meta, void *workspace, size_t workspace_bytes,
                 void *stream) {
  g_last_error.clear();
  if (rank_bytes != 4 && rank_bytes != 8)
    return fail(BEVPOOL_EINVAL, "rank_bytes must be 4 or 8, got %d", rank_bytes);
  if (n < 0 || n > int64_t(INT32_MAX)) return fail(BEVPOOL_EINVAL, "n out of range");
  if (!meta || !workspace) return fail(BEVPOOL_EINVAL, "null meta or workspace");
  if (workspace_bytes < bevpool_runs_workspace_bytes(n))
    return fail(BEVPOOL_ESPACE, "runs workspace %zu bytes < required %zu", workspace_bytes,
                bevpool_runs_workspace_bytes(n));
  if (n > 0 && (!ranks || !starts || !lengths))
    return fail(BEVPOOL_EINVAL, "null ranks / starts / lengths");
  hipStream_t s = static_cast<hipStream_t>(stream);
  int st;
  if (n == 0) {
    LaunchTimer t("init_meta", s);
    hipLaunchKernelGGL(init_meta_kernel, dim3(1), dim3(64), 0, s, meta);
    return check_launch("init_meta");
  }
  const int64_t blocks = ceil_div(n, int64_t(kRunTile));
  if ((st = check_grid(ceil_div(n, kThreads), kThreads, "runs"))) return st;
  int32_t *bcount = static_cast<int32_t *>(workspace);
  {
    LaunchTimer t("run_count", s);
    if (rank_bytes == 4)
      hipLaunchKernelGGL(run_count_kernel<int32_t>, dim3(unsigned(blocks)), dim3(kThreads), 0, s,
                         static_cast<const int32_t *>(ranks), n, bcount, meta);
    else
      hipLaunchKernelGGL(run_count_kernel<int64_t>, dim3(unsigned(blocks)), dim3(kThreads), 0, s,
                         static_cast<const int64_t *>(ranks), n, bcount, meta);
    if ((st = check_launch("run_count"))) return st;
  }
  {
    LaunchTimer t("scan_counts", s);
    hipLaunchKernelGGL(scan_counts_kernel, dim3(1), dim3(kThreads), 0, s, bcount, blocks,
                       meta + BEVPOOL_META_N_INTERVALS);
    if ((st = check_launch("scan_counts"))) return st;
  }
  {
    LaunchTimer t("run_write", s);
    if (rank_bytes == 4)
      hipLaunchKernelGGL(run_write_kernel<int32_t>, dim3(unsigned(blocks)), dim3(kThreads), 0, s,
                         static_cast<const int32_t *>(ranks), n, bcount, starts);
    else
      hipLaunchKernelGGL(run_write_kernel<int64_t>, dim3(unsigned(blocks)), dim3(kThreads), 0, s,
                         static_cast<const int64_t *>(ranks), n, bcount, starts);
    if ((st = check_launch("run_write"))) return st;
  }
  LaunchTimer t("run_length", s);
  hipLaunchKernelGGL(run_length_kernel, dim3(unsigned(ceil_div(n, kThreads))), dim3(kThreads), 0,
                     s, starts, n, meta + BEVPOOL_META_N_INTERVALS, lengths);
  return check_launch("run_length");
}


// Checks shared by the op-level entry points.
static int op_check_sizes(int64_t n_points, int32_t B, int32_t D, int32_t H, int32_t W,
                          int32_t C) {
  if (B < 1 || D < 1 || H < 1 || W < 1) return fail(BEVPOOL_EINVAL, "B, D, H, W must be positive");
  if (C < 1) return fail(BEVPOOL_EINVAL, "C must be positive");
  if (n_points < 0 || n_points > int64_t(INT32_MAX))
    return fail(BEVPOOL_EINVAL, "n_points=%lld out of range", (long long)n_points);
  if (int64_t(B) * D * H * W > int64_t(INT32_MAX))
    return fail(BEVPOOL_EINVAL, "B*D*H*W exceeds 2^31-1");
  return BEVPOOL_OK;
}

// bevpool_op_forward with the report destination already resolved to a
// device address (or null).
static int op_forward_impl(const void *feats, int32_t dtype, int64_t feats_row_stride, int32_t C,
                           const void *coords, int32_t coord_bytes, int64_t coords_row_stride,
                           int64_t n_points, int32_t B, int32_t D, int32_t H, int32_t W,
                           void *out, void *index, size_t index_bytes, void *scratch,
                           size_t scratch_bytes, int32_t *report_dev, void *stream) {
  if (int st = op_check_sizes(n_points, B, D, H, W, C)) return st;
  const int64_t cells = int64_t(B) * D * H * W;
  if (!index || !scratch) return fail(BEVPOOL_EINVAL, "null index or scratch buffer");
  const OpIndexLayout L = op_index_layout(n_points, cells);
  if (index_bytes < L.total)
    return fail(BEVPOOL_ESPACE, "op index buffer %zu bytes < required %zu", index_bytes, L.total);
  const OpScratchLayout S = op_scratch_layout(n_points, cells, C);
  if (scratch_bytes < S.total)
    return fail(BEVPOOL_ESPACE, "op scratch %zu bytes < required %zu", scratch_bytes, S.total);
  char *ix = static_cast<char *>(index);
  char *sc = static_cast<char *>(scratch);
  int32_t *meta = reinterpret_cast<int32_t *>(ix + L.meta);
  int32_t *rank = reinterpret_cast<int32_t *>(ix + L.rank);
  uint64_t *keys = reinterpret_cast<uint64_t *>(ix + L.keys);
  int32_t *cstart = reinterpret_cast<int32_t *>(ix + L.cstart);
  int32_t *cend = reinterpret_cast<int32_t *>(ix + L.cend);
  void *iws = sc + S.index_ws;
  const size_t iws_bytes = index_layout(n_points, cells).total;
  // meta is written by the first scatter (no separate initialising launch)
  int st = coord_ranks_impl(coords, coord_bytes, n_points, coords_row_stride, B, D, H, W, rank,
                            meta, iws, iws_bytes, stream, true);
  if (st) return st;
  if ((st = sort_impl(rank, n_points, cells, keys, cstart, cend, meta, iws, iws_bytes, stream,
                      true)))
    return st;
  const int64_t hw = int64_t(H) * W;
  MetaReport rep;
  rep.meta = meta;
  rep.dst = report_dev;
  return forward_impl(feats, dtype, feats_row_stride, C, n_points, keys, cstart, cend, meta, B, D,
                      hw, int64_t(C) * D * hw, int64_t(D) * hw, hw, out, sc + S.rows,
                      size_t(cells) * size_t(C) * sizeof(float), stream, rep);
}

size_t bevpool_op_index_bytes(int64_t n_points, int64_t n_cells) {
  if (n_points < 0 || n_cells < 0) return 0;
  return op_index_layout(n_points, n_cells).total;
}

size_t bevpool_op_scratch_bytes(int64_t n_points, int64_t n_cells, int32_t C) {
  if (n_points < 0 || n_cells < 0 || C < 0) return 0;
  return op_scratch_layout(n_points, n_cells, C).total;
}

size_t bevpool_op_workspace_bytes(int64_t n_points, int64_t n_cells, int32_t C) {
  if (n_points < 0 || n_cells < 0 || C < 0) return 0;
  return op_index_layout(n_points, n_cells).total + op_scratch_layout(n_points, n_cells, C).total;
}

int bevpool_op_forward(const void *feats, int32_t dtype, int64_t feats_row_stride, int32_t C,
                       const void *coords, int32_t coord_bytes, int64_t coords_row_stride,
                       int64_t n_points, int32_t B, int32_t D, int32_t H, int32_t W, void *out,
                       void *index, size_t index_bytes, void *scratch, size_t scratch_bytes,
                       int32_t *report, void *stream) {
  g_last_error.clear();
  int32_t *report_dev = nullptr;
  if (report) {
    if (int st = report_address(report, &report_dev)) return st;
  }
  return op_forward_impl(feats, dtype, feats_row_stride, C, coords, coord_bytes,
                         coords_row_stride, n_points, B, D, H, W, out, index, index_bytes,
                         scratch, scratch_bytes, report_dev, stream);
}

int bevpool_op_forward_noalloc(const void *feats, int32_t dtype, int64_t feats_row_stride,
                               int32_t C, const void *coords, int32_t coord_bytes,
                               int64_t coords_row_stride, int64_t n_points, int32_t B, int32_t D,
                               int32_t H, int32_t W, void *out, void *stream) {
  g_last_error.clear();
  if (int st = op_check_sizes(n_points, B, D, H, W, C)) return st;
  const int64_t cells = int64_t(B) * D * H * W;
  const size_t index_bytes = op_index_layout(n_points, cells).total;
  const size_t need = index_bytes + op_scratch_layout(n_points, cells, C).total;
  if (need > kNoAllocScratchBytes)
    return fail(BEVPOOL_ESPACE,
                "the allocation-free forward needs %zu bytes of scratch for n_points=%lld, "
                "B*D*H*W=%lld, C=%d; its static scratch holds %zu (use bevpool_op_forward)",
                need, (long long)n_points, (long long)cells, C, kNoAllocScratchBytes);
  char *ws = static_cast<char *>(noalloc_scratch());
  if (!ws) return BEVPOOL_EHIP;
  g_no_alloc_call = true;
  // index first (index_bytes is a multiple of 256), then the call's scratch
  const int st = op_forward_impl(feats, dtype, feats_row_stride, C, coords, coord_bytes,
                                 coords_row_stride, n_points, B, D, H, W, out, ws, index_bytes,
                                 ws + index_bytes, kNoAllocScratchBytes - index_bytes, nullptr,
                                 stream);
  g_no_alloc_call = false;
  return st;
}

int bevpool_op_backward(const void *grad, int32_t dtype, int64_t grad_stride_b,
                        int64_t grad_stride_c, int64_t grad_stride_z, int32_t C,
                        int64_t n_points, int32_t B, int32_t D, int32_t H, int32_t W,
                        void *x_grad, int64_t x_grad_row_stride, int32_t zero_dropped,
                        const void *index, size_t index_bytes, void *scratch,
                        size_t scratch_bytes, void *stream) {
  g_last_error.clear();
  if (int st = op_check_sizes(n_points, B, D, H, W, C)) return st;
  const int64_t cells = int64_t(B) * D * H * W;
  if (!index) return fail(BEVPOOL_EINVAL, "null index buffer");
  const OpIndexLayout L = op_index_layout(n_points, cells);
  if (index_bytes < L.total)
    return fail(BEVPOOL_ESPACE, "op index buffer %zu bytes < required %zu", index_bytes, L.total);
  const char *ix = static_cast<const char *>(index);
  return bevpool_backward(grad, dtype, grad_stride_b, grad_stride_c, grad_stride_z, C,
                          reinterpret_cast<const int32_t *>(ix + L.rank), n_points,
                          reinterpret_cast<const int32_t *>(ix + L.cstart),
                          reinterpret_cast<const int32_t *>(ix + L.cend), B, D, int64_t(H) * W,
                          x_grad, x_grad_row_stride, zero_dropped, scratch, scratch_bytes,
                          stream);
}

int bevpool_timing_enable(int enable) {
  std::lock_guard<std::mutex> lk(g_timing_mu);
  g_timing_enabled = enable != 0;
  return BEVPOOL_OK;
}

int bevpool_timing_reset(void) {
  std::lock_guard<std::mutex> lk(g_timing_mu);
  for (auto &r : g_timing_pending) {
    (void)hipEventSynchronize(r.stop);
    g_event_pool.push_back(r.start);
    g_event_pool.push_back(r.stop);
  }
  g_timing_pending.clear();
  g_timing_totals.clear();
  return BEVPOOL_OK;
}

int bevpool_timing_read(char *names, int name_stride, double *total_ms, int64_t *launches,
                        int max_entries) {
  std::lock_guard<std::mutex> lk(g_timing_mu);
  for (auto &r : g_timing_pending) {
    if (hipEventSynchronize(r.stop) != hipSuccess)
      return fail(BEVPOOL_EHIP, "hipEventSynchronize failed");
    float ms = 0.0f;
    if (hipEventElapsedTime(&ms, r.start, r.stop) != hipSuccess)
      return fail(BEVPOOL_EHIP, "hipEventElapsedTime failed");
    bool found = false;
    for (auto &kv : g_timing_totals) {
      if (kv.first == r.name) {
        kv.second.ms += ms;
        kv.second.launches += 1;
        found = true;
        break;
      }
    }
    if (!found) {
      TimingTotal tt;
      tt.ms = ms;
      tt.launches = 1;
      g_timing_totals.emplace_back(r.name, tt);
    }
    g_event_pool.push_back(r.start);
    g_event_pool.push_back(r.stop);
  }
  g_timing_pending.clear();
  int n = 0;
  for (auto &kv : g_timing_totals) {
    if (n >= max_entries) break;
    if (names && name_stride > 0) {
      snprintf(names + size_t(n) * name_stride, size_t(name_stride), "%s", kv.first.c_str());
    }
    if (total_ms) total_ms[n] = kv.second.ms;
    if (launches) launches[n] = kv.second.launches;
    ++n;
  }
  return n;
}

}  // extern "C"
