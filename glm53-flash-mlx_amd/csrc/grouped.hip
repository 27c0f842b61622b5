// Sorted grouped-expert prefill for the FP8 block-scaled MoE layer.
//
//  * Route plan (grouped_fp8.py:157-203; native_indexer_plan.metal:1878-1982):
//    per-block expert histograms, one scan workgroup (expert offsets, tile
//    offsets, expert-aligned descriptors, invalid-route count), and a stable
//    scatter that ranks each route among same-expert routes of its block.
//    No sorted-activation copy is made: the GEMM gathers token rows through
//    the sorted token index.
//  * Activation split (this build's MFMA operand format): every (row,
//    128-column block) gets a power-of-two scale s with amax/s <= 448, and
//    x/s is written as hi + lo/16 with hi, lo both E4M3.  A BF16 value has 8
//    significant bits: hi keeps 4 and lo the remaining 4, so the split is
//    exact whenever lo stays in E4M3's normal range, i.e. for every element
//    with |x/s| >= 2^-6 (|x| >= amax / 28672).  Smaller elements are rounded
//    on E4M3's subnormal grid, an absolute error of at most 2^-14 * s
//    (< 2.8e-7 * amax of the row block); the MFMA then multiplies these
//    operands by the raw weight codes with no further rounding of products.
//  * Grouped GEMM (grouped_fp8.py:30-140): gfx950 v_mfma_scale_f32_16x16x128
//    with raw E4M3 weight codes as the B operand (no decode) and the hi/lo
//    activation rows as the A operand, both streamed from HBM into an LDS
//    ring by direct global->LDS loads.  Two chained MFMAs (hi rows, then lo
//    rows) cover one 128-deep scale block, the activation scale riding as
//    the MFMA's E8M0 row scale; their result, times the weight block scale,
//    accumulates in FP32 registers.
//  * Reductions: grouped FP32 slot-order restore (grouped_fp8.py:273-276) or
//    the exact Direct ascending-expert BF16 order
//    (native_indexer_plan.metal:2174-2207), each with the shared-expert add.
#include "common.h"
#include "grouped.h"
#include "mfma_fp8.h"
#include "split_fp8.h"

namespace glm53 {

// ------------------------------------------------------------ route plan --

constexpr int kPlanWaves = 16;
static_assert(kPlanBlockRoutes == 64 * kPlanWaves, "a counted block is one batch of every wavefront");

// Ranks routes first + 64 B w + 64 b + lane (wavefront w of a workgroup of
// kPlanWaves, batch b < B) among the same expert's earlier routes of its
// wavefront; a lane's peers (same id in its batch) come from one ballot per
// id bit, so a batch costs ~12 ballots and one LDS counter round trip
// instead of a loop over the routes before it.  The wavefronts' counts then
// turn into their bases: hist[w][e] = routes of expert e in the wavefronts
// before w.  Returns the workgroup's routes of expert threadIdx.x (0 past the
// last).  id is -1 past the last route.
template <int B>
__device__ __forceinline__ unsigned rank_routes(const RoutePlanArgs& a, int64_t first, int id_bits, unsigned* hist,
                                                unsigned* invalid_total, int32_t (&id)[B], unsigned (&rank)[B]) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, E = a.experts;
  unsigned* mine = hist + w * E;
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const int64_t i = first + (static_cast<int64_t>(w) * B + b) * 64 + lane;
    id[b] = i < a.routes ? a.expert_ids[i] : -1;
  }
  for (int e = lane; e < E; e += 64) mine[e] = 0;
  if (t == 0) *invalid_total = 0;
  __syncthreads();
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const int64_t i = first + (static_cast<int64_t>(w) * B + b) * 64 + lane;
    const bool valid = id[b] >= 0 && id[b] < E;
    const unsigned long long bad = __ballot(i < a.routes && !valid);
    if (lane == 0 && bad != 0) atomicAdd(invalid_total, static_cast<unsigned>(__popcll(bad)));
    unsigned long long peers = __ballot(valid);
    for (int bit = 0; bit < id_bits; ++bit) {
      const bool one = (id[b] >> bit) & 1;
      const unsigned long long ones = __ballot(one);
      peers &= one ? ones : ~ones;
    }
    const unsigned before = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(peers >> 32),
                                                      __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(peers), 0u));
    rank[b] = valid ? mine[id[b]] + before : 0u;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // every peer has read the counter
    if (valid && before == 0) mine[id[b]] = rank[b] + static_cast<unsigned>(__popcll(peers));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // before the next batch reads it
  }
  __syncthreads();
  unsigned run = 0;
  if (t < E) {
    unsigned c[kPlanWaves];
#pragma unroll
    for (int j = 0; j < kPlanWaves; ++j) c[j] = hist[j * E + t];
#pragma unroll
    for (int j = 0; j < kPlanWaves; ++j) {
      hist[j * E + t] = run;
      run += c[j];
    }
  }
  __syncthreads();
  return run;
}

// Per block of kPlanBlockRoutes routes: the routes per expert, and each
// route's rank among its expert's routes of the block (inverse holds it until
// route_scatter_kernel; -1: id out of range), so that the scatter needs no
// look at other routes.  All three launches are bound by latency: blocks of
// 1,024 leave the scan a quarter of the rows that blocks of 256 did, and the
// scatter no loop over up to 255 routes.  Count / scan / scatter at 65,536
// routes over 288 experts 5.2 / 15.9 / 10.0 -> 5.2 / 10.2 / 6.7 us.
__global__ __launch_bounds__(64 * kPlanWaves) void route_count_kernel(RoutePlanArgs a, int id_bits) {
  extern __shared__ unsigned plan_hist[];  // [kPlanWaves][experts]
  __shared__ unsigned invalid;
  const int t = threadIdx.x, w = t >> 6;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * kPlanBlockRoutes;
  int32_t id[1];
  unsigned rank[1];
  const unsigned count = rank_routes<1>(a, first, id_bits, plan_hist, &invalid, id, rank);
  if (t < a.experts) a.block_counts[static_cast<int64_t>(blockIdx.x) * a.experts + t] = count;
  if (t == 0) a.block_invalid[blockIdx.x] = invalid;
  if (first + t >= a.routes) return;
  const bool valid = id[0] >= 0 && id[0] < a.experts;
  a.inverse[first + t] = valid ? static_cast<int32_t>(plan_hist[w * a.experts + id[0]] + rank[0]) : -1;
}

// Inclusive scans of a[0..n) and b[0..n) in LDS (n <= 1024, 1024 threads,
// all of them calling): a shuffle scan inside each wavefront, then each
// thread adds the totals of the wavefronts before it.
__device__ void block_scan2_inclusive(unsigned* a, unsigned* b, int n) {
  __shared__ unsigned wave_a[16], wave_b[16];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  unsigned x = t < n ? a[t] : 0u, y = t < n ? b[t] : 0u;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const unsigned xo = __shfl_up(x, off), yo = __shfl_up(y, off);
    if (lane >= off) {
      x += xo;
      y += yo;
    }
  }
  if (lane == 63) {
    wave_a[w] = x;
    wave_b[w] = y;
  }
  __syncthreads();
  for (int i = 0; i < w; ++i) {
    x += wave_a[i];
    y += wave_b[i];
  }
  if (t < n) {
    a[t] = x;
    b[t] = y;
  }
  __syncthreads();
}

// Offsets, status and descriptors from the inclusive scans in LDS (one
// workgroup of 1024 threads).
__device__ __forceinline__ void write_plan_tables(const RoutePlanArgs& a, const unsigned* route_cum,
                                                  const unsigned* tile_cum, unsigned invalid_total) {
  const int t = threadIdx.x;
  if (t < a.experts) {
    a.route_offsets[t + 1] = route_cum[t];
    a.tile_offsets[t + 1] = tile_cum[t];
  }
  if (t == 0) {
    a.route_offsets[0] = 0;
    a.tile_offsets[0] = 0;
    a.status[0] = invalid_total;                       // invalid route count
    a.status[1] = tile_cum[a.experts - 1];             // valid descriptors
  }
  // descriptors: owner by binary search over the inclusive tile scan
  const unsigned total_tiles = tile_cum[a.experts - 1];
  for (int64_t d = t; d < a.capacity; d += 1024) {
    if (d >= total_tiles) {
      a.tile_expert[d] = 0;
      a.tile_start[d] = static_cast<int32_t>(a.routes);
      a.tile_len[d] = 0;
      continue;
    }
    int lo = 0, hi = a.experts - 1;
    while (lo < hi) {  // first e with tile_cum[e] > d
      int mid = (lo + hi) >> 1;
      if (tile_cum[mid] > d) hi = mid; else lo = mid + 1;
    }
    const unsigned first_tile = lo == 0 ? 0 : tile_cum[lo - 1];
    const unsigned first_route = lo == 0 ? 0 : route_cum[lo - 1];
    const unsigned start = first_route + (static_cast<unsigned>(d) - first_tile) * a.tile_rows;
    const unsigned end = route_cum[lo];
    a.tile_expert[d] = lo;
    a.tile_start[d] = static_cast<int32_t>(start);
    a.tile_len[d] = static_cast<int32_t>(end - start < static_cast<unsigned>(a.tile_rows) ? end - start : a.tile_rows);
  }
}

__global__ __launch_bounds__(1024) void route_scan_kernel(RoutePlanArgs a) {
  __shared__ unsigned route_cum[kPlanMaxExperts];
  __shared__ unsigned tile_cum[kPlanMaxExperts];
  __shared__ unsigned invalid_total;
  const int t = threadIdx.x;
  if (t == 0) invalid_total = 0;
  __syncthreads();
  // per-expert running base over blocks (exclusive), totals per expert
  if (t < a.experts) {
    unsigned run = 0;
    int64_t b = 0;
    for (; b + 32 <= a.blocks; b += 32) {  // 32 loads in flight per round trip
      unsigned c[32];
#pragma unroll
      for (int j = 0; j < 32; ++j) c[j] = a.block_counts[(b + j) * a.experts + t];
#pragma unroll
      for (int j = 0; j < 32; ++j) {
        a.block_counts[(b + j) * a.experts + t] = run;
        run += c[j];
      }
    }
    for (; b + 8 <= a.blocks; b += 8) {
      unsigned c[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) c[j] = a.block_counts[(b + j) * a.experts + t];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        a.block_counts[(b + j) * a.experts + t] = run;
        run += c[j];
      }
    }
    for (; b < a.blocks; ++b) {
      unsigned c = a.block_counts[b * a.experts + t];
      a.block_counts[b * a.experts + t] = run;
      run += c;
    }
    route_cum[t] = run;
    tile_cum[t] = (run + a.tile_rows - 1) / a.tile_rows;
  }
  for (int64_t b = t; b < a.blocks; b += 1024) atomicAdd(&invalid_total, a.block_invalid[b]);
  __syncthreads();
  block_scan2_inclusive(route_cum, tile_cum, a.experts);
  write_plan_tables(a, route_cum, tile_cum, invalid_total);
}

__global__ __launch_bounds__(256) void route_scatter_kernel(RoutePlanArgs a) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= a.routes) return;
  const int32_t e = a.expert_ids[i], rank = a.inverse[i];
  if (rank < 0) return;  // an id out of range
  const int64_t pos = static_cast<int64_t>(a.route_offsets[e]) +
                      a.block_counts[i / kPlanBlockRoutes * a.experts + e] + rank;
  a.sorted_route[pos] = static_cast<int32_t>(i);
  a.inverse[i] = static_cast<int32_t>(pos);
  a.sorted_expert[pos] = e;
  a.sorted_token[pos] = static_cast<int32_t>(static_cast<uint32_t>(i) / static_cast<uint32_t>(a.top_k));
  if (a.scores != nullptr) a.sorted_score[pos] = a.scores[i];
}

// ------------------------------------------------ activation hi/lo split --

// Rounds V floats to BF16 and stores them (one 16-byte store for V = 8).
template <int V>
__device__ __forceinline__ void store_bf16_run(uint16_t* p, const float* v) {
  if constexpr (V == 8) {
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[i] = static_cast<uint32_t>(f32_to_bf16(v[2 * i])) | (static_cast<uint32_t>(f32_to_bf16(v[2 * i + 1])) << 16);
    *reinterpret_cast<uint4*>(p) = make_uint4(o[0], o[1], o[2], o[3]);
  } else {
#pragma unroll
    for (int i = 0; i < V; ++i) p[i] = f32_to_bf16(v[i]);
  }
}

// Wavefront = one row x (V / 2) consecutive 128-column blocks; lane l holds
// V columns of block l / (128 / V).  V = 8 (16-byte loads, each block's amax
// a reduction over one 16-lane DPP row) when the rows are 16-byte aligned,
// V = 2 (one block per wavefront) otherwise, into row-major planes or (V = 2
// only) planes in operand order.
template <int V, bool OPERAND>
__device__ __forceinline__ void split_unit(const SplitArgs& a, int64_t unit, int lane) {
  constexpr int kLanesPerBlock = kBlock / V;
  constexpr int kBlocksPerWave = 64 / kLanesPerBlock;
  const int64_t blocks_per_row = a.cols / kBlock;
  const int64_t groups = (blocks_per_row + kBlocksPerWave - 1) / kBlocksPerWave;
  if (unit >= a.rows * groups) return;
  const int64_t row = unit / groups;
  const int64_t blk = (unit % groups) * kBlocksPerWave + lane / kLanesPerBlock;
  const bool valid = blk < blocks_per_row;
  const int64_t col = blk * kBlock + V * (lane % kLanesPerBlock);
  Bf16Run<V> x;
  x.clear();
  if (valid) x.load(a.x + row * a.x_row_stride + col);
  bool has_nan;
  float amax = lane_amax<V>(x, has_nan);
  if constexpr (kLanesPerBlock == 64) {
    amax = wave_max(amax);
  } else {
    static_assert(kLanesPerBlock == 16, "a block spans one DPP row or the whole wavefront");
    amax = row16_amax(amax);
  }
  const SplitScale s = split_scale(amax);
  uint32_t hi[(V + 3) / 4], lo[(V + 3) / 4];
  split_encode<V>(x, s, has_nan, hi, lo);
  if (!valid) return;
  if constexpr (V == 8) {
    static_assert(!OPERAND, "split_operand_kernel");
    const int64_t off = row * a.cols + col;
    *reinterpret_cast<uint2*>(a.hi + off) = make_uint2(hi[0], hi[1]);
    *reinterpret_cast<uint2*>(a.lo + off) = make_uint2(lo[0], lo[1]);
  } else {
    static_assert(V == 2, "narrow split handles two columns per lane");
    const int64_t off = OPERAND ? operand_order_offset(row, col, a.rows, a.cols) : row * a.cols + col;
    *reinterpret_cast<uint16_t*>(a.hi + off) = static_cast<uint16_t>(hi[0]);
    *reinterpret_cast<uint16_t*>(a.lo + off) = static_cast<uint16_t>(lo[0]);
  }
  if (lane % kLanesPerBlock == 0) a.scale[row * blocks_per_row + blk] = s.s;
}

// The split into planes in operand order, 16-byte aligned rows: wavefront = 8
// rows x one 128-column block, lane l the 16 columns from 16 (l % 8) of row l
// / 8, which are one 16-byte piece of the operand, so that the 8 lanes of a
// piece write 128 consecutive bytes (one row per wavefront, as above, writes
// 8 bytes here and there, which cost the 300-row linear more than its kernel
// gained).
__global__ __launch_bounds__(256) void split_operand_kernel(SplitArgs a) {
  const int lane = threadIdx.x & 63, piece = lane & 7;
  const int64_t unit = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  const int64_t blocks_per_row = a.cols / kBlock;
  if (unit >= (a.rows + 7) / 8 * blocks_per_row) return;
  const int64_t blk = unit % blocks_per_row;
  const int64_t row = unit / blocks_per_row * 8 + (lane >> 3);
  const bool valid = row < a.rows;
  Bf16Run<8> x[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    x[j].clear();
    if (valid) x[j].load(a.x + row * a.x_row_stride + blk * kBlock + 16 * piece + 8 * j);
  }
  bool has_nan[2];
  float amax = lane_amax<8>(x[0], has_nan[0]);
  amax = fmaxf(amax, lane_amax<8>(x[1], has_nan[1]));
  amax = fmaxf(amax, dpp_f32<0xB1>(amax));
  amax = fmaxf(amax, dpp_f32<0x4E>(amax));
  amax = fmaxf(amax, dpp_f32<0x141>(amax));  // the row's amax in its 8 lanes
  const SplitScale s = split_scale(amax);
  uint32_t hi[2][2], lo[2][2];
#pragma unroll
  for (int j = 0; j < 2; ++j) split_encode<8>(x[j], s, has_nan[j], hi[j], lo[j]);
  if (!valid) return;
  const int64_t off = operand_order_offset(row, blk * kBlock + 16 * piece, a.rows, a.cols);
  *reinterpret_cast<u32x4*>(a.hi + off) = (u32x4){hi[0][0], hi[0][1], hi[1][0], hi[1][1]};
  *reinterpret_cast<u32x4*>(a.lo + off) = (u32x4){lo[0][0], lo[0][1], lo[1][0], lo[1][1]};
  if (piece == 0) a.scale[row * blocks_per_row + blk] = s.s;
}

template <int V, bool OPERAND>
__global__ __launch_bounds__(256) void split_activations_kernel(SplitArgs a) {
  split_unit<V, OPERAND>(a, static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6), threadIdx.x & 63);
}

// The whole route plan of up to kPlanOneLaunchRoutes routes in one workgroup,
// wavefront w's run of B batches held in registers from one round of loads.
// Bound by latency: 5.4 us at 512 routes and 8.4 at 2,048 over 288 experts,
// where the three launches of 256-route blocks took 11.7 and 12.3; at 3,072
// and 4,096 (11.7 and 13.7 with four batches against 13.3 and 13.0) one
// workgroup's batches cost what the launches do, so larger plans keep those.
template <int B>
__device__ __forceinline__ void route_plan_one(const RoutePlanArgs& a, int id_bits, unsigned* hist,
                                               unsigned* route_cum, unsigned* tile_cum, unsigned* invalid_total) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, E = a.experts;
  int32_t id[B];
  unsigned rank[B];
  const unsigned count = rank_routes<B>(a, 0, id_bits, hist, invalid_total, id, rank);
  if (t < E) {
    route_cum[t] = count;
    tile_cum[t] = (count + a.tile_rows - 1) / a.tile_rows;
  }
  __syncthreads();
  block_scan2_inclusive(route_cum, tile_cum, E);
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const int64_t i = (static_cast<int64_t>(w) * B + b) * 64 + lane;
    const int32_t e = id[b];
    if (i >= a.routes) continue;
    if (e < 0 || e >= E) {
      a.inverse[i] = -1;
      continue;
    }
    const int64_t pos = static_cast<int64_t>((e == 0 ? 0u : route_cum[e - 1]) + hist[w * E + e] + rank[b]);
    a.sorted_route[pos] = static_cast<int32_t>(i);
    a.inverse[i] = static_cast<int32_t>(pos);
    a.sorted_expert[pos] = e;
    a.sorted_token[pos] = static_cast<int32_t>(static_cast<uint32_t>(i) / static_cast<uint32_t>(a.top_k));
    if (a.scores != nullptr) a.sorted_score[pos] = a.scores[i];
  }
  write_plan_tables(a, route_cum, tile_cum, *invalid_total);
}

// Workgroup 0: the plan.  The others: the activation split of the same call
// (V as in split_activations_kernel; s.rows = 0: none), which needs nothing
// of the plan and would otherwise be a launch of its own.
template <int V>
__global__ __launch_bounds__(1024) void route_plan_one_kernel(RoutePlanArgs a, int id_bits, SplitArgs s) {
  extern __shared__ unsigned plan_hist[];  // [kPlanWaves][experts]
  __shared__ unsigned route_cum[kPlanMaxExperts];
  __shared__ unsigned tile_cum[kPlanMaxExperts];
  __shared__ unsigned invalid_total;
  if (blockIdx.x > 0) {
    split_unit<V, false>(s, static_cast<int64_t>(blockIdx.x - 1) * kPlanWaves + (threadIdx.x >> 6), threadIdx.x & 63);
    return;
  }
  static_assert(kPlanOneLaunchRoutes <= 2 * 64 * kPlanWaves, "two batches per wavefront at most");
  if (a.routes <= 64 * kPlanWaves) route_plan_one<1>(a, id_bits, plan_hist, route_cum, tile_cum, &invalid_total);
  else route_plan_one<2>(a, id_bits, plan_hist, route_cum, tile_cum, &invalid_total);
}

// --------------------------------------------------------- grouped GEMM --
//
// Workgroup = 4 wavefronts on one work item: one descriptor (32 GPW routes
// of one expert, 2 GPW pairs of 16) times one 128-row weight tile.  Per
// 128-deep K block (a "stage"):
//   * B: the tile's 128 weight rows of raw E4M3 codes (16 KB),
//   * A: per 16-route pair, one 16-row operand tile of the routes' hi rows
//     and one of their lo rows, gathered through the sorted token index
//     (2 x 2 KB),
// both brought straight from global memory into an LDS ring by direct loads
// (global_load_lds_dwordx4: lane l's 16 bytes land at base + 16 l), so no
// registers hold data in flight and the ring's other stages stream while
// one is multiplied.  Each direct load reads 8 rows as whole 128-byte lines
// (a 16-row operand tile takes two); in LDS a row's 16-byte pieces are
// permuted by an XOR of the row index, so the MFMA lane (r = l % 16, q =
// l / 16) reads its 32 operand bytes (row r, bytes 32 q .. 32 q + 31) as two
// conflict-free 16-byte LDS reads (operand_slots).  Whole lines per load
// stream weight tiles about 14% faster than 64 bytes of 16 rows per load.
// Per (pair, weight tile) two chained v_mfma_scale_f32_16x16x128_f8f6f4
// (pair_pass): hi rows x tile, then lo rows x tile added into the same
// result, with the route's activation block scale (a power of two) as the A
// rows' E8M0 scale and the lo pass's 1/16 as the B scale; the result, times
// the tile's weight block scale, accumulates in FP32 (one FMA per element).
// Lane l holds routes 4 (l / 16) .. 4 (l / 16) + 3 of the pair in column
// l % 16 of the tile.  Two shapes: GPW = 2 (64-route descriptors, 2-stage
// ring; wavefront w multiplies pair w against the 8 tiles) for many routes
// per expert, GPW = 1 (32 routes, 3-stage ring; wavefront w multiplies pair
// w / 2 against half of the tiles) otherwise.  Every shape computes each
// output element by the same sequence of operations, so all give the same
// bits.
//
// mode GEMM_PLAIN : the tile is output columns [128 tile, +128).
// mode GEMM_SWIGLU: the tile is gate rows j in [64 tile, +64) (tiles 0-3)
//   and the matching up rows (tiles 4-7), so h = SwiGLU(T(gate), T(up))
//   forms in registers.

namespace {

constexpr int kTileRows = 128;                     // weight rows per work item
constexpr int kStageB = (kTileRows / 16) * kOperand;  // 16 KB
// LDS ring depth of each shape: two slots (48 KB for 32-route
// descriptors, whose stages stream through registers kRegAhead stages
// ahead; 64 KB for 64-route descriptors, whose direct loads keep one stage
// in flight); two workgroups per CU either way.
template <int GPW>
constexpr int ring_stages() {
  return 2;
}
// Stages the register-staged shape (GPW = 1) keeps in flight in registers
constexpr int kRegAhead = 2;
// Descriptors of 32 GPW routes: 2 GPW pairs of 16, i.e. 4 GPW activation
// operand tiles (hi and lo rows of each pair) per stage
template <int GPW>
constexpr int stage_bytes() {
  return kStageB + 4 * GPW * kOperand;
}
static_assert(kGemmTileRows == 64 && kGemmMinTileRows == 32, "descriptor sizes of the two GEMM shapes");

// Direct global -> LDS load of 16 bytes per lane; lane l writes lds_base +
// 16 l (lds_base wave-uniform).  Written as inline assembly so that the only
// wait on it is the counted one in stage_barrier: the compiler otherwise
// drains every direct load before any LDS read it cannot prove disjoint.
__device__ __forceinline__ void lds_direct16(const uint8_t* g, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds_base) : "memory", "m0");
}

// The same load addressed as base + off: base wave-uniform (held in SGPRs),
// off a per-lane unsigned 32-bit offset, so a loop-invariant source costs
// one VGPR instead of a 64-bit address pair.
__device__ __forceinline__ void lds_direct16_at(const uint8_t* base, uint32_t off, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds_base)
               : "memory", "m0");
}

// Waits until at most N of this wavefront's vector-memory loads are in
// flight and its LDS reads have returned, then joins the workgroup barrier.
template <int N>
__device__ __forceinline__ void stage_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

}  // namespace

// What a work item reads and writes: the routed problem's operands or the
// dense problem's (GroupedGemmArgs.x_*), chosen per item.
struct ItemSource {
  const uint8_t* a_hi;
  const uint8_t* a_lo;
  const float* a_scale;
  const int32_t* a_row_index;
  int64_t routes;
  const int32_t* tile_expert;
  const int32_t* tile_start;
  const int32_t* tile_len;
  int64_t experts;
  const uint8_t* weight;
  const uint8_t* weight_up;
  int wg;  // row groups of the weight matrices (common.h)
  const float* scale;
  const float* scale_up;
  uint16_t* out;
  int64_t out_row_stride;
};

// Stores a wavefront's BF16 results: v[j][t][i / 2] holds, in its low half
// for even i and its high half for odd i, route 16 (p0 + pstep j) + 4 (l /
// 16) + i of the item and output column c0 + 16 t + l % 16.  Buffer stores
// against a record that ends after the item's len rows: a route past len
// lies outside it, a column past N is given an offset outside it, and the
// hardware drops both, so the stores need no branches.  (The host keeps
// out_row_stride below 2^22, so every offset fits 32 bits.)
template <int NP, int T>
__device__ __forceinline__ void store_item_rows(const ItemSource& src, int32_t start, int32_t len, int p0, int pstep,
                                                int64_t c0, int64_t N, const uint32_t (&v)[NP > 0 ? NP : 1][T][2],
                                                int lane) {
  const int n16 = lane & 15, kq = lane >> 4;
  const uint32_t stride2 = 2u * static_cast<uint32_t>(src.out_row_stride);
  const __amdgpu_buffer_rsrc_t rec = __builtin_amdgcn_make_buffer_rsrc(
      src.out + static_cast<int64_t>(start) * src.out_row_stride, 0, static_cast<int>(stride2 * len), 0x00020000);
  uint32_t coff[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int64_t c = c0 + 16 * t + n16;
    coff[t] = c < N ? 2u * static_cast<uint32_t>(c) : 0x80000000u;
  }
#pragma unroll
  for (int j = 0; j < NP; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t roff = stride2 * static_cast<uint32_t>(16 * (p0 + pstep * j) + 4 * kq + i);
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const uint16_t bits = static_cast<uint16_t>(i & 1 ? v[j][t][i >> 1] >> 16 : v[j][t][i >> 1]);
        __builtin_amdgcn_raw_buffer_store_b16(bits, rec, static_cast<int>(roff + coff[t]), 0, 0);
      }
    }
}

// SWIGLU epilogue of a wavefront: pair j of the wavefront is descriptor
// pair p0 + pstep j; lane l holds, for its routes 16 p + 4 (l / 16) + i,
// gate tiles 0 .. T - 1 in acc[j][t] and the matching up tiles in
// acc[j][t + T]; output column c0 + 16 t + l % 16.  Every value takes the
// straight-line form, two at a time; a wavefront with a value outside its
// range (|T(g)| > 87, NaN or T(g) = 0xC0DB: rare) recomputes all of its
// values with swiglu_mlx.
template <int NP, int T>
__device__ __forceinline__ void swiglu_epilogue(const GroupedGemmArgs& a, const ItemSource& src, int32_t start,
                                                int32_t len, int p0, int pstep, int64_t c0,
                                                const float (&acc)[NP > 0 ? NP : 1][2 * T][4], int lane) {
  uint32_t h[NP > 0 ? NP : 1][T][2];
  SwigluCheck check;
#pragma unroll
  for (int j = 0; j < NP; ++j)
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int q = 0; q < 2; ++q)
        h[j][t][q] = swiglu_mlx_straight2(acc[j][t][2 * q], acc[j][t + T][2 * q], acc[j][t][2 * q + 1],
                                          acc[j][t + T][2 * q + 1], a.limit, check);
  if (__builtin_amdgcn_ballot_w64(!swiglu_straight_ok(check, a.limit)) != 0) {
#pragma unroll
    for (int j = 0; j < NP; ++j)
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int q = 0; q < 2; ++q)
          h[j][t][q] = swiglu_mlx(acc[j][t][2 * q], acc[j][t + T][2 * q], a.limit) |
                       static_cast<uint32_t>(swiglu_mlx(acc[j][t][2 * q + 1], acc[j][t + T][2 * q + 1], a.limit)) << 16;
  }
  store_item_rows<NP, T>(src, start, len, p0, pstep, c0, a.N, h, lane);
}

// PLAIN epilogue of a wavefront: acc[j][t] holds output columns c0 + 16 t
// + l % 16 of routes 16 (p0 + pstep j) + 4 (l / 16) + i, stored as BF16.
template <int NP, int T>
__device__ __forceinline__ void plain_epilogue(const GroupedGemmArgs& a, const ItemSource& src, int32_t start,
                                               int32_t len, int p0, int pstep, int64_t c0,
                                               const float (&acc)[NP > 0 ? NP : 1][T][4], int lane) {
  uint32_t h[NP > 0 ? NP : 1][T][2];
#pragma unroll
  for (int j = 0; j < NP; ++j)
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int q = 0; q < 2; ++q) h[j][t][q] = f32x2_to_bf16x2(acc[j][t][2 * q], acc[j][t][2 * q + 1]);
  store_item_rows<NP, T>(src, start, len, p0, pstep, c0, a.N, h, lane);
}

// Wavefront w's share of a work item: it loads weight tiles 2 w, 2 w + 1 and
// activation tiles GPW w .. GPW w + GPW - 1 of every stage (NL of them: none
// when their pair has no routes), and multiplies one pair (NP = 1; NP = 0
// when the pair has no routes) against T weight tiles: GPW = 2 pair w
// against all 8 tiles, GPW = 1 pair w / 2 against the tiles of half h =
// w % 2 (PLAIN: tiles 4 h .. 4 h + 3; SWIGLU: gate tiles 2 h, 2 h + 1 and
// the matching up tiles).
// DETECT: found collects, in bit 7 of each byte, whether the weight codes the
// wavefront staged hold 0x7F / 0xFF (codes_480).
template <int MODE, bool FIX, int GPW, int NP, bool DETECT>
__device__ __forceinline__ void grouped_gemm_loop(const GroupedGemmArgs& a, const ItemSource src, int64_t ntile,
                                                  int32_t start, int32_t len, int64_t KB,
                                                  const uint8_t* const (&gb)[2][2], const uint8_t* const (&ga)[GPW][2],
                                                  uint8_t* lds, uint32_t lds_addr, const uint8_t* lds_se,
                                                  const float* lds_sw, int wave, int lane, uint32_t& found) {
  static_assert(!DETECT || GPW == 1, "codes are looked at where the weights stream through registers");
  constexpr int kStage = stage_bytes<GPW>();
  constexpr int kRoutes = 32 * GPW;
  constexpr int NL = GPW == 2 ? 2 * NP : NP;  // activation tiles this wavefront loads per stage
  constexpr int P = 4 + 2 * NL;               // its direct loads per stage
  constexpr int T = GPW == 2 ? 8 : 4;         // weight tiles it multiplies
  const int pair = GPW == 2 ? wave : wave >> 1;
  const int half = wave & 1;
  const OperandSlots slots = operand_slots(lane);
  auto issue = [&](int64_t kb, int slot) {
    const int64_t ko = kb * kBlock;        // activation rows: row-major
    const int64_t kw = kb << (7 + src.wg);  // weight rows: K block kb of the row group
    const uint32_t sb = lds_addr + slot * kStage + 2 * wave * kOperand;
    lds_direct16(gb[0][0] + kw, sb);
    lds_direct16(gb[0][1] + kw, sb + 1024);
    lds_direct16(gb[1][0] + kw, sb + kOperand);
    lds_direct16(gb[1][1] + kw, sb + kOperand + 1024);
    const uint32_t sa = lds_addr + slot * kStage + kStageB + GPW * wave * kOperand;
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      lds_direct16(ga[j][0] + ko, sa + j * kOperand);
      lds_direct16(ga[j][1] + ko, sa + j * kOperand + 1024);
    }
  };
  // the LDS weight tile of local tile tt, and whether it holds up rows
  auto tile_of = [&](int tt) {
    if (GPW == 2) return tt;
    return MODE == GEMM_PLAIN ? 4 * half + tt : (tt < 2 ? 2 * half + tt : 4 + 2 * half + tt - 2);
  };
  auto up_tile = [&](int tt) { return MODE == GEMM_SWIGLU && tt >= T / 2; };

  float acc[NP > 0 ? NP : 1][T][4];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[0][t][i] = 0.0f;

  // one stage's MFMAs on the operands in LDS slot `slot`
  auto compute = [&](int64_t kb, int slot) {
    if (NP > 0) {
      const uint8_t* st = lds + slot * kStage;
      const i32x8 ahi = lds_operand(st + kStageB + (2 * pair) * kOperand, slots);
      const i32x8 alo = lds_operand(st + kStageB + (2 * pair + 1) * kOperand, slots);
      const int se = lds_se[kb * kRoutes + 16 * pair + (lane & 15)];
      const float sw_lo = lds_sw[kb];
      const float sw_hi = MODE == GEMM_SWIGLU ? lds_sw[KB + kb] : sw_lo;
      i32x8 bq[T], bc[T];  // every weight tile read ahead: one LDS wait per stage
#pragma unroll
      for (int tt = 0; tt < T; ++tt) {
        bq[tt] = lds_operand(st + tile_of(tt) * kOperand, slots);
        weight_operand<FIX>(bq[tt], bc[tt]);
      }
      // Each tile's hi pass issues T MFMAs before its lo pass reads the
      // result, and tile tt is folded into the accumulators after tile
      // tt + 1's lo pass is issued: the MFMAs of a stage issue back to back
      // while the folding runs beside them.
      f32x4 c[T];
#pragma unroll
      for (int tt = 0; tt < T; ++tt)
        c[tt] = pair_pass<FIX, 0, 127>(ahi, bq[tt], bc[tt], (f32x4){0.0f, 0.0f, 0.0f, 0.0f}, se);
      auto fold = [&](int tt) {
        const float sw = up_tile(tt) ? sw_hi : sw_lo;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[0][tt][i] = fmaf(c[tt][i], sw, acc[0][tt][i]);
      };
#pragma unroll
      for (int tt = 0; tt < T; ++tt) {
        c[tt] = pair_pass<FIX, 0, 123>(alo, bq[tt], bc[tt], c[tt], se);
        if (tt > 0) fold(tt - 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      fold(T - 1);
    }
  };

  constexpr int kStages = ring_stages<GPW>();
  if constexpr (GPW == 1) {
    // Register-staged stream: each stage's operand bytes come with plain
    // 16-byte loads (the same 8 rows x 128 bytes per instruction as the
    // direct loads) kRegAhead stages ahead into registers and are written to
    // the LDS slot at the positions the direct loads would fill; a 2-slot
    // ring, one barrier per stage.  Every load is compiler-visible, so each
    // wait is the exact one.  A weight-streaming read probe moved 6.4-6.5
    // TB/s this way against 5.6-5.8 TB/s with direct loads.
    static_assert(kStages == 2, "the register-staged shape double-buffers its LDS");
    struct Staged {
      u32x4 b[4];
      u32x4 a[NL > 0 ? 2 * NL : 1];
    };
    auto load = [&](int64_t kb, Staged& r) {
      const int64_t ko = kb * kBlock;
      const int64_t kw = kb << (7 + src.wg);
      r.b[0] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(gb[0][0] + kw));
      r.b[1] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(gb[0][1] + kw));
      r.b[2] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(gb[1][0] + kw));
      r.b[3] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(gb[1][1] + kw));
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        r.a[2 * j] = *reinterpret_cast<const u32x4*>(ga[j][0] + ko);
        r.a[2 * j + 1] = *reinterpret_cast<const u32x4*>(ga[j][1] + ko);
      }
    };
    auto store = [&](int slot, const Staged& r) {
      if constexpr (DETECT) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) found |= codes_480(r.b[i][j]);
      }
      uint8_t* sb = lds + slot * kStage + 2 * wave * kOperand + 16 * lane;
      *reinterpret_cast<u32x4*>(sb) = r.b[0];
      *reinterpret_cast<u32x4*>(sb + 1024) = r.b[1];
      *reinterpret_cast<u32x4*>(sb + kOperand) = r.b[2];
      *reinterpret_cast<u32x4*>(sb + kOperand + 1024) = r.b[3];
      uint8_t* sa = lds + slot * kStage + kStageB + GPW * wave * kOperand + 16 * lane;
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        *reinterpret_cast<u32x4*>(sa + j * kOperand) = r.a[2 * j];
        *reinterpret_cast<u32x4*>(sa + j * kOperand + 1024) = r.a[2 * j + 1];
      }
    };
    // stage kb's bytes sit in r[kb % kRegAhead] until written to slot kb % 2;
    // stages past the last K block are never loaded or written
    // prologue loads are unconditional too: a block index past the last
    // K block re-reads the last one (only when KB <= kRegAhead), never stored
    auto clamp_kb = [&](int64_t kb) { return kb < KB ? kb : KB - 1; };
    Staged r[kRegAhead];
#pragma unroll
    for (int q = 0; q < kRegAhead; ++q) load(clamp_kb(q), r[q]);
    store(0, r[0]);
    load(clamp_kb(kRegAhead), r[0]);
    // Each stage: wait at the barrier (slot kb % 2 written by every
    // wavefront, all done reading slot (kb + 1) % 2, stage kb - 1), write
    // stage kb + 1 into that slot, load stage kb + 1 + kRegAhead into the
    // registers it leaves, multiply stage kb.  The main loop's loads are
    // unconditional, so the compiler's count of the loads in flight stays
    // exact (a conditional load made it wait for all of them).
    int64_t kb0 = 0;
    for (; kb0 + 2 * kRegAhead < KB; kb0 += kRegAhead) {
#pragma unroll
      for (int q = 0; q < kRegAhead; ++q) {
        const int64_t kb = kb0 + q;
        const int qn = (q + 1) % kRegAhead;
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        store(static_cast<int>((kb + 1) & 1), r[qn]);
        load(kb + 1 + kRegAhead, r[qn]);
        compute(kb, static_cast<int>(kb & 1));
      }
    }
    for (; kb0 < KB; kb0 += kRegAhead) {
#pragma unroll
      for (int q = 0; q < kRegAhead; ++q) {
        const int64_t kb = kb0 + q;
        if (kb >= KB) break;
        const int qn = (q + 1) % kRegAhead;
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (kb + 1 < KB) {
          store(static_cast<int>((kb + 1) & 1), r[qn]);
          if (kb + 1 + kRegAhead < KB) load(kb + 1 + kRegAhead, r[qn]);
        }
        compute(kb, static_cast<int>(kb & 1));
      }
    }
  } else {
#pragma unroll
    for (int s = 0; s < kStages - 1; ++s)
      if (s < KB) issue(s, s);
    int slot = 0;
    for (int64_t kb = 0; kb < KB; ++kb) {
      if (kb + kStages - 2 < KB) stage_barrier<P * (kStages - 2)>();
      else stage_barrier<0>();
      if (kb + kStages - 1 < KB) issue(kb + kStages - 1, slot == 0 ? kStages - 1 : slot - 1);
      compute(kb, slot);
      slot = slot == kStages - 1 ? 0 : slot + 1;
    }
  }

  // epilogue: lane holds routes 16 pair + 4 kq + i, column 16 tile + l % 16
  // (PLAIN: the wavefront's tiles tile_of(tt) are contiguous from tile_of(0))
  if (MODE == GEMM_PLAIN)
    plain_epilogue<NP, T>(a, src, start, len, pair, 1, ntile * kTileRows + tile_of(0) * 16, acc, lane);
  if (MODE == GEMM_SWIGLU)
    swiglu_epilogue<NP, T / 2>(a, src, start, len, pair, 1, ntile * (kTileRows / 2) + (GPW == 2 ? 0 : 32 * half), acc,
                               lane);
}

// Activation block scales of a work item's ROUTES routes into LDS as E8M0
// codes, K-block-major: [kb][r], or for the wide shape (WIDE)
// [kb][r % 16][r / 16], so that a lane reads the codes of its row in all
// eight pairs as one 8-byte word.  THREADS / ROUTES
// threads per route, each with its route's token row, eight loads in
// flight per thread, then the stores; indices past the last K block are
// clamped to it, so every load and store is unconditional (a clamped store
// writes the code that block's store writes) and the compiler's wait
// tracking sees every load consumed before the K loop.  Routes past the
// descriptor's end repeat its last route.
template <int ROUTES, int THREADS, bool WIDE>
__device__ __forceinline__ void load_activation_scales(const ItemSource& src, int32_t start, int32_t len,
                                                       int64_t KB, uint8_t* lds_se) {
  constexpr int TPR = THREADS / ROUTES;
  static_assert(TPR * ROUTES == THREADS, "threads split evenly over the routes");
  const int r = static_cast<int>(threadIdx.x) / TPR, sub = static_cast<int>(threadIdx.x) % TPR;
  const int64_t route = start + (r < len ? r : len - 1);
  const int64_t token = src.a_row_index != nullptr ? src.a_row_index[route] : route;
  const float* row = src.a_scale + token * KB;
  const int64_t pos = WIDE ? ((r & 15) * 8 + (r >> 4)) : r;
  constexpr int64_t kStride = WIDE ? 128 : ROUTES;  // bytes per K block
  for (int64_t kb0 = sub; kb0 < KB; kb0 += 8 * TPR) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int64_t kb = kb0 + u * TPR;
      v[u] = row[kb < KB ? kb : KB - 1];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int64_t kb = kb0 + u * TPR;
      lds_se[(kb < KB ? kb : KB - 1) * kStride + pos] = static_cast<uint8_t>(scale_e8m0(v[u]));
    }
  }
}

// routes start .. start + len - 1 (len <= 32 GPW) of one expert x column tile ntile
template <int MODE, bool FIX, int GPW, bool DETECT>
__device__ __forceinline__ uint32_t grouped_gemm_part(const GroupedGemmArgs& a, const ItemSource src, int64_t ntile,
                                                      int32_t expert, int32_t start, int32_t len, uint8_t* lds) {
  constexpr int kRoutes = 32 * GPW;
  constexpr int kStage = stage_bytes<GPW>();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int64_t K = a.K;
  const int64_t KB = K / kBlock;
  const int pairs = (len + 15) >> 4;
  uint8_t* lds_se = lds + ring_stages<GPW>() * kStage;                    // [KB][kRoutes]
  float* lds_sw = reinterpret_cast<float*>(lds_se + kRoutes * KB);        // [2][KB]

  // ---- block scales of the work item: activations of every route, weights
  // of the tile (one 128-row scale block: PLAIN tiles are 128-aligned, SWIGLU
  // tiles 64-aligned within one block)
  auto token_of = [&](int r) -> int64_t {
    const int64_t route = start + (r < len ? r : len - 1);
    return src.a_row_index != nullptr ? src.a_row_index[route] : route;
  };
  load_activation_scales<kRoutes, 256, false>(src, start, len, KB, lds_se);
  const int64_t srow = MODE == GEMM_PLAIN ? ntile : (ntile >> 1);
  const int64_t soff = static_cast<int64_t>(expert) * a.s_expert_stride + srow * a.s_cols;
  for (int64_t i = threadIdx.x; i < (MODE == GEMM_SWIGLU ? 2 : 1) * KB; i += 256)
    lds_sw[i] = i < KB ? src.scale[soff + i] : src.scale_up[soff + i - KB];
  __syncthreads();

  // ---- per-lane global sources of the direct loads: load h of a tile
  // fills its rows 8 h .. 8 h + 7, lane l reading row 8 h + l / 8
  auto b_row = [&](int t, int h) -> const uint8_t* {
    const int rr = 8 * h + (lane >> 3);
    int64_t row;
    const uint8_t* w;
    if (MODE == GEMM_PLAIN) {
      row = ntile * kTileRows + t * 16 + rr;
      w = src.weight;
    } else {
      row = ntile * (kTileRows / 2) + (t & 3) * 16 + rr;
      w = t < 4 ? src.weight : src.weight_up;
    }
    if (row >= a.N) row = a.N - 1;  // rows past the matrix: valid bytes, results never stored
    return w + static_cast<int64_t>(expert) * a.w_expert_stride + group_row_base(row, K, src.wg) +
           load_piece_offset(lane, h);
  };
  const uint8_t* gb[2][2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int h = 0; h < 2; ++h) gb[t][h] = b_row(2 * wave + t, h);
  // activation operand tile g: the hi rows (g even) or lo rows (g odd) of
  // pair g / 2; its row rho is route 16 (g / 2) + rho
  const uint8_t* ga[GPW][2];
#pragma unroll
  for (int j = 0; j < GPW; ++j) {
    const int g = GPW * wave + j;
    const uint8_t* plane = (g & 1) ? src.a_lo : src.a_hi;
#pragma unroll
    for (int h = 0; h < 2; ++h)
      ga[j][h] = plane + token_of(16 * (g >> 1) + 8 * h + (lane >> 3)) * K + load_piece_offset(lane, h);
  }
  const uint32_t lds_addr = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
  const bool active = (GPW == 2 ? wave : wave >> 1) < pairs;  // wave-uniform: this wavefront's pair holds routes
  uint32_t found = 0;
#define GLM53_LOOP(n)                                                                                            \
  grouped_gemm_loop<MODE, FIX, GPW, n, DETECT>(a, src, ntile, start, len, KB, gb, ga, lds, lds_addr, lds_se, lds_sw, \
                                               wave, lane, found)
  if (active) GLM53_LOOP(1);
  else GLM53_LOOP(0);
#undef GLM53_LOOP
  return found;
}

template <int MODE, bool FIX, int GPW>
__device__ __forceinline__ void grouped_gemm_body(const GroupedGemmArgs& a, const ItemSource src, int64_t ntile, int64_t d,
                                                  uint8_t* lds) {
  int32_t expert, start, len;
  if (!item_routes<32 * GPW>(src, d, expert, start, len)) return;
  grouped_gemm_part<MODE, FIX, GPW, false>(a, src, ntile, expert, start, len, lds);
}

template <int GPW>
size_t gemm_lds_bytes(int64_t K) {
  // ring, activation scale codes [KB][32 GPW], weight scales [2][KB]
  return static_cast<size_t>(ring_stages<GPW>()) * stage_bytes<GPW>() +
         (32 * GPW + 2 * sizeof(float)) * static_cast<size_t>(K / kBlock);
}

// The work item w of a launch: its column tile, its descriptor (of the
// routed problem or, past the routed descriptors, of the dense one), the
// operands it reads and whether its weights hold 0x7F/0xFF codes.
__device__ __forceinline__ ItemSource item_source(const GroupedGemmArgs& a, int64_t used, int64_t w, bool desc_major,
                                                  int64_t& ntile, int64_t& d, bool& fix) {
  const int64_t D = used + a.x_descriptors;
  ntile = desc_major ? w % a.n_tiles : w / D;
  d = desc_major ? w / a.n_tiles : w % D;
  const bool dense = d >= used;  // an item of the dense problem
  if (dense) d -= used;
  ItemSource src;
  src.a_hi = dense ? a.x_a_hi : a.a_hi;
  src.a_lo = dense ? a.x_a_lo : a.a_lo;
  src.a_scale = dense ? a.x_a_scale : a.a_scale;
  src.a_row_index = dense ? nullptr : a.a_row_index;
  src.routes = dense ? a.x_routes : a.routes;
  src.tile_expert = dense ? nullptr : a.tile_expert;
  src.tile_start = a.tile_start;
  src.tile_len = a.tile_len;
  src.experts = dense ? 1 : a.experts;
  src.weight = dense ? a.x_weight : a.weight;
  src.weight_up = dense ? a.x_weight_up : a.weight_up;
  src.wg = dense ? a.x_w_group_log2 : a.w_group_log2;
  src.scale = dense ? a.x_scale : a.scale;
  src.scale_up = dense ? a.x_scale_up : a.scale_up;
  src.out = dense ? a.x_out : a.out;
  src.out_row_stride = dense ? a.x_out_row_stride : a.out_row_stride;
  auto set = [](const int32_t* flag) { return flag != nullptr && *flag != 0; };
  fix = dense ? set(a.x_fixup) || set(a.x_fixup_up) : set(a.fixup) || set(a.fixup_up);
  return src;
}

// The descriptor's expert, first route and route count (at most R routes);
// false for an unused descriptor.
template <int R>
__device__ __forceinline__ bool item_routes(const ItemSource& src, int64_t d, int32_t& expert, int32_t& start,
                                            int32_t& len) {
  if (src.tile_expert != nullptr) {
    expert = src.tile_expert[d];
    start = src.tile_start[d];
    len = src.tile_len[d];
    if (start >= src.routes || len <= 0) return false;
    if (expert < 0 || expert >= src.experts) return false;
    if (len > R) len = R;
    if (start + len > src.routes) len = static_cast<int32_t>(src.routes - start);
  } else {
    expert = 0;
    start = static_cast<int32_t>(d * R);
    len = static_cast<int32_t>(src.routes - start < R ? src.routes - start : R);
    if (len <= 0) return false;
  }
  return true;
}

// The routed descriptors in use: the route plan's device count when given
// (clamped to the capacity), else all of them.
__device__ __forceinline__ int64_t used_descriptors(const GroupedGemmArgs& a) {
  if (a.used_descriptors == nullptr) return a.descriptors;
  const int64_t u = static_cast<int64_t>(*a.used_descriptors);
  return u < a.descriptors ? u : a.descriptors;
}

// Work items (column tile, descriptor in use) are dealt to the XCDs in
// contiguous runs: workgroup i runs on XCD i % 8, and item w = (i % 8) *
// ceil(W / 8) + i / 8 keeps neighbouring items on one XCD and its L2.  W
// counts the items of descriptors in use, so every XCD gets the same share
// of real work; the grid is sized for the capacity and its surplus
// workgroups exit at once.  This shape orders items descriptor-major (all
// column tiles of a descriptor, i.e. one expert's whole matrix, in a row:
// its weight rows stream in address order and its activation rows stay in
// L2; config 4 -9%); the wide shape tile-major (descriptors of one heavy
// expert side by side share each weight tile; descriptor-major was 4%
// slower there).
template <int MODE, int GPW>
__global__ __launch_bounds__(256) void grouped_gemm_kernel(GroupedGemmArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds_dyn[];
  const int64_t used = used_descriptors(a);
  const int64_t items = a.n_tiles * (used + a.x_descriptors);
  const int64_t per_xcd = (items + 7) / 8;
  if (static_cast<int64_t>(blockIdx.x / 8) >= per_xcd) return;
  const int64_t w = static_cast<int64_t>(blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (w >= items) return;
  int64_t ntile, d;
  bool fix;
  const ItemSource src = item_source(a, used, w, true, ntile, d, fix);
  if (fix) grouped_gemm_body<MODE, true, GPW>(a, src, ntile, d, lds_dyn);
  else grouped_gemm_body<MODE, false, GPW>(a, src, ntile, d, lds_dyn);
}

// A caller's own descriptors of up to kGemmTileRows routes
// (glm53_grouped_linear), on the 32-route shape (GPW = 1: a larger descriptor
// runs in 32-route parts, each streaming its weights again) or the 64-route
// one (GPW = 2); grouped_linear_narrow says which.  Bound by the weight
// stream at few routes per expert, where the 32-route shape streams deeper
// and past the caches (4,096 routes over 288 experts, [4096 x 4096] and [4096
// x 2048] in one chain of building blocks, 2,800 -> 2,612 us for the whole
// chain against the 64-route shape).
// Weights that come without a code flag (a.fixup null) are looked at as they
// stream through the 32-route shape's registers, 40 VALU instructions per
// wavefront and stage beside a stage's 8 MFMAs and loads, and an item that met
// 0x7F / 0xFF runs again in the FIX form; a scan of the bank beforehand, which
// the 64-route shape needs, reads every expert's bytes once more.
template <int GPW>
__global__ __launch_bounds__(256) void grouped_linear_kernel(GroupedGemmArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds_dyn[];
  // A caller's descriptors end in unused ones (a tile plan over 288 experts
  // and 4,096 routes holds 416, ~300 of them used) whose number only the
  // device knows: workgroup i runs on XCD i % 8, and descriptors go to the
  // XCDs in turn, a.deal at a time (one expert's neighbours share an L2),
  // each with all its column tiles.  In contiguous runs the last XCDs held
  // the unused ones: the chain above 1,569 us, 1,355 dealt in turn.
  const int64_t j = blockIdx.x / 8, turn = j / (a.deal * a.n_tiles), in_turn = j % (a.deal * a.n_tiles);
  int64_t ntile = in_turn % a.n_tiles, d = (8 * turn + blockIdx.x % 8) * a.deal + in_turn / a.n_tiles;
  if (d >= a.descriptors) return;
  bool fix;
  const ItemSource src = item_source(a, a.descriptors, d * a.n_tiles + ntile, true, ntile, d, fix);
  int32_t expert, start, len;
  if (!item_routes<kGemmTileRows>(src, d, expert, start, len)) return;
  if constexpr (GPW == 2) {
    if (fix) grouped_gemm_part<GEMM_PLAIN, true, 2, false>(a, src, ntile, expert, start, len, lds_dyn);
    else grouped_gemm_part<GEMM_PLAIN, false, 2, false>(a, src, ntile, expert, start, len, lds_dyn);
    return;
  }
  for (int32_t done = 0; done < len; done += kGemmMinTileRows) {
    if (done > 0) __syncthreads();  // every wavefront has read the part before out of LDS
    const int32_t part = len - done < kGemmMinTileRows ? len - done : kGemmMinTileRows;
    if (!fix) {
      const uint32_t found =
          grouped_gemm_part<GEMM_PLAIN, false, 1, true>(a, src, ntile, expert, start + done, part, lds_dyn);
      if (a.fixup == nullptr) fix = workgroup_any((found & 0x80808080u) != 0, lds_dyn);
      if (!fix) continue;
    }
    grouped_gemm_part<GEMM_PLAIN, true, 1, false>(a, src, ntile, expert, start + done, part, lds_dyn);
  }
}

// ------------------------------------------ grouped GEMM, wide shape --
//
// For plans whose experts carry many routes: work item = one 128-route
// descriptor (8 pairs of 16 routes) x 512 weight rows (PLAIN: 512 output
// columns; SWIGLU: 256 gate rows and the matching 256 up rows), one
// 512-thread workgroup per CU (8 wavefronts, two per SIMD).  Wavefront w
// multiplies every pair of the descriptor against its own four 16-row
// weight tiles (PLAIN: output columns 64 w .. 64 w + 63 of the item;
// SWIGLU: gate rows 32 w .. 32 w + 31 and the matching up rows), so all
// wavefronts carry the same work whatever the descriptor's route count.
// The wavefront loads its four tiles itself (direct loads into its own
// 8 KB of a single-buffered 64 KB B stage) and reads them into registers
// during the previous stage's last pair; once those reads have returned it
// issues the next stage's tiles into the same bytes, so the weight stream
// needs no workgroup barrier and runs a stage ahead.  The activations come
// through a 2-stage ring of 32 KB stages (wavefront w loads pair w's hi and
// lo tiles).  One barrier per stage, after each wavefront's last
// activation read of the stage and before its last pair's MFMAs, makes the
// next stage's activation tiles visible and frees this stage's slot; the
// wavefronts leave it with that pair's MFMAs in hand, so the MFMA pipes
// have work while the next stage starts (3-4% faster than a barrier at the
// stage start).  Per stage 8 KB of B and 32 KB of A operand reads for 64
// MFMAs per wavefront.  The arithmetic per output
// element is that of the narrower shapes, so every shape gives the same
// bits.  A dense launch may take T = 2 (PLAIN: or 1) weight tiles per
// wavefront instead of 4 (256 or 128 weight rows per item) where 512-row
// items would leave CUs without one.
namespace {
constexpr int kWidePairs = kGemmWideRows / 16;            // 8
constexpr int kWideTilesPerWave = 4;                      // weight tiles per wavefront (T)
constexpr int kWideBTiles = 8 * kWideTilesPerWave;        // 32 tiles: 512 rows
constexpr int kWideBBytes = kWideBTiles * kOperand;       // 64 KB
constexpr int kWideABytes = 2 * kWidePairs * kOperand;    // 32 KB per A stage
constexpr int kWidePlainRows = kWideBTiles * 16;          // 512
constexpr int kWideGateRows = kWidePlainRows / 2;         // 256
}  // namespace

size_t gemm_wide_lds_bytes(int64_t K, int tiles) {
  // B stage, 2-stage A ring, activation scale codes [KB][128 routes],
  // weight scales [4][KB]
  return static_cast<size_t>(8 * tiles * kOperand + 2 * kWideABytes) +
         (kGemmWideRows + 4 * sizeof(float)) * static_cast<size_t>(K / kBlock);
}

// Direct-load sources of a wavefront.  Load h of its tile q covers rows U +
// 0 .. 7 with U = (q < 2 ? rlo : rhi) + 16 (q % 2) + 8 h (a multiple of 8,
// clamped to rows - 8, rows being a multiple of 8); lane l reads row U + l /
// 8 at its piece, and since U is a multiple of 8, group_row_base(U + l / 8)
// = group_row_base(U) + group_row_base(l / 8).  So the wave-uniform part
// wrow[2 q + h] = group_row_base(U) (+ (kb << (7 + wg)) for stage kb) goes
// into the SGPR base and the lane adds woff (h = 0; h = 1 flips bit 4 of the
// piece: woff ^ 16).  Load h of its pair's hi / lo rows reads a_hi / a_lo at
// aoff[h] (token row tok[h] at the lane's piece) + 128 kb.
struct WideSources {
  const uint8_t* wlo;      // PLAIN: the expert's matrix; SWIGLU: its gate rows
  const uint8_t* whi;      // PLAIN: the same matrix; SWIGLU: its up rows
  const uint8_t* a_hi;
  const uint8_t* a_lo;
  int32_t wg;              // row groups of the matrices (common.h)
  int64_t wrow[2 * kWideTilesPerWave];
  uint32_t woff;
  uint32_t aoff[2];
};

// A wave-uniform pointer as the compiler can prove it uniform (so that it
// lives in SGPRs).
__device__ __forceinline__ const uint8_t* uniform_ptr(const uint8_t* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
  return reinterpret_cast<const uint8_t*>((static_cast<uint64_t>(hi) << 32) | lo);
}

template <int MODE, bool FIX, int NP, int T>
__device__ __forceinline__ void wide_gemm_loop(const GroupedGemmArgs& a, const ItemSource src, int64_t ntile,
                                                int32_t start, int32_t len, int64_t KB, const WideSources& ls,
                                                bool loads_pair, uint8_t* lds, uint32_t lds_addr, const uint8_t* lds_se,
                                                const float* lds_sw, int wave, int lane) {
  constexpr int kBBytes = 8 * T * kOperand;
  constexpr int kHalf = T > 1 ? T / 2 : 1;  // tiles of the lo rows (SWIGLU: gate), the others of the hi rows (up)
  const OperandSlots slots = operand_slots(lane);
  const uint32_t b_own = static_cast<uint32_t>(wave) * T * kOperand;  // this wavefront's tiles in the B stage
  auto issue_b = [&](int64_t kb) {
    const uint8_t* mlo = ls.wlo + (kb << (7 + ls.wg));
    const uint8_t* mhi = ls.whi + (kb << (7 + ls.wg));
#pragma unroll
    for (int q = 0; q < T; ++q)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        lds_direct16_at((q < kHalf ? mlo : mhi) + ls.wrow[2 * q + h], ls.woff ^ (16 * h),
                        lds_addr + b_own + q * kOperand + 1024 * h);
  };
  auto issue_b_tile = [&](int64_t kb, int q) {
    const uint8_t* m = (q < kHalf ? ls.wlo : ls.whi) + (kb << (7 + ls.wg));
#pragma unroll
    for (int h = 0; h < 2; ++h)
      lds_direct16_at(m + ls.wrow[2 * q + h], ls.woff ^ (16 * h), lds_addr + b_own + q * kOperand + 1024 * h);
  };
  auto issue_a = [&](int64_t kb, int slot) {
    if (loads_pair) {
      const uint32_t sa = lds_addr + kBBytes + slot * kWideABytes + 2 * wave * kOperand;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        lds_direct16_at(ls.a_hi + kb * kBlock, ls.aoff[h], sa + 1024 * h);
        lds_direct16_at(ls.a_lo + kb * kBlock, ls.aoff[h], sa + kOperand + 1024 * h);
      }
    }
  };
  // weight scale row (of lds_sw) of the wavefront's tile q: PLAIN its
  // 64 rows lie in block (64 w) / 128 of the item; SWIGLU gate tiles in
  // gate block (32 w) / 128, up tiles in the same up block
  const int sw_lo = MODE == GEMM_PLAIN ? (16 * T * wave) >> 7 : (8 * T * wave) >> 7;
  const int sw_hi = MODE == GEMM_PLAIN ? sw_lo : T / 2 + sw_lo;

  float acc[NP][T][4];
#pragma unroll
  for (int j = 0; j < NP; ++j)
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[j][t][i] = 0.0f;

  // Stage 0 (B and A) was issued by wide_gemm_body, before the block
  // scales, and has landed in every wavefront (the body waited for its own
  // loads before the barrier that published the scales).  The wavefront's
  // B tiles of a stage are read into registers during the previous stage's
  // last pair, each as soon as that pair's last MFMA on the tile has
  // issued (its own direct loads waited for; no barrier: no other
  // wavefront reads them), so a stage starts on its MFMAs at once and its
  // B bytes take the next stage.
  i32x8 bq[T];
#pragma unroll
  for (int q = 0; q < T; ++q) bq[q] = lds_operand(lds + b_own + q * kOperand, slots);
  i32x8 ahi_next = lds_operand(lds + kBBytes, slots);
  i32x8 alo_next = lds_operand(lds + kBBytes + kOperand, slots);
  int slot = 0;
  for (int64_t kb = 0; kb < KB; ++kb) {
    // the other slot's stage (kb - 1) was read out by every wavefront before
    // the barrier in its last pair, and this wavefront's B tiles of stage kb
    // are in registers: stage kb + 1 goes in, A first (the barrier's count
    // leaves B's 2 T loads in flight).  With more than T pairs the B tiles
    // go out one per pair instead, each after the pair's hi pass: twelve
    // direct loads at a stage start had the wavefronts stall on the vector
    // memory queue (gate/up -3%, down -4%).  Those issues are unconditional
    // (a branch in the pair loop made the compiler spill), so the last stage
    // reloads its own tiles, unused.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (kb + 1 < KB) {
      issue_a(kb + 1, slot ^ 1);
      if constexpr (NP <= T) issue_b(kb + 1);
    }
    const int64_t kb_next = kb + 1 < KB ? kb + 1 : kb;
    const float w_lo = lds_sw[sw_lo * KB + kb], w_hi = lds_sw[sw_hi * KB + kb];
    // bytes j: the E8M0 scales of this lane's route in pairs j (lo word) and 4 + j (hi word)
    const uint2 se2 = *reinterpret_cast<const uint2*>(lds_se + kb * kGemmWideRows + (lane & 15) * 8);
    const uint8_t* st = lds + kBBytes + slot * kWideABytes;
    f32x4 c[T];
    auto fold = [&](int j, int q) {
      const float sw = q < kHalf ? w_lo : w_hi;
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[j][q][i] = fmaf(c[q][i], sw, acc[j][q][i]);
    };
    const uint8_t* st_next = lds + kBBytes + (slot ^ 1) * kWideABytes;
    // A operands a whole pair ahead: pair j + 1's hi and lo rows (after the
    // last pair: the next stage's first) are read as pair j's lo pass
    // starts, so each pair's operands have had a whole pair's MFMAs to
    // arrive (8 VGPRs more than reading the lo rows at the pair's own start:
    // gate/up -3%, down -3.5%)
#pragma unroll
    for (int j = 0; j < NP; ++j) {
      const int se = static_cast<int>(j < 4 ? se2.x : se2.y);
      const i32x8 ahi = ahi_next;
      const i32x8 alo = alo_next;
      // Issue priority falls as a wavefront gets ahead in its stage, so of
      // the two on a SIMD the one behind gets the MFMA pipe and they reach
      // the barrier closer together (gate/up -2%).
      if (j == 0) __builtin_amdgcn_s_setprio(3);
      else if (j == 2) __builtin_amdgcn_s_setprio(2);
      else if (j == 4) __builtin_amdgcn_s_setprio(1);
      else if (j == 6) __builtin_amdgcn_s_setprio(0);
      // Every wavefront has read this stage's A and its own share of the
      // next stage's A has landed: the next stage's A is complete, and this
      // stage's slot is free for the stage after.  Each wavefront still
      // holds its last pair's MFMAs, so the pipes have work at the release.
      if (j == NP - 1) stage_barrier<2 * T>();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < T; ++q) {
        if (j > 0) fold(j - 1, q);
        i32x8 b = bq[q], bc;
        weight_operand<FIX>(b, bc);
        c[q] = pair_pass_byte<FIX, 127>(j & 3, ahi, b, bc, (f32x4){0.0f, 0.0f, 0.0f, 0.0f}, se);
      }
      if constexpr (!FIX) {
        // each tile's fold right before its first MFMA (the fold of tile q
        // waits only for tile q's last MFMA of the previous pair, not for
        // tile T - 1's)
        if (j > 0) {
#pragma unroll
          for (int q = 0; q < T; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);  // VALU: fold(j - 1, q)
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA: tile q's hi pass
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (NP > T) {  // tiles 0 .. T - 1 at pairs 0 .. T - 1: all before the last pair's barrier
        if (j < T) issue_b_tile(kb_next, j);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (j + 1 < NP) {
        ahi_next = lds_operand(st + (2 * j + 2) * kOperand, slots);
        alo_next = lds_operand(st + (2 * j + 3) * kOperand, slots);
      } else {  // unused after the last stage
        ahi_next = lds_operand(st_next, slots);
        alo_next = lds_operand(st_next + kOperand, slots);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < T; ++q) {
        i32x8 b = bq[q], bc;
        weight_operand<FIX>(b, bc);
        c[q] = pair_pass_byte<FIX, 123>(j & 3, alo, b, bc, c[q], se);
        if (j == NP - 1) {
          // unconditional (the last stage rereads its own tiles, unused),
          // so that no tile stays live beside its successor
          if (q == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the next stage's B landed
          bq[q] = lds_operand(lds + b_own + q * kOperand, slots);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int q = 0; q < T; ++q) fold(NP - 1, q);
    slot ^= 1;
  }

  // epilogue: lane holds columns 16 tile + l % 16 of routes 16 j + 4 kq + i
  if constexpr (MODE == GEMM_PLAIN) {
    plain_epilogue<NP, T>(a, src, start, len, 0, 1, ntile * (128 * T) + 16 * T * wave, acc, lane);
  } else {
    swiglu_epilogue<NP, T / 2>(a, src, start, len, 0, 1, ntile * (64 * T) + 8 * T * wave, acc, lane);
  }
}

template <int MODE, bool FIX, int T>
__device__ __forceinline__ void wide_gemm_body(const GroupedGemmArgs& a, const ItemSource src, int64_t ntile,
                                                int64_t d, uint8_t* lds) {
  constexpr int kBBytes = 8 * T * kOperand;
  constexpr int kHalf = T > 1 ? T / 2 : 1;  // tiles of the lo rows (SWIGLU: gate), the others of the hi rows (up)
  static_assert(MODE == GEMM_PLAIN || T % 2 == 0, "a SwiGLU item holds whole gate and up scale blocks");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  int32_t expert, start, len;
  if (!item_routes<kGemmWideRows>(src, d, expert, start, len)) return;
  const int64_t K = a.K;
  const int64_t KB = K / kBlock;
  const int pairs = (len + 15) >> 4;
  uint8_t* lds_se = lds + kBBytes + 2 * kWideABytes;                    // [KB][128]
  float* lds_sw = reinterpret_cast<float*>(lds_se + kGemmWideRows * KB);    // [4][KB]
  auto token_of = [&](int r) -> int64_t {
    const int64_t route = start + (r < len ? r : len - 1);
    return src.a_row_index != nullptr ? src.a_row_index[route] : route;
  };
  // direct-load sources: load h of a weight tile fills its rows 8 h .. 8 h
  // + 7, lane l reading row r = 8 h + l / 8 at piece (l % 8) ^ (l / 8) ^ h,
  // i.e. the h = 0 offset with bit 0 of the piece flipped for h = 1.  The
  // offsets fit 32 bits: the launcher takes this shape only for matrices
  // and activation planes under 2 GiB (and rows a multiple of 8).
  WideSources ls;
  {
    const uint8_t* e0 = src.weight + static_cast<int64_t>(expert) * a.w_expert_stride;
    ls.wlo = uniform_ptr(e0);
    ls.whi = MODE == GEMM_SWIGLU ? uniform_ptr(src.weight_up + static_cast<int64_t>(expert) * a.w_expert_stride)
                                 : ls.wlo;
    ls.a_hi = uniform_ptr(src.a_hi);
    ls.a_lo = uniform_ptr(src.a_lo);
    ls.wg = src.wg;
    const int64_t rows = a.N;
    const int32_t piece = load_piece_offset(lane, 0);
    const int64_t rlo = MODE == GEMM_PLAIN ? ntile * (128 * T) + 16 * T * wave : ntile * (64 * T) + 8 * T * wave;
    const int64_t rhi = MODE == GEMM_PLAIN ? rlo + 16 * kHalf : rlo;
#pragma unroll
    for (int q = 0; q < T; ++q)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        int64_t u = (q < kHalf ? rlo : rhi) + 16 * (q % kHalf) + 8 * h;
        u = u < rows - 8 ? u : rows - 8;
        ls.wrow[2 * q + h] = group_row_base(u, K, ls.wg);
      }
    ls.woff = static_cast<uint32_t>(group_row_base(lane >> 3, K, ls.wg) + piece);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      ls.aoff[h] = static_cast<uint32_t>(token_of(16 * wave + 8 * h + (lane >> 3)) * K + (piece ^ (16 * h)));
  }
  const bool loads_pair = wave < pairs;  // wave-uniform
  const uint32_t lds_addr = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
  // stage 0's direct loads fly while the block scales are gathered
  {
    const uint32_t b_own = static_cast<uint32_t>(wave) * T * kOperand;
#pragma unroll
    for (int q = 0; q < T; ++q)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        lds_direct16_at((q < kHalf ? ls.wlo : ls.whi) + ls.wrow[2 * q + h], ls.woff ^ (16 * h),
                        lds_addr + b_own + q * kOperand + 1024 * h);
    if (loads_pair) {
      const uint32_t sa = lds_addr + kBBytes + 2 * wave * kOperand;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        lds_direct16_at(ls.a_hi, ls.aoff[h], sa + 1024 * h);
        lds_direct16_at(ls.a_lo, ls.aoff[h], sa + kOperand + 1024 * h);
      }
    }
  }
  load_activation_scales<kGemmWideRows, 512, true>(src, start, len, KB, lds_se);
  // weight scale rows: PLAIN the item's four 128-row blocks; SWIGLU the two
  // blocks its 256 gate rows span, then the same up blocks
  const int64_t srows = (a.N + 127) / 128;
  const int64_t b0 = MODE == GEMM_PLAIN ? T * ntile : kHalf * ntile;
  for (int64_t i = threadIdx.x; i < T * KB; i += 512) {
    const int64_t r = i / KB, k = i - r * KB;
    int64_t blk = b0 + (MODE == GEMM_PLAIN ? r : r % kHalf);
    blk = blk < srows ? blk : srows - 1;
    const float* sc = (MODE == GEMM_SWIGLU && r >= kHalf) ? src.scale_up : src.scale;
    lds_sw[i] = sc[static_cast<int64_t>(expert) * a.s_expert_stride + blk * a.s_cols + k];
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's stage-0 loads landed
  __syncthreads();

#define GLM53_WIDE(n) \
  wide_gemm_loop<MODE, FIX, n, T>(a, src, ntile, start, len, KB, ls, loads_pair, lds, lds_addr, lds_se, lds_sw, wave, lane)
  // rows past the descriptor's routes (in its last pair) hold stale
  // activations: their products are never stored
  switch (pairs) {
    case 1: GLM53_WIDE(1); break;
    case 2: GLM53_WIDE(2); break;
    case 3: GLM53_WIDE(3); break;
    case 4: GLM53_WIDE(4); break;
    case 5: GLM53_WIDE(5); break;
    case 6: GLM53_WIDE(6); break;
    case 7: GLM53_WIDE(7); break;
    default: GLM53_WIDE(8); break;
  }
#undef GLM53_WIDE
}

template <int MODE, int T>
__global__ __launch_bounds__(512) void grouped_gemm_wide_kernel(GroupedGemmArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds_dyn[];
  const int64_t used = used_descriptors(a);
  const int64_t items = a.n_tiles * (used + a.x_descriptors);
  const int64_t per_xcd = (items + 7) / 8;
  if (static_cast<int64_t>(blockIdx.x / 8) >= per_xcd) return;
  const int64_t w = static_cast<int64_t>(blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (w >= items) return;
  int64_t ntile, d;
  bool fix;
  const ItemSource src = item_source(a, used, w, false, ntile, d, fix);
  if (fix) wide_gemm_body<MODE, true, T>(a, src, ntile, d, lds_dyn);
  else wide_gemm_body<MODE, false, T>(a, src, ntile, d, lds_dyn);
}

// Sets *flag (pre-cleared by clear_flag_kernel) when any byte of codes is
// 0x7F or 0xFF.
__global__ void clear_flag_kernel(int32_t* flag) { *flag = 0; }


__global__ __launch_bounds__(256) void scan_480_kernel(const uint8_t* codes, int64_t n, int32_t* flag) {
  const int64_t words = n / 16;
  bool hit = false;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < words;
       i += static_cast<int64_t>(gridDim.x) * 256) {
    u32x4 q = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(codes) + i);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t t = (q[j] & 0x7F7F7F7Fu) ^ 0x7F7F7F7Fu;
      hit |= (~((t | 0x80808080u) - 0x01010101u) & 0x80808080u) != 0u;
    }
  }
  if (blockIdx.x == 0) {
    for (int64_t i = words * 16 + threadIdx.x; i < n; i += 256) hit |= (codes[i] & 0x7Fu) == 0x7Fu;
  }
  if (hit) atomicOr(flag, 1);
}

// ------------------------------------------------------------ reductions --

// grouped_fp8.py:273-276: y[t] = T(sum_slot float(down[inv[t*k+slot]]) *
// score), FP32 products summed in slot order, optional BF16 shared add.
// Stores one thread's V MoE outputs (FP32 values already BF16-exact): the
// plain row, or the kHcBranches hyper-connection streams built from them
// (native_indexer_plan.metal:2362-2388: mixed = fma(comb[s][b], residual[s],
// mixed) over s in order from 0, then T(post[b] * moe + mixed)).
template <int V>
__device__ __forceinline__ void store_moe_row(const ReduceArgs& a, int64_t t, int64_t h0, const float (&moe)[V]) {
  if (a.hc_out == nullptr) {
    store_bf16_run<V>(a.out + t * a.H + h0, moe);
    return;
  }
  Bf16Run<V> res[kHcBranches];
#pragma unroll
  for (int s = 0; s < kHcBranches; ++s) res[s].load(a.hc_residual + (t * kHcBranches + s) * a.H + h0);
#pragma unroll
  for (int b = 0; b < kHcBranches; ++b) {
    const float post = a.hc_post[t * kHcBranches + b];
    float y[V];
#pragma unroll
    for (int i = 0; i < V; ++i) {
      float mixed = 0.0f;
#pragma unroll
      for (int s = 0; s < kHcBranches; ++s)
        mixed = __builtin_fmaf(a.hc_comb[(t * kHcBranches + s) * kHcBranches + b], res[s].get(i), mixed);
      y[i] = __fadd_rn(__fmul_rn(post, moe[i]), mixed);
    }
    store_bf16_run<V>(a.hc_out + (t * kHcBranches + b) * a.H + h0, y);
  }
}

// Thread = V consecutive columns of one token (V = 8: 16-byte loads and
// stores, when H and the row pointers allow it; V = 1 otherwise).  The
// token's positions and scores are read first (uniform across the
// workgroup), then every slot's row is requested before the first is summed,
// so the row loads overlap instead of each waiting behind the last.
template <int V, int K>
__global__ __launch_bounds__(256) void restore_reduce_kernel(ReduceArgs a) {
  constexpr int kSlots = K > 0 ? K : kMaxReduceTopK;  // K = 0: top_k known only at run time
  const int k = K > 0 ? K : a.top_k;
  const int64_t t = blockIdx.y;
  const int64_t h0 = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * V;
  if (h0 >= a.H) return;
  int32_t pos[kSlots];
  float score[kSlots];
#pragma unroll
  for (int s = 0; s < kSlots; ++s) pos[s] = s < k ? a.inverse[t * k + s] : 0;
#pragma unroll
  for (int s = 0; s < kSlots; ++s) score[s] = s < k ? a.sorted_score[pos[s] < 0 ? 0 : pos[s]] : 0.0f;
  Bf16Run<V> row[kSlots];
#pragma unroll
  for (int s = 0; s < kSlots; ++s) {  // a missing route (pos < 0) reads row 0 and sums NaN
    row[s].clear();
    if (s < k) row[s].load(a.route_out + static_cast<int64_t>(pos[s] < 0 ? 0 : pos[s]) * a.H + h0);
  }
  float total[V];
#pragma unroll
  for (int i = 0; i < V; ++i) total[i] = 0.0f;
#pragma unroll
  for (int s = 0; s < kSlots; ++s) {
    if (s >= k) continue;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const float v = pos[s] < 0 ? __builtin_nanf("") : row[s].get(i);
      total[i] = __fadd_rn(total[i], __fmul_rn(v, score[s]));
    }
  }
  Bf16Run<V> sh;
  sh.clear();
  if (a.shared != nullptr) sh.load(a.shared + t * a.H + h0);
#pragma unroll
  for (int i = 0; i < V; ++i) {
    total[i] = bf16_round(total[i]);
    if (a.shared != nullptr) total[i] = bf16_round(__fadd_rn(total[i], sh.get(i)));
  }
  store_moe_row<V>(a, t, h0, total);
}

// native_indexer_plan.metal:2174-2207 (fp8.py:384-397 order): per token,
// ascending expert id; contribution = T(down * score); total = T(total + c).
// Thread = V consecutive columns; loads are issued as above, in sorted order.
// The order comes from ranks (slots of a smaller id, and earlier slots of the
// same one, before it) and selects: every array index is static, and the
// ids, positions and scores are uniform.  K is top_k itself: a form for any
// top_k with all kMaxReduceTopK slots unrolled spends their ranks and loads
// on slots that are not there.  Measured (us; a sort in scratch memory / the
// form for any top_k / this): 64 tokens x 4096 columns 4.5 / 10.8 / 2.7 at
// top_k 2, 9.6 / 4.9 (as this) at 8, 20.8 / 15.3 / 12.8 at 16; 4,096 tokens
// 30.8 / 143 / 17.2 at top_k 2, 148 / 164 / 97 at 12; 64 x 1023 columns, one
// per thread, 8.9 / 12.1 / 3.9 at 8.
template <int V, int K>
__global__ __launch_bounds__(256) void direct_order_reduce_kernel(ReduceArgs a) {
  const int64_t t = blockIdx.y;
  const int64_t h0 = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * V;
  if (h0 >= a.H) return;
  int32_t id[K], slot_pos[K];
  float slot_score[K];
#pragma unroll
  for (int s = 0; s < K; ++s) {
    const int64_t i = t * K + s;
    id[s] = a.expert_ids[i];
    slot_pos[s] = a.inverse[i];
    slot_score[s] = a.route_score[i];
  }
  int32_t pos[K];
  float score[K];
#pragma unroll
  for (int r = 0; r < K; ++r) {
    pos[r] = 0;
    score[r] = 0.0f;
  }
#pragma unroll
  for (int s = 0; s < K; ++s) {
    int rank = 0;
#pragma unroll
    for (int o = 0; o < K; ++o) rank += o < s ? id[o] <= id[s] : id[o] < id[s];
#pragma unroll
    for (int r = 0; r < K; ++r) {
      const bool here = rank == r;
      pos[r] = here ? slot_pos[s] : pos[r];
      score[r] = here ? slot_score[s] : score[r];
    }
  }
  Bf16Run<V> row[K];
#pragma unroll
  for (int r = 0; r < K; ++r) row[r].load(a.route_out + static_cast<int64_t>(pos[r] < 0 ? 0 : pos[r]) * a.H + h0);
  Bf16Run<V> sh;
  sh.clear();
  if (a.shared != nullptr) sh.load(a.shared + t * a.H + h0);
  float total[V];
#pragma unroll
  for (int i = 0; i < V; ++i) total[i] = 0.0f;
#pragma unroll
  for (int r = 0; r < K; ++r) {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const float v = pos[r] < 0 ? __builtin_nanf("") : row[r].get(i);
      const float c = bf16_round(__fmul_rn(v, score[r]));
      total[i] = bf16_round(__fadd_rn(total[i], c));
    }
  }
#pragma unroll
  for (int i = 0; i < V; ++i)
    if (a.shared != nullptr) total[i] = bf16_round(__fadd_rn(total[i], sh.get(i)));
  store_moe_row<V>(a, t, h0, total);
}

// ------------------------------------------------------------- launchers --

namespace {
bool split_wide(const SplitArgs& a) { return a.x_row_stride % 8 == 0 && reinterpret_cast<uintptr_t>(a.x) % 16 == 0; }
int64_t split_units(const SplitArgs& a) {  // wavefronts
  const int64_t blocks_per_row = a.cols / kBlock;
  return a.rows * (split_wide(a) ? (blocks_per_row + 3) / 4 : blocks_per_row);
}
}  // namespace

hipError_t launch_route_plan(const RoutePlanArgs& a, const SplitArgs* split, hipStream_t st) {
  int id_bits = 0;
  while ((1 << id_bits) < a.experts) ++id_bits;
  const size_t lds = sizeof(unsigned) * static_cast<size_t>(kPlanWaves * a.experts);
  if (a.routes <= kPlanOneLaunchRoutes) {
    SplitArgs s{};
    if (split != nullptr) s = *split;
    if (s.cols % kBlock != 0 || s.operand_order) return hipErrorInvalidValue;
    const int64_t split_blocks = s.rows > 0 ? (split_units(s) + kPlanWaves - 1) / kPlanWaves : 0;
    const dim3 grid(static_cast<unsigned>(1 + split_blocks));
    if (split_wide(s)) hipLaunchKernelGGL(route_plan_one_kernel<8>, grid, dim3(64 * kPlanWaves), lds, st, a, id_bits, s);
    else hipLaunchKernelGGL(route_plan_one_kernel<2>, grid, dim3(64 * kPlanWaves), lds, st, a, id_bits, s);
    return hipGetLastError();
  }
  if (split != nullptr) {
    const hipError_t e = launch_split_activations(*split, st);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(route_count_kernel, dim3(static_cast<unsigned>(a.blocks)), dim3(64 * kPlanWaves), lds, st, a, id_bits);
  hipLaunchKernelGGL(route_scan_kernel, dim3(1), dim3(1024), 0, st, a);
  hipLaunchKernelGGL(route_scatter_kernel, dim3(static_cast<unsigned>((a.routes + 255) / 256)), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_split_activations(const SplitArgs& a, hipStream_t st) {
  if (a.rows == 0) return hipSuccess;
  if (a.cols % kBlock != 0) return hipErrorInvalidValue;
  const bool wide = split_wide(a);
  const int64_t units = wide && a.operand_order ? (a.rows + 7) / 8 * (a.cols / kBlock) : split_units(a);
  const dim3 grid(static_cast<unsigned>((units + 3) / 4));
  if (wide && a.operand_order) hipLaunchKernelGGL(split_operand_kernel, grid, dim3(256), 0, st, a);
  else if (wide) hipLaunchKernelGGL((split_activations_kernel<8, false>), grid, dim3(256), 0, st, a);
  else if (a.operand_order) hipLaunchKernelGGL((split_activations_kernel<2, true>), grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((split_activations_kernel<2, false>), grid, dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_grouped_gemm(const GroupedGemmArgs& a, int mode, int64_t descriptors, hipStream_t st) {
  if (descriptors == 0 && a.x_descriptors == 0) return hipSuccess;
  // the epilogues' buffer stores take 32-bit offsets of up to 128 rows
  if (a.out_row_stride < a.N || a.out_row_stride >= (int64_t{1} << 22) ||
      (a.x_descriptors > 0 && (a.x_out_row_stride < a.N || a.x_out_row_stride >= (int64_t{1} << 22))))
    return hipErrorInvalidValue;
  if (a.tile_rows == kGemmWideRows) {
    GroupedGemmArgs g = a;
    g.n_tiles = mode == GEMM_PLAIN ? (a.N + kWidePlainRows - 1) / kWidePlainRows : (a.N + kWideGateRows - 1) / kWideGateRows;
    g.descriptors = descriptors;
    const int64_t items = g.n_tiles * (descriptors + g.x_descriptors);
    const unsigned grid = static_cast<unsigned>(8 * ((items + 7) / 8));
    const size_t lds = gemm_wide_lds_bytes(a.K, kWideTilesPerWave);
    if (a.K % kBlock != 0 || a.K <= 0 || lds > 160 * 1024) return hipErrorInvalidValue;
    // its direct loads take 32-bit offsets into each matrix and activation plane
    if (!wide_offsets_fit(a.N, a.K, a.routes > a.x_routes ? a.routes : a.x_routes)) return hipErrorInvalidValue;
    if (mode == GEMM_PLAIN) hipLaunchKernelGGL((grouped_gemm_wide_kernel<GEMM_PLAIN, kWideTilesPerWave>), dim3(grid), dim3(512), lds, st, g);
    else hipLaunchKernelGGL((grouped_gemm_wide_kernel<GEMM_SWIGLU, kWideTilesPerWave>), dim3(grid), dim3(512), lds, st, g);
    return hipGetLastError();
  }
  GroupedGemmArgs g = a;
  g.n_tiles = mode == GEMM_PLAIN ? (a.N + 127) / 128 : (a.N + 63) / 64;
  g.descriptors = descriptors;
  const int64_t items = g.n_tiles * (descriptors + g.x_descriptors);
  const unsigned grid = static_cast<unsigned>(8 * ((items + 7) / 8));
  if (a.tile_rows != 0 && a.tile_rows != kGemmMinTileRows && a.tile_rows != kGemmTileRows)
    return hipErrorInvalidValue;
  const bool narrow = a.tile_rows == kGemmMinTileRows;
  const size_t lds = narrow ? gemm_lds_bytes<1>(a.K) : gemm_lds_bytes<2>(a.K);
  if (a.K % kBlock != 0 || a.K <= 0 || lds > 160 * 1024) return hipErrorInvalidValue;
#define GLM53_GEMM(m, w) hipLaunchKernelGGL((grouped_gemm_kernel<m, w>), dim3(grid), dim3(256), lds, st, g)
  if (mode == GEMM_PLAIN) {
    if (narrow) GLM53_GEMM(GEMM_PLAIN, 1);
    else GLM53_GEMM(GEMM_PLAIN, 2);
  } else {
    if (narrow) GLM53_GEMM(GEMM_SWIGLU, 1);
    else GLM53_GEMM(GEMM_SWIGLU, 2);
  }
#undef GLM53_GEMM
  return hipGetLastError();
}

hipError_t launch_wide_dense(const GroupedGemmArgs& a, int mode, int tiles, hipStream_t st) {
  if (a.out_row_stride < a.N || a.out_row_stride >= (int64_t{1} << 22)) return hipErrorInvalidValue;
  const int64_t cols = mode == GEMM_PLAIN ? 128 * tiles : 64 * tiles;
  GroupedGemmArgs g = a;
  g.n_tiles = (a.N + cols - 1) / cols;
  g.descriptors = (a.routes + kGemmWideRows - 1) / kGemmWideRows;
  const unsigned grid = static_cast<unsigned>(8 * ((g.n_tiles * g.descriptors + 7) / 8));
  const size_t lds = gemm_wide_lds_bytes(a.K, tiles);
  if (a.K % kBlock != 0 || a.K <= 0 || lds > 160 * 1024) return hipErrorInvalidValue;
  if (!wide_offsets_fit(a.N, a.K, a.routes)) return hipErrorInvalidValue;
#define GLM53_WIDE_DENSE(m, t) hipLaunchKernelGGL((grouped_gemm_wide_kernel<m, t>), dim3(grid), dim3(512), lds, st, g)
  if (mode == GEMM_PLAIN && tiles == 1) GLM53_WIDE_DENSE(GEMM_PLAIN, 1);
  else if (mode == GEMM_PLAIN && tiles == 2) GLM53_WIDE_DENSE(GEMM_PLAIN, 2);
  else if (mode == GEMM_PLAIN && tiles == kWideTilesPerWave) GLM53_WIDE_DENSE(GEMM_PLAIN, kWideTilesPerWave);
  else if (mode == GEMM_SWIGLU && tiles == 2) GLM53_WIDE_DENSE(GEMM_SWIGLU, 2);
  else if (mode == GEMM_SWIGLU && tiles == kWideTilesPerWave) GLM53_WIDE_DENSE(GEMM_SWIGLU, kWideTilesPerWave);
  else return hipErrorInvalidValue;
#undef GLM53_WIDE_DENSE
  return hipGetLastError();
}

// Whether the descriptors are as many as a tile plan of `rows` routes has
// (ceil(routes / rows) + experts, the last ones unused).
static bool plan_of(int64_t rows, int64_t routes, int64_t descriptors, int64_t experts) {
  return (descriptors - experts) * rows >= routes;
}

// Whether glm53_grouped_linear takes the 32-route shape: up to `most` routes
// per expert, beyond which experts fill the 64-route shape's items or have
// several descriptors, whose weights the 32-route shape streams again for each
// of them.  A code flag, which spares the 64-route shape its scan of the bank,
// brings the line down; so do descriptors too few for the plan of 32 routes,
// which may hold up to 64 routes, two parts of the 32-route shape, and a list
// without unused ones, which the 64-route shape takes in contiguous runs.
// Measured (us, 32-route / 64-route shape, 288 experts [3072 x 4096], uniform
// routing): flagged, plan of 32: 16 routes per expert 644 / 718, 24 738 / 763, 32
// 1,011 / 902, 96 2,393 / 1,668; plan of 64: 8 592 / 682, 16 644 / 717 (Zipf 774 /
// 704), 24 724 / 746 (Zipf 919 / 780), 192 4,546 / 2,076; none unused: 2 492 / 520,
// 8 596 / 634 (Zipf 611 / 598), 12 619 / 653 (Zipf 745 / 654); without a flag,
// plan of 32: 48 1,382 / 1,611, 64 1,725 / 1,784, 96 2,393 / 2,194; plan of 64: 40
// 1,281 / 1,317, 48 1,462 / 1,370, 192 4,545 / 2,498.
bool grouped_linear_narrow(int64_t routes, int64_t descriptors, int64_t experts, bool flagged) {
  const bool plan32 = plan_of(kGroupedTileRows, routes, descriptors, experts);
  const bool plan64 = plan_of(kGemmTileRows, routes, descriptors, experts);
  const int64_t most = flagged ? (plan32 ? 24 : plan64 ? 12 : 6) : plan32 ? 80 : 40;
  return routes <= most * experts;
}

hipError_t launch_grouped_linear(const GroupedGemmArgs& a, int64_t descriptors, hipStream_t st) {
  if (descriptors == 0) return hipSuccess;
  if (a.out_row_stride < a.N || a.out_row_stride >= (int64_t{1} << 22)) return hipErrorInvalidValue;
  GroupedGemmArgs g = a;
  g.n_tiles = (a.N + kTileRows - 1) / kTileRows;
  g.descriptors = descriptors;
  // Four at a time from 256 descriptors on (us, 4 / 1, 288 experts [3072 x
  // 4096]: 4 routes per expert 562 / 578, 8 590 / 609, 16 644 / 656); fewer leave
  // too few turns to even out (64-route shape, 64 experts [4096 x 2048], 24
  // routes per expert: 146 / 126).
  // The 64-route shape over a list without unused ones: contiguous runs (288
  // experts of 16 routes 665, four at a time 724; 64 routes 827 / 880).
  const bool narrow = a.tile_rows == kGemmMinTileRows;
  g.deal = descriptors >= 256 ? 4 : 1;
  if (!narrow && !plan_of(kGemmTileRows, a.routes, descriptors, a.experts)) g.deal = (descriptors + 7) / 8;
  const int64_t turns = (descriptors + 8 * g.deal - 1) / (8 * g.deal);
  const unsigned grid = static_cast<unsigned>(8 * turns * g.deal * g.n_tiles);
  const size_t lds = narrow ? gemm_lds_bytes<1>(a.K) : gemm_lds_bytes<2>(a.K);
  if (a.K % kBlock != 0 || a.K <= 0 || lds > 160 * 1024) return hipErrorInvalidValue;
  if (!narrow && (a.tile_rows != kGemmTileRows || a.fixup == nullptr)) return hipErrorInvalidValue;
  if (narrow) hipLaunchKernelGGL(grouped_linear_kernel<1>, dim3(grid), dim3(256), lds, st, g);
  else hipLaunchKernelGGL(grouped_linear_kernel<2>, dim3(grid), dim3(256), lds, st, g);
  return hipGetLastError();
}

hipError_t launch_scan_480(const uint8_t* codes, int64_t n, int32_t* flag, bool clear, hipStream_t st) {
  if (clear) hipLaunchKernelGGL(clear_flag_kernel, dim3(1), dim3(1), 0, st, flag);
  if (n > 0) {
    int64_t blocks = (n / 16 + 255) / 256;
    if (blocks < 1) blocks = 1;
    if (blocks > 2048) blocks = 2048;
    hipLaunchKernelGGL(scan_480_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st, codes, n, flag);
  }
  return hipGetLastError();
}

namespace {
// direct_order_reduce_kernel for a.top_k, 1 .. K
template <int V, int K = kMaxReduceTopK>
void launch_direct_order(const ReduceArgs& a, dim3 grid, hipStream_t st) {
  if constexpr (K > 1) {
    if (a.top_k < K) return launch_direct_order<V, K - 1>(a, grid, st);
  }
  hipLaunchKernelGGL((direct_order_reduce_kernel<V, K>), grid, dim3(256), 0, st, a);
}
}  // namespace

hipError_t launch_reduce(const ReduceArgs& a, bool direct_order, hipStream_t st) {
  if (a.tokens == 0) return hipSuccess;
  if (a.top_k < 1 || a.top_k > kMaxReduceTopK) return hipErrorInvalidValue;
  auto a16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const bool wide = a.H % 8 == 0 && a16(a.route_out) && a16(a.out) && a16(a.shared) && a16(a.hc_residual) &&
                    a16(a.hc_out);
  const int64_t per_thread = wide ? 8 : 1;
  const dim3 grid(static_cast<unsigned>((a.H / per_thread + 255) / 256), static_cast<unsigned>(a.tokens));
  if (wide) {
    if (direct_order) launch_direct_order<8>(a, grid, st);
    else if (a.top_k == 8) hipLaunchKernelGGL((restore_reduce_kernel<8, 8>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((restore_reduce_kernel<8, 0>), grid, dim3(256), 0, st, a);
  } else {
    if (direct_order) launch_direct_order<1>(a, grid, st);
    else hipLaunchKernelGGL((restore_reduce_kernel<1, 0>), grid, dim3(256), 0, st, a);
  }
  return hipGetLastError();
}

}  // namespace glm53
