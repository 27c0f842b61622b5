// Dense block-FP8 linear for few rows: y[m, n] = T(sum_k x[m, k] w[n, k]) on
// the split activations of grouped.hip, the contraction split over the
// wavefronts of a workgroup.
#include "common.h"
#include "dense.h"
#include "grouped.h"
#include "mfma_fp8.h"
#include "split_fp8.h"

namespace glm53 {

namespace {

constexpr int kDenseWaves = 8;
constexpr int64_t kWideDenseMaxK = 1 << 14;  // 128 x 512 items: 128 K blocks of scales beside their stages
constexpr int64_t kDenseMaxK = 1 << 18;  // its weight scales take 16 KB of LDS (gate and up)
template <int V>
struct Int {
  static constexpr int value = V;
};

// K steps (of kDenseWaves blocks) between two folds: their results wait in
// LDS, 1 KB per block and 16 x 16 output tile.
template <int P, int C>
constexpr int fold_steps() {
  return P * C <= 2 ? 4 : P * C <= 4 ? 2 : 1;
}
// K steps a wavefront keeps in flight in registers
template <int P, int C>
constexpr int load_depth() {
  return P * C <= 2 ? 4 : 2;
}
// Operand tiles a wavefront passes through its own LDS buffer: its weight
// tiles, and (RAW) the hi and lo tile it makes of its activations
template <int C, bool RAW>
constexpr int turn_tiles() {
  return C + (RAW ? 2 : 0);
}

template <int P, int C, bool RAW>
size_t dense_lds_bytes(int64_t K) {
  return static_cast<size_t>(kDenseWaves) * (fold_steps<P, C>() * P * C * 1024 + turn_tiles<C, RAW>() * kOperand) +
         2 * sizeof(float) * static_cast<size_t>(K / kBlock);
}

// Rows row0 .. row0 + 16 P - 1 x weight tiles 0 .. C - 1: columns col0 .. col0
// + 16 C - 1, or (SWIGLU) gate rows col0 .. col0 + 8 C - 1 in the first half
// of the tiles and the matching up rows in the second.  Wavefront w
// multiplies K blocks w, w + 8, ...: its operands come from global memory
// into registers (each byte of the item's rows and columns once per
// workgroup), load_depth steps ahead, so no barrier is waited at in between.
// The activations lie in operand order and are multiplied as loaded; the
// weight rows come 8 whole 128-byte lines per load and turn into operand
// order through an LDS buffer of the wavefront's own.  (Loading row-major
// bytes in operand order, 16 rows per load, ran at a third of this rate,
// neighbouring lanes in different lines; turning the activations through LDS
// too cost 300 x 1536 x 4096 13.9 us instead of 12.4, 16 x 4096 x 4096 7.2
// instead of 6.6.)
// A block's MFMA results (hi rows, then lo rows, before the weight scale) go
// to LDS, and wavefront t < P C adds tile t's results in block order, so
// every output goes through the operations of the grouped GEMM and has its
// bits.  Returns codes_480 of the weight bytes (DETECT).
//
// RAW (P = 1): the activations come as bf16 (a.x) and the wavefront splits
// each of its blocks itself on the way to LDS -- lanes 16 j .. 16 j + 15 hold
// 8 columns each of rows j, 4 + j, 8 + j and 12 + j -- instead of a launch of
// its own that writes planes and scales first.
template <int P, int C, bool SWIGLU, bool RAW, bool FIX, bool DETECT>
__device__ __forceinline__ uint32_t dense_ksplit_item(const DenseArgs& a, int64_t row0, int64_t col0, uint8_t* lds) {
  constexpr int D = FIX ? 1 : load_depth<P, C>(), F = FIX ? 1 : fold_steps<P, C>();
  constexpr int H = SWIGLU ? C / 2 : C;  // tiles of one matrix
  constexpr int U = D > F ? D : F;  // steps per loop turn: the registers rotate back, folds fall at its end
  const int lane = threadIdx.x & 63, r = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int64_t K = a.K;
  const int KB = static_cast<int>(K / kBlock);
  const int steps = (KB + kDenseWaves - 1) / kDenseWaves;
  constexpr int kFold = kDenseWaves * fold_steps<P, C>() * P * C * 1024;
  f32x4* lds_c = reinterpret_cast<f32x4*>(lds);                                          // [8 F][P C][64]
  constexpr int kTurn = turn_tiles<C, RAW>() * kOperand;
  uint8_t* turn = lds + kFold + wave * kTurn;                                            // this wavefront's
  float* lds_sw = reinterpret_cast<float*>(lds + kFold + kDenseWaves * kTurn);           // [2][KB]
  const OperandSlots slots = operand_slots(lane);

  // rows past the last repeat it, columns past the matrix its last row: valid
  // bytes whose results are never stored (offsets from wave-uniform bases;
  // the launcher keeps them below 2^32)
  static_assert(!RAW || P == 1, "a raw item holds one pair");
  uint32_t xoff[4];  // RAW: byte offsets of the lane's columns of row 4 i + lane / 16
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t m = row0 + 4 * i + kq;
    xoff[i] = static_cast<uint32_t>(2 * ((m < a.rows ? m : a.rows - 1) * K + 8 * r));
  }
  uint32_t aoff[P], srow[P], wrow[C][2];
  int64_t apair[P];  // the pair's bytes in the planes
  int arows[P];      // and rows
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int64_t last = a.rows - 1;
    int64_t pair = row0 / 16 + p;
    pair = pair < last / 16 ? pair : last / 16;
    const int64_t left = a.rows - 16 * pair;
    arows[p] = left < 16 ? static_cast<int>(left) : 16;
    apair[p] = 16 * pair * K;
    aoff[p] = static_cast<uint32_t>(16 * ((r < arows[p] ? r : arows[p] - 1) + arows[p] * kq));
    const int64_t m = row0 + 16 * p + r;
    srow[p] = static_cast<uint32_t>((m < last ? m : last) * KB);
  }
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t n = col0 + 16 * (c % H) + 8 * h + (lane >> 3);
      wrow[c][h] = static_cast<uint32_t>((n < a.N ? n : a.N - 1) * K + load_piece_offset(lane, h));
    }
  struct Step {
    u32x4 b[C][2], h[P][2], l[P][2];
    float s[P];
  };
  auto load = [&](int s, Step& v) {
    int kb = kDenseWaves * s + wave;
    kb = kb < KB ? kb : KB - 1;  // past the end: loaded, never folded
    const int64_t ko = static_cast<int64_t>(kb) * kBlock;  // wave-uniform
    const uint8_t *w = a.weight + ko, *up = SWIGLU ? a.weight_up + ko : w;
    if constexpr (RAW) {
      const uint8_t* x = reinterpret_cast<const uint8_t*>(a.x + ko);
#pragma unroll
      for (int i = 0; i < 4; ++i) (i < 2 ? v.h : v.l)[0][i & 1] = *reinterpret_cast<const u32x4*>(x + xoff[i]);
    }
    const float* se = a.a_scale + kb;
#pragma unroll
    for (int p = 0; p < (RAW ? 0 : P); ++p) {
      const int64_t block = apair[p] + ko * arows[p];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        v.h[p][h] = *reinterpret_cast<const u32x4*>(a.a_hi + block + 64 * h * arows[p] + aoff[p]);
        v.l[p][h] = *reinterpret_cast<const u32x4*>(a.a_lo + block + 64 * h * arows[p] + aoff[p]);
      }
      v.s[p] = se[srow[p]];
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) v.b[c][h] = *reinterpret_cast<const u32x4*>((c < H ? w : up) + wrow[c][h]);
  };
  auto vec = [](const u32x4 (&v)[2]) {
    return (i32x8){(int)v[0][0], (int)v[0][1], (int)v[0][2], (int)v[0][3],
                   (int)v[1][0], (int)v[1][1], (int)v[1][2], (int)v[1][3]};
  };
  auto put = [&](int tile, const u32x4 (&v)[2]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) *reinterpret_cast<u32x4*>(turn + tile * kOperand + 1024 * h + 16 * lane) = v[h];
  };
  // orders the wavefront's own LDS writes and reads (no other wavefront uses the buffer)
  auto turned = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
  Step v[D];
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < steps) load(d, v[d]);
  const int64_t scale_row = (col0 / kBlock) * KB;  // the item's columns lie in one scale block
  for (int kb = threadIdx.x; kb < KB; kb += 64 * kDenseWaves) {
    lds_sw[kb] = a.scale[scale_row + kb];
    if constexpr (SWIGLU) lds_sw[KB + kb] = a.scale_up[scale_row + kb];
  }

  uint32_t found = 0;
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  auto multiply = [&](int slot, const Step& v) {  // the step's results into slot (block slot of the fold)
    i32x8 b[C], bc[1], ah[P], al[P];
    int se[P];
#pragma unroll
    for (int c = 0; c < C; ++c) put(c, v.b[c]);
    if constexpr (RAW) {
      // byte (row, k) of a tile at 128 row + 16 (k / 16 ^ row % 8 ^ row / 8) + k % 16 (operand_slots)
      // The four rows side by side (one branch for all of them): each is a
      // chain of ~60 dependent instructions.
      Bf16Run<8> x[4];
      SplitScale sc[4];
      uint32_t hi[4][2], lo[4][2];
      bool plain = true;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) x[i].w[j] = (i < 2 ? v.h : v.l)[0][i & 1][j];
        // a lane with a NaN counts as infinite: no plain block
        sc[i] = split_scale(row16_amax(__uint_as_float(min(lane_amax_bits<8>(x[i]), 0x7F80u) << 16)));
        plain = plain && sc[i].plain;
      }
      if (__builtin_expect(__builtin_amdgcn_ballot_w64(!plain) == 0, 1)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) split_encode_plain<8>(x[i], sc[i], hi[i], lo[i]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          bool has_nan;
          sc[i] = split_scale(row16_amax(lane_amax<8>(x[i], has_nan)));
          split_encode_any<8>(x[i], sc[i], hi[i], lo[i]);
        }
      }
      uint32_t codes = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        codes |= scale_e8m0(sc[i].s) << (8 * i);
        const int row = 4 * i + kq;
        uint8_t* at = turn + C * kOperand + 128 * row + 16 * ((r >> 1) ^ (row & 7) ^ (row >> 3)) + 8 * (r & 1);
        *reinterpret_cast<uint2*>(at) = make_uint2(hi[i][0], hi[i][1]);
        *reinterpret_cast<uint2*>(at + kOperand) = make_uint2(lo[i][0], lo[i][1]);
      }
      // row r's scale code: byte r / 4 of the codes of lanes 16 (r % 4) ..
      codes = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(4 * 16 * (r & 3), static_cast<int>(codes)));
      se[0] = static_cast<int>((codes >> (8 * (r >> 2))) & 0xFFu);
    } else {
#pragma unroll
      for (int p = 0; p < P; ++p) {
        ah[p] = vec(v.h[p]);
        al[p] = vec(v.l[p]);
        se[p] = static_cast<int>(scale_e8m0(v.s[p]));
      }
    }
    turned();
#pragma unroll
    for (int c = 0; c < C; ++c) b[c] = lds_operand(turn + c * kOperand, slots);
    if constexpr (RAW) {
      ah[0] = lds_operand(turn + C * kOperand, slots);
      al[0] = lds_operand(turn + (C + 1) * kOperand, slots);
    }
    turned();
    if constexpr (DETECT) {
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int i = 0; i < 8; ++i) found |= codes_480(static_cast<uint32_t>(b[c][i]));
      asm volatile("" : "+v"(found));  // here, not after the loop with every operand kept
    }
    constexpr f32x4 kZero = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (FIX) {  // one tile at a time: its corrections take another operand's registers
#pragma unroll
      for (int c = 0; c < C; ++c) {
        weight_operand<FIX>(b[c], bc[0]);
#pragma unroll
        for (int p = 0; p < P; ++p) {
          const f32x4 x = pair_pass<FIX, 0, 127>(ah[p], b[c], bc[0], kZero, se[p]);
          lds_c[(slot * P * C + p * C + c) * 64 + lane] = pair_pass<FIX, 0, 123>(al[p], b[c], bc[0], x, se[p]);
        }
      }
    } else {
      f32x4 x[P][C];
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int c = 0; c < C; ++c)
          x[p][c] = pair_pass<FIX, 0, 127>(ah[p], b[c], b[c], kZero, se[p]);
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int c = 0; c < C; ++c)
          lds_c[(slot * P * C + p * C + c) * 64 + lane] =
              pair_pass<FIX, 0, 123>(al[p], b[c], b[c], x[p][c], se[p]);
    }
  };
  // adds the results of the K blocks of steps s0 .. s0 + F - 1, in block order
  auto fold = [&](int s0) {
    if (wave >= P * C) return;
    const int first = kDenseWaves * s0;
    const int count = KB - first < kDenseWaves * F ? KB - first : kDenseWaves * F;
    const f32x4* mine = lds_c + wave * 64 + lane;
    const float* my_sw = lds_sw + (wave % C < H ? 0 : KB);
    int i = 0;
    for (; i + 8 <= count; i += 8) {
      f32x4 x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = mine[(i + u) * P * C * 64];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float t = my_sw[first + i + u];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = fmaf(x[u][e], t, acc[e]);
      }
    }
    for (; i < count; ++i) {
      const f32x4 x = mine[i * P * C * 64];
      const float t = my_sw[first + i];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = fmaf(x[e], t, acc[e]);
    }
  };
  // R steps from s0 on (every register index static); LAST: none follows, so
  // nothing past them is loaded
  auto run = [&](auto R, auto LAST, int s0) {
#pragma unroll
    for (int f = 0; f < R.value; ++f) {
      multiply(kDenseWaves * (f % F) + wave, v[0]);
      __builtin_amdgcn_sched_barrier(0);  // the next loads take the registers this step leaves
#pragma unroll
      for (int d = 0; d + 1 < D; ++d) v[d] = v[d + 1];
      if (!LAST.value || f + D < R.value) load(s0 + f + D, v[D - 1]);
      if (f % F == F - 1 || f == R.value - 1) {
        __syncthreads();
        fold(s0 + f / F * F);
        if (!LAST.value || f < R.value - 1) __syncthreads();
      }
    }
  };
  int s0 = 0;
  for (; s0 + U < steps; s0 += U) run(Int<U>{}, Int<0>{}, s0);
  switch (steps - s0) {  // 1 .. U
    case 1: run(Int<1>{}, Int<1>{}, s0); break;
    case 2: if constexpr (U > 1) run(Int<2>{}, Int<1>{}, s0); break;
    case 3: if constexpr (U > 2) run(Int<3>{}, Int<1>{}, s0); break;
    default: if constexpr (U > 2) run(Int<4>{}, Int<1>{}, s0); break;
  }
  // lane holds rows 4 kq .. 4 kq + 3, column r of tile `wave`
  const int64_t n = col0 + 16 * (wave % C) + r;
  uint32_t y[2];
  if constexpr (SWIGLU) {
    f32x4* turned_up = lds_c + (wave % C < H ? wave + H : wave) * 64 + lane;  // the matching up tile's results
    __syncthreads();  // every fold has read its results
    if (wave < P * C && wave % C >= H) *turned_up = (f32x4){acc[0], acc[1], acc[2], acc[3]};
    __syncthreads();
    if (wave >= P * C || wave % C >= H) return found;
    const f32x4 up = *turned_up;
    SwigluCheck check;
#pragma unroll
    for (int q = 0; q < 2; ++q)
      y[q] = swiglu_mlx_straight2(acc[2 * q], up[2 * q], acc[2 * q + 1], up[2 * q + 1], a.limit, check);
    if (__builtin_amdgcn_ballot_w64(!swiglu_straight_ok(check, a.limit)) != 0) {
#pragma unroll
      for (int q = 0; q < 2; ++q)
        y[q] = swiglu_mlx(acc[2 * q], up[2 * q], a.limit) |
               static_cast<uint32_t>(swiglu_mlx(acc[2 * q + 1], up[2 * q + 1], a.limit)) << 16;
    }
  } else {
    if (wave >= P * C) return found;
#pragma unroll
    for (int q = 0; q < 2; ++q) y[q] = f32x2_to_bf16x2(acc[2 * q], acc[2 * q + 1]);
  }
  if (n < a.N) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t m = row0 + 16 * (wave / C) + 4 * kq + e;
      if (m < a.rows) a.out[m * a.N + n] = static_cast<uint16_t>(e & 1 ? y[e >> 1] >> 16 : y[e >> 1]);
    }
  }
  return found;
}

// Workgroup i runs on XCD i % 8; each XCD takes a contiguous run of items,
// row groups fastest, so the items that share weight columns meet in one L2.
template <int P, int C, bool SWIGLU, bool RAW>
__global__ __launch_bounds__(64 * kDenseWaves) void dense_ksplit_kernel(DenseArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds_dyn[];
  constexpr int kCols = SWIGLU ? 8 * C : 16 * C;
  const int64_t row_groups = (a.rows + 16 * P - 1) / (16 * P);
  const int64_t items = row_groups * ((a.N + kCols - 1) / kCols);
  const int64_t per_xcd = (items + 7) / 8;
  const int64_t i = static_cast<int64_t>(blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (i >= items) return;
  const int64_t row0 = 16 * P * (i % row_groups), col0 = kCols * (i / row_groups);
  const bool look = a.flag == nullptr || (SWIGLU && a.flag_up == nullptr);
  bool fix = (a.flag != nullptr && *a.flag != 0) || (SWIGLU && a.flag_up != nullptr && *a.flag_up != 0);
  if (!fix) {
    const uint32_t found = dense_ksplit_item<P, C, SWIGLU, RAW, false, true>(a, row0, col0, lds_dyn);
    if (look) fix = workgroup_any((found & 0x80808080u) != 0, lds_dyn);
  }
  if (fix) dense_ksplit_item<P, C, SWIGLU, RAW, true, false>(a, row0, col0, lds_dyn);
}

template <int P, int C, bool SWIGLU, bool RAW>
hipError_t launch_ksplit_t(const DenseArgs& a, hipStream_t st) {
  constexpr int kCols = SWIGLU ? 8 * C : 16 * C;
  const int64_t items = ((a.rows + 16 * P - 1) / (16 * P)) * ((a.N + kCols - 1) / kCols);
  const size_t lds = dense_lds_bytes<P, C, RAW>(a.K);
  if (a.K > kDenseMaxK || lds > 160 * 1024) return hipErrorInvalidValue;
  hipLaunchKernelGGL((dense_ksplit_kernel<P, C, SWIGLU, RAW>), dim3(static_cast<unsigned>(8 * ((items + 7) / 8))),
                     dim3(64 * kDenseWaves), lds, st, a);
  return hipGetLastError();
}

template <int P, int C, bool SWIGLU>
hipError_t launch_ksplit(const DenseArgs& a, hipStream_t st) {
  if constexpr (P == 1) {
    if (a.x != nullptr) return launch_ksplit_t<P, C, SWIGLU, true>(a, st);
  }
  return a.x != nullptr ? hipErrorInvalidValue : launch_ksplit_t<P, C, SWIGLU, false>(a, st);
}

}  // namespace

// The smallest tile whose items fit one round of a workgroup per CU: a
// larger tile brings fewer bytes per output but takes longer per round, and
// a second round mostly costs more than the larger tile does.  All figures
// are us per call, split included, of replayed graphs over weights that no
// cache holds.  N = 4096, K = 4096, each tile at its last one-round row count
// and just past it: 16 x 16 11.6 at 16 rows, 19.5 at 24, where 16 x 32 takes
// 12.4; 16 x 32 12.6 at 32, 21.7 at 48, where 32 x 32 takes 13.0; 32 x 32 14.2
// at 64, 21.5 at 96, where 32 x 64 takes 17.0; 32 x 64 17.7 at 128, 28.8 at
// 200 (32 x 128 32.0); 64 x 128 34.5 at 400 and 39.5 at 512 (256 items, where
// 128 x 128 takes 38.9: two workgroups per CU share the load path); 128 x 128
// 46.5 at 1,024; 128 x 256 57.4 at 1,500; 128 x 512 74.6 at 2,048 and 97.3 at
// 4,096 (kernel alone), one round of the matrix pipes at 2.8 PFLOP/s counting
// both passes.  (64 x 128 takes 25.6 at 16 rows, 32.5 at 128, 85.2 at 2,048.)
// Where a tile's items are not the whole of it:
// * 32 x 128 streams the weights past the caches, so row groups that read the
//   same columns again pay for it unless the matrix is small or the K loop
//   long: 32 x 128 / 64 x 128 at 256 x 4096 x 1536 18.6 / 17.3, 288 x 3072 x
//   3072 27.7 / 26.6; but 160 x 6144 x 2048 0.95 of it, 2,048 x 512 x 7168
//   50.7 / 58.3, 200 x 4096 x 8192 52.9 / 59.6.
// * 64 x 128 has two workgroups per CU.  Over few columns (activations are
//   most of the bytes) it beats the 128-row tiles up to 512 items: 4,096 x 512
//   x 512 13.3 / 15.5 (128 x 128), 2,048 x 1536 x 4096 42.3 / 44.1; and where
//   128 x 128 no longer fits, 128 x 256: 320 x 12288 x 4096 46.2 / 54.5.  Over
//   a matrix of more than 16 MB it wins up to 256 items (twice the CUs that
//   128 x 128 has busy: 256 x 8192 x 7168 63.0 / 67.5, 128 x 16384 x 4096 39.5 /
//   43.0; 256 x 8192 x 512 12.4 / 11.1), and from 32 MB on at 257 to 384 rows,
//   where 128 x 128 has three row groups (384 x 8192 x 7168 65.9 / 69.6).
// * Few rows over more columns than one round of 128 x 256 holds are a
//   stream of the weights: 32 x 128 (16 x 131072 x 4096 106 us, 128 x 512 133,
//   64 x 128 131; not for a few K blocks: 2 x 131072 x 512 21.8 / 18.1), and
//   128 x 256 for up to 64 rows where 128 x 512 needs a second round (48 x
//   151936 x 7168 231 / 253).
// The narrow tiles' offsets fit 32 bits, the wide shape's 31.
// A SwiGLU tile holds half as many output columns in the same time (gate and
// up tile side by side), so 16 x 16 and 128 x 128 have no SwiGLU form.
DenseTile dense_tile(int64_t rows, int64_t K, int64_t N, bool swiglu) {
  constexpr DenseTile kNarrow[] = {{16, 16}, {16, 32}, {32, 32}, {32, 64}};  // weight columns
  const bool narrow = K <= kDenseMaxK && N * K < (int64_t{1} << 32) && rows * K < (int64_t{1} << 32);
  const bool wide = K <= kWideDenseMaxK && wide_offsets_fit(N, K, rows);
  auto of = [&](DenseTile t) { return DenseTile{t.rows, swiglu ? t.cols / 2 : t.cols}; };
  auto items = [&](DenseTile t) {
    t = of(t);
    return ((rows + t.rows - 1) / t.rows) * ((N + t.cols - 1) / t.cols);
  };
  for (const DenseTile& t : kNarrow)
    if (narrow && !(swiglu && t.cols == 16) && items(t) <= 256) return of(t);
  if (items({32, 128}) <= 256 && (swiglu || rows <= 192 || N <= 2048 || K >= 4096)) return of({32, 128});
  if (!wide) return of({64, 128});
  int64_t most = 224;
  if (!swiglu) {
    if (N <= 2048 || (N <= 3072 && K >= 2048) || (rows > 128 && items({128, 128}) > 256)) most = 512;
    else if (rows > 256 && rows <= 384 && N * K >= (int64_t{1} << 25)) most = 384;
    else if (N * K > (int64_t{1} << 24)) most = 256;
  }
  if (items({64, 128}) <= most) return of({64, 128});
  if (!swiglu && items({128, 128}) <= 256) return of({128, 128});
  if (items({128, 256}) <= 256) return of({128, 256});
  if (!swiglu && rows <= 32 && K >= 1024) return of({32, 128});
  if (!swiglu && rows <= 64 && items({128, 512}) > 256) return of({128, 256});
  return of({128, 512});
}

// One-pair tiles split their own blocks: the conversion (~55 instructions per
// 8 columns, every workgroup for its 16 rows, the four rows of a lane side by
// side: one after the other they took 13.3 us) makes the kernel 11.6 us at 16
// x 4096 x 4096 where split and product take 3.7 + 7.0 and a launch between,
// and saves that launch and the workspace.  The conversion grows with K where
// the split's launch does not.  Eager calls of 16 rows over 4096 columns (us,
// in the kernel / by a launch): 11.4 / 15.4 at K = 4096, 14.5 / 15.4 at 6144,
// 16.0 / 15.5 at 7168, 18.1 / 15.5 at 8192: past ~6,700 it keeps the workspace
// away but no longer saves time, and longer rows keep the launch.  In a
// replayed graph, where a launch costs little, the launch is the quicker one:
// 11.6 / 9.4 at K = 4096, 19.4 / 15.2 at 8192.
bool dense_splits_x(DenseTile t, int64_t K, bool swiglu) {
  return t.rows == 16 && dense_ksplit(t, swiglu) && K <= 8192;
}

hipError_t launch_dense_linear(const DenseArgs& a, DenseTile t, bool swiglu, hipStream_t st) {
  if (a.x != nullptr && (!dense_splits_x(t, a.K, swiglu) || reinterpret_cast<uintptr_t>(a.x) % 16 != 0 ||
                         a.rows * a.K >= (int64_t{1} << 31)))
    return hipErrorInvalidValue;
  if (a.rows <= 0 || a.K <= 0 || a.K % kBlock != 0 || a.N <= 0 || a.N % 16 != 0) return hipErrorInvalidValue;
  if (a.N * a.K >= (int64_t{1} << 32) || a.rows * a.K >= (int64_t{1} << 32)) return hipErrorInvalidValue;
  const int cols = swiglu ? 2 * t.cols : t.cols;
  if (t.rows == 16 && cols == 16 && !swiglu) return launch_ksplit<1, 1, false>(a, st);
  if (t.rows == 16 && cols == 32) return swiglu ? launch_ksplit<1, 2, true>(a, st) : launch_ksplit<1, 2, false>(a, st);
  if (t.rows == 32 && cols == 32) return swiglu ? launch_ksplit<2, 2, true>(a, st) : launch_ksplit<2, 2, false>(a, st);
  if (t.rows == 32 && cols == 64) return swiglu ? launch_ksplit<2, 4, true>(a, st) : launch_ksplit<2, 4, false>(a, st);
  return hipErrorInvalidValue;
}

}  // namespace glm53
