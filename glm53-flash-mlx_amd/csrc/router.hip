// FP32 router logits for many tokens (patch.py:131-134 of the reference:
// logits = x.astype(float32) @ W.T, W FP32 [experts, hidden]) on BF16 MFMA.
//
// Every FP32 weight w is split exactly into three BF16 parts by truncation:
// hi = w with its low 16 bits cleared, mid = (w - hi) truncated the same
// way, lo = w - hi - mid (at most 8 significant bits, so exact in BF16);
// w = hi + mid + lo.  A BF16 activation times a BF16 part is exact in FP32,
// so three v_mfma_f32_16x16x32_bf16 per operand pair accumulate x . w in
// FP32 like an FP32 GEMM; only the order of the FP32 additions differs.
//
// Work item = 128 tokens x 96 experts (few tokens: 32 x 32) x one K chunk, 4
// wavefronts in a 2 x 2 grid (64 tokens x 48 experts each: 4 x 3 MFMA tiles).  Per 32-deep K step
// the workgroup loads the tokens' BF16 rows (8 KB) and the experts' FP32 rows
// (12 KB) once from global memory into registers, kAhead steps ahead, splits
// the weights into their three BF16 parts on the way into LDS (18 KB), and
// every wavefront reads its MFMA operands from LDS: each operand byte leaves
// L2 once per workgroup (the register-operand form read the token rows once
// per wavefront).  K chunks ("splits") write FP32 partial sums
// [split][token][expert]; topk_kernel adds them in split order.  Items run
// split-major in contiguous runs per XCD, so the items of one split share
// that chunk's weight rows in one L2.

#include "common.h"
#include "kernels.h"

namespace glm53 {

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// Tile = 32 MT tokens x 32 NT experts (2 x 2 wavefronts of MT x NT MFMA tiles).
constexpr int kWideMT = 4, kWideNT = 3;         // 128 x 96
constexpr int64_t kRouterSmallItems = 1152;     // 32 x 32 tiles up to this many work items
constexpr int kStep = 32;                       // K per step: one v_mfma_f32_16x16x32_bf16
constexpr int kRowBytes = kStep * 2;            // 64 B: one BF16 row of a step in LDS
template <int MT, int NT>
constexpr int stage_bytes() {                   // token rows, then three planes of expert rows
  return (32 * MT + 3 * 32 * NT) * kRowBytes;
}

// Octet q (8 BF16 = 16 B) of LDS row r sits at slot q ^ ((r >> 2) & 3): the
// 16 lanes reading octet q of rows r .. r + 15 then spread over all banks.
__device__ __forceinline__ int slot_offset(int r, int q) { return r * kRowBytes + 16 * (q ^ ((r >> 2) & 3)); }

// The upper halves of a and b as one word (a's below).
__device__ __forceinline__ uint32_t upper_halves(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

// The three BF16 parts of four FP32 weights, packed two per word.
__device__ __forceinline__ void split3(const f32x4_t& v, uint2& hi, uint2& mid, uint2& lo) {
  auto upper = [](float x) { return __uint_as_float(__float_as_uint(x) & 0xffff0000u); };
  float r1[4], r2[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    r1[j] = v[j] - upper(v[j]);
    r2[j] = r1[j] - upper(r1[j]);  // fits in BF16
  }
  hi = make_uint2(upper_halves(v[0], v[1]), upper_halves(v[2], v[3]));
  mid = make_uint2(upper_halves(r1[0], r1[1]), upper_halves(r1[2], r1[3]));
  lo = make_uint2(upper_halves(r2[0], r2[1]), upper_halves(r2[2], r2[3]));
}

// One step's global operands held by a thread: token rows (two 16-byte BF16
// octets) and expert rows (three 16-byte FP32 quads).
// ext_vector_type members: with HIP's uint4 / float4 the register copies
// became memcpy's that kept the prefetched activations in scratch memory,
// each written there right after its load was issued (that is, after
// waiting for it), and the many-token router ran ~10% longer.
template <int MT, int NT>
struct StepRegs {
  u32x4_t x[MT > 1 ? MT / 2 : 1];
  f32x4_t w[NT];
};

// kAhead: K steps of global loads in flight.
template <int MT, int NT, int kAhead>
__global__ __launch_bounds__(256, 2) void router_tile_kernel(RouterGemmArgs a, const float* __restrict__ weight) {
  constexpr int kTileTokens = 32 * MT, kTileExperts = 32 * NT;
  constexpr int kXBytes = kTileTokens * kRowBytes, kPlaneBytes = kTileExperts * kRowBytes;
  constexpr int kStageBytes = stage_bytes<MT, NT>();
  constexpr int kXLoads = MT > 1 ? MT / 2 : 1;  // octets per thread
  static_assert(MT == 1 || MT % 2 == 0, "whole octets per thread");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];  // 2 stages
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int64_t groups = a.token_groups * a.expert_groups;
  const int64_t items = groups * a.splits;
  const int64_t per_xcd = (items + 7) / 8;
  const int64_t item = static_cast<int64_t>(blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (item >= items) return;
  const int64_t split = item / groups;
  const int64_t t0 = (item % groups / a.expert_groups) * kTileTokens;
  const int64_t e0 = (item % a.expert_groups) * kTileExperts;
  const int64_t k_begin = split * a.k_chunk;
  const int64_t k_end = k_begin + a.k_chunk < a.hidden ? k_begin + a.k_chunk : a.hidden;
  const int64_t H = a.hidden;

  // ---- global load assignment (rows past the last token / expert re-read
  // the last one; their sums are never stored)
  // tokens: 32 MT rows x 4 octets, octet i = t + 256 j -> row i / 4, octet
  // i % 4: a load instruction takes whole 64-byte pieces of 16 rows (with two
  // neighbouring octets per thread it took half of each piece of 32 rows, and
  // the router and its top-k ran 91.3 us at 8,192 tokens x 288 experts, K =
  // 4,096, instead of 87.0).  MT = 1: 128 octets, which the second half of the
  // threads load again, unused.
  const int xr = (MT > 1 ? t : t & 127) >> 2, xq = t & 3;
  const bool stores_x = MT > 1 || t < 128;
  const uint16_t* xsrc[kXLoads];
#pragma unroll
  for (int j = 0; j < kXLoads; ++j) {
    const int64_t row = t0 + xr + 64 * j;
    xsrc[j] = a.x + (row < a.tokens ? row : a.tokens - 1) * H + 8 * xq;
  }
  // experts: 32 NT rows x 8 quads of 4 FP32, quad i = t + 256 j -> row i / 8, quad i % 8
  const float* wsrc[NT];
  int wr[NT], wq[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int i = t + 256 * j;
    wr[j] = i >> 3;
    wq[j] = i & 7;
    const int64_t e = e0 + wr[j];
    wsrc[j] = weight + (e < a.experts ? e : a.experts - 1) * H + 4 * wq[j];
  }
  auto load = [&](StepRegs<MT, NT>& r, int64_t k) {
#pragma unroll
    for (int j = 0; j < kXLoads; ++j) r.x[j] = *reinterpret_cast<const u32x4_t*>(xsrc[j] + k);
#pragma unroll
    for (int j = 0; j < NT; ++j) r.w[j] = *reinterpret_cast<const f32x4_t*>(wsrc[j] + k);
  };
  auto store = [&](const StepRegs<MT, NT>& r, uint8_t* stage) {
    if (stores_x) {
#pragma unroll
      for (int j = 0; j < kXLoads; ++j) *reinterpret_cast<u32x4_t*>(stage + slot_offset(xr + 64 * j, xq)) = r.x[j];
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      uint2 hi, mid, lo;
      split3(r.w[j], hi, mid, lo);
      // quad wq holds K 4 wq .. 4 wq + 3: half (wq & 1) of octet wq / 2
      const int off = slot_offset(wr[j], wq[j] >> 1) + 8 * (wq[j] & 1);
      uint8_t* planes = stage + kXBytes;
      *reinterpret_cast<uint2*>(planes + off) = hi;
      *reinterpret_cast<uint2*>(planes + kPlaneBytes + off) = mid;
      *reinterpret_cast<uint2*>(planes + 2 * kPlaneBytes + off) = lo;
    }
  };

  // ---- MFMA operand reads: lane reads row 16 tile + lane % 16, octet lane / 16
  const int wm = wave >> 1, wn = wave & 1;  // the wavefront's half of the tokens and of the experts
  const int r16 = lane & 15, q = lane >> 4;
  f32x4_t acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

  // kAhead register sets: step k's global loads are issued kAhead steps
  // before its operands go into LDS, so several steps' loads are in flight
  // behind each step's MFMAs (one step of 32 is too short to cover them).
  StepRegs<MT, NT> regs[kAhead];
#pragma unroll
  for (int d = 0; d < kAhead; ++d)
    if (k_begin + d * kStep < k_end) load(regs[d], k_begin + d * kStep);
  int s = 0;
  for (int64_t k0 = k_begin; k0 < k_end; k0 += kAhead * kStep) {
#pragma unroll
    for (int d = 0; d < kAhead; ++d) {
      const int64_t k = k0 + d * kStep;
      if (k >= k_end) break;
      uint8_t* stage = lds + s * kStageBytes;
      store(regs[d], stage);
      __syncthreads();  // the stage is complete; the other stage's readers are done
      if (k + kAhead * kStep < k_end) load(regs[d], k + kAhead * kStep);
      bf16x8_t xa[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m)
        xa[m] = __builtin_bit_cast(bf16x8_t,
                                   *reinterpret_cast<const uint4*>(stage + slot_offset(16 * MT * wm + 16 * m + r16, q)));
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int row = 16 * NT * wn + 16 * n + r16;
        bf16x8_t wb[3];
#pragma unroll
        for (int p = 0; p < 3; ++p)
          wb[p] = __builtin_bit_cast(
              bf16x8_t, *reinterpret_cast<const uint4*>(stage + kXBytes + p * kPlaneBytes + slot_offset(row, q)));
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
          for (int m = 0; m < MT; ++m)
            acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[m], wb[p], acc[m][n], 0, 0, 0);
      }
      s ^= 1;
    }
  }
  // D layout of the 16x16 MFMA: lane holds rows 4 (lane / 16) + i, column lane % 16.
  float* out = a.partial + split * a.tokens * a.experts;
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int64_t e = e0 + 16 * NT * wn + 16 * n + r16;
    if (e >= a.experts) continue;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t tok = t0 + 16 * MT * wm + 16 * m + 4 * q + i;
        if (tok < a.tokens) out[tok * a.experts + e] = acc[m][n][i];
      }
  }
}

}  // namespace

bool router_gemm_supported(int64_t hidden, int64_t experts, const void* x, const void* weight) {
  return hidden > 0 && hidden % 128 == 0 && experts > 0 && experts <= kMaxRouterExperts &&
         reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(weight) % 16 == 0;
}

RouterGemmShape router_gemm_shape(int64_t tokens, int64_t hidden, int64_t experts) {
  RouterGemmShape s{};
  const int64_t groups = ((tokens + 32 * kWideMT - 1) / (32 * kWideMT)) * ((experts + 32 * kWideNT - 1) / (32 * kWideNT));
  const int64_t blocks = hidden / 128;
  // At most 512 128 x 96 work items (two per CU, one round) where K allows: a
  // 513th item would cost a whole second round (e.g. 2,048 tokens x 288
  // experts, 48 groups over K = 4,096: 11 planes were 528 items, 8 planes are
  // 384), and at most kMaxRouterSplits partial planes.
  int64_t want = 512 / groups;
  if (want > kMaxRouterSplits) want = kMaxRouterSplits;
  if (want > blocks) want = blocks;
  if (want < 1) want = 1;
  const int64_t chunk_blocks = (blocks + want - 1) / want;
  s.k_chunk = chunk_blocks * 128;
  s.splits = (blocks + chunk_blocks - 1) / chunk_blocks;
  // The K chunks follow from the large tile alone, so the sums do not depend
  // on the tile.  Few tokens leave the large tile 48 workgroups of 8 steps
  // with three in flight; 32 x 32 tiles have a chunk's loads in flight all at
  // once over three times the workgroups, until their re-reads of the tokens
  // and weights outweigh it.  Measured (us, large / small tile), 288 experts,
  // K = 4,096: 8 tokens 9.8 / 5.1, 128 10.5 / 7.4, 256 (1,152 small items)
  // 10.9 / 9.5, 384 (1,728) 11.4 / 12.4; 256 experts, K = 7,168: 256 tokens
  // (896) 16.7 / 13.3, 384 (1,344) 17.1 / 17.7; 64 experts, K = 2,048: 1,024
  // tokens (1,024) 7.7 / 5.8.
  const int64_t small_items = ((tokens + 31) / 32) * ((experts + 31) / 32) * s.splits;
  s.few_tokens = small_items <= kRouterSmallItems;
  const int64_t tile_tokens = s.few_tokens ? 32 : 32 * kWideMT, tile_experts = s.few_tokens ? 32 : 32 * kWideNT;
  s.token_groups = (tokens + tile_tokens - 1) / tile_tokens;
  s.expert_groups = (experts + tile_experts - 1) / tile_experts;
  return s;
}

hipError_t launch_router_logits(const RouterGemmArgs& a, bool few_tokens, const float* weight, hipStream_t st) {
  if (a.tokens == 0) return hipSuccess;
  if (!router_gemm_supported(a.hidden, a.experts, a.x, weight) || a.k_chunk % 128 != 0 || a.splits < 1 ||
      a.splits > kMaxRouterSplits)
    return hipErrorInvalidValue;
  // item(b) = (b % 8) * ceil(items / 8) + b / 8 covers every item only over 8 * ceil(items / 8) workgroups
  const int64_t items = a.token_groups * a.expert_groups * a.splits;
  const dim3 grid(static_cast<unsigned>((items + 7) / 8 * 8));
  const size_t lds = few_tokens ? 2 * stage_bytes<1, 1>() : 2 * stage_bytes<kWideMT, kWideNT>();
  if (few_tokens) hipLaunchKernelGGL((router_tile_kernel<1, 1, 8>), grid, dim3(256), lds, st, a, weight);
  else hipLaunchKernelGGL((router_tile_kernel<kWideMT, kWideNT, 3>), grid, dim3(256), lds, st, a, weight);
  return hipGetLastError();
}

}  // namespace glm53
