// The FP8 MFMA step shared by the matrix kernels: operand vectors, the exact
// treatment of weight codes 0x7F / 0xFF, and the chained hi / lo pass of a
// 16-row pair over a 16-row weight tile.
#pragma once

#include "common.h"

namespace glm53 {

typedef int32_t i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// E4M3 codes 0x7F / 0xFF decode to +-480 in the reference's table but are
// NaN in the OCP E4M3 format the MFMA consumes.  Checkpoint quantisation
// never emits them (it saturates at +-448), so weights are scanned once and
// only a flagged matrix takes the FIX variant: such bytes are fed as
// 0x7E / 0xFE (+-448) and a second, chained MFMA adds +-32 at exactly those
// positions, reproducing +-480 without leaving the FP8 path.
__device__ __forceinline__ void split_480(uint32_t w, uint32_t& fixed, uint32_t& corr) {
  const uint32_t t = (w & 0x7F7F7F7Fu) ^ 0x7F7F7F7Fu;          // zero byte where |code| == 0x7F
  const uint32_t z = ~((t | 0x80808080u) - 0x01010101u) & 0x80808080u;  // exact per-byte zero test
  const uint32_t m = z >> 7;
  fixed = w ^ m;                                               // 0x7F -> 0x7E, 0xFF -> 0xFE
  corr = (m * 0x60u) | (w & z);                                // +-32 (code 0x60) where fixed
}

// Bit 7 of each byte set where the code is 0x7F or 0xFF (the other bits are
// not cleared): a byte's low 7 bits plus 1 reach 0x80 only from 0x7F.
__device__ __forceinline__ uint32_t codes_480(uint32_t w) { return (w & 0x7F7F7F7Fu) + 0x01010101u; }

constexpr int kOperand = 2048;  // one 16-row x 128-byte operand tile in LDS

// LDS layout of one 16-row x 128-byte operand tile: row r's 16-byte piece p
// sits in slot p ^ (r % 8) ^ (r / 8) of the row's 128 bytes, so the two
// direct loads that fill a tile each read 8 rows as whole 128-byte lines
// (lane l: row l / 8, slot l % 8).  The MFMA reads below (lane l: row
// l % 16, pieces 2 (l / 16) and 2 (l / 16) + 1) run at the LDS's full
// 16-byte read rate with this permutation: a read probe of the operand
// pattern measured ~210 bytes per clock per CU, the rate of 64 consecutive
// 16-byte reads, against ~120 for slot p ^ ((r / 2) % 8), though both give
// every 16 consecutive lanes distinct banks.
struct OperandSlots {
  uint32_t lo, hi;  // byte offsets of the lane's two pieces in a tile
};
__device__ __forceinline__ OperandSlots operand_slots(int lane) {
  const int r = lane & 15, kq = lane >> 4, g = (r & 7) ^ (r >> 3);
  return {static_cast<uint32_t>(128 * r + 16 * ((2 * kq) ^ g)), static_cast<uint32_t>(128 * r + 16 * ((2 * kq + 1) ^ g))};
}
// Byte offset, within its row's 128-byte K block, of the piece lane l loads
// in load h (0: rows 0-7, 1: rows 8-15) of a tile; its row is 8 h + l / 8,
// its slot l % 8, so the piece is (l % 8) ^ (l / 8) ^ h: load 1's offset is
// load 0's with bit 4 flipped.
__device__ __forceinline__ int load_piece_offset(int lane, int h) {
  return 16 * ((lane & 7) ^ (lane >> 3) ^ h);
}

__device__ __forceinline__ i32x8 lds_operand(const uint8_t* tile, OperandSlots o) {
  const u32x4 lo = *reinterpret_cast<const u32x4*>(tile + o.lo);
  const u32x4 hi = *reinterpret_cast<const u32x4*>(tile + o.hi);
  return (i32x8){(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
}

// E8M0 code of an activation block scale: the split's scales are powers of
// two 2^e, -126 <= e <= 127, whose FP32 exponent field e + 127 is the code.
__device__ __forceinline__ uint32_t scale_e8m0(float s) { return (__float_as_uint(s) >> 23) & 0xFFu; }

// A weight tile's B operand as the MFMA takes it: FIX feeds codes 0x7F /
// 0xFF as 0x7E / 0xFE and returns the +-32 corrections in bc.
template <bool FIX>
__device__ __forceinline__ void weight_operand(i32x8& b, i32x8& bc) {
  bc = (i32x8){0, 0, 0, 0, 0, 0, 0, 0};
  if (FIX) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      uint32_t f, cr;
      split_480(static_cast<uint32_t>(b[i]), f, cr);
      b[i] = static_cast<int>(f);
      bc[i] = static_cast<int>(cr);
    }
  }
}

// One pass of a 16-route pair over a weight tile: rows a (the pair's hi or
// lo rows) times b (FIX: plus the corrections bc) added into c.  The A rows'
// E8M0 scale is byte OPSEL of se (the lane's route), the B scale SB (127:
// 1 for the hi rows, 123: 1/16 for the lo rows).
template <bool FIX, int OPSEL, int SB>
__device__ __forceinline__ f32x4 pair_pass(const i32x8& a, const i32x8& b, const i32x8& bc, f32x4 c, int se) {
  c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, OPSEL, se, 0, SB);
  if (FIX) c = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, bc, c, 0, 0, OPSEL, se, 0, SB);
  return c;
}
// pair_pass with the scale byte chosen by a value that unrolling makes constant
template <bool FIX, int SB>
__device__ __forceinline__ f32x4 pair_pass_byte(int byte, const i32x8& a, const i32x8& b, const i32x8& bc, f32x4 c,
                                                int se) {
  switch (byte) {
    case 0: return pair_pass<FIX, 0, SB>(a, b, bc, c, se);
    case 1: return pair_pass<FIX, 1, SB>(a, b, bc, c, se);
    case 2: return pair_pass<FIX, 2, SB>(a, b, bc, c, se);
    default: return pair_pass<FIX, 3, SB>(a, b, bc, c, se);
  }
}

// True in every thread when any thread of the workgroup passes true.  Waits
// for the workgroup's earlier stores, so that what follows may write the
// same addresses; `lds` is free to be overwritten once all threads are here.
__device__ __forceinline__ bool workgroup_any(bool mine, uint8_t* lds) {
  uint32_t* word = reinterpret_cast<uint32_t*>(lds);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) *word = 0;
  __syncthreads();
  if (mine) atomicOr(word, 1u);
  __syncthreads();
  const bool any = *word != 0;
  __syncthreads();
  return any;
}

}  // namespace glm53
