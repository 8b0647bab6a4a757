// fp32 products on the bf16 matrix cores.  A value is the sum of three bf16
// parts, each the rounding of what the parts before it leave,
//   x = h + m + l,  |m| <= 2^-9 |x|,  |l| <= 2^-17 |x|,
// exact for every x whose parts neither overflow nor fall below the smallest
// normal (the three hold 24 bits).  The matrix core takes smaller parts as
// zero: products of rows or weights that are all below 2^-112 lose accuracy
// (relative to 64 bits 5.2e-8 down to 2^-108, 1.5e-7 at 2^-112, 2.2e-6 at
// 2^-116; the fp32 product 2.9e-7 throughout), smaller values beside larger
// ones nothing that their sum shows.  Of the nine products of two such sums the
// six largest are formed, each exact in fp32 and summed by the matrix core:
//   a b = ah bh + ah bm + am bh + am bm + ah bl + al bh  (+ < 2^-24 |a b|).
// gfx950 does 16x16x32 bf16 in 16 cycles against 32 for 16x16x4 fp32, so six
// of them take 96 cycles for what eight fp32 steps do in 256.
// The matrix core cuts what an accumulator operand and the products hold below
// its adder's last bit, towards minus infinity: a running sum as that operand
// drifts (16 steps of normal values: 3.4e-7 off in the 2-norm, mean -2.6e-8 of
// the size of the results).  So every chain starts from zero: the five smaller
// products in one, the largest alone, and their sum is added in fp32 (8.6e-8,
// mean -4e-10; eight fp32 matrix steps, added the same way, 1.3e-7).
// A value that is infinite, NaN or rounds to infinity leaves a NaN or an
// infinity in every result that it enters: callers recompute those.
#pragma once
#include "vc_common.h"

namespace vcs {

typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v2f __attribute__((ext_vector_type(2)));

// The three parts of two values, each pair packed (x0 in the low half).
__device__ __forceinline__ void split2(float x0, float x1, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{x0, x1}, v2bf));
  const float a0 = x0 - __builtin_bit_cast(float, h << 16);
  const float a1 = x1 - __builtin_bit_cast(float, h & 0xffff0000u);
  m = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{a0, a1}, v2bf));
  const float b0 = a0 - __builtin_bit_cast(float, m << 16);
  const float b1 = a1 - __builtin_bit_cast(float, m & 0xffff0000u);
  l = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{b0, b1}, v2bf));
}

// Eight values (consecutive k) into one 16-byte operand of each part.
__device__ __forceinline__ void split8(const float* x, uint4& h, uint4& m, uint4& l) {
  split2(x[0], x[1], h.x, m.x, l.x);
  split2(x[2], x[3], h.y, m.y, l.y);
  split2(x[4], x[5], h.z, m.z, l.z);
  split2(x[6], x[7], h.w, m.w, l.w);
}

// One 16x16x32 step.  Operand layout for lane l, g = l / 16, r = l % 16:
//   a[j] = A[row r][k 8 g + j], b[j] = B[k 8 g + j][col r],
//   acc[i] = D[row 4 g + i][col r].
template <class Operand>  // sixteen bytes
__device__ __forceinline__ v4f mfma_bf16(Operand a, Operand b, v4f acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a),
                                                 __builtin_bit_cast(v8bf, b), acc, 0, 0, 0);
}

// The six products' operand parts (0 = h, 1 = m, 2 = l), smallest first; the
// last one is the chain of its own.
constexpr int kPartA[6] = {2, 0, 1, 1, 0, 0};
constexpr int kPartB[6] = {0, 2, 1, 0, 1, 0};

// Loads with the base in scalar registers, a 32-bit byte offset per lane and
// a scalar one beside it; past the buffer's end (kOut) they return zero and
// stores are dropped, so that edges need no branches.
typedef __amdgpu_buffer_rsrc_t Buf;
constexpr uint32_t kOut = 0xffffffffu;
__device__ __forceinline__ Buf buffer(const float* p, int64_t bytes) {
  const int n = (int)(uint32_t)(bytes < 0xfffffff0ll ? bytes : 0xfffffff0ll);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, n, 0x00027000);
}
__device__ __forceinline__ float ldb(Buf b, uint32_t off, int soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(b, off, soff, 0));
}

__device__ __forceinline__ bool finite(float v) { return fabsf(v) <= 3.402823466e38f; }

}  // namespace vcs
