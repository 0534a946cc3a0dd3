// Device-side building blocks for the gfx950 (CDNA4) delta-rule kernels.
//
// Everything here is written for 64-wide wavefronts and the 16x16 MFMA tiles of CDNA4:
//   bf16:  v_mfma_f32_16x16x32_bf16   (8 bf16 of A and of B per lane, fp32 accumulate)
//   fp32:  v_mfma_f32_16x16x4_f32     (1 fp32 of A and of B per lane)
//
// Lane layout of one 16x16xK MFMA (lane l, group g = l / 16, column c = l % 16):
//   A operand:  A[row = c][k in the lane's K slice]
//   B operand:  B[k in the lane's K slice][col = c]
//   D result :  D[row = 4*g + i][col = c], i = 0..3 (a floatx4 per lane)
//
// "Permuted K".  A contraction does not care in which order its K indices are visited, as long
// as A and B agree.  We choose, per 16-row D block, the K order in which lane group g consumes
// exactly the four rows 4g..4g+3 that it already holds in its D registers.  Then the output
// of one MFMA chain (a [16R x 16] D tile) is directly the B operand of the next product that
// contracts over those R*16 rows — no LDS round trip, no cross-lane shuffle.  The matching A
// operand reads, for lane (row c, group g), the columns {4g..4g+3} of each 16-column block,
// i.e. short contiguous runs of the row-major A source.
//   bf16 (K = 32 per instruction): a K-block of 32 rows = D blocks (2kb, 2kb+1); lane group g
//        supplies rows {32kb + 4g + 0..3} and {32kb + 16 + 4g + 0..3}.
//   fp32 (K = 4 per instruction): a K-block of 16 rows = D block kb, consumed by 4 MFMAs; MFMA
//        i takes row 16kb + 4g + i from lane group g.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pf {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));   // one 16-byte vector
// The same at a caller's address that promises an element's alignment only (a contiguous view that starts
// inside a buffer): one instruction all the same, since global accesses need no more.
typedef float floatx4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned int u32x4_any __attribute__((ext_vector_type(4), aligned(2)));
typedef __bf16 bf16x4_any __attribute__((ext_vector_type(4), aligned(2)));

__device__ __forceinline__ float to_f32(float x) { return x; }
__device__ __forceinline__ float to_f32(bf16 x) { return (float)x; }

template <typename E> __device__ __forceinline__ E from_f32(float x);
template <> __device__ __forceinline__ float from_f32<float>(float x) { return x; }
template <> __device__ __forceinline__ bf16 from_f32<bf16>(float x) { return (bf16)x; }

__device__ __forceinline__ floatx4 zero4() { return floatx4{0.f, 0.f, 0.f, 0.f}; }

// Workgroup barrier that orders LDS traffic only.  __syncthreads() is a workgroup memory fence:
// it waits for every outstanding global load and store of the wave (vmcnt(0)) before the
// barrier, which turns register prefetches into synchronous HBM round trips.  Here the wave waits
// only for its own LDS operations (lgkmcnt(0); vmcnt and expcnt left at their maxima), so loads
// and stores to global memory stay in flight across the barrier.  Valid because no wave of these
// kernels reads global data that another wave of the same workgroup writes.
__device__ __forceinline__ void lds_barrier() {
  __asm__ __volatile__("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // gfx9 encoding: vmcnt 63, expcnt 7, lgkmcnt 0
  __builtin_amdgcn_s_barrier();
  __asm__ __volatile__("" ::: "memory");
}

// Index of the lower-triangular 16x16 tile (ib, jb), jb <= ib, of a 64 x 64 chunk matrix (T, the
// score) in a packed list of its ten tiles.
__device__ __forceinline__ constexpr int score_tile_index(int ib, int jb) { return ib * (ib + 1) / 2 + jb; }

// exp(x) for x <= 0, 0 for x > 0 (the reference's _safe_exp).
__device__ __forceinline__ float safe_exp(float x) { return x <= 0.f ? __expf(x) : 0.f; }

// --------------------------------------------------------------------------------------------
//  MFMA traits.  KB = contraction rows consumed per "K-block" step.
// --------------------------------------------------------------------------------------------
template <typename E> struct Mfma;

template <> struct Mfma<bf16> {
  static constexpr int KB = 32;
  // acc += A x B^T with both operands read as rows from memory (natural K order).
  // arow = row (lane c) of A, brow = row (lane c) of B, K-block kb.
  __device__ __forceinline__ static floatx4 rows(floatx4 acc, const bf16* arow, const bf16* brow,
                                                 int kb, int g) {
    bf16x8 a = *reinterpret_cast<const bf16x8*>(arow + kb * 32 + 8 * g);
    bf16x8 b = *reinterpret_cast<const bf16x8*>(brow + kb * 32 + 8 * g);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
  }
};

template <> struct Mfma<float> {
  static constexpr int KB = 16;
  __device__ __forceinline__ static floatx4 rows(floatx4 acc, const float* arow, const float* brow,
                                                 int kb, int g) {
    floatx4 a = *reinterpret_cast<const floatx4*>(arow + kb * 16 + 4 * g);
    floatx4 b = *reinterpret_cast<const floatx4*>(brow + kb * 16 + 4 * g);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[0], b[0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[1], b[1], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[2], b[2], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[3], b[3], acc, 0, 0, 0);
    return acc;
  }
};

// Store four consecutive values as one vector (8 bytes of bf16 or 16 bytes of fp32).
__device__ __forceinline__ void store4(bf16* p, float a, float b, float c, float d) {
  *reinterpret_cast<bf16x4*>(p) = bf16x4{(bf16)a, (bf16)b, (bf16)c, (bf16)d};
}
__device__ __forceinline__ void store4(float* p, float a, float b, float c, float d) {
  *reinterpret_cast<floatx4*>(p) = floatx4{a, b, c, d};
}

// 16-byte vector type of an element type (8 bf16 or 4 fp32).
template <typename E> struct Vec16;
template <> struct Vec16<bf16> { typedef uint4 T; static constexpr int N = 8; };
template <> struct Vec16<float> { typedef uint4 T; static constexpr int N = 4; };

}  // namespace pf
