// The score stages (pf_stages.h) at chunks of 16 and 32 tokens: one or two 16-token query blocks for the
// four waves of a workgroup.  The waves of a block (PARTS of them) share its work, key blocks of the score
// and columns of o, and all threads stage the query rows beside the key rows: one wave at work per
// block, with the rows loaded straight by every wave, took up to twice as long (fp32, 1024 chunks of 16 x 128:
// score 6.8 us, with prescales 10.4, chunk output 8.9; here 3.8, 4.5 and 6.0).  Bound by the call below
// about 500 chunks, by the chunk rows' way through LDS above.
#pragma once

#include "pf_stages.h"

namespace pf {

template <typename E, int C, int D>
struct SmallShape {
  static constexpr int VE = Vec16<E>::N, SLOTS = D / VE, NB = C / 16, PARTS = 4 / NB, NKB = D / Mfma<E>::KB;
  static constexpr int NV = C * SLOTS / 256;         // 16-byte vectors of a chunk's rows per thread
  static_assert((C == 16 || C == 32) && C * SLOTS % 256 == 0, "chunks of 16 or 32 rows that divide over 256 threads");
};

// Rows held as vectors u = tid + 256 i go to the key layout; query block ib's rows back as MFMA operands.
template <typename E, int C, int D, int NV>
__device__ __forceinline__ void put_rows(E* dst, const typename VecT<E>::T (&x)[NV], int tid) {
  constexpr int VE = Vec16<E>::N, SLOTS = D / VE;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int u = tid + 256 * i, row = u / SLOTS;
    *reinterpret_cast<typename VecT<E>::T*>(dst + row * D + VE * key_slot<E, D>(row, u % SLOTS)) = x[i];
  }
}
template <typename E, int D, int NKB>
__device__ __forceinline__ void get_block(typename VecT<E>::T (&q)[NKB], const E* src, int ib, int c, int g) {
#pragma unroll
  for (int kb = 0; kb < NKB; ++kb)
    q[kb] = *reinterpret_cast<const typename VecT<E>::T*>(src + (16 * ib + c) * D + Vec16<E>::N * key_slot<E, D>(c, 4 * kb + g));
}

template <typename E, int C, int D, bool MASK>
__global__ __launch_bounds__(256) void gated_qk_small_kernel(GatedQkArgs p) {
  using Sh = SmallShape<E, C, D>;
  typedef typename VecT<E>::T V;
  constexpr int VE = Sh::VE, SLOTS = Sh::SLOTS, NB = Sh::NB, NV = Sh::NV;
  __shared__ __attribute__((aligned(16))) E sa[C * D];
  __shared__ __attribute__((aligned(16))) E sb[C * D];
  __shared__ __attribute__((aligned(16))) float Gs[C], Ls[C];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), ib = w % NB, jb = w / NB;   // this wave's tile
  const int m = blockIdx.x, ch = m / p.H, h = m % p.H;
  const size_t rs = (size_t)p.H * D, base = ((size_t)ch * C * p.H + h) * D;
  const E* ag = static_cast<const E*>(p.a) + base;
  const E* bg = static_cast<const E*>(p.b) + base;

  V ar[NV], br[NV];
  auto off = [&](int i) {
    const int u = tid + 256 * i;
    return (u / SLOTS) * rs + (u % SLOTS) * VE;
  };
#pragma unroll
  for (int i = 0; i < NV; ++i) br[i] = load_vec(bg, off(i));
#pragma unroll
  for (int i = 0; i < NV; ++i) ar[i] = load_vec(ag, off(i));
  const int i = 16 * ib + c, j0 = 16 * jb + 4 * g;     // this lane's row and first column of its tile
  floatx4 mask = zero4();
  if (MASK && jb < NB) mask = *reinterpret_cast<const floatx4_any*>(p.mask + i * C + j0);
  if (p.b_scale) {
#pragma unroll
    for (int i = 0; i < NV; ++i) prescale<E>(br[i], p.b_scale + base, off(i));
  }
  if (p.a_scale) {
#pragma unroll
    for (int i = 0; i < NV; ++i) prescale<E>(ar[i], p.a_scale + base, off(i));
  }
  if (tid < C) {
    const size_t gi = ((size_t)ch * C + tid) * p.H + h;
    Gs[tid] = p.g ? p.g[gi] : 0.f;
    Ls[tid] = p.beta ? __logf(p.beta[gi]) : 0.f;
  }
  put_rows<E, C, D>(sb, br, tid);
  put_rows<E, C, D>(sa, ar, tid);
  lds_barrier();
  if (jb >= NB) return;
  V q[Sh::NKB];
  get_block<E, D>(q, sa, ib, c, g);
  floatx4 out = zero4();                               // strictly-upper tiles of a triangular mask are zero
  if (MASK || jb <= ib) {
    const floatx4 acc = score_tile<E, D>(sb, jb, q, c, g);
    const floatx4 gj = *reinterpret_cast<const floatx4*>(Gs + j0);
    const float gi = Gs[i] + Ls[i];
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
      const float mk = MASK ? mask[ii] : (i + p.causal > j0 + ii ? 1.f : 0.f);
      out[ii] = mk == 0.f ? 0.f : acc[ii] * __expf(fminf(gi - gj[ii], 0.f)) * mk;
    }
  }
  const size_t e = (((size_t)ch * C + i) * p.H + h) * C + j0;
  if (p.out_f32) *reinterpret_cast<floatx4_any*>(static_cast<float*>(p.L) + e) = out;
  else *reinterpret_cast<bf16x4_any*>(static_cast<bf16*>(p.L) + e) = bf16x4_any{(bf16)out[0], (bf16)out[1], (bf16)out[2], (bf16)out[3]};
}

template <typename E, int C, int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 8)))
void qkv_flash_small_kernel(QkvFlashArgs p) {
  using Sh = SmallShape<E, C, D>;
  typedef typename VecT<E>::T V;
  constexpr bool B16 = sizeof(E) == 2;
  constexpr int VE = Sh::VE, SLOTS = Sh::SLOTS, NB = Sh::NB, NV = Sh::NV;
  constexpr int NP = B16 ? (NB + 1) / 2 : NB, NR = D / 16 / Sh::PARTS;
  // fp32 rows of 32 tokens: v takes the query rows' place in LDS, which lets a CU hold one or two workgroups
  // more (2048 chunks of 32 x 128 with prescales: 32.0 us with three tiles, 29.7 with two)
  constexpr bool SHARE = !B16 && C == 32;
  typedef typename std::conditional<B16, bf16x8, floatx4>::type PV;
  __shared__ __attribute__((aligned(16))) E sk[C * D];
  __shared__ __attribute__((aligned(16))) E sq[C * D];
  __shared__ __attribute__((aligned(16))) E sv_own[SHARE ? 1 : C * D];
  E* sv = SHARE ? sq : sv_own;
  __shared__ __attribute__((aligned(16))) PV PX[NB * NP * 64];
  __shared__ __attribute__((aligned(16))) float Gs[C], Ls[C];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), ib = w % NB, part = w / NB;
  const size_t row0 = (size_t)blockIdx.x * C;
  const E* qg = static_cast<const E*>(p.q) + row0 * D;
  const E* kg = static_cast<const E*>(p.k) + row0 * D;
  const E* vg = static_cast<const E*>(p.v) + row0 * D;

  V kr[NV], qr[NV], vr[NV];
  auto off = [&](int i) { return (size_t)(tid + 256 * i) * VE; };
#pragma unroll
  for (int i = 0; i < NV; ++i) kr[i] = load_vec(kg, off(i));
#pragma unroll
  for (int i = 0; i < NV; ++i) qr[i] = load_vec(qg, off(i));
  if (tid < C) {
    Gs[tid] = p.g ? p.g[row0 + tid] : 0.f;
    Ls[tid] = p.beta ? __logf(p.beta[row0 + tid]) : 0.f;
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) vr[i] = load_vec(vg, off(i));
  if (p.k_scale) {
#pragma unroll
    for (int i = 0; i < NV; ++i) prescale<E>(kr[i], p.k_scale + row0 * D, off(i));
  }
  if (p.q_scale) {
#pragma unroll
    for (int i = 0; i < NV; ++i) prescale<E>(qr[i], p.q_scale + row0 * D, off(i));
  }
  put_rows<E, C, D>(sk, kr, tid);
  put_rows<E, C, D>(sq, qr, tid);
  lds_barrier();
  if (part == 0) {   // the first wave of a query block forms its score rows, in the operand type, for all of them
    V q[Sh::NKB];
    get_block<E, D>(q, sq, ib, c, g);
    const int i = 16 * ib + c;
    const float gi = Gs[i] + Ls[i];
    auto tile = [&](int jb) -> floatx4 {
      if (jb > ib) return zero4();
      const floatx4 acc = score_tile<E, D>(sk, jb, q, c, g);
      const floatx4 gj = *reinterpret_cast<const floatx4*>(Gs + 16 * jb + 4 * g);
      floatx4 out;
#pragma unroll
      for (int ii = 0; ii < 4; ++ii)
        out[ii] = i >= 16 * jb + 4 * g + ii ? acc[ii] * __expf(fminf(gi - gj[ii], 0.f)) : 0.f;
      return out;
    };
#pragma unroll
    for (int x = 0; x < NP; ++x) {
      if constexpr (B16) PX[(ib * NP + x) * 64 + lane] = pack8(tile(2 * x), tile(2 * x + 1));
      else PX[(ib * NP + x) * 64 + lane] = tile(x);
    }
  }
  if (SHARE) lds_barrier();                            // the query rows are read
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int u = tid + 256 * i, row = u / SLOTS;
    *reinterpret_cast<V*>(sv + row * D + VE * val_slot<E, D>(row, u % SLOTS)) = vr[i];
  }
  lds_barrier();
  // o^T tiles: lane (c, g) gets o[16 ib + c][16 r + 4g .. +3]
  PV P[NP];
#pragma unroll
  for (int x = 0; x < NP; ++x) P[x] = PX[(ib * NP + x) * 64 + lane];
  float* o = p.o + (row0 + 16 * ib + c) * D + 4 * g;
#pragma unroll
  for (int rr = 0; rr < NR; ++rr) {
    const int r = NR * part + rr;
    floatx4 acc = zero4();
#pragma unroll
    for (int x = 0; x < NP; ++x) {
      if constexpr (B16) {
        const int row = 32 * x + 4 * g + (c >> 2);
        const int vo = VE * val_slot<E, D>(c >> 2, 2 * r + ((c & 3) >> 1)) + 4 * (c & 1);
        acc = mfma_bf16(cat8(lds_read_tr(sv + row * D + vo), lds_read_tr(sv + (row + 16) * D + vo)), P[x], acc);
      } else if (x <= ib) {
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) {
          const float vx = sv[(16 * x + 4 * g + ii) * D + 4 * val_slot<E, D>(4 * g, 4 * r + (c >> 2)) + (c & 3)];
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(vx, P[x][ii], acc, 0, 0, 0);
        }
      }
    }
    *reinterpret_cast<floatx4_any*>(o + 16 * r) = acc;
  }
}

}  // namespace pf
