// Stage kernels behind the compile stack's fused nodes (the reference's FusedKernelRegistry keys,
// src/pto_fuser/fused.py:396-588).  Each is one launch over independent units, with no workspace:
//
//   gated_qk_kernel   L = (a' b'^T) * exp(min(G_i + log beta_i - G_j, 0)) * mask
//                     a' = a (.* a_scale), b' = b (.* b_scale) — the scalar-gate epilogue of
//                     kkt_fused.h:154-185 (kkt_gated*, gated_qk*) and, with the operand scales and
//                     no gate, the per-channel prologue of prologue_fused.h:37-107 (qk_prologue*).
//   qkv_flash_kernel  o = causal_incl(the same score) v, the score kept on chip
//                     (qkv_flash_native*, qkv_fused.h:62-175; qkvp_flash_native*,
//                     qkv_prologue_fused.h:99-187).
// (The third stage, the resident-state scan, is in pf_state_scan.h.)
//
// Row addressing.  The reference runs these stages on two layouts: the native batch [M, C, D]
// (heads outer) and the "mega" token layout [nc*C, H, D] (= [1, T, H, D]).  Both are described
// by one rule: chunk m = c*H + h, token i of it lives at row (c*C + i)*H + h.  H = 1 is the native
// layout.  Gates follow the same rule with row length 1, scores with row length C.
//
// gfx950 mapping (chunks of 64 and 128 tokens; of 16 and 32: pf_stages_small.h).  256-thread workgroups
// (4 waves), one per chunk.  A wave owns whole 16-token query blocks: their rows go straight from HBM into
// its registers as MFMA operands (no other wave reads them); only the key side (and v) is staged in LDS,
// unpadded with XOR-permuted 16-byte slots.
// Every score tile is formed transposed, P^T = k_jb q_ib^T, so a lane holds P[16 ib + c][16 jb + 4g ..
// +3]: four consecutive columns of one row, which is a vector to store (gated_qk) and, two tiles
// together, the B operand of o^T = v^T P^T as it stands (qkv_flash; v^T by transposed reads of the
// row-major tile, fp32 by element reads): the score never passes through LDS.
//
// What bounds them: the memory system (1024 chunks of C = D = 128 bf16: qkv_flash 30-37 us for 168 MB,
// 56-66 with the score and a transposed v staged in LDS by 2-byte writes; 2048 causal scores 37 us for
// 203 MB, 76 with 2-byte stores), below ~500 chunks the call itself.
#pragma once

#include <type_traits>

#include "pf_gfx950.h"

// Barriers are LDS-only (lds_barrier): waves exchange data through LDS alone, so a barrier need
// not wait for this wave's global stores to be acknowledged (a full __syncthreads would).

namespace pf {

template <typename E> struct VecT;
template <> struct VecT<bf16> { typedef bf16x8 T; };
template <> struct VecT<float> { typedef floatx4 T; };

// 16 bytes of operand rows at element offset `off`, and the same times their prescales (fp32, same
// addressing).  Callers load every vector first and prescale in one uniform branch: a branch per
// vector would make each load wait for the one before.
template <typename E>
__device__ __forceinline__ typename VecT<E>::T load_vec(const E* src, size_t off) {
  return *reinterpret_cast<const typename VecT<E>::T*>(src + off);
}
template <typename E>
__device__ __forceinline__ void prescale(typename VecT<E>::T& x, const float* scale, size_t off) {
#pragma unroll
  for (int e = 0; e < Vec16<E>::N; ++e) x[e] = from_f32<E>(to_f32(x[e]) * scale[off + e]);
}

// Physical slot of 16-byte slot `s` of row `row`: a key tile read one row per lane c, and a v tile
// read transposed (4 rows x 2 slots per lane group) or, fp32, as 4 rows x 16 floats.
template <typename E, int D>
__device__ __forceinline__ int key_slot(int row, int s) {
  return sizeof(E) == 2 && D == 64 ? s ^ ((row >> 1) & 7) : s ^ (row & 15);
}
template <typename E, int D>
__device__ __forceinline__ int val_slot(int row, int s) {
  if (sizeof(E) == 4) return s ^ (((row >> 2) & 3) << 2);
  return D == 64 ? s ^ (row & 2) : s ^ ((row & 3) << 1);
}

// The four-column score tile of query block rows `q` (one row per lane c, K-blocks in `q`) against key
// block jb of the staged tile.
template <typename E, int D>
__device__ __forceinline__ floatx4 score_tile(const E* ks, int jb, const typename VecT<E>::T* q, int c, int g) {
  floatx4 acc = zero4();
  const E* row = ks + (16 * jb + c) * D;
#pragma unroll
  for (int kb = 0; kb < D / Mfma<E>::KB; ++kb) {
    const auto k = *reinterpret_cast<const typename VecT<E>::T*>(row + Vec16<E>::N * key_slot<E, D>(c, 4 * kb + g));
    if constexpr (sizeof(E) == 2) {
      acc = mfma_bf16(k, q[kb], acc);
    } else {
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(k[ii], q[kb][ii], acc, 0, 0, 0);
    }
  }
  return acc;
}

// Query block s (0 or 1) of wave w: the last blocks, with most key blocks behind them, go to the
// waves with the first ones.
template <int NB>
__device__ __forceinline__ int query_block(int s, int w) { return s == 0 ? w : NB - 1 - w; }

struct GatedQkArgs {
  const void* a;        // rows of a  (E)
  const void* b;        // rows of b  (E)
  const float* a_scale; // same addressing as a, or null
  const float* b_scale; // same addressing as b, or null
  const float* g;       // per-token within-chunk cumulative log decay, or null (0)
  const float* beta;    // per-token beta, or null (1)
  const float* mask;    // [C, C] multiplier, or null (use `causal`)
  void* L;              // scores, row length C, fp32 or bf16
  int H;                // heads interleaved in the row index (1 = native [M, C, D])
  int causal;           // without mask: 1 keeps i >= j, 0 keeps i > j (0 or 1)
  int out_f32;          // 1: L is fp32, 0: bf16
};

template <typename E, int C, int D, bool MASK>
__global__ __launch_bounds__(256) void gated_qk_kernel(GatedQkArgs p) {
  static_assert(C >= 64, "smaller chunks: pf_stages_small.h");
  typedef typename VecT<E>::T V;
  constexpr int VE = Vec16<E>::N, SLOTS = D / VE, NB = C / 16, NKB = D / Mfma<E>::KB;
  constexpr int NBW = NB / 4, NV = C * SLOTS / 256;
  __shared__ __attribute__((aligned(16))) E sb[C * D];
  __shared__ __attribute__((aligned(16))) float Gs[C], Ls[C];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = blockIdx.x, ch = m / p.H, h = m % p.H;
  const size_t rs = (size_t)p.H * D, base = ((size_t)ch * C * p.H + h) * D;
  const E* ag = static_cast<const E*>(p.a) + base;
  const E* bg = static_cast<const E*>(p.b) + base;
  const float* as = p.a_scale ? p.a_scale + base : nullptr;
  const float* bs = p.b_scale ? p.b_scale + base : nullptr;

  V br[NV], q[NBW][NKB];
  auto b_off = [&](int i) {
    const int u = tid + 256 * i;                       // always in the tile; see the guard below
    return (min(u, C * SLOTS - 1) / SLOTS) * rs + (u % SLOTS) * VE;
  };
  auto a_off = [&](int s, int kb) {
    return (16 * (query_block<NB>(s, w) & (NB - 1)) + c) * rs + Mfma<E>::KB * kb + VE * g;
  };
#pragma unroll
  for (int i = 0; i < NV; ++i) br[i] = load_vec(bg, b_off(i));
#pragma unroll
  for (int s = 0; s < NBW; ++s)
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) q[s][kb] = load_vec(ag, a_off(s, kb));
  if (bs) {
#pragma unroll
    for (int i = 0; i < NV; ++i) prescale<E>(br[i], bs, b_off(i));
  }
  if (as) {
#pragma unroll
    for (int s = 0; s < NBW; ++s)
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) prescale<E>(q[s][kb], as, a_off(s, kb));
  }
  if (tid < C) {
    const size_t gi = ((size_t)ch * C + tid) * p.H + h;
    Gs[tid] = p.g ? p.g[gi] : 0.f;
    Ls[tid] = p.beta ? __logf(p.beta[gi]) : 0.f;
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int u = tid + 256 * i, row = u / SLOTS;
    *reinterpret_cast<V*>(sb + row * D + VE * key_slot<E, D>(row, u % SLOTS)) = br[i];
  }
  lds_barrier();
  // Never taken, as the min of the row offsets never acts (C >= 64).  Both shape what the compiler makes of
  // the score tiles: without them fp32 scores at C = D = 128 took up to 1.4 times as long (4096 chunks).
  if (w >= NB) return;
  const size_t lrs = (size_t)p.H * C, lbase = ((size_t)ch * C * p.H + h) * C;
#pragma unroll
  for (int s = 0; s < NBW; ++s) {
    const int ib = query_block<NB>(s, w), i = 16 * ib + c;
    const float gi = Gs[i] + Ls[i];
    auto tile = [&](int jb) -> floatx4 {   // strictly-upper tiles of a triangular mask are zero
      if (!MASK && jb > ib) return zero4();
      const floatx4 acc = score_tile<E, D>(sb, jb, q[s], c, g);
      const int j0 = 16 * jb + 4 * g;
      const floatx4 gj = *reinterpret_cast<const floatx4*>(Gs + j0);
      floatx4 out;
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        const float mk = MASK ? p.mask[i * C + j0 + ii] : (i + p.causal > j0 + ii ? 1.f : 0.f);
        out[ii] = mk == 0.f ? 0.f : acc[ii] * __expf(fminf(gi - gj[ii], 0.f)) * mk;
      }
      return out;
    };
    const size_t row = lbase + i * lrs;
    if (p.out_f32) {
#pragma unroll
      for (int jb = 0; jb < NB; ++jb)
        *reinterpret_cast<floatx4_any*>(static_cast<float*>(p.L) + row + 16 * jb + 4 * g) = tile(jb);
    } else {
      bf16* L = static_cast<bf16*>(p.L) + row;
#pragma unroll
      for (int jp = 0; jp < NB / 2; ++jp) {
        // lane groups 2x and 2x+1 exchange halves of two tiles: each lane then holds eight consecutive
        // columns, groups 0 and 2 of tile 2 jp and 1 and 3 of tile 2 jp + 1
        const floatx4 t0 = tile(2 * jp), t1 = tile(2 * jp + 1);
        typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
        const u32x2 x = __builtin_bit_cast(u32x2, bf16x4{(bf16)t0[0], (bf16)t0[1], (bf16)t0[2], (bf16)t0[3]});
        const u32x2 y = __builtin_bit_cast(u32x2, bf16x4{(bf16)t1[0], (bf16)t1[1], (bf16)t1[2], (bf16)t1[3]});
        const u32x2 e0 = __builtin_amdgcn_permlane16_swap(x[0], y[0], false, false);
        const u32x2 e1 = __builtin_amdgcn_permlane16_swap(x[1], y[1], false, false);
        *reinterpret_cast<u32x4_any*>(L + 32 * jp + 16 * (g & 1) + 8 * (g >> 1)) = u32x4{e0[0], e1[0], e0[1], e1[1]};
      }
    }
  }
}

struct QkvFlashArgs {
  const void* q;        // [M, C, D] E
  const void* k;        // [M, C, D] E
  const void* v;        // [M, C, D] E
  const float* q_scale; // [M, C, D] or null
  const float* k_scale; // [M, C, D] or null
  const float* g;       // [M, C] or null
  const float* beta;    // [M, C] or null
  float* o;             // [M, C, D] fp32
};

template <typename E, int C, int D>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(C * D * sizeof(E) > 32 * 1024 ? 1 : 2, 8)))
void qkv_flash_kernel(QkvFlashArgs p) {
  static_assert(C >= 64, "smaller chunks: pf_stages_small.h");
  typedef typename VecT<E>::T V;
  constexpr bool B16 = sizeof(E) == 2;
  constexpr int VE = Vec16<E>::N, SLOTS = D / VE, NB = C / 16, NKB = D / Mfma<E>::KB;
  constexpr int NBW = NB / 4, NV = C * SLOTS / 256;
  __shared__ __attribute__((aligned(16))) E sk[C * D];
  __shared__ __attribute__((aligned(16))) E sv[C * D];
  __shared__ __attribute__((aligned(16))) float Gs[C], Ls[C];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const size_t row0 = (size_t)blockIdx.x * C;
  const E* qg = static_cast<const E*>(p.q) + row0 * D;
  const E* kg = static_cast<const E*>(p.k) + row0 * D;
  const E* vg = static_cast<const E*>(p.v) + row0 * D;
  const float* qsc = p.q_scale ? p.q_scale + row0 * D : nullptr;
  const float* ksc = p.k_scale ? p.k_scale + row0 * D : nullptr;

  // every load is issued before the first LDS store; v's stay in flight while the score is formed
  V kr[NV], vr[NV], q[NBW][NKB];
  auto off = [&](int i) { return (size_t)min(tid + 256 * i, C * SLOTS - 1) * VE; };
  auto q_off = [&](int s, int kb) {
    return (size_t)(16 * (query_block<NB>(s, w) & (NB - 1)) + c) * D + Mfma<E>::KB * kb + VE * g;
  };
#pragma unroll
  for (int i = 0; i < NV; ++i) kr[i] = load_vec(kg, off(i));
#pragma unroll
  for (int s = 0; s < NBW; ++s)
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) q[s][kb] = load_vec(qg, q_off(s, kb));
  if (tid < C) {
    Gs[tid] = p.g ? p.g[row0 + tid] : 0.f;
    Ls[tid] = p.beta ? __logf(p.beta[row0 + tid]) : 0.f;
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) vr[i] = load_vec(vg, off(i));
  if (ksc) {
#pragma unroll
    for (int i = 0; i < NV; ++i) prescale<E>(kr[i], ksc, off(i));
  }
  if (qsc) {
#pragma unroll
    for (int s = 0; s < NBW; ++s)
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) prescale<E>(q[s][kb], qsc, q_off(s, kb));
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int u = tid + 256 * i, row = u / SLOTS;
    *reinterpret_cast<V*>(sk + row * D + VE * key_slot<E, D>(row, u % SLOTS)) = kr[i];
  }
  lds_barrier();

  // the score rows of this wave's query blocks, in the operand type
  constexpr int NP = B16 ? NB / 2 : NB;
  typedef typename std::conditional<B16, bf16x8, floatx4>::type PV;
  PV P[NBW][NP];
#pragma unroll
  for (int s = 0; s < NBW; ++s) {
    const int ib = query_block<NB>(s, w), i = 16 * ib + c;
    if (w < NB) {
      const float gi = Gs[i] + Ls[i];
      auto tile = [&](int jb) -> floatx4 {
        if (jb > ib) return zero4();
        const floatx4 acc = score_tile<E, D>(sk, jb, q[s], c, g);
        const floatx4 gj = *reinterpret_cast<const floatx4*>(Gs + 16 * jb + 4 * g);
        floatx4 out;
#pragma unroll
        for (int ii = 0; ii < 4; ++ii)
          out[ii] = i >= 16 * jb + 4 * g + ii ? acc[ii] * __expf(fminf(gi - gj[ii], 0.f)) : 0.f;
        return out;
      };
#pragma unroll
      for (int x = 0; x < NP; ++x) {
        if constexpr (B16) P[s][x] = pack8(tile(2 * x), tile(2 * x + 1));
        else P[s][x] = tile(x);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int u = tid + 256 * i, row = u / SLOTS;
    *reinterpret_cast<V*>(sv + row * D + VE * val_slot<E, D>(row, u % SLOTS)) = vr[i];
  }
  lds_barrier();
  if (w >= NB) return;                                 // never taken, as in gated_qk_kernel
  // o^T tiles: lane (c, g) gets o[16 ib + c][16 r + 4g .. +3]
#pragma unroll
  for (int s = 0; s < NBW; ++s) {
    const int ib = query_block<NB>(s, w);
    float* o = p.o + (row0 + 16 * ib + c) * D + 4 * g;
#pragma unroll
    for (int r = 0; r < D / 16; ++r) {
      floatx4 acc = zero4();
#pragma unroll
      for (int x = 0; x < NP; ++x) {
        if constexpr (B16) {
          if (2 * x <= ib) {
            const int row = 32 * x + 4 * g + (c >> 2);
            const int off = VE * val_slot<E, D>(c >> 2, 2 * r + ((c & 3) >> 1)) + 4 * (c & 1);
            acc = mfma_bf16(cat8(lds_read_tr(sv + row * D + off), lds_read_tr(sv + (row + 16) * D + off)), P[s][x], acc);
          }
        } else {
          if (x <= ib) {
#pragma unroll
            for (int ii = 0; ii < 4; ++ii) {
              const float vx = sv[(16 * x + 4 * g + ii) * D + 4 * val_slot<E, D>(4 * g, 4 * r + (c >> 2)) + (c & 3)];
              acc = __builtin_amdgcn_mfma_f32_16x16x4f32(vx, P[s][x][ii], acc, 0, 0, 0);
            }
          }
        }
      }
      *reinterpret_cast<floatx4_any*>(o + 16 * r) = acc;
    }
  }
}

}  // namespace pf
