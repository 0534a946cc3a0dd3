// chunk_h_scan — the resident-state chunk recurrence of the compile stack:
//
//   h_out[c] = S;   S <- decay (.) S + k_c^T (u_c - w_c S)
//
// with a scalar decay per chunk or one per state row (key channel); scan_fused.h:198-262,
// vec_recurrence_perdim :143-180.  Operands are token-major [B, nc, C, H, D]: the rows of one
// chain (b, h) lie H*D elements apart.
//
// Mapping on gfx950.  State columns are independent, so a wave owns 16 of them for the whole chain
// and every product feeds the next from registers: S (D-layout tiles) is the B operand of w S as it
// stands, u - w S (D layout again) the B operand of k^T (u - w S).  Waves share only the chunk's
// read-only w and k images in LDS; there is no exchange between them.  A workgroup is 256 threads
// over one chain and 16*NCW columns; all four waves copy, NCW of them compute.  The next chunk
// is loaded into registers while the current one is computed and written to LDS between two
// barriers.
//
// LDS images are unpadded (16-byte slots XOR-permuted by row bits, scan_w_slot / scan_k_slot), so
// that the bf16 C = D = 128 workgroup of 64 columns takes exactly 80 KiB and two share a CU: one
// computes while the other waits for its loads.  With bf16 operands a state tile pair (2kb, 2kb+1)
// holds rows 32kb + 8g + 0..7 per lane group (scan_row), so w rows are read as natural-order 16-byte
// fragments and k^T by transposed reads straight from the row-major image.  bf16 snapshots pass
// through the wave's own u tile (dead by then) and leave as 8-byte pieces of rows.
//
// What bounds it: many chains, the memory system (bf16, 256 chains x 16 chunks, C = D = 128: 138 us
// for 553 MB, 4.0 TB/s; 596 us for the earlier form, which copied each chunk with the products
// waiting, transposed k by 2-byte LDS writes, read w and k once per 32 columns and stored
// snapshots by 2-byte elements).  Few chains, the chunk step's latency: 2.7 us, of which a wave's 64
// products and 68 KiB of LDS reads are the larger part (16 chains x 8 chunks: 22 us, 97 before).
// fp32 operands, fp32 product issue (512 products of 32 cycles per wave and chunk: 430 us).
#pragma once

#include "pf_gfx950.h"

namespace pf {

struct ScanStateArgs {
  const void* w;        // [B, nc, C, H, D] E
  const void* u;        // [B, nc, C, H, D] E
  const void* k;        // [B, nc, C, H, D] E
  const float* decay;   // [B, H, nc] (scalar) or [B, H, nc, D] (per row)
  const float* h0;      // [B, H, D, D] or null (zero)
  void* h_out;          // [B, nc, H, D, D] fp32 or bf16
  float* final_state;   // [B, H, D, D] or null
  int BH, H, NC, out_f32;
};

// Physical 16-byte slot of logical slot `s` in row `row` of the w image (read one row per lane c)
// and of the k image (read as 4 rows x 4 slots per lane group, or fp32: 4 rows x 16 floats).
template <typename E, int D>
__device__ __forceinline__ int scan_w_slot(int row, int s) {
  return sizeof(E) == 2 && D == 64 ? s ^ ((row >> 1) & 7) : s ^ (row & 15);
}
template <typename E, int D>
__device__ __forceinline__ int scan_k_slot(int row, int s) {
  if (sizeof(E) == 4) return s ^ (((row >> 2) & 3) << 2);
  return D == 64 ? s ^ (((row >> 1) & 1) << 2) : s ^ ((row & 3) << 2);
}
// Slot permutation of the bf16 snapshot tile [16 columns][D]: conflict free for both the 16-byte
// writes (16 rows, one slot) and the transposed reads (4 rows x 2 slots).
template <int D>
__device__ __forceinline__ int scan_x_slot(int n, int s) {
  return D == 64 ? s ^ ((n & 2) | (n & 4) | (n >> 3)) : s ^ (((n << 1) & 15) | (n >> 3));
}
// Row of the u tile [C][16] that holds token t: fp32 lane groups read tokens 4g + ii, kept adjacent.
template <typename E>
__device__ __forceinline__ constexpr int scan_u_row(int t) {
  return sizeof(E) == 2 ? t : (t & ~15) | ((t & 3) << 2) | ((t >> 2) & 3);
}
// State row held in register ii of lane group g of D tile r.
template <typename E>
__device__ __forceinline__ constexpr int scan_row(int r, int g, int ii) {
  return sizeof(E) == 2 ? 32 * (r >> 1) + 8 * g + 4 * (r & 1) + ii : 16 * r + 4 * g + ii;
}

template <typename E, int C, int D, int NCW>
struct ScanStateShape {
  static constexpr int NCOL = 16 * NCW, NS = D / NCOL;
  static constexpr int VE = 16 / (int)sizeof(E), SLOTS = D / VE;
  static constexpr int NV = C * SLOTS / 256;                         // w (or k) vectors per thread
  static constexpr int UT = sizeof(E) == 2 ? 16 * (C > D ? C : D) : 16 * C;   // u tile of a wave
  static constexpr size_t lds = ((size_t)2 * C * D + (size_t)NCW * UT) * sizeof(E);
  static constexpr int wg_per_cu = lds <= 80 * 1024 ? 2 : 1;
  static_assert(NV >= 1 && C * SLOTS % 256 == 0, "a chunk image divides over the workgroup");
};

template <typename E, int C, int D, int NCW, bool PERDIM>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(ScanStateShape<E, C, D, NCW>::wg_per_cu,
                                   ScanStateShape<E, C, D, NCW>::wg_per_cu)))
void scan_state_kernel(ScanStateArgs p) {
  using Sh = ScanStateShape<E, C, D, NCW>;
  constexpr bool B16 = sizeof(E) == 2;
  constexpr int VE = Sh::VE, SLOTS = Sh::SLOTS, NV = Sh::NV, NS = Sh::NS, NCOL = Sh::NCOL;
  constexpr int MB = C / 16, RB = D / 16;
  __shared__ __attribute__((aligned(16))) E ws[C * D];
  __shared__ __attribute__((aligned(16))) E ks[C * D];
  __shared__ __attribute__((aligned(16))) E us[NCW * Sh::UT];

  int bh, slice;
  const int bid = blockIdx.x;
  if (p.BH % 8 == 0) {   // the slices of one chain on one XCD: they read the same w and k
    const int grp = bid / (8 * NS), within = bid % (8 * NS);
    bh = grp * 8 + (within % 8);
    slice = within / 8;
  } else {
    bh = bid / NS;
    slice = bid % NS;
  }
  const int b = bh / p.H, h = bh % p.H;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool compute = w < NCW;
  const int col = slice * NCOL + 16 * w + c;            // this lane's state column (compute waves)
  const size_t rs = (size_t)p.H * D;                    // token row stride
  const size_t chain0 = ((size_t)b * p.NC * C * p.H + h) * D;
  const E* wg = static_cast<const E*>(p.w) + chain0;
  const E* kg = static_cast<const E*>(p.k) + chain0;
  const E* ug = static_cast<const E*>(p.u) + chain0;

  // ---- chunk copies: thread tid holds rows tid / SLOTS + i * 256 / SLOTS, slot tid % SLOTS ----
  constexpr int RSTEP = 256 / SLOTS;
  const int vrow = tid / SLOTS, vslot = tid % SLOTS;
  constexpr int UVR = NCOL / VE, U_VECS = C * UVR, NU = (U_VECS + 255) / 256;   // u tile
  u32x4 wr[NV], kr[NV], ur[NU];
  auto load = [&](int ch) {
    const size_t t0 = (size_t)ch * C * rs;
#pragma unroll
    for (int i = 0; i < NV; ++i)
      wr[i] = *reinterpret_cast<const u32x4*>(wg + t0 + (size_t)(vrow + i * RSTEP) * rs + vslot * VE);
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int x = min(tid + 256 * i, U_VECS - 1);     // lanes past the tile repeat its last vector
      ur[i] = *reinterpret_cast<const u32x4_any*>(ug + t0 + (size_t)(x / UVR) * rs + slice * NCOL + (x % UVR) * VE);
    }
#pragma unroll
    for (int i = 0; i < NV; ++i)
      kr[i] = *reinterpret_cast<const u32x4*>(kg + t0 + (size_t)(vrow + i * RSTEP) * rs + vslot * VE);
  };
  auto store = [&]() {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int row = vrow + i * RSTEP;
      *reinterpret_cast<u32x4*>(ws + row * D + VE * scan_w_slot<E, D>(row, vslot)) = wr[i];
    }
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int x = tid + 256 * i, v = x % UVR;
      if (U_VECS >= 256 * (i + 1) || x < U_VECS)
        *reinterpret_cast<u32x4*>(us + v * VE / 16 * Sh::UT + scan_u_row<E>(x / UVR) * 16 + v * VE % 16) = ur[i];
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int row = vrow + i * RSTEP;
      *reinterpret_cast<u32x4*>(ks + row * D + VE * scan_k_slot<E, D>(row, vslot)) = kr[i];
    }
  };

  floatx4 S[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int ii = 0; ii < 4; ++ii)
      S[r][ii] = p.h0 && compute ? p.h0[((size_t)bh * D + scan_row<E>(r, g, ii)) * D + col] : 0.f;
  bf16x8 Sb[B16 ? RB / 2 : 1];                          // bf16 S: tile pairs as B fragments

  // snapshot of chunk ch (the state before it); bf16 operands leave S packed in Sb
  auto snapshot = [&](int ch) {
    const size_t hb = (((size_t)b * p.NC + ch) * p.H + h) * D * D;
    if constexpr (B16) {
#pragma unroll
      for (int kb = 0; kb < RB / 2; ++kb) Sb[kb] = pack8(S[2 * kb], S[2 * kb + 1]);
      if (!p.out_f32) {
        bf16* x = reinterpret_cast<bf16*>(us) + w * Sh::UT;   // this wave's tile: no barrier
        bf16* ho = static_cast<bf16*>(p.h_out) + hb;
#pragma unroll
        for (int kb = 0; kb < RB / 2; ++kb)
          *reinterpret_cast<bf16x8*>(x + c * D + 8 * scan_x_slot<D>(c, 4 * kb + g)) = Sb[kb];
        const int n = 4 * g + (c >> 2);                 // transposed read: row n, 4 state rows
#pragma unroll
        for (int r = 0; r < RB; ++r) {
          const bf16x4 t = lds_read_tr(x + n * D + 8 * scan_x_slot<D>(n, 2 * r + ((c & 3) >> 1)) + 4 * (c & 1));
          *reinterpret_cast<bf16x4_any*>(ho + (size_t)(16 * r + c) * D + slice * NCOL + 16 * w + 4 * g) = t;
        }
        return;
      }
    }
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        const size_t e = hb + (size_t)scan_row<E>(r, g, ii) * D + col;
        if (p.out_f32) static_cast<float*>(p.h_out)[e] = S[r][ii];
        else static_cast<bf16*>(p.h_out)[e] = (bf16)S[r][ii];
      }
  };

  load(0);
  if (compute) snapshot(0);
  for (int ch = 0; ch < p.NC; ++ch) {
    lds_barrier();                                      // the last images and snapshot tiles are read
    store();
    lds_barrier();
    load(min(ch + 1, p.NC - 1));                        // past the end: the last chunk again, unused
    if (!compute) continue;
    // decay of state tile r: one value per chunk, or per row, loaded two tiles ahead of its use (all
    // of a chunk's 32 would spill beside the prefetched chunk)
    floatx4 dec[PERDIM ? RB + 2 : 1];
    float dec1 = 0.f;
    if constexpr (!PERDIM) dec1 = p.decay[(size_t)bh * p.NC + ch];
    auto load_decay = [&](int r) {
      if constexpr (PERDIM)
        if (r < RB) dec[r] = *reinterpret_cast<const floatx4_any*>(p.decay + ((size_t)bh * p.NC + ch) * D + scan_row<E>(r, g, 0));
    };
    auto decayed = [&](int r) {
      if constexpr (PERDIM) return S[r] * dec[r];
      else return S[r] * dec1;
    };
    load_decay(0);
    load_decay(1);
    if constexpr (B16) {
      bf16x8 Vb[MB / 2 > 0 ? MB / 2 : 1];
#pragma unroll
      for (int mb2 = 0; mb2 < MB / 2; ++mb2) {
        floatx4 V[2];
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          const int mb = 2 * mb2 + hh;
          floatx4 X = zero4();
#pragma unroll
          for (int kb = 0; kb < RB / 2; ++kb)
            X = mfma_bf16(*reinterpret_cast<const bf16x8*>(ws + (16 * mb + c) * D + 8 * scan_w_slot<E, D>(c, 4 * kb + g)), Sb[kb], X);
          const bf16x4 u4 = lds_read_tr(us + w * Sh::UT + (16 * mb + 4 * g + (c >> 2)) * 16 + 4 * (c & 3));
#pragma unroll
          for (int ii = 0; ii < 4; ++ii) V[hh][ii] = (float)u4[ii] - X[ii];
        }
        Vb[mb2] = pack8(V[0], V[1]);
        __builtin_amdgcn_sched_barrier(0);
      }
      const int tr = 4 * g + (c >> 2);                  // transposed read of k: token row, slot c & 3
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        load_decay(r + 2);
        floatx4 acc = decayed(r);
        const int off = tr * D + 8 * scan_k_slot<E, D>(c >> 2, 4 * (r >> 1) + (c & 3)) + 4 * (r & 1);
#pragma unroll
        for (int tb = 0; tb < MB / 2; ++tb)
          acc = mfma_bf16(cat8(lds_read_tr(ks + off + 32 * tb * D), lds_read_tr(ks + off + (32 * tb + 16) * D)),
                          Vb[tb], acc);
        S[r] = acc;
        if (r & 1) __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      floatx4 V[MB];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        floatx4 X = zero4();
#pragma unroll
        for (int r = 0; r < RB; ++r) {
          const floatx4 a = *reinterpret_cast<const floatx4*>(ws + (16 * mb + c) * D + 4 * scan_w_slot<E, D>(c, 4 * r + g));
#pragma unroll
          for (int ii = 0; ii < 4; ++ii) X = __builtin_amdgcn_mfma_f32_16x16x4f32(a[ii], S[r][ii], X, 0, 0, 0);
        }
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) V[mb][ii] = us[w * Sh::UT + scan_u_row<E>(16 * mb + 4 * g + ii) * 16 + c] - X[ii];
        if (mb & 1) __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        load_decay(r + 2);
        floatx4 acc = decayed(r);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int ii = 0; ii < 4; ++ii) {
            const int row = 16 * mb + 4 * g + ii;       // (row >> 2) & 3 == g
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(
                ks[row * D + 4 * scan_k_slot<E, D>(4 * g, 4 * r + (c >> 2)) + (c & 3)], V[mb][ii], acc, 0, 0, 0);
          }
        S[r] = acc;
        if (r & 1) __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (ch + 1 < p.NC) snapshot(ch + 1);
  }
  if (p.final_state && compute) {
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int ii = 0; ii < 4; ++ii)
        p.final_state[((size_t)bh * D + scan_row<E>(r, g, ii)) * D + col] = S[r][ii];
  }
}

}  // namespace pf
