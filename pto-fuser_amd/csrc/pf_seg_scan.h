// Segmented chains (bf16 operands, few long chains): what turns one chain of NC sequential chunks into
// SEG segments that run side by side.
//
// Over a segment of chunks the delta rule is affine in its incoming state, H_out = M H_in + D, so
//
//   1. seg_map_kernel     for every segment but the last, D (128 columns, from a zero state; the first
//                         segment from h0, which makes its D the true state) and M (the state
//                         recurrence without v, from the identity; not needed for the first);
//   2. seg_compose_kernel H_{s+1} = D_s + M_s H_s along each chain, fp32 products, in place of D_s;
//   3. the scan (pf_scan_split.h) over all segments at once, each from its own H_s.
//
// Step 1 repeats the state part of the chunk loop on 256 columns instead of 128, so segments pay
// where chains leave the chip idle or their length is the bound, not where every CU is busy
// (pf_segments.h has the rule and its measurements).
//
// seg_map_kernel: state columns are independent, so a wave owns 16 NT of them for the whole segment and
// every product feeds the next from registers: S (packed pairs of D tiles) is the B operand of k S,
// r = beta v - beta e^G (k S) that of T r, v_new e^{G_last - G} that of the update
// S <- e^{G_last} S + k^T (.).  Workgroups of eight waves: NT = 1, D or M of a segment each (the shorter
// step, while they fit one generation); NT = 2, four waves on D and four on M (half the LDS reads).
// M runs the same code with v masked to zero, so a chunk is straight-line code.  Waves share only the
// chunk's k, T, v and gate images in LDS (two), loaded into registers two chunks ahead.  Tile pair (2x, 2x + 1) holds
// rows (state rows or tokens) 32x + 8g + 0..7 per lane group, so k and T rows are read as
// natural-order 16-byte fragments and k^T by transposed reads of the same image; a fragment read
// serves all of the wave's column tiles.  fp32 state and accumulators, bf16 operands, as in the scan
// itself.  A chunk step takes 2.4 us (NT = 1, 128 columns) or 3.3 us (NT = 2, 256 columns): 336 KB of LDS
// reads, 76 products and about 300 vector instructions per wave at NT = 2, two waves per SIMD.
#pragma once

#include "pf_gfx950.h"
#include "pf_scan_args.h"

namespace pf {

// Row of tile t (a pair's half t & 1) held in register ii of lane group g, and the row lane c supplies
// as the A operand of that tile.
__device__ __forceinline__ constexpr int seg_row(int t, int g, int ii) { return 32 * (t >> 1) + 8 * g + 4 * (t & 1) + ii; }

// Physical 16-byte slot of slot `s` of row `row`: k (16 slots a row; read as 16 rows x one slot and,
// transposed, as 4 rows x 4 slots) and T (8 slots a row; 16 rows x one slot).
__device__ __forceinline__ int seg_k_slot(int row, int s) { return s ^ (((row & 3) << 2) | ((row >> 3) & 3)); }
__device__ __forceinline__ int seg_t_slot(int row, int s) { return s ^ ((((row >> 1) & 1) << 2) | ((row >> 3) & 3)); }

// M is kept in the operand order of seg_compose_kernel: 16x16 tiles, each 64 lanes x four consecutive
// columns, so that its loads are contiguous (row-major, 64-byte pieces of 16 rows, a step took 2.6 us).
__device__ __forceinline__ constexpr int seg_m_index(int row, int col) {
  return (((row >> 4) * 8 + (col >> 4)) * 64 + ((col >> 2) & 3) * 16 + (row & 15)) * 4 + (col & 3);
}

struct SegImage {                                      // one chunk in LDS
  bf16 ks[64 * 128], ts[64 * 64], vs[8 * 64 * 16];     // v: per 16 columns [64][16]
  struct {
    float BT[64], BEG[64], EL[64];                     // beta, beta e^G, e^{G_last - G}
  } gate[8];                                           // per wave: no branch around the tables
};

template <int C, int DK, int DV, int NT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void seg_map_kernel(SegMapArgs a) {
  static_assert(C == 64 && DK == 128 && DV == 128, "the forward's tile: C 64, dk = dv = 128");
  __shared__ __attribute__((aligned(16))) SegImage img[2];
  // NT = 2: one workgroup per segment; NT = 1: two, eight ids apart (one XCD: they read the same k and T)
  const int bid = blockIdx.x;
  const int unit = NT == 2 ? bid : bid / 16 * 8 + bid % 8;
  if (unit >= a.BH * (a.SEG - 1)) return;
  const int bh = unit / (a.SEG - 1), seg = unit % (a.SEG - 1);
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool map = NT == 2 ? w >= 4 : bid % 16 >= 8;   // M, else D
  if (NT == 1 && map && seg == 0) return;              // the first segment's D is the state itself
  const int wt = NT == 2 ? NT * (w & 3) : w;           // this wave's first column tile
  const int col = 16 * wt + c;                         // this lane's column of tile nt: + 16 nt
  const unsigned vmask = map ? 0u : ~0u;
  const size_t m0 = (size_t)bh * a.NC + (size_t)seg * a.L, t0 = m0 * C;
  const bf16* kg = a.k + t0 * DK;
  const bf16* vg = a.v + t0 * DV;
  const bf16* tg = a.Tm + m0 * C * C;
  const float* Gg = a.G + t0;
  const float* Bg = a.beta + t0;

  // one chunk in registers: 16-byte vectors u = tid + 512 i of k and v (16 a row), tid of T (8 a row)
  struct Regs {
    u32x4 k[2], t, v[2];
    float g, b;
  };
  auto load = [&](Regs& x, int ch) {
    ch = min(ch, a.L - 1);                             // past the end: the last chunk again, unused
#pragma unroll
    for (int i = 0; i < 2; ++i) x.k[i] = *reinterpret_cast<const u32x4*>(kg + (size_t)ch * C * DK + (tid + 512 * i) * 8);
    x.t = *reinterpret_cast<const u32x4*>(tg + (size_t)ch * C * C + tid * 8);
#pragma unroll
    for (int i = 0; i < 2; ++i) x.v[i] = *reinterpret_cast<const u32x4*>(vg + (size_t)ch * C * DV + (tid + 512 * i) * 8);
    x.g = Gg[(size_t)ch * C + lane];
    x.b = Bg[(size_t)ch * C + lane];
  };
  auto store = [&](SegImage& im, const Regs& x) -> float {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int u = tid + 512 * i, row = u >> 4, s = u & 15;
      *reinterpret_cast<u32x4*>(im.ks + row * DK + 8 * seg_k_slot(row, s)) = x.k[i];
      *reinterpret_cast<u32x4*>(im.vs + (s >> 1) * C * 16 + row * 16 + 8 * (s & 1)) = x.v[i];
    }
    *reinterpret_cast<u32x4*>(im.ts + (tid >> 3) * C + 8 * seg_t_slot(tid >> 3, tid & 7)) = x.t;
    const float gl = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x.g), C - 1));
    im.gate[w].BT[lane] = x.b;                         // lane = token
    im.gate[w].BEG[lane] = x.b * __expf(x.g);
    im.gate[w].EL[lane] = __expf(gl - x.g);
    return __expf(gl);                                 // the chunk's decay
  };

  floatx4 S[8][NT];
#pragma unroll
  for (int r = 0; r < 8; ++r)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) S[r][nt][ii] = map && seg_row(r, g, ii) == col + 16 * nt ? 1.f : 0.f;
  if (!map && seg == 0 && a.h0) {                      // one branch around all loads
    const float* h = a.h0 + (size_t)bh * DK * DV + col;
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) S[r][nt][ii] = h[seg_row(r, g, ii) * DV + 16 * nt];
    if (a.keep_h0) {
      float* keep = a.M + (size_t)unit * DK * DK + col;
#pragma unroll
      for (int r = 0; r < 8; ++r)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int ii = 0; ii < 4; ++ii) keep[seg_row(r, g, ii) * DV + 16 * nt] = S[r][nt][ii];
    }
  }

  const int crow = 8 * (c >> 2) + (c & 3);             // + 32x + 4h: the row lane c supplies
  const int trow = 8 * g + (c >> 2);                   // transposed reads: + 32x + 4h
  // chunk m in register set m & 1 until it is written to LDS
  Regs r0, r1;
  load(r0, 0);
  load(r1, 1);
  float dl = store(img[0], r0), dl_next = 0.f;
  load(r0, 2);
  lds_barrier();
  auto chunk = [&](Regs& nx, int ch) {                 // nx holds chunk ch + 1
    const SegImage& im = img[ch & 1];
    const bf16 *ks = im.ks, *ts = im.ts, *vs = im.vs + wt * C * 16;
    bf16x8 Sb[4][NT];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) Sb[kb][nt] = pack8(S[2 * kb][nt], S[2 * kb + 1][nt]);
    // r = beta v - beta e^G (k S)
    bf16x8 Rb[2][NT];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      floatx4 r[2][NT];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        floatx4 Y[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) Y[nt] = zero4();
        const int row = 32 * x + 4 * h + crow;
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
          const bf16x8 kf = *reinterpret_cast<const bf16x8*>(ks + row * DK + 8 * seg_k_slot(row, 4 * kb + g));
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) Y[nt] = mfma_bf16(kf, Sb[kb][nt], Y[nt]);
        }
        const int t4 = 32 * x + 8 * g + 4 * h;
        const floatx4 beg = *reinterpret_cast<const floatx4*>(im.gate[w].BEG + t4);
        const floatx4 bt = *reinterpret_cast<const floatx4*>(im.gate[w].BT + t4);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
          const u32x2 vx = __builtin_bit_cast(u32x2, lds_read_tr(vs + nt * C * 16 + (32 * x + 4 * h + trow) * 16 + 4 * (c & 3)));
          const bf16x4 v4 = __builtin_bit_cast(bf16x4, u32x2{vx[0] & vmask, vx[1] & vmask});
#pragma unroll
          for (int ii = 0; ii < 4; ++ii) r[h][nt][ii] = fmaf(-beg[ii], Y[nt][ii], bt[ii] * (float)v4[ii]);
        }
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) Rb[x][nt] = pack8(r[0][nt], r[1][nt]);
    }
    dl_next = store(img[(ch + 1) & 1], nx);            // last read a barrier ago
    load(nx, ch + 3);
    // v_new = T r (T lower triangular by 32-token blocks), scaled by e^{G_last - G}
    bf16x8 Vb[2][NT];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      floatx4 V[2][NT];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) V[h][nt] = zero4();
        const int row = 32 * x + 4 * h + crow;
#pragma unroll
        for (int xb = 0; xb <= x; ++xb) {
          const bf16x8 tf = *reinterpret_cast<const bf16x8*>(ts + row * C + 8 * seg_t_slot(row, 4 * xb + g));
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) V[h][nt] = mfma_bf16(tf, Rb[xb][nt], V[h][nt]);
        }
        const floatx4 el = *reinterpret_cast<const floatx4*>(im.gate[w].EL + 32 * x + 8 * g + 4 * h);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) V[h][nt] *= el;
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) Vb[x][nt] = pack8(V[0][nt], V[1][nt]);
    }
    // S <- e^{G_last} S + k^T (.)
#pragma unroll
    for (int r = 0; r < 8; ++r) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) S[r][nt] *= dl;
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int r0 = 32 * x + trow, off = 8 * seg_k_slot(trow, 4 * (r >> 1) + (c & 3)) + 4 * (r & 1);
        // rows r0 and r0 + 4 share their slot permutation (row bits 0, 1, 3, 4)
        const bf16x8 kt = cat8(lds_read_tr(ks + r0 * DK + off), lds_read_tr(ks + (r0 + 4) * DK + off));
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) S[r][nt] = mfma_bf16(kt, Vb[x][nt], S[r][nt]);
      }
    }
    dl = dl_next;
    lds_barrier();                                     // the next image written, this one read
  };
  int ch = 0;
  for (; ch + 1 < a.L; ch += 2) {
    chunk(r1, ch);
    chunk(r0, ch + 1);
  }
  if (ch < a.L) chunk(r1, ch);
  if (map && seg == 0) return;
  float* out = (map ? a.M : a.D) + (size_t)unit * DK * DV;
#pragma unroll
  for (int r = 0; r < 8; ++r)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        const int row = seg_row(r, g, ii), cl = col + 16 * nt;
        out[map ? seg_m_index(row, cl) : row * DV + cl] = S[r][nt][ii];
      }
}

// The KDA form of seg_map_kernel: v_new = TB v - W S, S <- e^{G_last} (.) (S + KB^T v_new) over stage 1's
// images (pf_kda.h); the organisation of NT = 1 (D or M of a segment per workgroup, 16 columns a wave), the
// decay one factor per state row.  2.3-2.5 us a chunk step.  (32 columns a wave spill: the image is 114 KiB
// and its prefetch half the registers.)
struct KdaSegImage {
  bf16 ws[64 * 128], ks[64 * 128], ts[64 * 64], vs[8 * 64 * 16];
  float dec[128];
};

template <int C, int DK, int DV>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void kda_seg_map_kernel(KdaSegMapArgs a) {
  static_assert(C == 64 && DK == 128 && DV == 128, "the forward's tile: C 64, dk = dv = 128");
  __shared__ __attribute__((aligned(16))) KdaSegImage img[2];
  const int bid = blockIdx.x;
  const int unit = bid / 16 * 8 + bid % 8;             // D and M of a segment eight ids apart: one XCD
  if (unit >= a.BH * (a.SEG - 1)) return;
  const int bh = unit / (a.SEG - 1), seg = unit % (a.SEG - 1);
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool map = bid % 16 >= 8;                      // M, else D
  if (map && seg == 0) return;                         // the first segment's D is the state itself
  const int col = 16 * w + c;                          // this lane's column
  const unsigned vmask = map ? 0u : ~0u;
  const size_t m0 = (size_t)bh * a.NC + (size_t)seg * a.L, t0 = m0 * C;

  struct Regs {
    u32x4 w[2], k[2], t, v[2];
    floatx4 d;
  };
  auto load = [&](Regs& x, int ch) {
    ch = min(ch, a.L - 1);                             // past the end: the last chunk again, unused
    const size_t e = (t0 + (size_t)ch * C) * DK;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      x.w[i] = *reinterpret_cast<const u32x4*>(a.W + e + (tid + 512 * i) * 8);
      x.k[i] = *reinterpret_cast<const u32x4*>(a.KB + e + (tid + 512 * i) * 8);
      x.v[i] = *reinterpret_cast<const u32x4*>(a.v + e + (tid + 512 * i) * 8);
    }
    x.t = *reinterpret_cast<const u32x4*>(a.TB + (m0 + ch) * C * C + tid * 8);
    x.d = *reinterpret_cast<const floatx4*>(a.DEC + (m0 + ch) * DK + 4 * (tid & 31));
  };
  auto store = [&](KdaSegImage& im, const Regs& x) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int u = tid + 512 * i, row = u >> 4, s = u & 15;
      *reinterpret_cast<u32x4*>(im.ws + row * DK + 8 * seg_k_slot(row, s)) = x.w[i];
      *reinterpret_cast<u32x4*>(im.ks + row * DK + 8 * seg_k_slot(row, s)) = x.k[i];
      *reinterpret_cast<u32x4*>(im.vs + (s >> 1) * C * 16 + row * 16 + 8 * (s & 1)) = x.v[i];
    }
    *reinterpret_cast<u32x4*>(im.ts + (tid >> 3) * C + 8 * seg_t_slot(tid >> 3, tid & 7)) = x.t;
    if (tid < 32) *reinterpret_cast<floatx4*>(im.dec + 4 * tid) = x.d;
  };

  floatx4 S[8];
#pragma unroll
  for (int r = 0; r < 8; ++r)
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) S[r][ii] = map && seg_row(r, g, ii) == col ? 1.f : 0.f;
  if (!map && seg == 0 && a.h0) {                      // one branch around all loads
    const float* h = a.h0 + (size_t)bh * DK * DV + col;
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) S[r][ii] = h[seg_row(r, g, ii) * DV];
    if (a.keep_h0) {
      float* keep = a.M + (size_t)unit * DK * DK + col;
#pragma unroll
      for (int r = 0; r < 8; ++r)
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) keep[seg_row(r, g, ii) * DV] = S[r][ii];
    }
  }

  const int crow = 8 * (c >> 2) + (c & 3);             // + 32x + 4h: the row lane c supplies
  const int trow = 8 * g + (c >> 2);                   // transposed reads: + 32x + 4h
  Regs r0, r1;                                         // chunk m in set m & 1 until it is written to LDS
  load(r0, 0);
  load(r1, 1);
  store(img[0], r0);
  load(r0, 2);
  lds_barrier();
  auto chunk = [&](Regs& nx, int ch) {                 // nx holds chunk ch + 1
    const KdaSegImage& im = img[ch & 1];
    const bf16 *ws = im.ws, *ks = im.ks, *ts = im.ts, *vs = im.vs + w * C * 16;
    bf16x8 Sb[4], Vt[2];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) Sb[kb] = pack8(S[2 * kb], S[2 * kb + 1]);
    // v's tokens 32x + 8g .. +7 of this lane's column, zero for M
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const bf16* vp = vs + (32 * x + trow) * 16 + 4 * (c & 3);
      u32x4 vx = __builtin_bit_cast(u32x4, cat8(lds_read_tr(vp), lds_read_tr(vp + 4 * 16)));
      vx &= u32x4{vmask, vmask, vmask, vmask};
      Vt[x] = __builtin_bit_cast(bf16x8, vx);
    }
    // v_new = TB v - W S (TB lower triangular by 32-token blocks)
    bf16x8 Vb[2];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      floatx4 V[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        floatx4 Y = zero4(), U = zero4();
        const int row = 32 * x + 4 * h + crow;
#pragma unroll
        for (int xb = 0; xb <= x; ++xb) {
          const bf16x8 tf = *reinterpret_cast<const bf16x8*>(ts + row * C + 8 * seg_t_slot(row, 4 * xb + g));
          U = mfma_bf16(tf, Vt[xb], U);
        }
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
          const bf16x8 wf = *reinterpret_cast<const bf16x8*>(ws + row * DK + 8 * seg_k_slot(row, 4 * kb + g));
          Y = mfma_bf16(wf, Sb[kb], Y);
        }
        V[h] = U - Y;
      }
      Vb[x] = pack8(V[0], V[1]);
    }
    store(img[(ch + 1) & 1], nx);                      // last read a barrier ago
    load(nx, ch + 3);
    // S <- e^{G_last} (.) (S + KB^T v_new)
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const floatx4 d4 = *reinterpret_cast<const floatx4*>(im.dec + seg_row(r, g, 0));
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int r0 = 32 * x + trow, off = 8 * seg_k_slot(trow, 4 * (r >> 1) + (c & 3)) + 4 * (r & 1);
        const bf16x8 kt = cat8(lds_read_tr(ks + r0 * DK + off), lds_read_tr(ks + (r0 + 4) * DK + off));
        S[r] = mfma_bf16(kt, Vb[x], S[r]);
      }
      S[r] *= d4;
    }
    lds_barrier();                                     // the next image written, this one read
  };
  int ch = 0;
  for (; ch + 1 < a.L; ch += 2) {
    chunk(r1, ch);
    chunk(r0, ch + 1);
  }
  if (ch < a.L) chunk(r1, ch);
  float* out = (map ? a.M : a.D) + (size_t)unit * DK * DV;
#pragma unroll
  for (int r = 0; r < 8; ++r)
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
      const int row = seg_row(r, g, ii);
      out[map ? seg_m_index(row, col) : row * DV + col] = S[r][ii];
    }
}

// H_{s+1} = D_s + M_s H_s for s = 1 .. SEG - 2 (H_1 = D_0 is final), written over D_s.  One workgroup per
// (chain, 16 columns); wave w forms rows 32w .. 32w+31 with fp32 products (two 16-row tiles, the
// four-element K order of the D layout), its rows of M_s loaded a step ahead; H_s passes through LDS as
// D tiles.
//
// A segment's map can leave fp32 range where the states it is applied to do not (they are zero, or small):
// then Inf * 0 is NaN.  A state that is not finite stays so in every row of its column through the later
// products, so the last one shows it; its row 0 is set to NaN in all of the slice's columns, which is
// where the scan looks before it splits the chain.
template <int DK, int DV>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void seg_compose_kernel(float* D, const float* M, int BH, int SEG) {
  constexpr int NS = DV / 16;
  __shared__ __attribute__((aligned(16))) floatx4 H[2][8 * 64];
  __shared__ int bad[4];
  // the slices of one chain on one XCD: they read the same M
  const int bh = (blockIdx.x / (8 * NS)) * 8 + blockIdx.x % 8, col0 = 16 * (blockIdx.x % (8 * NS) / 8);
  if (bh >= BH) return;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  float* Dc = D + (size_t)bh * (SEG - 1) * DK * DV + col0 + c;
  const float* Mc = M + (size_t)bh * (SEG - 1) * DK * DK;
  struct Step {
    floatx4 m[2][8], d[2];
  };
  auto load = [&](Step& x, int s) {
    s = min(s, SEG - 2);                               // past the end: the last step again, unused
#pragma unroll
    for (int r = 0; r < 2; ++r) {
#pragma unroll
      for (int kk = 0; kk < 8; ++kk)
        x.m[r][kk] = *reinterpret_cast<const floatx4*>(Mc + (size_t)s * DK * DK + (((2 * w + r) * 8 + kk) * 64 + lane) * 4);
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) x.d[r][ii] = Dc[((size_t)s * DK + 32 * w + 16 * r + 4 * g + ii) * DV];
    }
  };
  Step st[3];                                          // step s in set (s - 1) % 3: two steps of lead
  load(st[0], 1);
  load(st[1], 2);
  load(st[2], 3);
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    floatx4 x;
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) x[ii] = Dc[(size_t)(32 * w + 16 * r + 4 * g + ii) * DV];
    H[1][(2 * w + r) * 64 + lane] = x;
  }
  lds_barrier();
  floatx4 last[2];                                     // this wave's rows of the newest state
  auto step = [&](Step& x, int s) {
    const floatx4* h = H[s & 1];
    floatx4 acc[2][2] = {{x.d[0], zero4()}, {x.d[1], zero4()}}, hv[8];
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) hv[kk] = h[kk * 64 + lane];
    __builtin_amdgcn_sched_barrier(0);                 // all eight reads issued before the first use
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int ii = 0; ii < 4; ++ii)
          acc[r][ii & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.m[r][kk][ii], hv[kk][ii], acc[r][ii & 1], 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const floatx4 y = acc[r][0] + acc[r][1];
      H[(s + 1) & 1][(2 * w + r) * 64 + lane] = y;
      last[r] = y;
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) Dc[((size_t)s * DK + 32 * w + 16 * r + 4 * g + ii) * DV] = y[ii];
    }
    load(x, s + 3);
    lds_barrier();                                     // H of the next step written, this step's read
  };
  int s = 1;
  for (; s + 2 < SEG - 1; s += 3) {
    step(st[0], s);
    step(st[1], s + 1);
    step(st[2], s + 2);
  }
  if (s < SEG - 1) step(st[0], s);
  if (s + 1 < SEG - 1) step(st[1], s + 1);
  bool off = false;
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) off = off || !__builtin_isfinite(last[r][ii]);
  const bool any_off = __any(off);
  if (lane == 0) bad[w] = any_off;
  lds_barrier();
  if (w == 0 && g == 0 && (bad[0] | bad[1] | bad[2] | bad[3]))
    Dc[(size_t)(SEG - 2) * DK * DV] = __builtin_nanf("");   // row 0, which this lane stored
}

}  // namespace pf
