// KDA forward for fp32 operands: the two stages of the bf16 kernels (pf_kda.h) with fp32 tiles and
// the fp32 MFMA (v_mfma_f32_16x16x4f32).  Mathematics (examples/attention/_kda_full.py:42-76), per
// chain and chunk of C tokens, G = within-chunk cumsum of g [C, dk], a = k e^G, b = k e^-G:
//
//   A = strictly_lower(beta_i (a b^T)_ij),  T = (I + A)^-1,  W = T diag(beta) a,  U = T diag(beta) v
//   stage 2:  v_new = U - W S,  o = QE S + P v_new,  S <- diag(e^{G_last}) S + KR^T v_new
//
// with QE = scale q e^G, KR = k e^{G_last - G}, P = causal_incl(QE b^T).
//
// Stage 1 (kda_local_f32_kernel): one 256-thread workgroup per chunk; a, b and qe in LDS (fp32,
// 68-float rows, so that the 16 rows of an MFMA operand read fall in 16 different bank groups),
// the 20 score blocks over the GDN chunk-local kernel's lists, the inverse in place, then W and U
// with the T rows as the A operand.  Stage 2 (kda_scan_f32_kernel): one workgroup of four waves per
// (chain, 16-column slice), the products of every chunk split over the state rows.
#pragma once

#include <type_traits>

#include "pf_chunk_local.h"
#include "pf_gfx950.h"

namespace pf {

struct KdaLocalF32Args {
  const float* q;       // [M*C, DK]
  const float* k;       // [M*C, DK]
  const float* v;       // [M*C, DV]
  const float* g;       // [M*C, DK] per-token, per-channel log decay (cumsummed here)
  const float* beta;    // [M*C]
  float scale;
  float* W;             // [M, C, DK]
  float* U;             // [M, C, DV]
  float* QE;            // [M*C, DK]
  float* KR;            // [M*C, DK]
  float* P;             // [M, C, C]   lower blocks only (the scan reads no other)
  float* DEC;           // [M, DK]     e^{G_last}
};

// The row tiles hold 64 of the 128 channels at a time (69.8 KB of LDS with A): two workgroups share a
// CU, so that one's loads and stores run beside the other's products: 1024 chunks (287 MB) in 66 us,
// 83 with full-width tiles and one workgroup per CU.
template <int C, int DK>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void kda_local_f32_kernel(KdaLocalF32Args a) {
  static_assert(C == 64 && DK == 128, "the fp32 KDA kernels are written for C 64, dk = dv = 128");
  constexpr int HD = DK / 2, RP = HD + 4;   // half-width row tiles
  constexpr int CP = C + 4;                 // A / T
  constexpr int TILE = C * RP;
  // LDS: a | b | qe row tiles of one channel half, then A; the g staging [C][DK] aliases the tiles
  // until the gated operands are formed; after the scores T replaces A in place and the tiles
  // hold a (second half), a (first half) and v.
  static_assert(C * DK <= 3 * TILE, "g staging fits the tiles");
  __shared__ __attribute__((aligned(16))) float tiles[3 * TILE];
  __shared__ __attribute__((aligned(16))) float As[C * CP];
  __shared__ __attribute__((aligned(16))) float Bs[C];
  float* at = tiles;
  float* bt = tiles + TILE;
  float* qt = tiles + 2 * TILE;
  float* gsm = tiles;

  const int m = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const size_t row0 = (size_t)m * C;
  const int rb = tid >> 4, vc = (tid & 15) * 4;    // rows rb + 16 i, columns 64 h + vc .. vc+3

  // ---- 1. loads; g to LDS ----------------------------------------------------------------
  floatx4 kr[4][2], qr[4][2], vr[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const size_t e = (row0 + rb + 16 * i) * DK + HD * h + vc;
      kr[i][h] = *reinterpret_cast<const floatx4*>(a.k + e);
      qr[i][h] = *reinterpret_cast<const floatx4*>(a.q + e);
      vr[i][h] = *reinterpret_cast<const floatx4*>(a.v + e);
      *reinterpret_cast<floatx4*>(gsm + (rb + 16 * i) * DK + HD * h + vc) =
          *reinterpret_cast<const floatx4*>(a.g + e);
    }
  if (tid < C) Bs[tid] = a.beta[row0 + tid];
  lds_barrier();

  // ---- 2. within-chunk cumsum per channel (thread = column x half of the rows; the second
  //         half's entries get the first half's total when read below) ------------------------
  {
    const int col = tid & (DK - 1), h = tid >> 7;
    float x[C / 2];
#pragma unroll
    for (int r = 0; r < C / 2; ++r) x[r] = gsm[(h * (C / 2) + r) * DK + col];
#pragma unroll
    for (int r = 1; r < C / 2; ++r) x[r] += x[r - 1];
#pragma unroll
    for (int r = 0; r < C / 2; ++r) gsm[(h * (C / 2) + r) * DK + col] = x[r];
  }
  lds_barrier();

  // ---- 3. the cumulative gates of this thread's elements ------------------------------------
  floatx4 G[4][2], gl[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const floatx4 half = *reinterpret_cast<const floatx4*>(gsm + (C / 2 - 1) * DK + HD * h + vc);
    gl[h] = *reinterpret_cast<const floatx4*>(gsm + (C - 1) * DK + HD * h + vc) + half;   // G_last
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      G[i][h] = *reinterpret_cast<const floatx4*>(gsm + (rb + 16 * i) * DK + HD * h + vc);
      if (i >= 2) G[i][h] += half;
    }
    if (tid < 16)
      *reinterpret_cast<floatx4*>(a.DEC + (size_t)m * DK + HD * h + vc) =
          floatx4{__expf(gl[h][0]), __expf(gl[h][1]), __expf(gl[h][2]), __expf(gl[h][3])};
  }

  // ---- 4. gated operands and scores, one channel half at a time: the GDN chunk-local kernel's block
  //         lists (score_code with P): A = beta_i (a_i . b_j) strictly lower into As,
  //         P = qe_i . b_j (lower, with its diagonal) to HBM
  floatx4 a0[4];                                       // a of the first half, for W
  constexpr int N = 5;
  floatx4 acc[N];
#pragma unroll
  for (int b = 0; b < N; ++b) acc[b] = zero4();
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    lds_barrier();                                     // the g staging / the first half is read
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = rb + 16 * i;
      floatx4 av, bv, qv, rv;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float gg = G[i][h][e];
        const float eg = __expf(gg), ebg = __expf(-gg);
        av[e] = kr[i][h][e] * eg;
        bv[e] = kr[i][h][e] * ebg;
        qv[e] = a.scale * qr[i][h][e] * eg;
        rv[e] = kr[i][h][e] * __expf(gl[h][e] - gg);
      }
      const size_t e0 = (row0 + r) * DK + HD * h + vc;
      *reinterpret_cast<floatx4*>(a.QE + e0) = qv;
      *reinterpret_cast<floatx4*>(a.KR + e0) = rv;
      *reinterpret_cast<floatx4*>(at + r * RP + vc) = av;
      *reinterpret_cast<floatx4*>(bt + r * RP + vc) = bv;
      *reinterpret_cast<floatx4*>(qt + r * RP + vc) = qv;
      if (h == 0) a0[i] = av;
    }
    lds_barrier();
    auto products = [&](auto wtag) {
      constexpr int WW = decltype(wtag)::value;
#pragma unroll
      for (int kb = 0; kb < HD / 16; ++kb) {
#pragma unroll
        for (int b = 0; b < N; ++b) {
          const int code = score_code(kScoreAP, WW, b);
          const float* jrow = bt + (16 * (code & 3) + c) * RP;
          const float* irow = ((code & 16) ? qt : at) + (16 * ((code >> 2) & 3) + c) * RP;
          acc[b] = Mfma<float>::rows(acc[b], jrow, irow, kb, g);
        }
      }
    };
    switch (w) {
      case 0: products(std::integral_constant<int, 0>{}); break;
      case 1: products(std::integral_constant<int, 1>{}); break;
      case 2: products(std::integral_constant<int, 2>{}); break;
      default: products(std::integral_constant<int, 3>{}); break;
    }
  }
  // each product is formed transposed: acc[ii] = (x_i . b_j), i = 16 bi + c, j = 16 bj + 4g + ii
#pragma unroll
  for (int b = 0; b < N; ++b) {
    const int code = score_code(kScoreAP, w, b);
    const int i = 16 * ((code >> 2) & 3) + c, j0 = 16 * (code & 3) + 4 * g;
    floatx4 out;
    if (!(code & 16)) {
      const float bi = Bs[i];
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) out[ii] = (i > j0 + ii) ? bi * acc[b][ii] : 0.f;
      *reinterpret_cast<floatx4*>(As + i * CP + j0) = out;
    } else {
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) out[ii] = (i >= j0 + ii) ? acc[b][ii] : 0.f;
      *reinterpret_cast<floatx4*>(a.P + (size_t)m * C * C + i * C + j0) = out;
    }
  }
  lds_barrier();

  // ---- 5. a (first half) and v (first half) into the b and qe tiles; T = (I + A)^-1 in place -----
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    *reinterpret_cast<floatx4*>(bt + (rb + 16 * i) * RP + vc) = a0[i];
    *reinterpret_cast<floatx4*>(qt + (rb + 16 * i) * RP + vc) = vr[i][0];
  }
  unit_lower_inverse64(As, As);

  // ---- 6. W = T diag(beta) a, U = T diag(beta) v: wave w owns column block w of each tile ---------
  //         (A operand = T rows, lane (c, g) T[16 ib + c][4 kk + g]; B = beta_j x[j][16 w + c])
  auto wy = [&](auto ntag, const float* const (&tile)[decltype(ntag)::value],
                float* const (&dst)[decltype(ntag)::value]) {
    constexpr int NT = decltype(ntag)::value;
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) {
      floatx4 d[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) d[t] = zero4();
#pragma unroll 4
      for (int kk = 0; kk < 4 * ib + 4; ++kk) {        // T lower triangular: j <= 16 ib + 15
        const int j = 4 * kk + g;
        const float tv = As[(16 * ib + c) * CP + j], bj = Bs[j];
#pragma unroll
        for (int t = 0; t < NT; ++t)
          d[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(tv, bj * tile[t][j * RP + 16 * w + c], d[t], 0, 0, 0);
      }
      // lane (c, g) holds D[4g + ii][c] of the tile: rows 16 ib + 4g + ii, column 16 w + c
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) dst[t][(row0 + 16 * ib + 4 * g + ii) * DK + 16 * w + c] = d[t][ii];
    }
  };
  wy(std::integral_constant<int, 3>{}, {at, bt, qt}, {a.W + HD, a.W, a.U});
  lds_barrier();
#pragma unroll
  for (int i = 0; i < 4; ++i) *reinterpret_cast<floatx4*>(at + (rb + 16 * i) * RP + vc) = vr[i][1];
  lds_barrier();
  wy(std::integral_constant<int, 1>{}, {at}, {a.U + HD});
}

struct KdaScanF32Args {
  const float* W;       // [BH*NC, C, DK]
  const float* U;       // [BH*NC, C, DV]
  const float* QE;      // [BH*T, DK]
  const float* KR;      // [BH*T, DK]
  const float* P;       // [BH*NC, C, C]  (lower blocks read)
  const float* DEC;     // [BH*NC, DK]
  const float* h0;      // [BH, DK, DV] or null
  float* o;             // [BH*T, DV]
  float* h_final;       // [BH, DK, DV] or null
  int BH, NC;
};

// One workgroup per (chain, 16-column slice), four waves; wave w owns state rows 32w .. 32w+31 (MFMA
// D layout, in registers for the whole chain).  Per chunk:
//
//   1.  partial (W S)_w and (QE S)_w over the wave's rows for all 64 tokens              -> LDS
//   2a. wave w: v_new of token tile w = U - sum of the partials -> LDS; the QE S partials of its
//       o tile 3 - w summed
//   2b. every wave reads all of v_new; wave w: o of token tile 3 - w = QE S + P v_new -> HBM;
//       S_w <- e^{G_last} (.) S_w + KR[:, rows of w]^T v_new
//
// (64 + 4..16 + 32 products per wave and chunk).  Wave w reads only columns 32w .. 32w+31 of the W, QE
// and KR rows, so it loads those slices itself and refills them after its own last read, with no
// barrier; P is written between the barriers (its readers are past the first one), U after the
// second.  Two barriers per chunk, the next chunk's loads in flight across both.  Bound by the chunk
// step's chain, 3.25 us, of which the fp32 products take 1.4 (32 chains x 32 chunks: 104 us; 480
// for the earlier two-wave form, which copied every image with the products waiting).
template <int C, int DK, int DV>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void kda_scan_f32_kernel(KdaScanF32Args a) {
  static_assert(C == 64 && DK == 128 && DV == 128, "the fp32 KDA kernels are written for C 64, dk = dv = 128");
  constexpr int RP = DK + 4, UP = 16 + 4;
  constexpr int TR = 20, TT = 16 * TR;                 // P: its ten lower 16x16 tiles, 20-float rows
  __shared__ __attribute__((aligned(16))) float Ws[C * RP];
  __shared__ __attribute__((aligned(16))) float Qs[C * RP];
  __shared__ __attribute__((aligned(16))) float Ks[C * RP];
  __shared__ __attribute__((aligned(16))) float Ps[10 * TT];
  __shared__ __attribute__((aligned(16))) float Us[C * UP];
  __shared__ __attribute__((aligned(16))) floatx4 YP[4 * 4 * 64];   // [wave][token tile][lane]
  __shared__ __attribute__((aligned(16))) floatx4 QP[4 * 4 * 64];
  __shared__ __attribute__((aligned(16))) floatx4 VX[4 * 64];       // v_new, [token tile][lane]

  constexpr int NS = DV / 16;
  int bh, slice;
  const int bid = blockIdx.x;
  if (a.BH % 8 == 0) {  // the slices of one chain share an XCD: they read the same W, QE, KR, P
    const int grp = bid / (8 * NS), within = bid % (8 * NS);
    bh = grp * 8 + (within % 8);
    slice = within / 8;
  } else {
    bh = bid / NS;
    slice = bid % NS;
  }
  const int col0 = 16 * slice;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int NC = a.NC, last = NC - 1;
  const size_t m0 = (size_t)bh * NC, t0 = m0 * C;

  // chunk data: global -> registers -> LDS.  Lane u of a wave's slice: row u / 8, columns 32w + 4 (u % 8)
  floatx4 rw[8], rq[8], rk[8], rp[4], ru, rd[2];
  const int srow = lane >> 3, scol = 32 * w + 4 * (lane & 7);
  auto load_slice = [&](floatx4 (&r)[8], const float* src, int ch) {
    const float* s = src + (t0 + (size_t)ch * C + srow) * DK + scol;
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = *reinterpret_cast<const floatx4*>(s + i * 8 * DK);
  };
  auto store_slice = [&](float* dst, const floatx4 (&r)[8]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) *reinterpret_cast<floatx4*>(dst + (srow + 8 * i) * RP + scol) = r[i];
  };
  // thread tid holds P rows 16 i + tid / 16, columns 4 (tid % 16) ..: tile (i, (tid % 16) / 4)
  const int p_row = tid >> 4, p_jb = (tid & 15) >> 2, p_col = 4 * (tid & 3);
  auto load_p = [&](int ch) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      rp[i] = *reinterpret_cast<const floatx4*>(a.P + ((m0 + ch) * C + 16 * i + p_row) * C + 4 * (tid & 15));
  };
  auto store_p = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (p_jb <= i) *reinterpret_cast<floatx4*>(Ps + score_tile_index(i, p_jb) * TT + p_row * TR + p_col) = rp[i];
  };
  auto load_u = [&](int ch) {
    ru = *reinterpret_cast<const floatx4*>(a.U + (t0 + (size_t)ch * C + (tid >> 2)) * DV + col0 + 4 * (tid & 3));
  };
  auto store_u = [&]() { *reinterpret_cast<floatx4*>(Us + (tid >> 2) * UP + 4 * (tid & 3)) = ru; };
  auto load_d = [&](int ch) {
#pragma unroll
    for (int r = 0; r < 2; ++r)
      rd[r] = *reinterpret_cast<const floatx4*>(a.DEC + (m0 + ch) * DK + 32 * w + 16 * r + 4 * g);
  };

  floatx4 S[2];                                        // rows 32w + 16r + 4g + ii, column col0 + c
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int ii = 0; ii < 4; ++ii)
      S[r][ii] = a.h0 ? a.h0[((size_t)bh * DK + 32 * w + 16 * r + 4 * g + ii) * DV + col0 + c] : 0.f;

  load_slice(rw, a.W, 0);
  load_slice(rq, a.QE, 0);
  load_slice(rk, a.KR, 0);
  load_u(0);
  store_slice(Ws, rw);
  store_slice(Qs, rq);
  store_slice(Ks, rk);
  store_u();
  load_p(0);
  load_d(0);
  load_slice(rw, a.W, min(1, last));
  load_slice(rq, a.QE, min(1, last));
  load_slice(rk, a.KR, min(1, last));
  load_u(min(1, last));
  lds_barrier();

  // Past the end the loads repeat the last chunk and the copies write what no one reads again, so
  // the loop is straight-line code and a copy waits only for its own loads.
  for (int ch = 0; ch < NC; ++ch) {
    const int nx1 = min(ch + 1, last), nx2 = min(ch + 2, last);
    // ---- 1. partial products over this wave's 32 state rows ----
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) {
      floatx4 y = zero4(), qy = zero4();
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int off = (16 * ib + c) * RP + 32 * w + 16 * r + 4 * g;
        const floatx4 wa = *reinterpret_cast<const floatx4*>(Ws + off);
        const floatx4 qa = *reinterpret_cast<const floatx4*>(Qs + off);
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) {
          y = __builtin_amdgcn_mfma_f32_16x16x4f32(wa[ii], S[r][ii], y, 0, 0, 0);
          qy = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[ii], S[r][ii], qy, 0, 0, 0);
        }
      }
      YP[(w * 4 + ib) * 64 + lane] = y;
      QP[(w * 4 + ib) * 64 + lane] = qy;
    }
    store_slice(Ws, rw);                               // this wave's W and QE slices are read
    store_slice(Qs, rq);
    load_slice(rw, a.W, nx2);
    load_slice(rq, a.QE, nx2);
    lds_barrier();                                     // B1: partials written; P and VX read
    store_p();
    load_p(nx1);
    // ---- 2a. v_new of token tile w; the QE S partials of o tile 3 - w ----
    const int ot = 3 - w;
    floatx4 O = QP[ot * 64 + lane];
#pragma unroll
    for (int w2 = 1; w2 < 4; ++w2) O += QP[(w2 * 4 + ot) * 64 + lane];
    {
      floatx4 Y = YP[w * 64 + lane];
#pragma unroll
      for (int w2 = 1; w2 < 4; ++w2) Y += YP[(w2 * 4 + w) * 64 + lane];
      floatx4 V;
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) V[ii] = Us[(16 * w + 4 * g + ii) * UP + c] - Y[ii];
      VX[w * 64 + lane] = V;
    }
    lds_barrier();                                     // B2: v_new and P written, U read
    store_u();
    load_u(nx2);
    // ---- 2b. o of token tile 3 - w; the update of rows 32w .. ----
    floatx4 VN[4];
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) VN[ib] = VX[ib * 64 + lane];
    {
      floatx4 O2 = zero4();
#pragma unroll
      for (int jb = 0; jb < 4; ++jb) {
        if (jb <= ot) {
          const floatx4 pa = *reinterpret_cast<const floatx4*>(Ps + score_tile_index(ot, jb) * TT + c * TR + 4 * g);
#pragma unroll
          for (int ii = 0; ii < 4; ++ii) {
            if (ii & 1) O2 = __builtin_amdgcn_mfma_f32_16x16x4f32(pa[ii], VN[jb][ii], O2, 0, 0, 0);
            else O = __builtin_amdgcn_mfma_f32_16x16x4f32(pa[ii], VN[jb][ii], O, 0, 0, 0);
          }
        }
      }
      O += O2;
#pragma unroll
      for (int ii = 0; ii < 4; ++ii)
        a.o[(t0 + (size_t)ch * C + 16 * ot + 4 * g + ii) * DV + col0 + c] = O[ii];
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      floatx4 acc, acc2 = zero4();                     // two accumulators: shorter chains
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) acc[ii] = rd[r][ii] * S[r][ii];
#pragma unroll
      for (int jb = 0; jb < 4; ++jb)
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) {
          const float kx = Ks[(16 * jb + 4 * g + ii) * RP + 32 * w + 16 * r + c];
          if (ii & 1) acc2 = __builtin_amdgcn_mfma_f32_16x16x4f32(kx, VN[jb][ii], acc2, 0, 0, 0);
          else acc = __builtin_amdgcn_mfma_f32_16x16x4f32(kx, VN[jb][ii], acc, 0, 0, 0);
        }
      S[r] = acc + acc2;
    }
    load_d(nx1);
    store_slice(Ks, rk);                               // this wave's KR slice is read
    load_slice(rk, a.KR, nx2);
    // no third barrier: the next step 1 writes YP and QP (last read before B2), its B1 precedes the
    // next writes of VX and P
  }
  if (a.h_final) {
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int ii = 0; ii < 4; ++ii)
        a.h_final[((size_t)bh * DK + 32 * w + 16 * r + 4 * g + ii) * DV + col0 + c] = S[r][ii];
  }
}

}  // namespace pf
