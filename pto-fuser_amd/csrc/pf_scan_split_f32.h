// Stage 2 for fp32 operands: the state scan fused with the output, eight waves per chunk so that the
// chain's latency (the forward's time at few chains) is the state's own products and no more.
//
// Workgroup = one chain bh x one 16-column slice (grid BH * DV / 16).  Waves 0..3 carry the state, wave
// w its rows 32w .. 32w+31 (fp32, MFMA D layout, in registers for the whole chain); waves 4..7 form the
// output, one token tile each, beside them.  Per chunk (T, P, G from stage 1; fp32 MFMA 16x16x4):
//
//   state waves                                          output waves
//   1.  partial Y_w = k[:, rows of w] S_w -> LDS
//   ------------------------------------- B1 -------------------------------------
//   2a. Y = sum of the partials and r = beta v -         (q S) of the token tile from the published
//       beta e^G Y for token tiles 0..w, v_new of        state
//       tile w = sum_jb T[w][jb] r_jb -> LDS
//   ------------------------------------- B2 -------------------------------------
//   2b. S_w <- e^{G_last} S_w + k[:, rows of w]^T        o = scale e^G (q S) + P v_new -> HBM
//       (e^{G_last - G} v_new), published to LDS
//
// 32 + 4..16 + 32 products per state wave and 32 + 4..16 per output wave, one of each on every SIMD (token
// tile 3 - w beside wave w: the longer sums share a SIMD with the shorter ones).  q, T and P rows go from
// HBM straight to registers as MFMA operands (no other wave reads them); only k and v pass through
// LDS, wave w's own columns of k refilled after its last read of them with no barrier, v after B2.
//
// The chunk step is bound by the state waves' chain, about 3.2 us, of which their products take 1.1 (four
// waves carrying the output's products too, with q S exchanged as partial sums: 3.8 us).  B1 H4 T512 40.6
// -> 36.5 us whole forward, B1 H4 T4096 251 -> 214, B8 H64 T128 233 -> 210.  Two such workgroups per CU
// (128 registers a wave) were not faster: 282 against 288 us at 32 chains x 64 chunks, 211 against 236 at
// 512 x 2.
#pragma once

#include "pf_scan_args.h"

namespace pf {

template <int C, int DK, int DV>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void scan_split_f32_kernel(ScanOutArgs a) {
  static_assert(C == 64 && DK == 128 && DV % 16 == 0, "tile shapes of the fp32 split scan: C 64, DK 128");
  constexpr int KP = DK + 4, VP = 16 + 4;
  __shared__ __attribute__((aligned(16))) float ks[C * KP];
  __shared__ __attribute__((aligned(16))) float vs[C * VP];
  __shared__ __attribute__((aligned(16))) float Bs[2][C], BEG[2][C], EG[2][C], EL[2][C], DL[2][4];
  __shared__ __attribute__((aligned(16))) floatx4 YP[4 * 4 * 64];   // [wave][token tile][lane]
  __shared__ __attribute__((aligned(16))) floatx4 VX[4 * 64];       // v_new, [token tile][lane]
  __shared__ __attribute__((aligned(16))) floatx4 SB[8 * 64];       // the state, [16-row tile][lane]

  constexpr int NS = DV / 16;
  const int bh = blockIdx.x / NS, col0 = 16 * (blockIdx.x % NS);
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int NC = a.NC, last = NC - 1;
  const size_t t0 = (size_t)bh * NC * C, m0 = (size_t)bh * NC;

  // Past the end the loads repeat the last chunk and the copies write what no one reads again: every
  // chunk is straight-line code, so the compiler's wait counts stay exact.
  if (wv < 4) {
    // =========================== state waves ===========================
    const int w = wv;
    const float* kg = static_cast<const float*>(a.k) + t0 * DK;
    const float* vg = static_cast<const float*>(a.v) + t0 * DV;
    const float* tg = static_cast<const float*>(a.Tm) + m0 * C * C;
    const float oscale = *a.scale;
    floatx4 rk[8], rt[4], rv;
    float rg, rb;
    auto load_k = [&](int ch) {                          // rows u / 8, columns 32w + 4 (u % 8)
#pragma unroll
      for (int i = 0; i < 8; ++i)
        rk[i] = *reinterpret_cast<const floatx4*>(kg + ((size_t)ch * C + (lane >> 3) + 8 * i) * DK + 32 * w + 4 * (lane & 7));
    };
    auto store_k = [&]() {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        *reinterpret_cast<floatx4*>(ks + ((lane >> 3) + 8 * i) * KP + 32 * w + 4 * (lane & 7)) = rk[i];
    };
    auto load_t = [&](int ch) {                          // T[16w + c][16 jb + 4g ..], jb <= w
#pragma unroll
      for (int jb = 0; jb < 4; ++jb)
        rt[jb] = *reinterpret_cast<const floatx4*>(tg + ((size_t)ch * C + 16 * w + c) * C + 16 * min(jb, w) + 4 * g);
    };
    auto load_v = [&](int ch) {
      rv = *reinterpret_cast<const floatx4*>(vg + ((size_t)ch * C + (tid >> 2)) * DV + col0 + 4 * (tid & 3));
    };
    auto store_v = [&]() { *reinterpret_cast<floatx4*>(vs + (tid >> 2) * VP + 4 * (tid & 3)) = rv; };
    auto load_g = [&](int ch) {                          // lane = token
      rg = a.G[t0 + (size_t)ch * C + lane];
      rb = a.beta[t0 + (size_t)ch * C + lane];
    };
    auto store_g = [&](int b) {
      if (w == 0) {
        const float gl = __shfl(rg, C - 1);
        Bs[b][lane] = rb;
        BEG[b][lane] = rb * __expf(rg);
        EG[b][lane] = oscale * __expf(rg);
        EL[b][lane] = __expf(gl - rg);
        if (lane == 0) DL[b][0] = __expf(gl);
      }
    };

    floatx4 S[2];                                        // rows 32w + 16r + 4g + ii, column col0 + c
#pragma unroll
    for (int r = 0; r < 2; ++r) S[r] = zero4();
    if (a.h0) {
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int ii = 0; ii < 4; ++ii)
          S[r][ii] = a.h0[((size_t)bh * DK + 32 * w + 16 * r + 4 * g + ii) * DV + col0 + c];
    }
    auto publish = [&]() {
#pragma unroll
      for (int r = 0; r < 2; ++r) SB[(2 * w + r) * 64 + lane] = S[r];
    };
    load_k(0);
    load_v(0);
    load_g(0);
    load_t(0);
    store_k();
    store_v();
    store_g(0);
    publish();
    load_k(min(1, last));
    load_v(min(1, last));
    load_g(min(1, last));
    lds_barrier();                                       // start

    for (int ch = 0; ch < NC; ++ch) {
      const int cb = ch & 1, nx1 = min(ch + 1, last), nx2 = min(ch + 2, last);
      // ---- 1. partial products over this wave's 32 state rows ----
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) {
        floatx4 y[2] = {zero4(), zero4()};
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const floatx4 ka = *reinterpret_cast<const floatx4*>(ks + (16 * ib + c) * KP + 32 * w + 16 * r + 4 * g);
#pragma unroll
          for (int ii = 0; ii < 4; ++ii) y[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[ii], S[r][ii], y[r], 0, 0, 0);
        }
        YP[(w * 4 + ib) * 64 + lane] = y[0] + y[1];
      }
      lds_barrier();                                     // B1: partials written
      store_g((ch + 1) & 1);                             // the other gate tables are free
      load_g(nx2);
      // ---- 2a. r for token tiles 0..w, v_new tile w = sum_jb T[w][jb] r_jb -> VX ----
      {
        floatx4 V = zero4(), V2 = zero4();               // two accumulators: shorter chains
#pragma unroll
        for (int jb = 0; jb < 4; ++jb) {
          if (jb <= w) {
            floatx4 Y = YP[jb * 64 + lane];
#pragma unroll
            for (int w2 = 1; w2 < 4; ++w2) Y += YP[(w2 * 4 + jb) * 64 + lane];
            floatx4 R;
#pragma unroll
            for (int ii = 0; ii < 4; ++ii) {
              const int t = 16 * jb + 4 * g + ii;
              R[ii] = Bs[cb][t] * vs[t * VP + c] - BEG[cb][t] * Y[ii];
            }
#pragma unroll
            for (int ii = 0; ii < 4; ++ii) {
              if (ii & 1) V2 = __builtin_amdgcn_mfma_f32_16x16x4f32(rt[jb][ii], R[ii], V2, 0, 0, 0);
              else V = __builtin_amdgcn_mfma_f32_16x16x4f32(rt[jb][ii], R[ii], V, 0, 0, 0);
            }
          }
        }
        VX[w * 64 + lane] = V + V2;
      }
      load_t(nx1);
      lds_barrier();                                     // B2: v_new written, v and the state read
      store_v();
      load_v(nx2);
      // ---- 2b. the update of rows 32w .. ----
      floatx4 VN[4];
#pragma unroll
      for (int jb = 0; jb < 4; ++jb) {
        VN[jb] = VX[jb * 64 + lane];
        VN[jb] *= *reinterpret_cast<const floatx4*>(EL[cb] + 16 * jb + 4 * g);
      }
      const float dl = DL[cb][0];
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        floatx4 acc = S[r] * dl, acc2 = zero4();
#pragma unroll
        for (int jb = 0; jb < 4; ++jb)
#pragma unroll
          for (int ii = 0; ii < 4; ++ii) {
            const float kx = ks[(16 * jb + 4 * g + ii) * KP + 32 * w + 16 * r + c];
            if (ii & 1) acc2 = __builtin_amdgcn_mfma_f32_16x16x4f32(kx, VN[jb][ii], acc2, 0, 0, 0);
            else acc = __builtin_amdgcn_mfma_f32_16x16x4f32(kx, VN[jb][ii], acc, 0, 0, 0);
          }
        S[r] = acc + acc2;
      }
      publish();
      store_k();                                         // this wave's k columns are read
      load_k(nx2);
      // no third barrier: the next step 1 writes YP (last read before B2), its B1 orders the published
      // state and the next VX; the gate tables alternate
    }
    if (a.h_final) {
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int ii = 0; ii < 4; ++ii)
          a.h_final[((size_t)bh * DK + 32 * w + 16 * r + 4 * g + ii) * DV + col0 + c] = S[r][ii];
    }
  } else {
    // =========================== output waves ===========================
    const int tt = 7 - wv;                               // token tile
    const float* qg = static_cast<const float*>(a.q) + (t0 + 16 * tt + c) * DK + 4 * g;
    const float* pg = static_cast<const float*>(a.P) + (m0 * C + 16 * tt + c) * C + 4 * g;
    float* og = a.o + (t0 + 16 * tt + 4 * g) * DV + col0 + c;
    floatx4 q0[8], q1[8], rp[4];
    auto load_q = [&](floatx4 (&q)[8], int ch) {         // q[16 tt + c][16 r + 4g ..]
#pragma unroll
      for (int r = 0; r < 8; ++r) q[r] = *reinterpret_cast<const floatx4*>(qg + (size_t)ch * C * DK + 16 * r);
    };
    auto load_p = [&](int ch) {                          // P[16 tt + c][16 jb + 4g ..], jb <= tt
#pragma unroll
      for (int jb = 0; jb < 4; ++jb)
        rp[jb] = *reinterpret_cast<const floatx4*>(pg + (size_t)ch * C * C + 16 * min(jb, tt));
    };
    load_q(q0, 0);
    load_p(0);
    load_q(q1, min(1, last));
    lds_barrier();                                       // start
    auto chunk = [&](floatx4 (&q)[8], int ch) {
      lds_barrier();                                     // B1: the state published
      floatx4 O[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) O[i] = zero4();
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const floatx4 s = SB[r * 64 + lane];
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) O[ii] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[r][ii], s[ii], O[ii], 0, 0, 0);
      }
      load_q(q, min(ch + 2, last));
      const floatx4 eg = *reinterpret_cast<const floatx4*>(EG[ch & 1] + 16 * tt + 4 * g);
      O[0] = ((O[0] + O[1]) + (O[2] + O[3])) * eg;
      O[1] = zero4();
      lds_barrier();                                     // B2: v_new written
#pragma unroll
      for (int jb = 0; jb < 4; ++jb) {
        if (jb <= tt) {
          const floatx4 vn = VX[jb * 64 + lane];
#pragma unroll
          for (int ii = 0; ii < 4; ++ii) O[ii & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(rp[jb][ii], vn[ii], O[ii & 1], 0, 0, 0);
        }
      }
      load_p(min(ch + 1, last));
      O[0] += O[1];
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) __builtin_nontemporal_store(O[0][ii], og + ((size_t)ch * C + ii) * DV);
    };
    int ch = 0;
    for (; ch + 1 < NC; ch += 2) {
      chunk(q0, ch);
      chunk(q1, ch + 1);
    }
    if (ch < NC) chunk(q0, ch);
  }
}

}  // namespace pf
