// Launch arguments of the stage-2 kernels (the state scan fused with the output): the bf16 split
// scan (pf_scan_split.h) and the fp32 split scan (pf_scan_split_f32.h).
#pragma once

#include "pf_device.h"

namespace pf {

struct ScanOutArgs {
  const void* q;        // [BH*T, DK]  E
  const void* k;        // [BH*T, DK]  E
  const void* v;        // [BH*T, DV]  E
  const float* beta;    // [BH*T]
  const float* G;       // [BH*T] within-chunk cumsum of the log decay, from stage 1
  const void* Tm;       // [M, C, C]   E  (I + A)^-1 per chunk, from stage 1
  const void* P;        // [M, C, C]   E  gated causal score (fp32 operands only), from stage 1
  const float* h0;      // [BH, DK, DV] or null
  float* o;             // [BH*T, DV]
  float* h_final;       // [BH, DK, DV] or null
  int BH;
  int NC;               // chunks per chain
  // segmented chains (bf16): each chain runs as SEG segments of L chunks (the last may have fewer),
  // segment s > 0 from the state hseg[bh][s - 1]; SEG = 1, L = NC otherwise.  h0_stride (SEG > 1): elements
  // between two chains' h0 (DK * DV, or more where h0 is the maps' copy of it)
  int SEG, L;
  const float* scale;   // device scalar: the output scale (written by stage 1)
  const float* hseg;    // [BH, SEG - 1, DK, DV]
  size_t h0_stride;
};

// Arguments of the segmented chains' first two steps (pf_seg_scan.h) and their launch (pf_seg.hip).
struct SegMapArgs {
  const bf16* k;        // [BH*T, DK]
  const bf16* v;        // [BH*T, DV]
  const float* beta;    // [BH*T]
  const float* G;       // [BH*T] within-chunk cumsum of the log decay, from stage 1
  const bf16* Tm;       // [M, C, C] (I + A)^-1, from stage 1
  const float* h0;      // [BH, DK, DV] or null
  float* D;             // [BH, SEG - 1, DK, DV]
  float* M;             // [BH, SEG - 1, DK, DK]   (segment 0's slot: the copy of h0, or not written)
  int BH, NC;           // chains, chunks per chain
  int SEG, L;           // segments per chain, chunks per segment (the last may have fewer)
  int keep_h0;          // copy h0 to M's slots of segment 0: the final state is written over h0 itself, by
                        // another workgroup than the one that starts from it
};
void seg_states_launch(const SegMapArgs& m, hipStream_t stream);

// The same for the KDA forward (stage 1's images instead of k, T and the scalar gate).
struct KdaSegMapArgs {
  const bf16* W;        // [BH*NC, C, DK]
  const bf16* TB;       // [BH*NC, C, C]
  const bf16* KB;       // [BH*T, DK]
  const bf16* v;        // [BH*T, DV]
  const float* DEC;     // [BH*NC, DK]
  const float* h0;      // [BH, DK, DV] or null
  float* D;             // [BH, SEG - 1, DK, DV]
  float* M;             // [BH, SEG - 1, DK, DK]
  int BH, NC, SEG, L, keep_h0;
};
void kda_seg_states_launch(const KdaSegMapArgs& m, hipStream_t stream);

}  // namespace pf
