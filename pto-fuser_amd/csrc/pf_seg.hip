// Launches of the segmented-chain kernels (pf_seg_scan.h), in a source of their own: they are compiled
// with the default machine scheduler.
#include <hip/hip_runtime.h>

#include "pf_seg_scan.h"
#include "pf_segments.h"
#include "pf_status.h"

namespace pf {

namespace {
void compose_launch(float* D, const float* M, int BH, int SEG, hipStream_t stream) {
  if (SEG > 2)
    seg_compose_kernel<128, 128><<<dim3((unsigned)((BH + 7) / 8 * 64)), dim3(256), 0, stream>>>(D, M, BH, SEG);
}
}  // namespace

void seg_states_launch(const SegMapArgs& m, hipStream_t stream) {
  const unsigned units = (unsigned)(m.BH * (m.SEG - 1));
  if (seg_map_split(m.BH, m.SEG, device_cu_count()))
    seg_map_kernel<64, 128, 128, 1><<<dim3((units + 7) / 8 * 16), dim3(512), 0, stream>>>(m);
  else
    seg_map_kernel<64, 128, 128, 2><<<dim3(units), dim3(512), 0, stream>>>(m);
  compose_launch(m.D, m.M, m.BH, m.SEG, stream);
}

void kda_seg_states_launch(const KdaSegMapArgs& m, hipStream_t stream) {
  const unsigned units = (unsigned)(m.BH * (m.SEG - 1));
  kda_seg_map_kernel<64, 128, 128><<<dim3((units + 7) / 8 * 16), dim3(512), 0, stream>>>(m);
  compose_launch(m.D, m.M, m.BH, m.SEG, stream);
}

}  // namespace pf
