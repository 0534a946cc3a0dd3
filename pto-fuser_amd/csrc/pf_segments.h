// Host rules of the bf16 scans: how many columns a workgroup takes and when a chain runs in segments
// (pf_seg_scan.h).  Plain C++ on plain numbers, no HIP: workspace sizes follow from it without a
// device.  `cus` is the number of CUs, one scan workgroup each.
#pragma once

namespace pf {

constexpr int kCus = 256;   // MI355X; what workspaces are sized for

// How a chain of NC chunks is run: `seg` segments of `len` chunks (the last may have fewer).
struct Segments {
  int seg, len;
};

inline int generations(long wgs, int cus) { return (int)((wgs + cus - 1) / cus); }

// D and M of a segment in workgroups of their own (the shorter chunk step), while those fit one generation.
inline bool seg_map_split(int BH, int SEG, int cus) { return BH * (2L * SEG - 3) <= cus; }

// Column slices of the bf16 scan, one workgroup per CU: 16 columns (a chunk step of 1.2 us) while eight
// slices per unit (a chain or a segment) fit one generation of workgroups, 32 (1.45 us) while four do, else
// 64 (2.0-2.3 us, half the workgroups of 32 and half their reads of k, q and T).  Whole forward at
// 16 / 32 / 64 columns: 32 chains x 128 chunks 176 / 193 / 272 us, 64 x 64 178 / 113 / 150, 65 x 64
// 339 / 250 / 150, 96 x 64 265 / 207 / 160, 128 x 64 349 / 240 / 194, 192 x 32 283 / 180 / 164, 512 x 8
// 235 / 157 / 116.  The three give the same bits.
inline int gdn_slice_columns(long units, int cus) { return units * 8 <= cus ? 16 : units * 4 <= cus ? 32 : 64; }
inline double gdn_scan_us(long units, int chunks, int cus) {
  const int cols = gdn_slice_columns(units, cus);
  return (cols == 16 ? 1.2 : cols == 32 ? 1.45 : 2.25) * chunks * generations(units * (128 / cols), cus);
}

// The same for KDA, 32 columns while four slices per unit fit one generation, else 64.  Whole forward at
// 32 / 64 columns: 65 chains x 32 chunks 177 / 122 us, 96 x 32 181 / 150, 128 x 64 394 / 352, 512 x 8
// 238 / 206, but 64 x 64 203 / 228 and 32 x 128 283 / 343.  The same bits.
// The scan's time: a chunk step of 1.25 us at 32 columns (1.8 at 64) alone on the chip and 0.4 (1.0) more
// with every CU pulling its chunk images.
inline int kda_slice_columns(long units, int cus) { return units * 4 <= cus ? 32 : 64; }
inline double kda_scan_us(long units, int chunks, int cus) {
  const int cols = kda_slice_columns(units, cus);
  const double wgs = (double)units * (128 / cols), full = wgs < cus ? wgs / cus : 1.0;
  return (cols == 32 ? 1.25 + 0.4 * full : 1.8 + full) * chunks * generations((long)wgs, cus);
}

// The segment counts weighed: 4, 6, then in steps of a quarter, of at least four chunks each.  `time` gives
// the estimate of a count (its own segments' length included) or a negative number to stop; whole chains
// are kept unless one comes out below `limit`.
template <class Time>
inline Segments best_segments(int NC, double limit, Time&& time) {
  Segments best{1, NC};
  if (NC < 16) return best;
  for (int want = 4; want <= 64 && want * 4 <= NC; want += want < 8 ? 2 : want / 4) {
    const int len = (NC + want - 1) / want;
    const Segments s{(NC + len - 1) / len, len};
    const double x = time(s);
    if (x < 0) break;
    if (x < limit) {
      limit = x;
      best = s;
    }
  }
  return best;
}

// Segments of a bf16 GDN chain.  A chain's time is its chunk count while chains leave CUs idle; in
// segments it is the segment's length twice (its map, 2.45 or 3.35 us per chunk step, and the scan) plus a
// composition step of 1.9 us per segment, 9 us for the two more launches, and what short segments of
// many chains lose at their starts (2 us per chain and chunk of length).  No more segments than let every
// map run in one generation of workgroups, which also bounds their states and maps to 128 KiB per CU.  They
// are taken where they come out 5 % ahead.  Whole forward, whole chains and the segments taken (us):
//   1 chain x 128 chunks 149, 69;  4 x 512 578, 153;  8 x 64 82, 60;  8 x 256 301, 128;  16 x 128 160, 109;
//   32 x 512 692, 567;  1 x 32 42.7, 40.6;  20 x 96 125, 104
// and what the segments would have taken where chains stay whole:
//   12 x 40 55.2, 56.4;  33 x 192 286, 311;  64 x 256 434, 552
inline Segments gdn_segments(int BH, int NC, int cus) {
  return best_segments(NC, 0.95 * gdn_scan_us(BH, NC, cus), [&](Segments s) {
    if ((long)BH * (s.seg - 1) > cus) return -1.0;
    const double map = (seg_map_split(BH, s.seg, cus) ? 2.45 : 3.35) * s.len;
    return 9.0 + 2.0 * BH / s.len + map + 1.9 * (s.seg - 2) + gdn_scan_us((long)BH * s.seg, s.len, cus);
  });
}

// Segments of a bf16 KDA chain, by the same reasoning: 2.3 us per chunk of a segment's map (D and M in
// workgroups of their own, and only as many segments as let those run at once: more were never faster),
// 10 us for the launches, taken where that is ahead of whole chains.  Whole forward, whole chains and the
// segments taken (us):
//   1 chain x 128 chunks 168, 76;  4 x 128 176, 84;  8 x 64 98, 71;  16 x 128 220, 154;  24 x 128 258, 232;
//   32 x 256 555, 497
// and what the segments would have taken where chains stay whole:
//   9 x 24 45.7, 50.1;  16 x 32 59.8, 62.9;  32 x 64 142, 143
inline Segments kda_segments(int BH, int NC, int cus) {
  return best_segments(NC, kda_scan_us(BH, NC, cus), [&](Segments s) {
    if (!seg_map_split(BH, s.seg, cus)) return -1.0;
    return 10.0 + 2.0 * BH / s.len + 2.3 * s.len + 1.9 * (s.seg - 2) + kda_scan_us((long)BH * s.seg, s.len, cus);
  });
}

}  // namespace pf
