// Which full-attention calls the short-call kernels (gqa_rows.h) serve, and their scratch: code from sizes alone, for the engine and
// the launches (and a CPU test, which compiles it without a GPU).
#pragma once
#include <algorithm>

#include "ha_kernels.h"

namespace ha {

// 32-bit byte offsets of a sequence's input and output rows, rows past the call's end (up to 64 on) included, do not wrap.
inline bool gqa_offsets_fit(const GqaArgs& a) {
  const size_t esz = a.dtype == 0 ? 4 : 2, rows = (size_t)a.L + 64;
  return rows * a.stride * esz <= 0xFFFFFFFFull && rows * a.HQ * a.HD * esz <= 0xFFFFFFFFull;
}

namespace gqa_rows {

constexpr int kG = 32;           // query rows of a group
constexpr int kTile = 64;        // keys of a tile
constexpr int kMaxPieces = 8;    // waves of a values workgroup with split key ranges
constexpr int kPUnit = 2048;     // bytes of P of one 32-key half: [k-step][lane] 16 bytes
constexpr int kSUnit = 32 * 8;   // bytes of a half's row statistics: [row] (alpha, sum)
constexpr int kMUnit = 32 * 4;   // bytes of a half's row maxima, and of its reference maxima
constexpr size_t kUnitBytes = kPUnit + kSUnit + 2 * kMUnit;

// Scratch of a call: per chain unit u = ((pair * ngrp + group) * 4 + head) * nh + half all P, then all statistics, all
// maxima, all reference maxima. The marks [pair][group][tile] are a buffer of their own, so that no other data ever lies where a mark is
// looked for. They are zero between calls: a scores workgroup sets its own, the values kernel clears them again, so a
// launch that a graph replays waits for its own marks and not for those of the replay before.
constexpr unsigned kMark = 1;
struct RowsLayout {
  int ngrp, nt, nh;  // query groups, tiles of the longest group, halves
  unsigned units;    // chain units in all
};
__host__ __device__ inline RowsLayout rows_layout(const GqaArgs& a) {
  RowsLayout r;
  r.ngrp = (a.L + kG - 1) / kG;
  r.nt = (a.P + a.L - 1) / kTile + 1;
  r.nh = 2 * r.nt;
  r.units = (unsigned)(a.B * a.HK * r.ngrp * 4) * (unsigned)r.nh;
  return r;
}

}  // namespace gqa_rows

// The longest call taken, rows a sequence. gqa_attn_kernel has one workgroup per 64 rows and pair (pieces of 8 tiles in
// engines of one or two pairs), so it catches up as rows and pairs fill the chip; the lines lie where it does. Measured at
// 0 to 3000 cached keys, its time over this one's: 2 pairs 1.02 .. 2.6 at up to 256 rows (0.99 .. 1.02 at 400); 4 to 16
// pairs 1.02 .. 3.1 at up to 128; 32 pairs 1.00 .. 1.5 at up to 64 but 0.5 .. 1.0 at 128; 64 pairs 0.5 .. 1.1 at any.
inline int gqa_rows_max(int pairs) { return pairs <= 2 ? 256 : pairs <= 16 ? 128 : pairs <= 32 ? 64 : 0; }

// Marks and scratch bytes an engine holds. The scratch is what its longest short call on a full context needs, but no more
// than one layer's K/V cache, or 64 MiB: calls that would need more are gqa_attn_kernel's (8 sequences of 4096 positions:
// above 102 rows on a full context).
inline size_t gqa_rows_marks(int pairs, int max_ctx) {
  return (size_t)pairs * ((gqa_rows_max(pairs) + gqa_rows::kG - 1) / gqa_rows::kG) * ((max_ctx + gqa_rows::kTile - 1) / gqa_rows::kTile);
}
inline size_t gqa_rows_bytes(int pairs, int max_ctx) {
  const size_t groups = (gqa_rows_max(pairs) + gqa_rows::kG - 1) / gqa_rows::kG;
  const size_t halves = 2 * (size_t)((max_ctx + gqa_rows::kTile - 1) / gqa_rows::kTile);
  const size_t all = pairs * groups * 4 * halves * gqa_rows::kUnitBytes, cache = (size_t)pairs * max_ctx * 256 * 2 * 2;
  return std::min(all, std::max(cache, (size_t)64 << 20));
}

// Whether launch_gqa_rows can run a call: its shape (as launch_gqa checks it), and its scratch, which may be missing or too
// small. Maxima are addressed by 32-bit byte offsets.
inline bool gqa_rows_takes(const GqaArgs& a) {
  if (!a.rows || !a.row_marks || a.L < 1 || a.L > gqa_rows_max(a.B * a.HK)) return false;
  if (a.HD != 256 || a.RD != 64 || a.HQ != 4 * a.HK || a.LT % gqa_rows::kTile || a.P + a.L > a.LT || !gqa_offsets_fit(a)) return false;
  if (a.split > 0 && (a.LT / gqa_rows::kTile + a.split - 1) / a.split > gqa_rows::kMaxPieces) return false;
  const gqa_rows::RowsLayout r = gqa_rows::rows_layout(a);
  const size_t units = (size_t)a.B * a.HK * r.ngrp * 4 * r.nh;
  return units * gqa_rows::kMUnit <= 0x7fffffff && units * gqa_rows::kUnitBytes <= a.rows_bytes &&
         (size_t)a.B * a.HK * r.ngrp * r.nt * sizeof(unsigned) <= a.marks_bytes;
}

}  // namespace ha
