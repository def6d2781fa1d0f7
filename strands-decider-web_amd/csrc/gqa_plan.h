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

// The longest call taken, rows a sequence (gqa_rows_faster: which of them are served).
inline int gqa_rows_max(int pairs) { return pairs <= 2 ? 256 : pairs <= 16 ? 128 : pairs <= 32 ? 64 : 0; }

// Whether the short-call kernels are expected to be the faster ones. gqa_attn_kernel has one workgroup per 64 rows and pair
// that walks the key tiles, so its time hardly depends on the pairs; here every tile is a workgroup, which also replays the
// maxima of the tiles before it, so the time grows with pairs x groups x tiles and, in long contexts, with their square.
// Measured, gqa_attn_kernel's time over this one's, f16 rows, at 300 / 3000 / 12000 / 48000 cached keys:
//   4 pairs   1 row 1.28 / 2.68 / 3.04 / 2.67   64 rows 2.38 / 3.06 / 3.42 / 2.60   128 rows 2.40 / 2.40 / 2.52 / 1.59
//   16 pairs  1 row 1.27 / 1.96 / 1.84 / 1.18   64 rows 2.24 / 1.83 / 1.52 / 1.00   128 rows 1.53 / 1.04 / 0.78 / 0.49
//   32 pairs  1 row 1.28 / 1.42 / 1.13 / 0.69   64 rows 1.49 / 0.99 / 0.78 / 0.48
//   2 pairs, whose key ranges are split: 1 row 1.30 / 1.25 / 1.15 / 1.04 (96000: 0.97)   64 rows 2.40 / 2.23 / 1.58 / 1.18 (0.94)
//             128 rows 2.42 / 1.64 / 1.12 / 0.82   256 rows 2.61 / 1.03 / 0.66 / 0.42
// f32 rows are read directly by every tile's workgroup, twice (16 pairs, 3000 keys: 1 row 1.77, 32 rows 1.17, 64 rows 1.18, 96
// rows 0.74; 32 pairs: 1.21, 0.73, 0.61; an empty context: 32 rows 0.82 .. 0.85).
inline bool gqa_rows_faster(int pairs, bool split, bool f32, int L, int nt) {
  const int ngrp = (L + gqa_rows::kG - 1) / gqa_rows::kG;
  const bool some = f32 && L > 8;  // f32 rows whose loads count
  if (split) {  // by row groups: the tiles up to which this is the faster
    constexpr int kTiles[8] = {1200, 1200, 750, 300, 150, 80, 65, 55}, kTiles32[8] = {150, 350, 150, 90, 60, 35, 30, 25};
    return ngrp <= 8 && nt <= (some ? kTiles32 : f32 ? kTiles + 3 : kTiles)[ngrp - 1] && !(some && ngrp == 1 && nt < 3);
  }
  const double wg = (double)pairs * ngrp * nt, replay = 0.055 * nt * wg;  // ns, as below
  if (some)  // the chip takes 192 such workgroups in one go
    return 27000.0 + 250.0 * nt + 75.0 * std::max(0.0, wg - 192.0) + replay <= (L <= 32 ? 21000.0 + 1680.0 * nt : 33000.0 + 2570.0 * nt);
  // 45 ns a workgroup and 0.055 more for each tile of the context, against 1700 a tile (2800 with both 32-row halves; a few
  // rows cost this side less too) and 12000 that the launches and the K/V rows take less
  return 45.0 * wg + replay <= (L <= 8 ? 1850.0 : L <= 32 ? 1700.0 : 2800.0) * nt + 12000.0;
}
inline bool gqa_rows_faster(const GqaArgs& a) {
  return gqa_rows_faster(a.B * a.HK, a.split > 0, a.dtype == 0, a.L, gqa_rows::rows_layout(a).nt);
}

// Marks and scratch bytes an engine holds: what the calls need that gqa_rows_faster serves. (8 sequences of 4096 positions 66 MB
// beside 67 MB of K/V a layer, of 32768 336 beside 537 MB; four pairs at most 1.25 times a layer's K/V.)
inline size_t gqa_rows_marks(int pairs, int max_ctx) {
  return (size_t)pairs * ((gqa_rows_max(pairs) + gqa_rows::kG - 1) / gqa_rows::kG) * ((max_ctx + gqa_rows::kTile - 1) / gqa_rows::kTile);
}
inline size_t gqa_rows_bytes(int pairs, int max_ctx, bool split, bool f32) {
  size_t units = 0;
  const int all = (max_ctx + gqa_rows::kTile - 1) / gqa_rows::kTile;
  for (int L = 8; L <= gqa_rows_max(pairs); L = L == 8 ? gqa_rows::kG : L + gqa_rows::kG) {
    int lo = std::min(all, 4), hi = all;  // the most tiles served: beyond a few, more tiles never make it the faster again
    while (lo < hi) {
      const int nt = (lo + hi + 1) / 2;
      if (gqa_rows_faster(pairs, split, f32, L, nt)) lo = nt;
      else hi = nt - 1;
    }
    units = std::max(units, (size_t)pairs * ((L + gqa_rows::kG - 1) / gqa_rows::kG) * 4 * 2 * lo);
  }
  return units * gqa_rows::kUnitBytes;
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
