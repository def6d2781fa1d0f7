// Which MatMulNBits kernel serves a call, with which tiles: host code from sizes and formats alone (no HIP, so that a test can
// compile it by itself). Kernels: mnb.hip, mnb_strip.h, mnb_tiles.h.
#pragma once
#include <algorithm>

namespace ha {

enum MnbPath { kMnbGemv, kMnbStrip, kMnbTiles, kMnbGemm };

struct MnbShape {
  int M, N, K, bits, group;
  bool asym;
  bool dma;  // the strip and tile kernels' DMAs can move the operands (mnb_strip_takes)
};

namespace strip {

// Tile counts the strip kernel is built for: all for what the exporter writes (4 bits, groups of 32, symmetric), fewer
// shapes for the other formats.
inline bool every_tile(const MnbShape& p) { return p.bits == 4 && p.group == 32 && !p.asym; }
inline bool built(bool every, int mt, int nt) {
  if (!every) return (mt == 1 || mt == 2 || mt == 4) && nt >= 1 && nt <= 3;
  return mt >= 1 && mt <= 8 && mt != 7 && nt >= 1 && nt <= (mt <= 6 ? 4 : 3);
}

// The tile counts (mt, nt) of a shape; returns their cost. One workgroup fits a CU's LDS once to four times and its time
// grows with mt + nt (rows of a and columns of W it reads), so: over every shape built, the least rounds of 256 workgroups
// x (mt + nt + 2). Measured choices (M, N, K: mt x nt us, next best): 61, 2048, 6144: 2 x 1 8.0, 3 x 1 9.0; 61, 12288,
// 2048: 4 x 3 9.9, 2 x 3 10.4; 128, 5120, 2048: 3 x 4 8.9, 4 x 3 9.1; 192, 8256, 2048: 4 x 4 18.0, 3 x 3 18.7.
inline long pick_tiles(int M, int N, bool every, int* mt, int* nt) {
  const long tm = (M + 15) / 16, tn = N / 16;
  long best = -1;
  for (int n = 1; n <= 4; n++)
    for (int m = 8; m >= 1; m--) {  // (of equal costs the fewest rounds)
      if (!built(every, m, n)) continue;
      const long rounds = ((tn + n - 1) / n * ((tm + m - 1) / m) + 255) / 256, cost = rounds * (m + n + 2);
      if (best < 0 || cost < best) best = cost, *mt = m, *nt = n;
    }
  return best;
}

// Expected us. 4 bits: 0.35 and 0.55 for every 2048 of K, a unit of cost (measured 0.8 to 1.1 of this). 3 and 2 bits, which
// read narrower words but have fewer shapes: fitted to 65 to 384 rows of 2048 to 151936 columns at K = 512, 2048 and 6144
// (r.m.s. error 9 %).
inline float us(const MnbShape& p) {
  int mt, nt;
  const float cost = (float)pick_tiles(p.M, p.N, every_tile(p), &mt, &nt);
  if (p.bits == 4) return cost * (0.35f + 0.55f * p.K / 2048.0f);
  return 2.2f + cost * (p.bits == 3 ? 0.142f + 0.61f * p.K / 2048.0f : 0.123f + 0.47f * p.K / 2048.0f);
}

}  // namespace strip

namespace tiles {

enum Shape { k256x256, k128x256, k128x128 };
// Columns [0, n1) by 256 x 256 tiles, [n1, n2) by `rest`, [n2, N) by the strip kernel; us: the time this is expected to take.
struct Plan {
  int n1, n2;
  Shape rest;
  float us;
};
// Measured, K = 2048: a round (at most one tile on each of the 256 CUs) takes 57, 29 and 20.5 us, plus a launch's own few;
// full rounds end up at about 920 TFLOP/s whatever the shape (the clock falls: 256 tiles of 256 x 256 take 75 us, 160 59).
inline Plan plan_tiles(int M, int N, int K) {
  const int m256 = (M + 255) / 256, m128 = (M + 127) / 128, tail = N > 256 && N % 256 <= 64 ? N % 256 : 0, nt = N - tail;
  auto rounds = [](long t) { return (float)((t + 255) / 256); };
  Plan best{0, nt, k128x128, 1e30f};
  for (int r = 0; r <= 64; r++) {
    const int c1 = std::min(256 * r / m256, nt / 256);  // tile columns that fill r rounds
    const int left = nt - 256 * c1;
    const float t1 = c1 ? 57.0f * rounds((long)m256 * c1) : 0.0f;
    const float tb = 29.0f * rounds((long)m128 * ((left + 255) / 256)), tc = 20.5f * rounds((long)m128 * ((left + 127) / 128));
    const float busy = (float)M * nt * (2 * 2048 / 920e6f);
    const float t = K / 2048.0f * std::max(t1 + std::min(tb, tc), busy) + (c1 ? 2.0f : 0.0f) + (left ? 3.0f : 0.0f) + (tail ? 5.0f : 0.0f);
    if (t < best.us) best = {256 * c1, nt, tb <= tc ? k128x256 : k128x128, t};
    if (c1 == nt / 256) break;
  }
  return best;
}

}  // namespace tiles

namespace gemm {

constexpr int kTN = 128;  // columns of an output tile
// Whether the 256-row tiles still give every CU a workgroup (else 128-row tiles).
inline bool tall(int M, int N) { return (long)((N + kTN - 1) / kTN) * ((M + 255) / 256) >= 256; }

// K ranges of a product. Fewer output tiles than CUs leave CUs idle behind one long K loop each (about 0.85 us per 64-deep
// k tile): split K so that about 384 workgroups run, each over at least 4 k tiles, with at most 64 MiB of fp32 partials.
inline int split(int M, int N, int K) {
  const long ntn = (N + kTN - 1) / kTN, tiles = tall(M, N) ? ntn * ((M + 255) / 256) : ntn * ((M + 127) / 128);
  const int nkt = (K / 32 + 1) / 2;
  if (tiles >= 256) return 1;
  long sp = std::min<long>((384 + tiles - 1) / tiles, nkt / 4);
  while (sp > 1 && sp * M * (long)N * 4 > (64L << 20)) sp--;
  return (int)std::max<long>(sp, 1);
}

// Expected us, 3 and 2 bits, fitted to the same shapes as strip::us (r.m.s. error 5 %). 256-row tiles take turns on the
// CUs one at a time; 128-row tiles up to two. With K split, the sum of the partials besides.
inline float us(int M, int N, int K, int bits) {
  const long ntn = (N + kTN - 1) / kTN;
  const int sp = split(M, N, K);
  const float k = (bits == 2 ? 0.91f : 1.0f) * K / sp;
  if (tall(M, N)) {
    const long t = ntn * ((M + 255) / 256);
    return std::max((float)((t + 255) / 256) * (5.8f + 0.0172f * k), (float)t / 256.0f * (5.9f + 0.0192f * k));
  }
  const long wg = ntn * ((M + 127) / 128) * sp;
  const float t = wg <= 256 ? 8.1f + 0.0126f * k : (float)((wg + 511) / 512) * (10.4f + 0.0187f * k);
  return sp > 1 ? t + 2.3f + 0.5e-6f * sp * M * (float)N : t;
}

}  // namespace gemm

// One or two rows: from kLaneWide columns the lanes kernel takes four columns a wave instead of two. Measured here and below as
// the mean of weights read long ago (rotating through 700 MB) and of eight rotating matrices, us a call; one row, 4 bits, two
// columns : four: 6144 x 2048 4.5 : 4.7, 8192 x 2048 5.2 : 4.9, 12288 x 2048 6.5 : 6.2, 49152 x 2048 17.9 : 14.8. (A lane
// with three blocks a column puts the line higher: 8192 x 6144 8.7 : 9.3, 24576 x 6144 21.1 : 20.6.)
constexpr int kLanesRows = 2, kLaneWide = 8192;

// One or two rows by the strip kernel rather than the lanes kernel, lanes : strip:
//   4 bits, one row: 5120 x 2048 4.3 : 4.7, 8192 x 2048 4.9 : 4.9, 12288 x 2048 6.2 : 6.0, 16384 x 2048 7.2 : 7.3, 24576 x
//     2048 8.9 : 9.9, 8192 x 6144 9.3 : 9.2, 12288 x 4096 9.3 : 9.0, 12288 x 6144 12.6 : 13.8
//   4 bits, two rows: 5120 x 2048 4.8 : 4.7, 8192 x 2048 5.2 : 4.9, 8192 x 6144 10.3 : 9.2, 12288 x 6144 14.2 : 13.9,
//     49152 x 2048 17.1 : 19.1, 24576 x 6144 24.2 : 29.3
//   3 bits, one row: 12288 x 2048 6.9 : 7.8, 8192 x 6144 11.6 : 12.4; two rows: 5120 x 2048 5.5 : 5.9, 8192 x 2048 6.2 : 6.1,
//     16384 x 2048 9.9 : 9.2, 12288 x 6144 18.5 : 18.0
//   2 bits, one row: 12288 x 2048 5.8 : 5.8, 16384 x 2048 6.8 : 6.3, 12288 x 6144 12.1 : 11.5, 24576 x 6144 20.4 : 23.0
//   K = 512, where most lanes have no block: from 8192 columns strip (16384, 4 bits, 5.9 : 4.4), 2 and 3 bits from 5120
inline bool strip_for_few(const MnbShape& p) {
  if (p.K <= 1024) return p.N >= (p.bits == 4 ? 8192 : 5120);
  if (p.N < 8192) return p.bits == 4 && p.M == 2 && p.K <= 2048 && p.N >= 5120;
  const double w = (double)p.N * p.K;
  if (p.M == 2) return p.bits != 4 || w <= 80e6;
  return p.bits == 4 ? w <= 45e6 : p.bits == 2 && w <= 101e6;
}

inline MnbPath mnb_path(const MnbShape& p) {
  // Operands that the DMAs of the strip and tile kernels cannot move (K % 64, alignment): the lanes kernel, the
  // register-operand kernel up to 64 rows (10 - 28 us at 64 rows against 27 - 71 us for the GEMM), then the GEMM.
  if (p.M <= kLanesRows) return p.dma && strip_for_few(p) ? kMnbStrip : kMnbGemv;
  if (!p.dma) return p.M <= 64 ? kMnbGemv : kMnbGemm;
  if (p.M <= 48) return kMnbStrip;
  if (p.bits == 4) {
    // 49 to 256 rows of at most 12800 columns: strip, so that a row's bits there depend on neither M nor the tiles (from 3
    // rows on; the tile kernel's order of sums is another one). Beyond 12800 columns, where the strip kernel needs several
    // rounds, the tile kernel where it is expected to be the faster by 1.1 (200 rows: 16384 x 2048 30 : 24 us, 49152 x 2048
    // 86 : 64, 151936 x 2048 270 : 192), and above 256 rows the one expected to take less.
    const float s = strip::us(p), t = tiles::plan_tiles(p.M, p.N, p.K).us;
    if (p.M <= 256) return p.N <= 12800 || s <= 1.1f * t ? kMnbStrip : kMnbTiles;
    return s < t ? kMnbStrip : kMnbTiles;
  }
  // 2 and 3 bits: strip up to 64 rows, the GEMM above 384, between them the one expected to take less (200 rows, 3 bits,
  // strip : GEMM: 12288 x 2048 29 : 35 us, 24576 x 2048 53 : 48, 16384 x 6144 106 : 87, 248320 x 2048 551 : 352)
  if (p.M <= 64) return kMnbStrip;
  return p.M <= 384 && strip::us(p) <= 1.04f * gemm::us(p.M, p.N, p.K, p.bits) ? kMnbStrip : kMnbGemm;
}

}  // namespace ha
