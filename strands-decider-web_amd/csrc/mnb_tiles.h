// MatMulNBits projection of many rows with 4-bit weights, gfx950, part of mnb.hip: y[M][N] = a[M][K] x W^T on
// matrix-core tiles.
//
// Bound: the matrix cores and, beside them, LDS reads. mnb_gemm_kernel dequantises a weight tile into LDS, so each MFMA
// costs 1 KiB of LDS reads (two operands for two 32 x 32 tiles each way) on top of the tile's writes: 550 - 600 TFLOP/s.
// Here only a goes through LDS (DMA, three stages). A wave holds whole packed blocks of its own columns in registers (lane
// half h the block 2 kt + h of column l % 32), dequantises a slice right before the MFMAs that use it, and multiplies it
// into RT row tiles; with CT column tiles a wave an MFMA costs 1 / CT KiB of LDS reads, and there is no dequantise-store-
// barrier chain. K order: MFMA j of a 64-k tile takes k 8 j .. + 7 of both blocks; it is the same for every tile shape, so
// the shape chosen never changes a bit.
//
// Tiles: 256 x 256 (8 waves, 4 x 2 tiles each, one workgroup a CU), 128 x 256 (8 waves, 4 x 1), 128 x 128 (4 waves, 4 x 1).
// A launch takes whole rounds of the 256 CUs whatever its last round holds, so columns are given to 256 x 256 tiles only
// in whole rounds, and the rest to the smaller tiles (plan_tiles). An N just over a multiple of 256 (8256 = 32 x 256 + 64)
// would buy a round for its last columns: those go to the strip kernel.
//
// Measured, us a call over a long run of calls, weights rotating through eight matrices, mnb_gemm_kernel -> this (or the strip
// kernel where that is the faster, *):
//   N x K          M = 333     512         1024        1531        2048
//   12288 x 2048   42 -> 31    44 -> 34    79 -> 65    122 -> 102  135 -> 114
//   8256 x 2048    34 -> 27*   41 -> 29    79 -> 45    80 -> 71    122 -> 85
//   2048 x 6144    28 -> 20*   33 -> 24*   52 -> 45*   70 -> 58    78 -> 68
//   5120 x 2048    26 -> 17*   32 -> 22    43 -> 32    49 -> 40    79 -> 60
// In a run of 20 calls of one matrix (HIP events; a kernel trace agrees) M = 2048 takes 124, 92, 77 and 69: the clock differs.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ha_kernels.h"
#include "lds_dma.h"
#include "mnb_common.h"

namespace ha {
namespace tiles {
namespace {

typedef float f16v __attribute__((ext_vector_type(16)));
template <typename T>
using gptr = const __attribute__((address_space(1))) T*;
template <typename T>
__device__ __forceinline__ gptr<T> gp(const void* p) { return (gptr<T>)(p); }

constexpr int kStages = 3;  // a tiles in LDS

// wave (wm, wn) of WM x WN: rows 32 RT wm .., columns 32 CT wn .. of the workgroup's tile
template <int GROUP, bool ASYM, int RT, int CT, int WM, int WN, int kMinWaves>
__global__ __launch_bounds__(64 * WM * WN, kMinWaves) void mnb_tiles_kernel(MnbArgs a) {
  constexpr int kTM = 32 * RT * WM, kTN = 32 * CT * WN, kStage = kTM * 128;
  constexpr int kCopies = kTM / 8 / (WM * WN);  // DMA instructions of a wave for one a tile, 8 rows each
  constexpr int kWLoads = (ASYM ? 3 : 2) * CT;  // loads of a wave for one tile's weights
  extern __shared__ __attribute__((aligned(16))) unsigned char sm[];
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 31, fh = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wm = w / WN, wn = w % WN;
  const int ntn = (a.N + kTN - 1) / kTN, ntm = (a.M + kTM - 1) / kTM, ntiles = ntn * ntm;
  // workgroups go to the 8 XCDs in turn: XCD x takes a contiguous range of tiles, in bands of 4 tile rows, rows fastest,
  // so that neighbours share rows of a and columns of W in its L2
  int id = blockIdx.x;
  {
    const int q = ntiles / 8, r = ntiles % 8, x = id % 8;
    id = x * q + min(x, r) + id / 8;
  }
  constexpr int kBand = 4;
  const int band = id / (kBand * ntn), in_band = id - band * kBand * ntn, rows = min(kBand, ntm - band * kBand);
  const int tm = band * kBand + in_band % rows, tn = in_band / rows;
  const int nblk = a.K / 32, nkt = a.K / 64, ng = a.K / GROUP;
  // rows past M and columns past N repeat the last one and are not stored; a wave whose columns all lie past N only copies
  const int n0 = tn * kTN + 32 * CT * wn;
  const bool active = n0 < a.N;
  unsigned ao[kCopies];
#pragma unroll
  for (int i = 0; i < kCopies; i++) {
    const int r = 8 * (kCopies * w + i) + (lane >> 3), j = (lane & 7) ^ (r & 7);  // chunk j of row r in slot j ^ (r & 7)
    ao[i] = (unsigned)min(r, a.M - 1 - tm * kTM) * (unsigned)a.K * 2u + 16u * j;
  }
  const char* ap = (const char*)a.a + (size_t)tm * kTM * a.K * 2;
  const unsigned lds = lds_addr(sm) + 1024u * kCopies * w;
  auto copy_a = [&](int kt, int stage) {
    kt = min(kt, nkt - 1);  // (past the last tile: that one again, not read)
#pragma unroll
    for (int i = 0; i < kCopies; i++) dma16(lds + (unsigned)(stage * kStage + 1024 * i), ao[i], ap + (size_t)kt * 128);
  };
  gptr<unsigned> wp[CT];
  gptr<unsigned short> sp[CT], bp[CT];
#pragma unroll
  for (int c = 0; c < CT; c++) {
    const int col = min(n0 + 32 * c + fr, a.N - 1);
    wp[c] = gp<unsigned>(a.q) + ((size_t)col * nblk + fh) * 4;
    sp[c] = gp<unsigned short>(a.s) + (size_t)col * ng;
    bp[c] = ASYM ? gp<unsigned short>(a.b) + (size_t)col * ng : sp[c];
  }
  typedef unsigned u4 __attribute__((ext_vector_type(4)));
  u4 wr[2][CT];
  unsigned sr[2][CT], br[2][CT];
  auto load_w = [&](int kt, int q) {
    kt = min(kt, nkt - 1);
#pragma unroll
    for (int c = 0; c < CT; c++) {
      wr[q][c] = *(gptr<u4>)(wp[c] + (size_t)kt * 8);
      sr[q][c] = sp[c][(2 * kt + fh) * 32 / GROUP];
      if constexpr (ASYM) br[q][c] = bp[c][(2 * kt + fh) * 32 / GROUP];
    }
  };
  f16v acc[RT][CT];
#pragma unroll
  for (int i = 0; i < RT; i++)
#pragma unroll
    for (int c = 0; c < CT; c++) acc[i][c] = f16v{};
  const unsigned arow = (unsigned)(32 * RT * wm + fr) * 128u;
  // Tile kt, in stage kt % 3, its weights in registers kt % 2. Loads complete in order: in flight at the top are the weights of
  // tile kt, this wave's part of the copy of tile kt + 1 (a whole tile's time old) and the weights of tile kt + 1, so waiting
  // for all but the last kWLoads lands the first two; the barrier at the end then makes tile kt + 1 everybody's. The wait is
  // written out: the compiler's own, for the weights, is none in a wave that uses no weights. The copy of tile kt + 2 goes
  // into the stage that tile kt - 1 left before the last barrier.
  auto step = [&](int kt, int stage, int q) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kWLoads) : "memory");
#pragma unroll
    for (int c = 0; c < CT; c++) {
      asm volatile("" : "+v"(wr[q][c]), "+v"(sr[q][c])::"memory");
      if constexpr (ASYM) asm volatile("" : "+v"(br[q][c])::"memory");
    }
    copy_a(kt + 2, (stage + 2) % kStages);
    if (active) {
      const unsigned char* as = sm + stage * kStage + arow;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        h8 bf[CT], af[RT];
#pragma unroll
        for (int i = 0; i < RT; i++) af[i] = *(const h8*)(as + 32 * 128 * i + 16 * ((4 * fh + j) ^ (fr & 7)));
#pragma unroll
        for (int c = 0; c < CT; c++)
          bf[c] = dequant8_nat4<ASYM>(wr[q][c][j], splat2u(sr[q][c]), splat2u(ASYM ? br[q][c] : 0u));
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
          for (int c = 0; c < CT; c++) acc[i][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], bf[c], acc[i][c], 0, 0, 0);
      }
    }
    load_w(kt + 2, q);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's reads of the stage are done
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  copy_a(0, 0);
  load_w(0, 0);
  copy_a(1, 1);
  load_w(1, 1);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kCopies + 2 * kWLoads) : "memory");  // tile 0 has landed
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  int kt = 0;
  for (; kt + 6 <= nkt; kt += 6) {
#pragma unroll
    for (int u = 0; u < 6; u++) step(kt + u, u % kStages, u & 1);
  }
#pragma unroll
  for (int u = 0; u < 6; u++)
    if (kt + u < nkt) step(kt + u, u % kStages, u & 1);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // copies past the end land before the LDS is given up
  if (!active) return;
#pragma unroll
  for (int i = 0; i < RT; i++)
#pragma unroll
    for (int c = 0; c < CT; c++) {
      const int n = n0 + 32 * c + fr;
      if (n >= a.N) continue;
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int m = tm * kTM + 32 * (RT * wm + i) + 8 * (v >> 2) + 4 * fh + (v & 3);
        if (m < a.M) ((_Float16*)a.y)[(size_t)m * a.ldy + n] = (_Float16)acc[i][c][v];
      }
    }
}

template <int GROUP, bool ASYM, int RT, int CT, int WM, int WN, int kMinWaves>
hipError_t launch_shape(const MnbArgs& a, hipStream_t s) {
  constexpr int kTM = 32 * RT * WM, kTN = 32 * CT * WN, lds = kStages * kTM * 128;
  auto k = mnb_tiles_kernel<GROUP, ASYM, RT, CT, WM, WN, kMinWaves>;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k, dim3((unsigned)(((a.N + kTN - 1) / kTN) * ((a.M + kTM - 1) / kTM))), dim3(64 * WM * WN), lds, s, a);
  return hipGetLastError();
}

template <int GROUP, bool ASYM>
hipError_t launch_fmt(const MnbArgs& a, Shape sh, hipStream_t s) {
  if (sh == k256x256) return launch_shape<GROUP, ASYM, 4, 2, 2, 4, 2>(a, s);
  if (sh == k128x256) return launch_shape<GROUP, ASYM, 4, 1, 1, 8, 2>(a, s);
  return launch_shape<GROUP, ASYM, 4, 1, 1, 4, 2>(a, s);
}
hipError_t launch(const MnbArgs& a, Shape sh, hipStream_t s) {
  if (a.group == 32) return a.asym ? launch_fmt<32, true>(a, sh, s) : launch_fmt<32, false>(a, sh, s);
  return a.asym ? launch_fmt<64, true>(a, sh, s) : launch_fmt<64, false>(a, sh, s);
}

}  // namespace
}  // namespace tiles

bool mnb_tiles_takes(const MnbArgs& a) { return a.bits == 4 && mnb_strip_takes(a); }

hipError_t launch_mnb_tiles(const MnbArgs& a, hipStream_t s) {
  if (a.M < 1 || !a.a || !a.y || !mnb_tiles_takes(a)) return hipErrorInvalidValue;
  const tiles::Plan p = tiles::plan_tiles(a.M, a.N, a.K);
  auto columns = [&](int from, int to) {
    MnbArgs b = a;
    const size_t per_col = (size_t)(a.K / a.group) * 2;
    b.N = to - from;
    b.q = (const char*)a.q + (size_t)from * (a.K / 32) * 16;
    b.s = (const char*)a.s + from * per_col;
    b.b = a.b ? (const char*)a.b + from * per_col : nullptr;
    b.y = (_Float16*)a.y + from;
    return b;
  };
  hipError_t e = hipSuccess;
  if (p.n1 > 0) e = tiles::launch(columns(0, p.n1), tiles::k256x256, s);
  if (e == hipSuccess && p.n2 > p.n1) e = tiles::launch(columns(p.n1, p.n2), p.rest, s);
  if (e == hipSuccess && a.N > p.n2) e = launch_mnb_strip(columns(p.n2, a.N), s);
  return e;
}

}  // namespace ha
