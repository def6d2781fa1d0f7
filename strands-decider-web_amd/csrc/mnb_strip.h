// MatMulNBits projection of a few hundred rows or less, gfx950, part of torso.hip: y[M][N] = a[M][K] x W^T (formats: mnb.hip).
//
// Bound: moving a. Each workgroup needs all of its rows of a, so M x K x 2 bytes pass through the L2 once per column
// tile; the packed weights (0.56 bytes each) are read once or twice. A wave cannot load its MFMA operands from a
// straight into registers: consecutive lanes hold different rows, so every lane of a 16-byte load is a cache line of
// its own (64 address cycles per 1 KiB; the kernel that did so took 25 us for 61 x 2048 x 6144). Here a wave copies
// whole 128-byte row pieces into LDS by DMA, eight lanes to a row, and reads the operands from there.
//
// One workgroup makes 16 MT rows x 16 NT columns. Its 8 waves split K (128-k groups w, w + 8, ...) and never meet
// before their partial sums do: each copies into LDS of its own and waits for its own DMAs only, so there is no
// barrier in the loop. A wave handles one 64-k half of a group at a time: wait for its DMAs, read the operands into
// registers, start the next half's DMAs into the same place, then dequantise and multiply. Other waves' arithmetic
// covers the wait; a second stage per wave cost more (fewer workgroups on a CU) than it hid (9.6 against 10.4 us for
// 61 x 12288 x 2048). The K order of a row does not depend on M, so its bits do not either.
//
// v_mfma_f32_16x16x32_f16: lane (g = l / 16, c = l % 16) holds row c of a tile (A operand) or column c (B operand); of a
// half's 64 k it takes k 16 g + 8 j .. + 7 for MFMA j = 0, 1. D: rows 4 g + e, column c.
//
// Measured, us per call back to back, weights rotating through eight matrices, with the kernels this replaced (the
// register-operand kernel up to 64 rows, the tiled GEMM with K split over workgroups above) -> now:
//   N x K          M = 3       17         61          68          128         256
//   12288 x 2048   7.5 -> 5.7  13.3->6.4  25.8->9.1   22.1->9.9   25.8->13.5  35.4->25.1
//   2048 x 6144    7.7 -> 6.3  13.9->6.3  25.0->7.5   21.7->8.5   23.1->9.3   24.6->14.7
//   2048 x 2048    4.0 -> 3.8  5.8 ->3.9  9.8 ->4.2   13.7->4.4   14.3->4.5   15.8->6.1
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ha_kernels.h"
#include "lds_dma.h"
#include "mnb_common.h"

namespace ha {
namespace strip {
namespace {

constexpr int kSW = 8;  // waves of a workgroup

// A wave's LDS stage: a rows, packed words, scales (, biases) of one 64-k half; at the end its partial sums.
template <int BITS, bool ASYM, int MT, int NT>
struct Strip {
  static constexpr int kA = MT * 16 * 128;
  static constexpr int kWBytes = NT * 16 * 8 * BITS;  // two packed blocks of each column
  static constexpr int kWLanes = kWBytes / (BITS == 4 ? 16 : 4), kWUnits = (kWLanes + 63) / 64;
  static constexpr int kSc = NT * 64;  // one word of two scales per column
  static constexpr int kStage = kA + kWBytes + kSc * (ASYM ? 2 : 1);
  static constexpr size_t kLds = std::max(kSW * kStage, kSW / 2 * MT * NT * 1024);
};

template <int BITS, int GROUP, bool ASYM, int MT, int NT>
__global__ __launch_bounds__(64 * kSW) void mnb_strip_kernel(MnbArgs a) {
  using C = Strip<BITS, ASYM, MT, NT>;
  extern __shared__ __attribute__((aligned(16))) unsigned char sm[];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = 16 * NT * blockIdx.x, m0 = 16 * MT * blockIdx.y;
  const int nh = a.K / 64, nblk = a.K / 32, ng = a.K / GROUP;
  // this wave's halves, two per 128-k group (one where the last group has no second)
  const int ngrp = (nh + 1) / 2, mine = w < ngrp ? (ngrp - 1 - w) / kSW + 1 : 0;
  const int T = 2 * mine - ((nh & 1) && mine > 0 && (ngrp - 1) % kSW == w ? 1 : 0);
  auto half_of = [&](int t) { return 2 * (w + kSW * (t >> 1)) + (t & 1); };
  unsigned char* const st = sm + w * C::kStage;
  const unsigned lds = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)sm + w * C::kStage;
  // byte offsets of the lane's pieces from the workgroup's first row / column; rows past M and columns past N repeat
  // the last one and are not stored. a: instruction i copies rows 8 i .. + 7, 16-byte chunk j of row r into slot
  // j ^ (r & 7), so that the operand reads of 16 rows at one chunk fall in distinct banks
  unsigned ao[2 * MT], wo[C::kWUnits];
#pragma unroll
  for (int i = 0; i < 2 * MT; i++) {
    const int r = 8 * i + (lane >> 3), j = (lane & 7) ^ (r & 7);
    ao[i] = (unsigned)min(r, a.M - 1 - m0) * (unsigned)a.K * 2u + 16u * j;
  }
#pragma unroll
  for (int i = 0; i < C::kWUnits; i++) {
    const int u = 64 * i + lane;
    const int col = BITS == 4 ? u >> 1 : u / (2 * BITS), part = BITS == 4 ? u & 1 : u % (2 * BITS);
    wo[i] = (unsigned)min(col, a.N - 1 - n0) * (unsigned)(nblk * BITS * 4) + (BITS == 4 ? 16u : 4u) * part;
  }
  const unsigned so = (unsigned)min(lane, a.N - 1 - n0) * (unsigned)ng * 2u;
  const char* ap = (const char*)a.a + (size_t)m0 * a.K * 2;
  const char* wp = (const char*)a.q + (size_t)n0 * nblk * BITS * 4;
  const char* sp = (const char*)a.s + (size_t)n0 * ng * 2;
  const char* bp = ASYM ? (const char*)a.b + (size_t)n0 * ng * 2 : sp;
  auto issue = [&](int t) {
    const int h = half_of(t);
#pragma unroll
    for (int i = 0; i < 2 * MT; i++) dma16(lds + 1024 * i, ao[i], ap + (size_t)h * 128);
#pragma unroll
    for (int i = 0; i < C::kWUnits; i++) {
      if (64 * i + lane < C::kWLanes) {
        if constexpr (BITS == 4) dma16(lds + C::kA + 1024 * i, wo[i], wp + (size_t)h * (8 * BITS));
        else dma4(lds + C::kA + 256 * i, wo[i], wp + (size_t)h * (8 * BITS));
      }
    }
    // the two scales of the half's blocks, or with groups of 64 those of the 128-k group's halves
    const size_t sb = GROUP == 32 ? (size_t)h * 4 : (size_t)(h >> 1) * 4;
    static_assert(NT <= 4, "one lane per column");
    if (lane < 16 * NT) {
      dma4(lds + C::kA + C::kWBytes, so, sp + sb);
      if constexpr (ASYM) dma4(lds + C::kA + C::kWBytes + C::kSc, so, bp + sb);
    }
  };
  f4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
  if (T > 0) issue(0);
  for (int t = 0; t < T; t++) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    h8 af[MT][2];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) af[i][j] = *(const h8*)(st + (16 * i + c) * 128 + 16 * ((2 * g + j) ^ (c & 7)));
    unsigned wd[NT][2], scw[NT], biw[NT];
#pragma unroll
    for (int n = 0; n < NT; n++) {
      // the words that hold the lane's two 8-element slices 2 (g & 1), + 1 of block g / 2
      const unsigned char* wc = st + C::kA + (16 * n + c) * (8 * BITS);
      if constexpr (BITS == 4) {
        const uint2 v = *(const uint2*)(wc + 8 * g);
        wd[n][0] = v.x;
        wd[n][1] = v.y;
      } else {
        wd[n][0] = *(const unsigned*)(wc + (g >> 1) * 4 * BITS + (g & 1) * 4);
        wd[n][1] = BITS == 3 ? *(const unsigned*)(wc + (g >> 1) * 12 + 8) >> (16 * (g & 1)) : 0u;
      }
      scw[n] = *(const unsigned*)(st + C::kA + C::kWBytes + 4 * (16 * n + c));
      biw[n] = ASYM ? *(const unsigned*)(st + C::kA + C::kWBytes + C::kSc + 4 * (16 * n + c)) : 0u;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the stage has been read: refill it
    if (t + 1 < T) issue(t + 1);
    const int sel = GROUP == 32 ? 16 * (g >> 1) : 16 * (half_of(t) & 1);
#pragma unroll
    for (int n = 0; n < NT; n++) {
      const h2 sc = splat2u(scw[n] >> sel), bi = splat2u(ASYM ? biw[n] >> sel : 0u);
#pragma unroll
      for (int j = 0; j < 2; j++) {
        h8 b;
        if constexpr (BITS == 4) b = dequant8_nat4<ASYM>(wd[n][j], sc, bi);
        else b = dequant8_nat<BITS, ASYM>((wd[n][0] >> (16 * j)) & 0xFFFFu, (wd[n][1] >> (8 * j)) & 0xFFu, sc, bi);
#pragma unroll
        for (int i = 0; i < MT; i++) acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i][j], b, acc[i][n], 0, 0, 0);
      }
    }
  }
  // y = sum over w < 4 of (wave w + wave w + 4), in this order for every shape
  __syncthreads();  // every wave has drained and read its stage: the partial sums take its place
  f4* red = (f4*)sm;
  auto slot = [&](int v, int i, int j) { return ((v * MT + i) * NT + j) * 64 + lane; };
  if (w >= kSW / 2) {
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int j = 0; j < NT; j++) red[slot(w - kSW / 2, i, j)] = acc[i][j];
  }
  __syncthreads();
  if (w < kSW / 2) {
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int j = 0; j < NT; j++) red[slot(w, i, j)] = acc[i][j] + red[slot(w, i, j)];
  }
  __syncthreads();
  for (int q = w; q < MT * NT; q += kSW) {
    f4 s = red[q * 64 + lane];
#pragma unroll
    for (int j = 1; j < kSW / 2; j++) s += red[(j * MT * NT + q) * 64 + lane];
    const int n = n0 + 16 * (q % NT) + c;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int m = m0 + 16 * (q / NT) + 4 * g + e;
      if (m < a.M && n < a.N) ((_Float16*)a.y)[(size_t)m * a.ldy + n] = (_Float16)s[e];
    }
  }
}

template <int BITS, int GROUP, bool ASYM, int MT, int NT>
hipError_t launch_one(const MnbArgs& a, hipStream_t s) {
  constexpr size_t lds = Strip<BITS, ASYM, MT, NT>::kLds;
  static_assert(lds <= 160 * 1024, "LDS of one CU");
  auto k = mnb_strip_kernel<BITS, GROUP, ASYM, MT, NT>;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  const int tiles_n = a.N / 16, tiles_m = (a.M + 15) / 16;
  hipLaunchKernelGGL(k, dim3((tiles_n + NT - 1) / NT, (tiles_m + MT - 1) / MT), dim3(64 * kSW), lds, s, a);
  return hipGetLastError();
}

// The tile counts of mnb_plan.h's built().
template <int BITS, int GROUP, bool ASYM>
constexpr bool kEveryTile = BITS == 4 && GROUP == 32 && !ASYM;
template <int BITS, int GROUP, bool ASYM>
hipError_t launch_fmt(const MnbArgs& a, int mt, int nt, hipStream_t s) {
#define HA_STRIP(MT, NT) \
  if (mt == MT && nt == NT) return launch_one<BITS, GROUP, ASYM, MT, NT>(a, s);
#define HA_STRIP3(MT) HA_STRIP(MT, 1) HA_STRIP(MT, 2) HA_STRIP(MT, 3)
  HA_STRIP3(1) HA_STRIP3(2) HA_STRIP3(4)
  if constexpr (kEveryTile<BITS, GROUP, ASYM>) {
    HA_STRIP3(3) HA_STRIP3(5) HA_STRIP3(6) HA_STRIP3(8)
    HA_STRIP(1, 4) HA_STRIP(2, 4) HA_STRIP(3, 4) HA_STRIP(4, 4) HA_STRIP(5, 4) HA_STRIP(6, 4)
  }
#undef HA_STRIP3
#undef HA_STRIP
  return hipErrorInvalidValue;
}

}  // namespace
}  // namespace strip

// The DMAs move whole 64-k halves: 16 bytes at a time of a and of 4-bit rows, 4 of the others, and two scales at once.
bool mnb_strip_takes(const MnbArgs& a) {
  const uintptr_t q = (uintptr_t)a.q, sb = (uintptr_t)a.s | (a.asym ? (uintptr_t)a.b : 0);
  return a.K % 64 == 0 && (a.group == 32 || a.K % 128 == 0) && (uintptr_t)a.a % 16 == 0 &&
         q % (a.bits == 4 ? 16 : 4) == 0 && sb % 4 == 0;
}

hipError_t launch_mnb_strip(const MnbArgs& a, hipStream_t s) {
  if (a.M < 1 || !a.a || !a.y || !mnb_strip_takes(a)) return hipErrorInvalidValue;
  int mt = 0, nt = 0;
  strip::pick_tiles(a.M, a.N, strip::every_tile(mnb_shape(a)), &mt, &nt);
#define HA_STRIP_CASE(B, G, S) \
  if (a.bits == B && a.group == G && a.asym == S) return strip::launch_fmt<B, G, S>(a, mt, nt, s);
  HA_STRIP_CASE(4, 32, false) HA_STRIP_CASE(4, 32, true) HA_STRIP_CASE(4, 64, false) HA_STRIP_CASE(4, 64, true)
  HA_STRIP_CASE(3, 32, false) HA_STRIP_CASE(3, 32, true) HA_STRIP_CASE(3, 64, false) HA_STRIP_CASE(3, 64, true)
  HA_STRIP_CASE(2, 32, false) HA_STRIP_CASE(2, 32, true) HA_STRIP_CASE(2, 64, false) HA_STRIP_CASE(2, 64, true)
#undef HA_STRIP_CASE
  return hipErrorInvalidValue;
}

}  // namespace ha
