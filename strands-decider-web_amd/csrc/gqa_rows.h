// Full attention of a short call (a decode step, a resumed question), gfx950, part of gqa.hip: the same arithmetic as gqa.hip, row
// for row and bit for bit (gqa_common.h writes out the roundings the two share), in two launches that put every
// key tile and every slice of output dims on a workgroup of its own.
//
// A short call has one or two 32-row query groups per (sequence, KV head), so gqa_attn_kernel has a handful of workgroups
// that walk the key tiles one after another: 51 us for a decode step of 8 sequences at 1536 keys, 50 us for 61 rows after
// 1531 (plus 5 - 11 us for the K/V rows). What has to be serial is little: the reference maximum of a row (one compare per
// 32-key half), the sum, and O's accumulation over the keys. So:
//   gqa_scores_kernel  one workgroup per (tile of 64 keys, query group, (sequence, KV head)): K and V^T rows of the call's
//     new positions in the tile (gqa_kv_kernel's work; V^T in groups of 8 absolute positions, so the 16-byte stores stay
//     aligned wherever the call starts), S^T = K Q^T, the halves' row maxima to scratch; then it waits for the maxima of
//     the earlier tiles of its chain, replays the reference-maximum rule over them, and writes P (f16, in the lane order
//     of the P V operand), alpha, the row sums and the reference maximum of its two halves.
//   gqa_values_kernel  one wave per (32 output dims, query group, query head), and with split key ranges per piece:
//     O = alpha O + P V over the halves in order, the pieces merged in LDS, 1 / l and the gate.
// The chain of a piece (split engines) starts afresh, as there. A tile that is masked for every row of a group adds exact
// zeros in gqa_attn_kernel; here it is left out.
//
// Bound: latency (a dependent chain of launches, loads and one cross-workgroup hand-off); the K/V cache is read once.
// Waits: a workgroup waits only for workgroups of lower index in its grid. Each XCD takes its blocks in order, so the
// lowest unfinished block is always resident and waits for finished ones: every wait ends, and each is bounded besides.
// Measured, f16 rows, us a call, gqa_attn_kernel -> this: 61 rows after 1531 (1 sequence) 61 -> 23 (traced: scores 12.8, values
// 9.5); one row after 1536 (8 sequences) 56 -> 30 (18.0, 14.3), after 3000 93 -> 48; 64 rows of an empty context 27 -> 19. Where
// it is the faster one and where not: gqa_plan.h.
#pragma once
#include <algorithm>

#include "gqa_common.h"
#include "gqa_plan.h"
#include "ha_kernels.h"
#include "lds_dma.h"

namespace ha {
namespace gqa_rows {
namespace {

constexpr int kSW = 8;           // waves of a scores workgroup: query head w & 3, 32-key half w >> 2 of the tile
static_assert(kTile == kBK, "the tiles of gqa_attn_kernel");
typedef float f2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ unsigned unit_of(const RowsLayout& r, int pair, int grp, int head, int half) {
  return (((unsigned)pair * r.ngrp + grp) * 4 + head) * r.nh + half;
}
// key tiles that query group grp of the call sees
__device__ __forceinline__ int group_tiles(const GqaArgs& a, int grp) {
  return min(a.P + grp * kG + kG - 1, a.P + a.L - 1) / kBK + 1;
}

// Q as the B operand of S^T = K Q^T: qreg[ks] = q[row c32 of the group][16 ks + 8 half .. + 7] after RMSNorm, gain, RoPE
// and the scale 2^-4, with gqa_attn_kernel's roundings and order of sums. A row past the call's end repeats the last one.
// load() issues an f16 row's loads (an f32 row is read in pieces later).
template <typename T>
struct QRow {
  f4 rz[2][4];  // (cos, sin) pairs of dims 16 ks + 8 half + e, ks < 2
  h8 raw[sizeof(T) == 2 ? 16 : 1];
  gptr<T> src;
  gptr<float> rp;
  template <bool kStaged>
  __device__ __forceinline__ void load(const GqaArgs& a, int b, int h, int q0, int half, int c32) {
    const int tc = min(q0 + c32, a.L - 1);
    src = gp<T>(a.in) + ((size_t)b * a.L + tc) * a.stride + (size_t)h * 2 * kHD + 8 * half;
    if constexpr (sizeof(T) == 2 && !kStaged) {
#pragma unroll
      for (int ks = 0; ks < 16; ks++) raw[ks] = *(gptr<h8>)(src + 16 * ks);
    }
    rp = gp<float>(a.rope) + (size_t)(a.P + tc) * a.RD + 16 * half;
  }
  // the same from the group's staged rows of this head: row r at 512 r, 16-byte chunk j in slot j ^ r
  __device__ __forceinline__ void take(const unsigned char* ql, int half, int c32) {
    if constexpr (sizeof(T) == 2) {
#pragma unroll
      for (int ks = 0; ks < 16; ks++) raw[ks] = *reinterpret_cast<const h8*>(ql + 512 * c32 + 16 * ((2 * ks + half) ^ c32));
    }
  }
  __device__ __forceinline__ void load_rope() {
#pragma unroll
    for (int ks = 0; ks < 2; ks++)
#pragma unroll
      for (int j = 0; j < 4; j++) rz[ks][j] = *(gptr<f4>)(rp + 32 * ks + 4 * j);
  }
  __device__ __forceinline__ void prepare(const float* qw, int half, h8* qreg) {
    const h8 scale = h8{} + (_Float16)0.0625f;
    float ss = 0.0f;
    auto finish = [&](int ks, const float* x, float inv) {
      const f4 w0 = lds4(qw + 16 * ks + 8 * half), w1 = lds4(qw + 16 * ks + 8 * half + 4);
      h8 n;
#pragma unroll
      for (int e = 0; e < 8; e++) n[e] = (_Float16)(x[e] * inv * (e < 4 ? w0[e] : w1[e - 4]));
      qreg[ks] = n * scale;
    };
    auto rotate = [&](int ks, const float* x1, const float* x2, float inv) {
      const f4 w10 = lds4(qw + 16 * ks + 8 * half), w11 = lds4(qw + 16 * ks + 8 * half + 4);
      const f4 w20 = lds4(qw + 16 * ks + 8 * half + 32), w21 = lds4(qw + 16 * ks + 8 * half + 36);
      h8 r1, r2;
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float n1 = x1[e] * inv * (e < 4 ? w10[e] : w11[e - 4]), n2 = x2[e] * inv * (e < 4 ? w20[e] : w21[e - 4]);
        const f4 c = rz[ks][e >> 1];
        const float cs = c[2 * (e & 1)], sn = c[2 * (e & 1) + 1];
        r1[e] = fma_f16(n1, cs, -(n2 * sn));
        r2[e] = fma_f16(n2, cs, n1 * sn);
      }
      qreg[ks] = r1 * scale;
      qreg[ks + 2] = r2 * scale;
    };
    if constexpr (sizeof(T) == 2) {
#pragma unroll
      for (int ks = 0; ks < 16; ks++)
#pragma unroll
        for (int e = 0; e < 8; e++) ss += (float)raw[ks][e] * (float)raw[ks][e];
      const float inv = rsqrtf(sum_halves(ss) / kHD + 1e-6f);
      // the f32 values of the squares are not kept for the second use
#pragma unroll
      for (int ks = 0; ks < 16; ks++) asm volatile("" : "+v"(raw[ks])::"memory");
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        float x1[8], x2[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
          x1[e] = (float)raw[ks][e];
          x2[e] = (float)raw[ks + 2][e];
        }
        rotate(ks, x1, x2, inv);
        asm volatile("" : "+v"(qreg[ks]), "+v"(qreg[ks + 2])::"memory");
      }
#pragma unroll
      for (int ks = 4; ks < 16; ks++) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = (float)raw[ks][e];
        finish(ks, x, inv);
        asm volatile("" : "+v"(qreg[ks])::"memory");
      }
    } else {
      // two passes over the row slice, four 32-byte loads in flight at a time
#pragma unroll
      for (int bt = 0; bt < 4; bt++) {
        float qv[4][8];
#pragma unroll
        for (int k = 0; k < 4; k++) load8f<T>(src + 16 * (4 * bt + k), qv[k]);
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
          for (int e = 0; e < 8; e++) ss += qv[k][e] * qv[k][e];
        asm volatile("" : "+v"(ss)::"memory");
      }
      const float inv = rsqrtf(sum_halves(ss) / kHD + 1e-6f);
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        float x1[8], x2[8];
        load8f<T>(src + 16 * ks, x1);
        load8f<T>(src + 16 * (ks + 2), x2);
        rotate(ks, x1, x2, inv);
        asm volatile("" : "+v"(qreg[ks]), "+v"(qreg[ks + 2])::"memory");
      }
#pragma unroll
      for (int bt = 0; bt < 6; bt++) {
        float qv[2][8];
#pragma unroll
        for (int k = 0; k < 2; k++) load8f<T>(src + 16 * (4 + 2 * bt + k), qv[k]);
#pragma unroll
        for (int k = 0; k < 2; k++) finish(4 + 2 * bt + k, qv[k], inv);
        asm volatile("" : "+v"(qreg[4 + 2 * bt]), "+v"(qreg[5 + 2 * bt])::"memory");
      }
    }
  }
};

// 4 dims of a row as loaded
template <typename T>
struct Raw4;
template <>
struct Raw4<_Float16> { h4 v; };
template <>
struct Raw4<float> { f4 v; };
__device__ __forceinline__ f4 wide(const Raw4<_Float16>& x) { return f4{(float)x.v[0], (float)x.v[1], (float)x.v[2], (float)x.v[3]}; }
__device__ __forceinline__ f4 wide(const Raw4<float>& x) { return x.v; }

// 128 VGPRs: two workgroups a CU, so that a batch's tiles all run at once. kStaged (f16 rows, more than kDirect rows): the
// group's q rows of the four heads come through LDS, copied once in whole lines; read directly, a lane's 16 bytes are a
// cache line of their own, for both waves of a head (8K address cycles a workgroup against 1K). 64 KiB more LDS leaves one
// workgroup a CU, so only in launches of at most one for each: 64 rows after 1531, B = 1 (104 workgroups) 25.4 -> 22.8 us
// for both launches, after 500 24.4 -> 21.1; but 9 rows after 1531, B = 8 (400) 30 -> 34. Up to kDirect rows the lanes of a
// direct load share lines: no gain.
constexpr int kDirect = 8;
constexpr int kQLds = 4 * 32 * 512;
template <typename T, bool kStaged>
__global__ __launch_bounds__(64 * kSW, 4) void gqa_scores_kernel(GqaArgs a) {
  // K tile as gqa_attn_kernel stages it: key r at [r][32 chunks of 8 dims], chunk j in slot j ^ (r & 31)
  // then, once S is made, the maxima of earlier halves
  __shared__ __attribute__((aligned(16))) unsigned char kt_l[kBK * kHD * 2];
  __shared__ __attribute__((aligned(16))) float qw_l[kHD];
  __shared__ f4 rope_l[kBK][16];  // the RoPE rows of the tile's positions, in a tile with new keys
  __shared__ float mx_l[4][32];   // the first half's row maxima, for the waves of the second
  extern __shared__ __attribute__((aligned(16))) unsigned char q_l[];
  const RowsLayout r = rows_layout(a);
  const int npair = a.B * a.HK;
  const int id = blockIdx.x, pair = id % npair, grp = (id / npair) % r.ngrp, kt = id / npair / r.ngrp;
  if (kt >= group_tiles(a, grp)) return;
  const int b = pair / a.HK, kh = pair % a.HK;
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int hh = w & 3, kk = w >> 2, half = lane >> 5, c32 = lane & 31, q0 = grp * kG;
  const size_t kvb = ((size_t)b * a.HK + kh) * a.LT * kHD;

  f4 qwv = {};
  if (tid < kHD / 4) qwv = *(gptr<f4>)(gp<float>(a.qw) + 4 * tid);
  QRow<T> q;
  q.template load<kStaged>(a, b, kh * 4 + hh, q0, half, c32);
  if constexpr (kStaged) {
    // 16 of 64 copy instructions a head, two rows each: waves w and w + 4 share head w & 3
    const char* qg = reinterpret_cast<const char*>(a.in) + ((size_t)b * a.L * a.stride + (size_t)(kh * 4 + hh) * 2 * kHD) * 2;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int ins = 8 * kk + i, rr = 2 * ins + half;
      dma16(lds_addr(q_l) + hh * 16384 + ins * 1024,
            (unsigned)min(q0 + rr, a.L - 1) * (unsigned)a.stride * 2u + 16u * (unsigned)(c32 ^ rr), qg);
    }
  }
  // cached keys of the tile: 4 of 32 copy instructions a wave, 2 keys each
  if (kt * kBK < a.P) {
    const char* kg = (const char*)(a.K + kvb + (size_t)kt * kBK * kHD);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int ins = w + kSW * i, rr = 2 * ins + half, js = c32, j = js ^ (rr & 31);
      dma16(lds_addr(kt_l) + ins * 1024, (unsigned)(rr * kHD + 8 * j) * 2u, kg);
    }
  }
  // the call's positions in this tile: raw k, 8 rows a wave, a lane 4 dims
  const int p0 = kt * kBK + 8 * w;  // the wave's first position
  const bool fresh = kt * kBK + kBK > a.P, mine = p0 + 8 > a.P && p0 < a.P + a.L;
  auto kv_row = [&](int i) {
    return gp<T>(a.in) + ((size_t)b * a.L + min(max(p0 + i - a.P, 0), a.L - 1)) * a.stride + (size_t)a.HQ * 2 * kHD +
           (size_t)kh * kHD + 4 * lane;
  };
  typedef decltype(Raw4<T>::v) R4;
  Raw4<T> x[8];
  if (mine) {
#pragma unroll
    for (int i = 0; i < 8; i++) x[i].v = *(gptr<R4>)(kv_row(i));
  }
  if (fresh) {
    const int pr = tid >> 3, c = 2 * (tid & 7);
    gptr<float> rp = gp<float>(a.rope) + (size_t)min(kt * kBK + pr, a.LT - 1) * a.RD + 4 * c;
    const f4 r0 = *(gptr<f4>)(rp), r1 = *(gptr<f4>)(rp + 4);
    rope_l[pr][c] = r0;
    rope_l[pr][c + 1] = r1;
  }
  if (tid < kHD / 4) *reinterpret_cast<f4*>(qw_l + 4 * tid) = qwv;
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __syncthreads();  // q's weights, the cached keys and the RoPE rows are in LDS
  const bool last = grp == r.ngrp - 1;  // the group that sees every tile writes the caches
  if (mine) {
    const f4 kw = *(gptr<f4>)(gp<float>(a.kw) + 4 * lane);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int pos = p0 + i, rr = 8 * w + i;
      const f4 k = key_row(wide(x[i]), kw, rope_l[rr][2 * (lane & 7)], rope_l[rr][2 * (lane & 7) + 1], lane);
      const h4 kf = h4{(_Float16)k[0], (_Float16)k[1], (_Float16)k[2], (_Float16)k[3]};
      if (pos >= a.P && pos < a.P + a.L) {
        *reinterpret_cast<h4*>(kt_l + rr * (kHD * 2) + 16 * ((lane >> 1) ^ (rr & 31)) + 8 * (lane & 1)) = kf;
        if (last) *(__attribute__((address_space(1))) h4*)(gpw<_Float16>(a.K) + kvb + (size_t)pos * kHD + 4 * lane) = kf;
      }
    }
  }
  h8 qreg[16];
  if constexpr (kStaged) q.take(q_l + hh * 16384, half, c32);
  q.load_rope();
  q.prepare(qw_l, half, qreg);
  if (fresh) __syncthreads();  // the new keys are in LDS

  // S^T of the wave's 32-key half: row i holds key pi(i) (bits 2 and 3 swapped), a lane's st[v] is key
  // 16 (v / 8) + 8 half + v % 8 of the half, query row c32
  f16v st = f16v{};
  {
    const int pr = (c32 & 19) | ((c32 & 4) << 1) | ((c32 & 8) >> 1);
    const unsigned kb = (unsigned)(kk * 32 * kHD * 2) + (unsigned)pr * (kHD * 2) + 16u * (unsigned)(pr ^ half);
#pragma unroll
    for (int ks = 0; ks < 16; ks++) {
      const h8 ka = *reinterpret_cast<const h8*>(kt_l + (kb ^ (32u * ks)));
      st = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka, qreg[ks], st, 0, 0, 0);
    }
  }
  const int rowpos = a.P + q0 + c32;
  const float log2e = 1.4426950408889634f;
#pragma unroll
  for (int v = 0; v < 16; v++) {
    const int key = kt * kBK + 32 * kk + 16 * (v >> 3) + 8 * half + (v & 7);
    st[v] = key <= rowpos ? st[v] : -INFINITY;
  }
  float mx = -INFINITY;
#pragma unroll
  for (int v = 0; v < 16; v++) mx = fmaxf(mx, st[v]);
  mx = max_halves(mx) * log2e;

  // publish the maxima, unless no later tile's chain reads them
  char* const base = reinterpret_cast<char*>(a.rows);
  float* const maxima = reinterpret_cast<float*>(base + (size_t)r.units * (kPUnit + kSUnit));
  unsigned* const marks = a.row_marks + ((size_t)pair * r.ngrp + grp) * r.nt;
  const int first = a.split > 0 ? kt / a.split * a.split : 0;  // the first tile of this chain
  const unsigned u = unit_of(r, pair, grp, hh, 2 * kt + kk);
  const __amdgpu_buffer_rsrc_t rm = __builtin_amdgcn_make_buffer_rsrc(maxima, 0, 0x7fffffff, 0x00020000);
  if (half == 0) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, mx), rm, (u * 32 + c32) * 4, 0, kCacheSc1);
  if (kk == 0 && half == 0) mx_l[hh][c32] = mx;
  __builtin_amdgcn_s_waitcnt(0);  // this wave's maxima have reached the device-coherent level
  __syncthreads();                // ... and every wave's
  if (tid == 0) __hip_atomic_store(marks + kt, kMark, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  float mref = -INFINITY;
  auto raise = [&](float m) { mref = m > mref + kRescale ? m : mref; };
  if (first < kt) {
    if (w == 0) {
      // bounded; a wait that runs out is reported through the engine's error word (a test's skew makes every mark this
      // wait looks for one that no workgroup writes)
      const unsigned want = kMark + a.wait.skew;
      for (int j0 = first; j0 < kt; j0 += 64) {
        const int j = min(j0 + lane, kt - 1);
        int i = 0;
        for (; i < a.wait.polls; i++) {
          if (__all(__hip_atomic_load(marks + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == want)) break;
          __builtin_amdgcn_s_sleep(1);
        }
        if (i == a.wait.polls && a.wait.err && lane == 0)
          __hip_atomic_store(a.wait.err, kErrGqaRows, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
    __syncthreads();  // the marks are seen; every wave is done with the K tile
    // the earlier halves' maxima of the four heads through LDS (16 KiB at a time: 32 halves), then the rule over them
    f4* const m_l = reinterpret_cast<f4*>(kt_l);  // [head][half][8]
    const unsigned m0 = unit_of(r, pair, grp, 0, 0) * 8u;
    for (int j0 = 2 * first; j0 < 2 * kt; j0 += 32) {
      const int n = min(32, 2 * kt - j0);
      f4 m[2];
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const int e = tid + 512 * i, j = e >> 3 & 31;  // head e / 256, half j0 + j, rows 4 (e % 8) ..
        m[i] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(
            rm, (m0 + (unsigned)(((e >> 8) * r.nh + j0 + min(j, n - 1)) * 8 + (e & 7))) * 16, 0, kCacheSc1));
      }
      if (j0 > 2 * first) __syncthreads();
#pragma unroll
      for (int i = 0; i < 2; i++) m_l[tid + 512 * i] = m[i];
      __syncthreads();
      const float* mh = reinterpret_cast<const float*>(m_l) + hh * 1024 + c32;
#pragma unroll 8
      for (int j = 0; j < n; j++) raise(mh[32 * j]);
    }
  }
  if (kk == 1) raise(mx_l[hh][c32]);
  const float mnew = mx > mref + kRescale ? mx : mref;
  const float alpha = mnew == mref ? 1.0f : __builtin_amdgcn_exp2f(mref - mnew);
  const float msub = mnew == -INFINITY ? 0.0f : mnew;  // masked scores give exp2(-inf) = 0, never NaN
  float sum = 0.0f;
  h8 pa[2];
#pragma unroll
  for (int v = 0; v < 16; v++) {
    const float pv = __builtin_amdgcn_exp2f(fmaf(st[v], log2e, -msub));
    sum += pv;
    pa[v >> 3][v & 7] = (_Float16)pv;
  }
  const float s2 = sum_halves(sum);
  if (q0 + c32 < a.L) {  // rows of the call; the others' lanes are neither written nor read
    h8* const pp = reinterpret_cast<h8*>(base + (size_t)u * kPUnit);
    pp[lane] = pa[0];
    pp[64 + lane] = pa[1];
    if (half == 0) {
      reinterpret_cast<f2*>(base + (size_t)r.units * kPUnit)[u * 32 + c32] = f2{alpha, s2};
      reinterpret_cast<float*>(base + (size_t)r.units * (kPUnit + kSUnit + kMUnit))[u * 32 + c32] = mnew;
    }
  }
  // V^T of the wave's 8 positions: a lane holds its 4 dims, per dim one 16-byte store where all 8 are the call's
  if (mine && last) {
    Raw4<T> v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i].v = *(gptr<R4>)(kv_row(i) + (size_t)a.HK * kHD);
    __attribute__((address_space(1))) _Float16* vt = gpw<_Float16>(a.V) + kvb + (size_t)(4 * lane) * a.LT + p0;
    if (p0 >= a.P && p0 + 8 <= a.P + a.L) {
#pragma unroll
      for (int c = 0; c < 4; c++) {
        h8 v8;
#pragma unroll
        for (int i = 0; i < 8; i++) v8[i] = (_Float16)v[i].v[c];
        *(__attribute__((address_space(1))) h8*)(vt + (size_t)c * a.LT) = v8;
      }
    } else {
#pragma unroll
      for (int c = 0; c < 4; c++)
#pragma unroll
        for (int i = 0; i < 8; i++)
          if (p0 + i >= a.P && p0 + i < a.P + a.L) vt[(size_t)c * a.LT + i] = (_Float16)v[i].v[c];
    }
  }
}

// V^T tiles in LDS: dim d (of the workgroup's 32) at [d][8 chunks of 8 positions], chunk c in slot c ^ ((d >> 1) & 7)
constexpr int kVTile = 32 * kBK * 2;  // bytes of one tile's slice
constexpr int kVLds = 128 * 1024;

// kSplit: waves are the pieces of one query head's key range; else the four query heads over the whole range.
template <typename T, bool kSplit>
__global__ __launch_bounds__(kSplit ? 64 * kMaxPieces : 256) void gqa_values_kernel(GqaArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char vl[];
  constexpr int kRing = 8;  // (even: a half's parity is its place's)
  const RowsLayout r = rows_layout(a);
  const int npair = a.B * a.HK;
  int id = blockIdx.x;
  const int pair = id % npair;
  id /= npair;
  const int sl = id % 8, grp = id / 8 % r.ngrp;  // 32 output dims 32 sl ..
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int hh = kSplit ? id / 8 / r.ngrp : w;
  const int b = pair / a.HK, kh = pair % a.HK, h = kh * 4 + hh;
  const int half = lane >> 5, c32 = lane & 31, q0 = grp * kG;
  const int nt = group_tiles(a, grp);
  // every scores workgroup has ended: its pair's and group's marks are cleared for the next call (first of all, beside the loads:
  // at the end the stores are 0.2 us of a decode step)
  if (sl == 0 && w == 0 && (!kSplit || hh == 0))
    for (int j = lane; j < r.nt; j += 64)
      __hip_atomic_store(a.row_marks + ((size_t)pair * r.ngrp + grp) * r.nt + j, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int t0 = kSplit ? w * a.split : 0, t1 = kSplit ? min(t0 + a.split, nt) : nt;  // the wave's tiles; none if t0 >= t1
  const size_t kvb = ((size_t)b * a.HK + kh) * a.LT * kHD;
  const char* vg = (const char*)(a.V + kvb + (size_t)(32 * sl) * a.LT);
  const char* const base = reinterpret_cast<const char*>(a.rows);
  const unsigned u0 = unit_of(r, pair, grp, hh, 0);
  const h8* const pp = reinterpret_cast<const h8*>(base) + (size_t)u0 * (kPUnit / 16);
  const f2* const sp = reinterpret_cast<const f2*>(base + (size_t)r.units * kPUnit) + (size_t)u0 * 32 + (q0 + c32 < a.L ? c32 : 0);
  // a lane whose row is past the call's end reads a live row's P and statistics: its products are its own row's only
  const bool live = q0 + c32 < a.L;
  const int plane = live ? lane : 32 * half;
  // V^T in chunks of tiles that fit LDS: a share per piece, or one for all heads
  const int nw = blockDim.x >> 6;
  const int cap = kSplit ? min(a.split, kVLds / kVTile / nw) : kVLds / kVTile;
  unsigned char* const vb = vl + (kSplit ? w * cap * kVTile : 0);
  f16v O = f16v{};
  float mref = -INFINITY, lsum = 0.0f;
  const unsigned vrow = (unsigned)c32 * (kBK * 2) + 16u * (unsigned)((c32 >> 1) & 7);
  constexpr int kParts = kSplit ? 4 : 1;
  unsigned vo[kParts];  // byte offsets of the lane's pieces of a tile from the tile's first dim and position
#pragma unroll
  for (int j = 0; j < kParts; j++) {
    const int d = 8 * (kSplit ? j : w) + (lane >> 3), c = (lane & 7) ^ ((d >> 1) & 7);
    vo[j] = ((unsigned)d * (unsigned)a.LT + 8u * c) * 2u;
  }
  const int last = kSplit ? a.split : nt;  // every wave runs the same number of chunks
  for (int k0 = 0; k0 < last; k0 += cap) {
    if (k0) __syncthreads();  // the chunk before has been read
    // a tile's slice is four copy instructions of 8 dims x 128 bytes (one from each wave where they share the tiles)
    const int n = min(cap, t1 - t0 - k0);
    const char* vt0 = vg + (size_t)(t0 + k0) * (kBK * 2);
    unsigned to = lds_addr(vb);
    for (int i = 0; i < n; i++, vt0 += kBK * 2, to += kVTile) {
#pragma unroll
      for (int j = 0; j < kParts; j++) dma16(to + 1024 * (kSplit ? j : w), vo[j], vt0);
    }
    // P and the row statistics of kRing halves in flight; a half's registers are refilled as soon as it is used. One small
    // loop: code that runs once is fetched as slowly as it runs (batches of 8 unrolled three deep took 18.1 us for one row of 8 sequences after 1536, this 12.3)
    h8 p[kRing][2];
    f2 st[kRing];
    auto load = [&](int j, int q) {
      const int hf = 2 * (t0 + k0) + min(j, 2 * n - 1);  // (past the end: the last half again)
      p[q][0] = pp[hf * (kPUnit / 16) + plane];
      p[q][1] = pp[hf * (kPUnit / 16) + 64 + plane];
      st[q] = sp[hf * 32];
    };
    if (n > 0) {
#pragma unroll
      for (int q = 0; q < kRing; q++) load(q, q);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();  // the chunk's tiles are in LDS
      for (int j0 = 0; j0 < 2 * n; j0 += kRing) {
#pragma unroll
        for (int q = 0; q < kRing; q++) {
          if (j0 + q >= 2 * n) break;
          const float alpha = st[q][0];
          lsum = lsum * alpha + st[q][1];
          // alpha is 1 unless the reference max was raised (then at most 2^-8) or the row meets its first keys (0: O is 0)
          if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int v = 0; v < 16; v++) O[v] *= __shfl(alpha, 8 * (v >> 2) + 4 * half + (v & 3));
          }
          const unsigned char* vt = vb + ((j0 + q) >> 1) * kVTile;
#pragma unroll
          for (int kb = 0; kb < 2; kb++) {
            const h8 ve = *reinterpret_cast<const h8*>(vt + (vrow ^ (unsigned)(16 * (4 * (q & 1) + 2 * kb + half))));
            O = __builtin_amdgcn_mfma_f32_32x32x16_f16(p[q][kb], ve, O, 0, 0, 0);
          }
          load(j0 + q + kRing, q);
        }
      }
    }
    if (n <= 0) __syncthreads();  // (meets the others' barrier above)
  }
  // lane: query rows 8 (v / 4) + 4 half + v % 4 of dim c32 of the slice; statistics by row c32
  float l = lsum;
  if constexpr (kSplit) {
    if (nw > 1) {
      if (live && t0 < t1)
        mref = reinterpret_cast<const float*>(base + (size_t)r.units * (kPUnit + kSUnit + kMUnit))[(u0 + 2 * t1 - 1) * 32 + c32];
      // merge the pieces, in order, with merge_block's arithmetic
      __syncthreads();
      float* const po = reinterpret_cast<float*>(vl);        // [piece][v][lane]
      float* const pm = po + nw * 16 * 64;                   // [piece][(reference max, sum)][row]
#pragma unroll
      for (int v = 0; v < 16; v++) po[(w * 16 + v) * 64 + lane] = O[v];
      if (half == 0) {
        pm[(2 * w) * 32 + c32] = mref;
        pm[(2 * w + 1) * 32 + c32] = lsum;
      }
      __syncthreads();
      if (w) return;
      float M = -INFINITY;
      for (int j = 0; j < nw; j++) M = fmaxf(M, pm[2 * j * 32 + c32]);
      O = f16v{};
      l = 0.0f;
      for (int j = 0; j < nw; j++) {
        const float mj = pm[2 * j * 32 + c32];
        const float wt = mj == M ? 1.0f : __builtin_amdgcn_exp2f(mj - M);
#pragma unroll
        for (int v = 0; v < 16; v++) O[v] = O[v] + __shfl(wt, 8 * (v >> 2) + 4 * half + (v & 3)) * po[(j * 16 + v) * 64 + lane];
        l = l + wt * pm[(2 * j + 1) * 32 + c32];
      }
    }
  }
  const float rinv = 1.0f / l;
  const int d = h * kHD + 32 * sl + c32;
  T gt[16];  // the output gates of the lane's 16 rows, needed last
#pragma unroll
  for (int v = 0; v < 16; v++) {
    const int t = min(q0 + 8 * (v >> 2) + 4 * half + (v & 3), a.L - 1);
    gt[v] = gp<T>(a.in)[((size_t)b * a.L + t) * a.stride + (size_t)h * 2 * kHD + kHD + 32 * sl + c32];
  }
#pragma unroll
  for (int v = 0; v < 16; v++) {
    const int rr = 8 * (v >> 2) + 4 * half + (v & 3), t = q0 + rr;
    const float o = O[v] * __shfl(rinv, rr);
    float y = o * sigmoid((float)gt[v]);
    asm volatile("" : "+v"(y));  // rounded to f32 before f16, as gqa_attn_kernel rounds it, not by one mixed-precision fma
    if (t < a.L) gpw<T>(a.out)[((size_t)b * a.L + t) * (size_t)(a.HQ * kHD) + d] = (T)y;
  }
}

template <typename T>
hipError_t launch(const GqaArgs& a, hipStream_t s) {
  const RowsLayout r = rows_layout(a);
  const int npair = a.B * a.HK;
  const dim3 grid(npair * r.ngrp * r.nt), block(64 * kSW);
  hipError_t e;
  // the staging copies move 16 bytes at a time: rows that are not 16-byte aligned are read directly
  const bool aligned = a.stride % 8 == 0 && (uintptr_t)a.in % 16 == 0;
  if (sizeof(T) == 2 && a.L > kDirect && grid.x <= 256 && aligned) {  // (never with f32 rows)
    if ((e = hipFuncSetAttribute(reinterpret_cast<const void*>(gqa_scores_kernel<T, true>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, kQLds)) != hipSuccess)
      return e;
    hipLaunchKernelGGL((gqa_scores_kernel<T, true>), grid, block, kQLds, s, a);
  } else {
    hipLaunchKernelGGL((gqa_scores_kernel<T, false>), grid, block, 0, s, a);
  }
  if ((e = hipGetLastError()) != hipSuccess) return e;
  const int np = a.split > 0 ? (r.nt + a.split - 1) / a.split : 1;
  auto k = a.split > 0 ? gqa_values_kernel<T, true> : gqa_values_kernel<T, false>;
  if ((e = hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, kVLds)) != hipSuccess)
    return e;
  // LDS: the tiles of a whole range where they fit, and at least the merge's partial results (4.25 KiB a piece)
  const int tiles = a.split > 0 ? std::min(a.split, kVLds / kVTile / np) * np : std::min(r.nt, kVLds / kVTile);
  const int lds = std::max(tiles * kVTile, np * (16 * 64 + 64) * 4);
  hipLaunchKernelGGL(k, dim3(npair * 8 * r.ngrp * (a.split > 0 ? 4 : 1)), dim3(64 * (a.split > 0 ? np : 4)), lds, s, a);
  return hipGetLastError();
}

}  // namespace
}  // namespace gqa_rows

hipError_t launch_gqa_rows(const GqaArgs& a, hipStream_t s) {
  if (!gqa_rows_takes(a)) return hipErrorInvalidValue;
  return a.dtype == 0 ? gqa_rows::launch<float>(a, s) : gqa_rows::launch<_Float16>(a, s);
}

}  // namespace ha
