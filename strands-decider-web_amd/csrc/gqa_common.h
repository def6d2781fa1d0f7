// Shared by the full-attention kernels (gqa.hip, gqa_rows.h), gfx950.
#pragma once
#include <hip/hip_runtime.h>

namespace ha {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));

template <typename T>
using gptr = const __attribute__((address_space(1))) T*;
template <typename T>
__device__ __forceinline__ gptr<T> gp(const void* p) { return (gptr<T>)(p); }
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* gpw(void* p) { return (__attribute__((address_space(1))) T*)(p); }

constexpr int kHD = 256, kBK = 64;  // head dim, keys per tile
constexpr float kRescale = 8.0f;    // log2 headroom before the reference max is raised
constexpr int kCacheSc1 = 16;       // cache-policy operand of buffer instructions: device-coherent (sc1)
typedef int i4v __attribute__((ext_vector_type(4)));
typedef int i2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f4 ld4(gptr<float> p) { return *(gptr<f4>)(p); }
__device__ __forceinline__ f4 ld4(gptr<_Float16> p) {
  const h4 x = *(gptr<h4>)(p);
  return f4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]};
}
__device__ __forceinline__ void store4(__attribute__((address_space(1))) float* p, const f4& v) {
  *(__attribute__((address_space(1))) f4*)(p) = v;
}
__device__ __forceinline__ void store4(__attribute__((address_space(1))) _Float16* p, const f4& v) {
  *(__attribute__((address_space(1))) h4*)(p) = h4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
}

__device__ __forceinline__ f4 lds4(const float* p) { return *reinterpret_cast<const f4*>(p); }

// Orders a wave's LDS writes before its later reads of other lanes' entries (no workgroup barrier).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// max / sum of x over lanes l and l ^ 32: v_permlane32_swap hands every lane both values (in an order that depends
// on the half, which neither a max nor a two-term sum sees)
__device__ __forceinline__ void both_halves(float x, float& u, float& v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, x), false, false);
  u = __builtin_bit_cast(float, (unsigned)r[0]);
  v = __builtin_bit_cast(float, (unsigned)r[1]);
}
__device__ __forceinline__ float max_halves(float x) {
  float u, v;
  both_halves(x, u, v);
  return fmaxf(u, v);
}
__device__ __forceinline__ float sum_halves(float x) {
  float u, v;
  both_halves(x, u, v);
  return u + v;
}

__device__ __forceinline__ float sigmoid(float x) { return __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }

template <typename T>
__device__ __forceinline__ void load8f(gptr<T> p, float* o);
template <>
__device__ __forceinline__ void load8f<float>(gptr<float> p, float* o) {
  const f4 x = *(gptr<f4>)(p), y = *(gptr<f4>)(p + 4);
  o[0] = x[0]; o[1] = x[1]; o[2] = x[2]; o[3] = x[3]; o[4] = y[0]; o[5] = y[1]; o[6] = y[2]; o[7] = y[3];
}
template <>
__device__ __forceinline__ void load8f<_Float16>(gptr<_Float16> p, float* o) {
  const h8 x = *(gptr<h8>)(p);
#pragma unroll
  for (int i = 0; i < 8; i++) o[i] = (float)x[i];
}

// Sum over the 64 lanes of a wave without LDS: row rotations inside each 16-lane row, then v_permlane16_swap
// (rows 2r <-> 2r+1) and v_permlane32_swap (halves). Every lane ends with the same bits (each step adds two values
// that the lanes it pairs see in the other order).
template <int kCtrl>
__device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), kCtrl, 0xf, 0xf, false));
}
__device__ __forceinline__ float wave_sum64(float v) {
  v += dpp<0x128>(v);  // row_ror:8
  v += dpp<0x124>(v);  // row_ror:4
  v += dpp<0x122>(v);  // row_ror:2
  v += dpp<0x121>(v);  // row_ror:1
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, v), __builtin_bit_cast(unsigned, v), false, false);
  v = __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
  return sum_halves(v);
}

// The general and the short-call kernels have to give the same bits, so every rounding that the compiler could choose is written
// out: which of two products a sum fuses (it has chosen differently in two kernels of the same source), and whether an f16
// result is rounded to f32 first.
// f16(a b + c), one rounding.
__device__ __forceinline__ _Float16 fma_f16(float a, float b, float c) {
  unsigned r;
  asm("v_fma_mixlo_f16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return __builtin_bit_cast(_Float16, (unsigned short)r);
}

// Key row of one position from a lane's 4 raw dims x (dims 4 lane .. + 3 of the wave's 64 lanes): RMSNorm, gain kw and
// rotate-half RoPE on dims [0, 64) (dim i < 32 pairs with i + 32, held by lane l ^ 8); cs0, cs1: the lane's four
// (cos, sin) pairs, used by lanes < 16.
__device__ __forceinline__ f4 key_row(const f4& x, const f4& kw, const f4& cs0, const f4& cs1, int lane) {
  const float ss = wave_sum64(__builtin_fmaf(x[0], x[0], x[1] * x[1]) + __builtin_fmaf(x[2], x[2], x[3] * x[3]));
  const float inv = rsqrtf(ss / kHD + 1e-6f);
  f4 k = x * inv * kw;
  f4 pk;
#pragma unroll
  for (int c = 0; c < 4; c++) pk[c] = dpp<0x128>(k[c]);  // lane l ^ 8: row_ror:8 within each 16-lane row
  if (lane < 16) {
    const float cs[4] = {cs0[0], cs0[2], cs1[0], cs1[2]}, sn[4] = {cs0[1], cs0[3], cs1[1], cs1[3]};
#pragma unroll
    for (int c = 0; c < 4; c++) k[c] = __builtin_fmaf(k[c], cs[c], lane < 8 ? -(pk[c] * sn[c]) : pk[c] * sn[c]);
  }
  return k;
}

}  // namespace
}  // namespace ha
