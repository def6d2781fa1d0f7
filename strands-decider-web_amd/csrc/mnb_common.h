// Weight decoding shared by the MatMulNBits kernels (mnb.hip, mnb_strip.h), gfx950.
#pragma once
#include <hip/hip_runtime.h>

namespace ha {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ h2 splat2(_Float16 v) { return h2{v, v}; }
// the low 16 bits of u as an f16, in both halves
__device__ __forceinline__ h2 splat2u(unsigned u) { return splat2(__builtin_bit_cast(_Float16, (unsigned short)u)); }

// The eight 4-bit codes of one word, dequantised to f16 in element order. v_perm puts a byte (two codes) in both
// half-words; one mask keeps the even code in the low half at bit 0 and the odd one in the high half at bit 4. In the
// mantissa of 1024.0 (0x6400) bit 0 is worth 1, in that of 64.0 (0x5400) bit 4 is: the halves are 1024 + q and 64 + q
// exactly. Subtracting 1024 + 8 and 64 + 8 leaves q - 8 exactly, and one f16 multiply by the scale (one f16 fma with
// the bias when asymmetric) rounds each weight once. 16 VALU instructions for 8 weights.
template <bool ASYM>
__device__ __forceinline__ h8 dequant8_nat4(unsigned u, h2 sc, h2 bi) {
  const h2 off = ASYM ? h2{(_Float16)1024.0f, (_Float16)64.0f} : h2{(_Float16)1032.0f, (_Float16)72.0f};
  h8 r;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const unsigned p = __builtin_amdgcn_perm(u, u, 0x01010101u * i);
    const h2 q = __builtin_bit_cast(h2, (p & 0x00F0000Fu) | 0x54006400u) - off;
    const h2 v = ASYM ? __builtin_elementwise_fma(q, sc, bi) : q * sc;
    r[2 * i] = v[0];
    r[2 * i + 1] = v[1];
  }
  return r;
}

// Eight 2- or 3-bit codes in element order: lo holds their low two bits (element e at bits 2 e), hi their third bits
// (element e at bit e; 3 bits only).
template <int BITS, bool ASYM>
__device__ __forceinline__ h8 dequant8_nat(unsigned lo, unsigned hi, h2 sc, h2 bi) {
  const h2 off = ASYM ? h2{(_Float16)1024.0f, (_Float16)1024.0f}
                      : h2{(_Float16)(1024 + (1 << (BITS - 1))), (_Float16)(1024 + (1 << (BITS - 1)))};
  h8 r;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const unsigned x = lo >> (4 * i);  // elements 2 i (bits 0..1) and 2 i + 1 (bits 2..3)
    unsigned p = (x & 3u) | ((x & 12u) << 14);
    if constexpr (BITS == 3) {
      const unsigned t = hi >> (2 * i);
      p |= ((t & 1u) << 2) | ((t & 2u) << 17);
    }
    const h2 q = __builtin_bit_cast(h2, p | 0x64006400u) - off;
    const h2 v = ASYM ? __builtin_elementwise_fma(q, sc, bi) : q * sc;
    r[2 * i] = v[0];
    r[2 * i + 1] = v[1];
  }
  return r;
}

}  // namespace
}  // namespace ha
