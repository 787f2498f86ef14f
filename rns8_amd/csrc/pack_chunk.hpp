// The residue planes of 8 consecutive 64-bit elements: the inner step of
// pack.hip's native pack kernel.
//
// Residue of a 64-bit value without 64-bit division (tables.hpp): split u into
// bytes, s = dot(lo bytes, 2^(8b) mod m) + dot(hi bytes, 2^(32+8b) mod m) + off
// with two v_dot4_u32_u8 (s < 2^19), then the full-rate 24-bit quotient.
// Signed inputs are biased by 2^63 (flip the top bit) and the bias is folded
// into `off`, so int64 and uint64 share the same arithmetic. A plane with
// m = 256 needs no arithmetic: its centered residue is the low byte of x read
// as int8.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "int_ops.hpp"
#include "plane_consts.hpp"
#include "tables.hpp"

namespace rns8x {

typedef uint32_t v8u __attribute__((ext_vector_type(8)));

// A ladder plane's pack constants as one record {pow_lo, pow_hi, shift, recip,
// offset - H, H << shift, 256 - m, 0}, by form: [narrow (32-bit elements),
// wide][signed, unsigned]. The offsets less H: the dot product gives s - H
// (centered_byte).
struct PackTable {
  v8u form[2][2][kMaxPrefix];
};
constexpr PackTable make_pack_table() {
  PackTable t{};
  for (uint32_t p = 0; p < kMaxPrefix; ++p) {
    const ModulusConsts c = make_modulus_consts(kLadder[p]);
    for (uint32_t wide = 0; wide < 2; ++wide)
      for (uint32_t uns = 0; uns < 2; ++uns) {
        const uint32_t shift = wide ? c.pq_shift : c.q_shift;
        const uint32_t off = uns ? c.off_u64 : wide ? c.off_i64 : c.off_i32;
        t.form[wide][uns][p] = v8u{c.pow_lo, c.pow_hi, shift, wide ? c.pq_recip : c.q_recip, off - c.half,
                                   c.half << shift, 256u - c.m, 0};
      }
  }
  return t;
}
static __device__ const PackTable kPackTable = make_pack_table();

// Writes the centered residues of the elements (lo[e], hi[e]) (32-bit halves;
// padding columns hold 0) for planes 0 .. nplanes-1, one aligned 8-byte run
// per plane at out + p * plane_pitch, when `store` is set. Every lane of the
// wave must call it: when every element of the wave fits 32 bits (int32 for
// signed input, uint32 for unsigned), one byte dot product per residue covers
// it (u = x + 2^31 (signed) or x (unsigned) against the int32 reduction
// constants, whose s_max covers both offsets: off_u64 = H <= off_i32).
// Lanes that do not store must hold elements that fit 32 bits (zeros do).
template <bool Signed, bool kStream>
__device__ __forceinline__ void pack_chunk8(uint32_t (&lo)[8], uint32_t (&hi)[8], int8_t* out, int64_t plane_pitch,
                                            uint32_t nplanes, bool store) {
  typedef int v2i __attribute__((ext_vector_type(2)));
  constexpr int kCols = 8;
  bool fits = true;
#pragma unroll
  for (int e = 0; e < kCols; ++e)
    fits &= hi[e] == (Signed ? static_cast<uint32_t>(static_cast<int32_t>(lo[e]) >> 31) : 0u);
  const bool narrow = __all(fits);
  if (Signed) {
#pragma unroll
    for (int e = 0; e < kCols; ++e) {
      hi[e] ^= 0x80000000u;
      if (narrow) lo[e] ^= 0x80000000u;
    }
  }
  auto put = [&](uint32_t p, const uint32_t (&r)[kCols]) {
    const v2i w = {static_cast<int>(pack_low_bytes(r[0], r[1], r[2], r[3])),
                   static_cast<int>(pack_low_bytes(r[4], r[5], r[6], r[7]))};
    if (store) {
      v2i* const dst = reinterpret_cast<v2i*>(out + static_cast<int64_t>(p) * plane_pitch);
      if constexpr (kStream)
        __builtin_nontemporal_store(w, dst);
      else
        *dst = w;
    }
  };
  // The ladder's plane 0 has m = 256: x mod 256 is the low byte, and its
  // centered value is that byte as int8 (the narrow path's bias 2^31 leaves
  // the low byte alone).
  put(0, lo);
  // The other planes' constants are one 32-byte record each, four scalar loads
  // issued together (a plane's scattered fields were loaded, and waited for,
  // plane by plane), and the eight elements go through each operation
  // together, which covers the wait states between a dot product and the
  // reader of its result.
  auto planes = [&](auto narrow_c) {
    constexpr bool kNarrow = decltype(narrow_c)::value;
    const v8u* const table = kPackTable.form[kNarrow ? 0 : 1][Signed ? 0 : 1];
    auto plane = [&](uint32_t p, v8u c) {
      const uint32_t pow_lo = c[0], pow_hi = c[1], shift = c[2], recip = c[3], off = c[4], m_comp = c[6];
      const uint32_t h_sh = in_vgpr(c[5]);
      uint32_t r[kCols];
#pragma unroll
      for (int e = 0; e < kCols; ++e) r[e] = __builtin_amdgcn_udot4(lo[e], pow_lo, off, false);
      if constexpr (!kNarrow) {
#pragma unroll
        for (int e = 0; e < kCols; ++e) r[e] = __builtin_amdgcn_udot4(hi[e], pow_hi, r[e], false);
      }
#pragma unroll
      for (int e = 0; e < kCols; ++e) r[e] = centered_byte(r[e], shift, h_sh, recip, m_comp);
      put(p, r);
    };
    uint32_t p = 1;
    for (; p + 4 <= nplanes; p += 4) {
      const v8u c0 = table[p], c1 = table[p + 1], c2 = table[p + 2], c3 = table[p + 3];
      plane(p, c0);
      plane(p + 1, c1);
      plane(p + 2, c2);
      plane(p + 3, c3);
    }
    for (; p < nplanes; ++p) plane(p, table[p]);
  };
  if (narrow)
    planes(std::true_type{});
  else
    planes(std::false_type{});
}

}  // namespace rns8x
