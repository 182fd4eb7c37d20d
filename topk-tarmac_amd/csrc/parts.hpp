// fp32 operands in 16-bit parts for the 32 x 32 matrix instructions: splits,
// tile layout, and the transposing LDS read. Used by the dense fp32 kernels
// (forward and backward).
//
// Three bf16 parts carry fp32's 24 significand bits and its exponent range;
// products of 2^-16 of the whole or more are six of nine. Two fp16 parts carry
// 22 bits of a value whose hi part is normal, in half the instructions; the lo
// part is kept scaled by 2^11, so that it is normal where hi is.
#pragma once

#include "frag.hpp"

namespace tarmac {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef short i16x4_t __attribute__((ext_vector_type(4)));

constexpr float kLoScale = 0x1p11f;  // of the lo part of two fp16 parts

__device__ __forceinline__ f32x16 mfma_bf16_32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma_f16_32(f16x8 a, f16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// Element i of a 32 x 32 tile is row tile_row(i) + 4 (l / 32) of column l % 32.
__device__ constexpr int tile_row(int i) { return 8 * (i / 4) + i % 4; }

// Maximum (sum) over the two lanes l, l + 32 of a column.
__device__ __forceinline__ float max_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// A wave-uniform offset in scalar registers: row offsets computed behind a
// divergent branch's join are otherwise kept, per lane, in vector registers.
__device__ __forceinline__ size_t uniform_offset(size_t x) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(x));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(x >> 32));
  return static_cast<size_t>(hi) << 32 | lo;
}

// A wave-uniform value in a scalar register.
__device__ __forceinline__ float uniform_value(float x) {
  return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x)));
}

// A barrier that orders LDS accesses only: global loads in flight stay so.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Two values as three bf16 pairs: one packed conversion a part, and each
// residual as one v_dot2_f32_bf16 of the packed pair with (-1, 0) or (0, -1)
// onto the value: exact, since the residual is an fp32 number (checked on the
// device over 2^25 values of exponents 2^-107 to 2^113). 7 VALU a pair. A value
// that is not finite makes its pair's residuals NaN. The two constants are
// scalar copies that the compiler cannot see through: as a literal, the low
// form is encoded as the inline constant of the other half.
__device__ __forceinline__ void split3_dot(float x0, float x1, uint32_t& hi, uint32_t& mid,
                                           uint32_t& lo) {
  typedef __bf16 pair_t __attribute__((ext_vector_type(2)));
  uint32_t c0, c1;
  asm("s_mov_b32 %0, 0xbf80" : "=s"(c0));
  asm("s_mov_b32 %0, 0xbf800000" : "=s"(c1));
  const pair_t m0 = __builtin_bit_cast(pair_t, c0), m1 = __builtin_bit_cast(pair_t, c1);
  const pair_t h = {static_cast<__bf16>(x0), static_cast<__bf16>(x1)};
  hi = __builtin_bit_cast(uint32_t, h);
  asm("" : "+v"(hi));  // the packed word, not a second conversion
  const pair_t hp = __builtin_bit_cast(pair_t, hi);
  const float r0 = __builtin_amdgcn_fdot2_f32_bf16(hp, m0, x0, false);
  const float r1 = __builtin_amdgcn_fdot2_f32_bf16(hp, m1, x1, false);
  const pair_t m = {static_cast<__bf16>(r0), static_cast<__bf16>(r1)};
  mid = __builtin_bit_cast(uint32_t, m);
  asm("" : "+v"(mid));
  const pair_t mp = __builtin_bit_cast(pair_t, mid);
  const pair_t l = {static_cast<__bf16>(__builtin_amdgcn_fdot2_f32_bf16(mp, m0, r0, false)),
                    static_cast<__bf16>(__builtin_amdgcn_fdot2_f32_bf16(mp, m1, r1, false))};
  lo = __builtin_bit_cast(uint32_t, l);
}

// Two values below 2^16 as two fp16 pairs: hi rounded to nearest, lo what is left
// of it times 2^11, so that a value keeps 22 bits down to 2^-14 and is held to
// 2^-36 below (unscaled, 2^-25: a weight of 2^-20 beside one of 1 had 10 bits).
// v_fma_mix_f32 subtracts a half of the packed word; 6 VALU a pair (v_fma_mixlo
// and mixhi for the last four save one and run no faster).
__device__ __forceinline__ void split2_pair(float a, float b, uint32_t& hi, uint32_t& lo) {
  const f16x2 h = {static_cast<_Float16>(a), static_cast<_Float16>(b)};
  hi = __builtin_bit_cast(uint32_t, h);
  asm("" : "+v"(hi));  // the packed word, not a second conversion
  const f16x2 hp = __builtin_bit_cast(f16x2, hi);
  float m1;  // -1, opaque: a multiply by a known -1 becomes two conversions and two subtractions
  asm("s_mov_b32 %0, -1.0" : "=s"(m1));
  const f16x2 l = {static_cast<_Float16>(fmaf(static_cast<float>(hp[0]), m1, a) * kLoScale),
                   static_cast<_Float16>(fmaf(static_cast<float>(hp[1]), m1, b) * kLoScale)};
  lo = __builtin_bit_cast(uint32_t, l);
}

// One row of D channels in three bf16 parts, as the B operand of score tiles:
// lane l holds channels 16 g + 8 (l / 32) .. + 7 of its column's row.
template <int D>
struct RowParts {
  bf16x8 hi[D / 16], mid[D / 16], lo[D / 16];
  // c: a factor applied in fp32 before the split
  __device__ __forceinline__ void load(const float* row, int half, float c) {
#pragma unroll
    for (int g = 0; g < D / 16; ++g) {
      float x[8];
      ld_f32<8>(x, row + 16 * g + 8 * half);
      uint32_t h[4], m[4], l[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) split3_dot(x[2 * e] * c, x[2 * e + 1] * c, h[e], m[e], l[e]);
      hi[g] = __builtin_bit_cast(bf16x8, h);
      mid[g] = __builtin_bit_cast(bf16x8, m);
      lo[g] = __builtin_bit_cast(bf16x8, l);
    }
  }
};

// s + (32 staged rows) . (the columns' rows): rows at R (lane l: row l % 32 of
// the tile plus 8 (l / 32) channels), stored as hi[D] mid[D] lo[D]. A bf16 MFMA
// cuts what it adds at the accumulator's last place, so the products of the
// parts go in from the smallest up, over all channel groups before the next
// larger ones, and a chain starts at 0 rather than at a large offset: only the
// D / 16 products of the hi parts are rounded at the sum's own magnitude.
// SWAP: what are columns otherwise are rows here; the products keep their order,
// so a score has the same bits either way.
template <int D, bool SWAP = false>
__device__ __forceinline__ f32x16 tile_dot(const RowParts<D>& q, const bf16* R, f32x16 s) {
  constexpr int G = D / 16;
  // d = 64 reads the rows' hi and mid parts again for the larger products:
  // kept, they would take 32 registers that the kernels do not have. The
  // opaque copy is of the LDS address (of a generic pointer it would make the
  // reads flat ones, which wait for the global loads in flight).
  using lds_t = const __attribute__((address_space(3))) bf16x8;
  using lds_row = const __attribute__((address_space(3))) bf16;
  lds_row* L = (lds_row*)R;
  auto again = [&]() {
    if constexpr (D > 32) asm volatile("" : "+v"(L));
  };
  auto part = [&](int p, int g) { return *(lds_t*)(L + p * D + 16 * g); };
#pragma unroll
  for (int g = 0; g < G; ++g) {
    s = SWAP ? mfma_bf16_32(part(0, g), q.lo[g], s) : mfma_bf16_32(part(2, g), q.hi[g], s);
    s = SWAP ? mfma_bf16_32(part(2, g), q.hi[g], s) : mfma_bf16_32(part(0, g), q.lo[g], s);
    s = mfma_bf16_32(part(1, g), q.mid[g], s);
  }
  again();
#pragma unroll
  for (int g = 0; g < G; ++g) {
    s = SWAP ? mfma_bf16_32(part(0, g), q.mid[g], s) : mfma_bf16_32(part(1, g), q.hi[g], s);
    s = SWAP ? mfma_bf16_32(part(1, g), q.hi[g], s) : mfma_bf16_32(part(0, g), q.mid[g], s);
  }
  again();
#pragma unroll
  for (int g = 0; g < G; ++g) s = mfma_bf16_32(part(0, g), q.hi[g], s);
  return s;
}

// Four fp32 values as hi, mid, lo at p, p + D, p + 2 D.
template <int D>
__device__ __forceinline__ void store_parts3(bf16* p, f32x4 x) {
  uint2 hi, mid, lo;
  split3_dot(x[0], x[1], hi.x, mid.x, lo.x);
  split3_dot(x[2], x[3], hi.y, mid.y, lo.y);
  *reinterpret_cast<uint2*>(p) = hi;
  *reinterpret_cast<uint2*>(p + D) = mid;
  *reinterpret_cast<uint2*>(p + 2 * D) = lo;
}

// X^T operand (A) of a 32x32x16 product over 16 row-major staged rows of LD
// halves: slot 8 (l / 32) + e of lane l is row 4 (l / 32) + e (e < 4) or
// 8 + 4 (l / 32) + e - 4, the order in which a lane holds half a tile's
// elements. piece: the lane's 8 bytes of row 4 (l / 32) + (l % 16) / 4, at
// columns 4 (l % 4) of the 16 that lanes (l / 16) % 2 take; the transposing read
// hands each 16-lane group the columns of its 4 x 16 block.
template <int LD>
__device__ __forceinline__ uint4 load_t(const bf16* piece) {
  using lds_t = __attribute__((address_space(3))) i16x4_t;
  i16x4_t w[2] = {__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t*)piece),
                  __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t*)(piece + 8 * LD))};
  return __builtin_bit_cast(uint4, w);
}

}  // namespace tarmac
