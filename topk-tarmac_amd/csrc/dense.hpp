// The block loop of dense_kernel (dense.hip): scores, self and chunk-end masks,
// exponents, row sums and the P.V product over one staged key chunk, for
// operands in their own type (fp32 or bf16 MFMA). The split-operand kernel
// (dense_split.hip) takes its constants and query_max4 from here.
#pragma once

#include "frag.hpp"
#include "select.hpp"
#include "tarmac_internal.hpp"

namespace tarmac {

constexpr float kLog2e = 1.4426950408889634f;
constexpr int kDenseBlockTiles = 4;  // 64 keys per score block
constexpr int kDenseQueryTiles = 2;  // 16-query tiles per wavefront

template <typename T, int D>
struct PvOperand;

// fp32: O^T block h (channels 16h..16h+15) += V^T(16 x 4 keys) * P^T(4 keys x 16 q),
// four steps per 16-key tile. The V^T fragment of a (tile, h) is read once
// and used by every query tile.
template <int D>
struct PvOperand<float, D> {
  static constexpr int NH = (D + 15) / 16;  // output blocks of 16 channels
  static constexpr int CP = NH * 16;        // padded channel count in LDS
  static constexpr int TILES = 1;           // 16-key tiles per step
  template <int QT>
  __device__ __forceinline__ static void pv_step(f32x4 (&acc)[QT][NH], const float* Vt, int ldv,
                                                 int kb, int lane, const float (&p)[QT][TILES][4]) {
    const int col = lane & 15, grp = lane >> 4;
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      const f32x4 vv = *reinterpret_cast<const f32x4*>(Vt + (16 * h + col) * ldv + kb + 4 * grp);
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) acc[qt][h] = mfma_f32_16x16x4(vv[u], p[qt][0][u], acc[qt][h]);
    }
  }
};

// Four probabilities as bf16 (round to nearest even, the rounding of
// Tensor.to(torch.bfloat16)), two hardware conversions.
__device__ __forceinline__ bf16x8 pack_p_pair(const float (&a)[4], const float (&b)[4]) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    bf16x2_t lo = {static_cast<__bf16>(a[2 * i]), static_cast<__bf16>(a[2 * i + 1])};
    bf16x2_t hi = {static_cast<__bf16>(b[2 * i]), static_cast<__bf16>(b[2 * i + 1])};
    w[i] = __builtin_bit_cast(uint32_t, lo);
    w[2 + i] = __builtin_bit_cast(uint32_t, hi);
  }
  return __builtin_bit_cast(bf16x8, w);
}

// bf16: one 16x16x32 MFMA per output block and pair of 16-key tiles. The
// contraction index j = 8 (l/16) + e of lane l maps to key 4 (l/16) + e of the
// first tile (e < 4) and of the second (e >= 4): the B operand is the lane's
// own eight probabilities, the A operand two 8-byte V^T reads.
template <int D>
struct PvOperand<bf16, D> {
  static constexpr int NH = D / 16;
  static constexpr int CP = NH * 16;
  static constexpr int TILES = 2;  // 16-key tiles per step
  // pb: each query tile's eight probabilities, packed (pack_p_pair)
  template <int QT>
  __device__ __forceinline__ static void pv_step_packed(f32x4 (&acc)[QT][NH], const bf16* Vt,
                                                        int ldv, int kb, int lane,
                                                        const bf16x8 (&pb)[QT]) {
    const int col = lane & 15, grp = lane >> 4;
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      const bf16* r = Vt + (16 * h + col) * ldv + kb + 4 * grp;
      uint2 w[2] = {*reinterpret_cast<const uint2*>(r), *reinterpret_cast<const uint2*>(r + 16)};
      const bf16x8 vv = __builtin_bit_cast(bf16x8, w);
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) acc[qt][h] = mfma_bf16_16x16x32(vv, pb[qt], acc[qt][h]);
    }
  }
};

// Row sum of eight bf16 probabilities (the PV operand) into an fp32 sum: four
// v_dot2 against (1, 1). The softmax then normalises by the sum of exactly
// the weights the PV product uses.
__device__ __forceinline__ float sum_bf16x8(bf16x8 p, float acc) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  const uint4 w = __builtin_bit_cast(uint4, p);
  const bf16x2_t one = {static_cast<__bf16>(1.f), static_cast<__bf16>(1.f)};
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w.x), one, acc, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w.y), one, acc, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w.z), one, acc, false);
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w.w), one, acc, false);
}

// Maximum over the four lanes of a query (lanes l, l + 16, l + 32, l + 48):
// two row swaps, VALU only.
__device__ __forceinline__ float query_max4(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = max_plain(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return max_plain(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// Softmax terms are 2^(c s - off). Where the whole row is staged at once
// (one key chunk), off is fixed per query before the first block:
// off = c |q| max_j |k_j| >= c s for every key (Cauchy-Schwarz), so no term
// exceeds 1 and a block needs no maximum. The bound can sit far above the
// row's true maximum; terms then shrink by 2^-(gap) and the query's sum shows
// it: a sum below 2^-64 (a gap of more than 64 - log2 N) makes the wave run
// the row again with the running maximum below, the path every multi-chunk
// row takes. With the sum at or above 2^-64 the largest term is at least
// 2^-74 (N <= 1024 keys in one chunk), so only terms below 2^-52 of it can
// leave the fp32 (and bf16) normal range.
// The running maximum of c s is only raised when a block's maximum exceeds it
// by more than 2^kDenseLag: terms then stay below 2^kDenseLag (no overflow,
// no loss of precision in fp32), and after the first block a raise -- a
// rescale of the query's sum and accumulator -- is rare.
constexpr float kDenseLag = 8.f;
constexpr float kDenseTinySum = 0x1p-64f;

// All-ones bf16 A operand (0x3f80 = 1.0).
constexpr bf16x8 kOnesBf16x8 = {1.0, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0, 1.0};

// The query's softmax sum: fp32 lanes hold a quarter each (element 0), bf16
// lanes the whole sum (every element).
template <typename T>
__device__ __forceinline__ float row_total(f32x4 l) {
  if constexpr (sizeof(T) == 2) return l[0];
  float t = l[0] + __shfl_xor(l[0], 16);
  return t + __shfl_xor(t, 32);
}

// Fixed-offset exponents (fp32) of QT query tiles against BT key tiles: the
// fragments hold c q, and every MFMA chain starts at -off, so the product
// returns c s - off itself -- no VALU between the product and exp2. (bf16
// would need c q as a bf16 pair, twice the products: measured slower than the
// fma it saves.)
template <typename F, int QT, int BT, typename T>
__device__ __forceinline__ void block_exponents(const F (&frag)[QT], const T* Ks, int kb, int lane,
                                                const float (&neg)[QT], f32x4 (&s)[QT][BT]) {
  const int col = lane & 15, grp = lane >> 4;
  typename F::KF kf[BT];
#pragma unroll
  for (int t = 0; t < BT; ++t) kf[t] = F::load_k(Ks + (kb + 16 * t + col) * F::LDK, grp);
#pragma unroll
  for (int qt = 0; qt < QT; ++qt)
#pragma unroll
    for (int t = 0; t < BT; ++t) s[qt][t] = f32x4{neg[qt], neg[qt], neg[qt], neg[qt]};
#pragma unroll
  for (int i = 0; i < F::NI; ++i)
#pragma unroll
    for (int t = 0; t < BT; ++t)
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) s[qt][t] = frag[qt].step(kf[t], i, s[qt][t]);
}

// The block loop over one staged chunk (rows [0, cnp) of Ks / Vt, keys
// c0 + row): scores, the self and chunk-end masks, exponents, row sums and
// the P.V product. ONLINE: off follows the running maximum; otherwise off
// is the fixed per-query bound.
template <bool ONLINE, typename T, int D, int QT>
__device__ __forceinline__ void dense_blocks(const Frag<T, D> (&frag)[QT], const T* Ks, const T* Vt,
                                             int ldv, int c0, int cn, int cnp, int q0,
                                             const bool (&self_r)[4], int lane, int grp, float post,
                                             f32x4 (&acc)[QT][PvOperand<T, D>::NH],
                                             float (&off)[QT], f32x4 (&l_run)[QT]) {
  using F = Frag<T, D>;
  using PV = PvOperand<T, D>;
  constexpr int LDK = F::LDK;
  constexpr int NH = PV::NH;
  constexpr int BT = kDenseBlockTiles;
  constexpr int BK = 16 * BT;
  const int kend = c0 + cn;  // rows past the chunk end are zero padding
  float neg[QT];             // the exponent's offset
  if constexpr (!ONLINE) {
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) neg[qt] = -off[qt];
  }
  for (int kb0 = 0; kb0 < cnp; kb0 += BK) {
    f32x4 s[QT][BT];
    constexpr bool FOLDED = !ONLINE && sizeof(T) == 4;  // s is already c s - off
    if constexpr (FOLDED) block_exponents<F, QT, BT>(frag, Ks, kb0, lane, neg, s);
    else block_scores<F, QT, BT>(frag, Ks, kb0, LDK, lane, s);
    const int kabs = c0 + kb0;
    // the self pair (one select per element of a diagonal tile, on the
    // loop-invariant lane predicates) and keys past the chunk end
    mask_block<QT, BT>(s, self_r, q0, kabs, kend, grp, -INFINITY);
    if constexpr (ONLINE) {
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        float mloc = -INFINITY;
#pragma unroll
        for (int t = 0; t < BT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) mloc = fmaxf(mloc, s[qt][t][r]);
        const float m_blk = query_max4(mloc) * post;
        if (m_blk > off[qt] + kDenseLag) {  // rare after the first block
          const float alpha = fast_exp2(off[qt] - m_blk);  // 0 while nothing has been seen
          l_run[qt] *= alpha;
#pragma unroll
          for (int h = 0; h < NH; ++h) acc[qt][h] *= alpha;
          off[qt] = m_blk;
        }
        neg[qt] = off[qt] == -INFINITY ? 0.f : -off[qt];  // a block of masked keys only
      }
    }
    constexpr int TS = PV::TILES;
    static_assert(BT % TS == 0, "whole PV steps per block");
#pragma unroll
    for (int t0 = 0; t0 < BT; t0 += TS) {
      float p[QT][TS][4];
#pragma unroll
      for (int qt = 0; qt < QT; ++qt)
#pragma unroll
        for (int t = 0; t < TS; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            p[qt][t][r] = FOLDED ? fast_exp2(s[qt][t0 + t][r])
                                 : fast_exp2(fmaf(s[qt][t0 + t][r], post, neg[qt]));
      if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
#pragma unroll
          for (int t = 0; t < TS; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) l_run[qt][0] += p[qt][t][r];
        PV::template pv_step<QT>(acc, Vt, ldv, kb0 + 16 * t0, lane, p);
      } else {
        bf16x8 pb[QT];
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
          pb[qt] = pack_p_pair(p[qt][0], p[qt][1]);
          // the row sum on the matrix core: an all-ones A operand adds the
          // step's 32 weights of the query into every output element
          l_run[qt] = mfma_bf16_16x16x32(kOnesBf16x8, pb[qt], l_run[qt]);
        }
        PV::template pv_step_packed<QT>(acc, Vt, ldv, kb0 + 16 * t0, lane, pb);
      }
    }
  }
}

// A fixed-offset row whose softmax sum is below 2^-64 (the bound sat too far
// above its maximum), above 2N (each term is at most 1) or not a number must
// run again with the online softmax.
template <typename T, int QT>
__device__ __forceinline__ bool sum_out_of_range(const f32x4 (&l_run)[QT], int N) {
  bool out = false;
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const float l_tot = row_total<T>(l_run[qt]);
    out |= !(l_tot >= kDenseTinySum && l_tot <= 2.f * static_cast<float>(N));
  }
  return out;
}

}  // namespace tarmac
