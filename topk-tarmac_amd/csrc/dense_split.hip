// Dense attention in fp32 on 16-bit matrix instructions (d = 16, 32, 64),
// every fp32 operand split into parts, sums in fp32.
//
// Why: the fp32 MFMA runs at 64 FLOP a cycle and SIMD and blocks the VALU
// meanwhile; the bf16 / fp16 one at 1024, and its 32 x 32 form beside the
// VALU (24 half-rate VALU operations and one 32x32x16: 46 ns against 43 for
// the VALU alone and 14 for the MFMA; two 16x16x32 in its place: 53).
//
//   S^T = K Q^T      K and q in three bf16 parts (24 significand bits, fp32's
//       exponent range): the six products of 2^-16 or more.
//   O^T += V^T P^T   V and P in two fp16 parts (22 bits): all products at
//       d = 16, where one 32-row operand holds V's hi and lo parts, three of
//       four above. Three bf16 parts of each (24 bits, no range to see to) cost
//       21% at d = 16 and gave the same error. V is scaled by a power of two that
//       puts the row's largest magnitude below 2^15; P = 2^(c s - off) is kept
//       below 2^15 with a sum of 2^4 or more. Both lo parts are scaled by 2^11
//       more, and the products with one of them are summed apart: without that,
//       weights of 2^-20 of the largest were off by 4e-4 of themselves, which a
//       channel that only they feed shows (now 1e-6, fp32 MFMA 3e-6), for 5% more
//       time at d = 16 (B=1024 N=256 30.9 -> 32.5 us; d = 32 and 64 unchanged).
//   Error against 64 bits, N(0, 1) inputs, N = 256: 1.8, 1.9, 2.0e-7 at d = 16,
//   32, 64 (fp32 MFMA: 6.1, 10.2, 4.0e-7); logsumexp 3e-8 off on average (5e-8).
//   The A operand V^T comes from row-major rows by the transposing LDS read.
//
// Exponents: off is fixed per query before the first block, the maximum over
// the row's first 32 keys less 5. A block whose terms add up to 2^15 or more
// raises off first, which scales by a power of two (rare: 7 nats above the first
// keys); one whose terms overflow (85 nats above) raises it by 120 and is formed
// again, up to eight times. With q 32 and 64 times N(0, 1), where many waves meet
// that, B=1024 N=256 d=16 takes 36 and 40 us (84 and 114 when such waves went to
// the rerun), d=64 107 and 118 (284 and 589). Score chains start at 0 and off is
// subtracted after: a chain that starts at off is cut at off's magnitude in every
// product, which the backward sees at scores of 2^5 and more.
//
// The result decides whether the parts kept what fp32 keeps: P and scaled V are
// held to 2^-36 below 2^-14. A query whose sum is out of range, whose values are
// not finite, whose largest channel is small beside what such rounding adds up
// to, or that has a channel of the size of the smallest parts in a row that
// holds such elements, runs again on fp32 MFMA with a running maximum, from
// global memory (B=1024 N=256: the queries of one batch row of 1024 add 18, 48,
// 72 us at d = 16, 32, 64, those of all take 114, 214, 578; N(0, 1) inputs, also
// with q 8 times as large and half the values 64 times, meet none).
//
// Loads: a workgroup's items (query blocks) and their key chunks form one
// stream. The next chunk's K and V are loaded into registers while the current
// one is computed on.
//
// Measured against the fp32 MFMA kernel (us): B=1024 N=256 d=16 45.0 -> 32.5,
// d=32 85.5 -> 47.7, d=64 153 -> 103; B=256 N=1024 d=16 166 -> 102; B=36 N=1000
// d=64 152 -> 81. About 115 VALU and 10 MFMA per 32 x 32 tile and wave at d = 16,
// 36 MFMA at d = 64. Bound by issue at d = 16 and 32 (B=1024 N=256: VALU 22.9 and
// MFMA 10.1 of 33.4 us traced, 29.0 and 19.3 of 50.4), at d = 64 (37.9 and 36.6 of
// 113) also by LDS latency at two waves a SIMD. At d = 32 with two vectors a thread 8 lane addresses, each
// written once and read back once a chunk, do not fit the 128 registers of four
// waves a SIMD and stay in scratch; the tile loops use none.
#include <algorithm>

#include "dense.hpp"
#include "parts.hpp"

namespace tarmac {

constexpr float kSplitWindow = 5.f;      // log2 of the first tile's largest term
constexpr float kSplitBlockMax = 0x1p15f;
constexpr int kSplitAgain = 8;            // times a tile is formed again; then the rerun decides

template <int D>
struct DenseSplit {
  static constexpr int NB = D > 32 ? D / 32 : 1;  // 32-row blocks of O^T
  static constexpr int LDK = 3 * D + 8;     // halves per staged K row: hi, mid, lo
  static constexpr int LDV = 2 * D + 8;     // halves per staged V row: hi, lo
  static constexpr int VPR = D / 4;         // 16-byte vectors per fp32 row
  static constexpr int KC = 2048 / D;       // most keys per chunk
  static constexpr size_t lds_bytes(int kc) {
    return static_cast<size_t>(kc) * (LDK + LDV) * 2 + 16;
  }
};

// The rerun: 16 queries of a wave on fp32 MFMA, K and V^T fragments straight
// from global memory, the running maximum raised per 16-key tile; writes the
// outputs of the queries whose bit of want is set.
template <int D>
__device__ __forceinline__ void dense_online_global(const float* __restrict__ Qb,
                                                    const float* __restrict__ Kb,
                                                    const float* __restrict__ Vb,
                                                    float* __restrict__ Ob, float* lse, int N,
                                                    int q0, int lane, float c,
                                                    uint32_t want) {
  using F = Frag<float, D>;
  constexpr int NH = D / 16;
  const int col = lane & 15, grp = lane >> 4, qi = q0 + col;
  F frag;
  frag.load_q(Qb + static_cast<size_t>(min(qi, N - 1)) * D, grp, c);
  f32x4 acc[NH];
#pragma unroll
  for (int h = 0; h < NH; ++h) acc[h] = f32x4{0.f, 0.f, 0.f, 0.f};
  float off = -INFINITY, l = 0.f;
#pragma unroll 1
  for (int k0 = 0; k0 < N; k0 += 16) {
    const typename F::KF kf = F::load_k(Kb + static_cast<size_t>(min(k0 + col, N - 1)) * D, grp);
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < F::NI; ++i) s = frag.step(kf, i, s);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int key = k0 + 4 * grp + r;
      if (key >= N || key == qi) s[r] = -INFINITY;
    }
    const float m = query_max4(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])));
    if (m > off + kDenseLag) {
      const float alpha = fast_exp2(off - m);
      l *= alpha;
#pragma unroll
      for (int h = 0; h < NH; ++h) acc[h] *= alpha;
      off = m;
    }
    const float neg = off == -INFINITY ? 0.f : -off;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s[r] = fast_exp2(s[r] + neg);
      l += s[r];
    }
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int row = k0 + 4 * grp + u;
        const float x = row < N ? Vb[static_cast<size_t>(row) * D + 16 * h + col] : 0.f;
        acc[h] = mfma_f32_16x16x4(x, s[u], acc[h]);
      }
  }
  l = add_xor32(add_xor16(l));
  if (qi >= N || (want >> col & 1u) == 0u) return;
  if (lse != nullptr && grp == 0) lse[qi] = off + log2f(l);
  const float inv = __builtin_amdgcn_rcpf(l);
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    float o[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = acc[h][r] * inv;
    st_f32<4>(Ob + static_cast<size_t>(qi) * D + 16 * h + 4 * grp, o);
  }
}

// U: 16-byte vectors of K, and of V, per thread and chunk.
template <int D, int U>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(D == 64 ? 2 : 4)))
dense_split_kernel(const float* __restrict__ Q, const float* __restrict__ Kx,
                   const float* __restrict__ V, float* __restrict__ O, float* __restrict__ lse,
                   int N, int n_qblk, int kc, float scale, int nblocks) {
  using DS = DenseSplit<D>;
  constexpr int NB = DS::NB, LDK = DS::LDK, LDV = DS::LDV, VPR = DS::VPR;
  constexpr bool STACKED = D == 16;  // hi and lo rows of V^T in one operand
  extern __shared__ __align__(16) unsigned char smem_raw[];
  bf16* const Ks = reinterpret_cast<bf16*>(smem_raw);
  bf16* const Vs = Ks + static_cast<size_t>(kc) * LDK;
  // per parity of the item: the row's largest |v| (bits), and whether some
  // element is too small beside it for two parts
  uint32_t* const vmax = reinterpret_cast<uint32_t*>(Vs + static_cast<size_t>(kc) * LDV);
  uint32_t* const tiny = vmax + 2;

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = blockDim.x >> 6, bd = blockDim.x;
  const int col = lane & 31, half = lane >> 5;
  const int self = col - 4 * half;  // tile_row of the self pair in a diagonal tile
  const bf16* const Kl = Ks + col * LDK + 8 * half;
  // this lane's 8-byte piece of the transposing reads: row 4 half + (l % 16) / 4
  const bf16* const Vl = Vs + (4 * half + ((lane & 15) >> 2)) * LDV +
                         ((lane >> 4) & 1) * (STACKED ? D : 16) + 4 * (lane & 3);

  f32x4 xk[U], xv[U];  // the next chunk's vectors of this thread
  auto load_chunk = [&](int b, int c0) {
    // uniform bases, so a thread's address is a 32-bit offset
    const size_t base = uniform_offset((static_cast<size_t>(b) * N + c0) * D);
    const char* const Kb = reinterpret_cast<const char*>(Kx + base);
    const char* const Vb = reinterpret_cast<const char*>(V + base);
    const int avail = min(kc, N - c0) * VPR;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int v = threadIdx.x + u * bd;
      xk[u] = xv[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (v < avail) {
        xk[u] = *reinterpret_cast<const f32x4*>(Kb + static_cast<uint32_t>(v) * 16u);
        xv[u] = *reinterpret_cast<const f32x4*>(Vb + static_cast<uint32_t>(v) * 16u);
      }
    }
  };
  // item numbers are uniform; kept in SGPRs, so row bases are too
  const int grid = gridDim.x;
  int blk = __builtin_amdgcn_readfirstlane(xcd_logical_block(blockIdx.x, grid));
  if (blk >= nblocks) return;
  load_chunk(blk / n_qblk, 0);
  if (threadIdx.x < 4) vmax[threadIdx.x] = 0u;
  lds_barrier();
  for (int par = 0; blk < nblocks; blk = __builtin_amdgcn_readfirstlane(blk + grid), par ^= 1) {
    const int b = __builtin_amdgcn_readfirstlane(blk / n_qblk), qblk = blk - b * n_qblk;
    const int q0 = __builtin_amdgcn_readfirstlane((qblk * nw + wave) * 32);
    const size_t boff = uniform_offset(static_cast<size_t>(b) * N * D);
    // opaque copies of the lane number, here and after the loops: addresses
    // formed from them are not kept in registers across the loops
    int pl = lane;
    asm volatile("" : "+v"(pl));
    RowParts<D> q;
    q.load(Q + boff + static_cast<size_t>(min(q0 + (pl & 31), N - 1)) * D, pl >> 5, scale * kLog2e);
    // acc: V^T P of the hi parts; accl, scaled by 2^11: hi by lo and lo by hi.
    // Stacked: acc's elements 8..15 are V's lo by P's hi, accl's are lo by lo.
    f32x16 acc[NB], accl[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) acc[n] = accl[n] = f32x16{};
    float off = 0.f, l = 0.f, vs = 0.f;  // vs: the scale of V so far (0: none yet)
    int again = kSplitAgain;
    for (int c0 = 0; c0 < N; c0 += kc) {
      const int cn = min(kc, N - c0), kend = c0 + cn;
      // V's largest magnitude so far in the row
      float mx = 0.f;
#pragma unroll
      for (int u = 0; u < U; ++u)
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(xv[u][0]), fabsf(xv[u][1])),
                             fmaxf(fabsf(xv[u][2]), fabsf(xv[u][3]))));
      mx = row16_reduce(mx, [](float a, float y) { return fmaxf(a, y); });
      mx = query_max4(mx);
      if (lane == 0) atomicMax(vmax + par, __float_as_uint(mx));
      lds_barrier();  // also: the last chunk has been computed on
      const uint32_t ef = max(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(vmax[par])) >> 23, 27u);
      const float vs_new = __uint_as_float((268u - ef) << 23);  // 2^(14 - exponent)
      if (c0 == 0 && threadIdx.x == 0) vmax[par ^ 1] = tiny[par ^ 1] = 0u;
      uint32_t low = 0xffffffffu;  // the smallest nonzero |v|, scaled, less one ulp
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int v = threadIdx.x + u * bd, row = v / VPR, cv = v - row * VPR;
        if (row < kc) {
          store_parts3<D>(Ks + row * LDK + 4 * cv, xk[u]);
          f16x2 vh[2], vl[2];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float x = xv[u][e] * vs_new;
            low = min(low, (__float_as_uint(x) & 0x7fffffffu) - 1u);
            vh[e / 2][e % 2] = static_cast<_Float16>(x);
            vl[e / 2][e % 2] =
                static_cast<_Float16>((x - static_cast<float>(vh[e / 2][e % 2])) * kLoScale);
          }
          bf16* vd = Vs + row * LDV + 4 * cv;
          *reinterpret_cast<uint2*>(vd) = __builtin_bit_cast(uint2, vh);
          *reinterpret_cast<uint2*>(vd + D) = __builtin_bit_cast(uint2, vl);
        }
      }
      if (__any(low < 0x38800000u - 1u) && lane == 0) tiny[par] = 1u;  // below 2^-14
      if (kend < N) load_chunk(b, kend);
      else if (blk + grid < nblocks) load_chunk(__builtin_amdgcn_readfirstlane((blk + grid) / n_qblk), 0);
      lds_barrier();
      if (q0 < N) {
        if (vs != vs_new) {  // uniform: the first chunk, or one with a larger |v|
          const float r = vs == 0.f ? 0.f : vs_new * __uint_as_float((254u << 23) - __float_as_uint(vs));
          vs = vs_new;
#pragma unroll
          for (int n = 0; n < NB; ++n) {
            acc[n] *= r;
            accl[n] *= r;
          }
        }
        for (int kb = 0; kb < cn; kb += 32) {
          f32x16 s = tile_dot<D>(q, Kl + kb * LDK, f32x16{});
          const int kabs = c0 + kb;
          if (kabs == q0) {  // the diagonal tile
#pragma unroll
            for (int i = 0; i < 16; ++i)
              if (tile_row(i) == self) s[i] = -INFINITY;
          }
          if (kabs + 32 > kend) {
#pragma unroll
            for (int i = 0; i < 16; ++i)
              if (tile_row(i) >= kend - kabs - 4 * half) s[i] = -INFINITY;
          }
          if (kabs == 0) {  // the first tile: off from its maximum
            float m = -INFINITY;
#pragma unroll
            for (int i = 0; i < 16; ++i) m = fmaxf(m, s[i]);
            m = max_xor32(m);
            off = m == -INFINITY ? 0.f : m - kSplitWindow;
          }
          float e[16], lb = 0.f;
#pragma unroll
          for (int i = 0; i < 16; ++i) e[i] = fast_exp2(s[i] - off);
#pragma unroll
          for (int i = 0; i < 16; ++i) lb += e[i];
          if (__any(!(lb < kSplitBlockMax))) {  // rare: raise off where the sum is out of range
            // to a sum of 2^9 to 2^10 (a term of 2^5 or more); by 120 where it
            // overflows, and then the tile is formed again
            const uint32_t mb = __float_as_uint(max_xor32(lb)), em = mb >> 23;
            const bool over = mb == 0x7f800000u;
            const uint32_t x = over ? 120u : em >= 142u && em < 255u ? em - 136u : 0u;
            const float r = __uint_as_float((127u - x) << 23);
            off += static_cast<float>(x);
            l *= r;
#pragma unroll
            for (int n = 0; n < NB; ++n) {
              acc[n] *= r;
              accl[n] *= r;
            }
            if (__any(over) && again > 0) {
              --again;
              kb -= 32;
              continue;
            }
            lb *= r;
#pragma unroll
            for (int i = 0; i < 16; ++i) e[i] *= r;
          }
          l += lb;
          again = kSplitAgain;
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            uint32_t ph[4], pl[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) split2_pair(e[8 * t + 2 * i], e[8 * t + 2 * i + 1], ph[i], pl[i]);
            const f16x8 p_hi = __builtin_bit_cast(f16x8, ph), p_lo = __builtin_bit_cast(f16x8, pl);
            const bf16* vp = Vl + (kb + 16 * t) * LDV;
#pragma unroll
            for (int n = 0; n < NB; ++n) {
              const f16x8 vh = __builtin_bit_cast(f16x8, load_t<LDV>(vp + 32 * n));
              accl[n] = mfma_f16_32(vh, p_lo, accl[n]);
              acc[n] = mfma_f16_32(vh, p_hi, acc[n]);
              if constexpr (!STACKED)
                accl[n] = mfma_f16_32(__builtin_bit_cast(f16x8, load_t<LDV>(vp + D + 32 * n)), p_hi, accl[n]);
            }
          }
        }
      }
    }
    if (q0 < N) {
      l = add_xor32(l);
      float a = 0.f, big = 0.f, small = INFINITY;
#pragma unroll
      for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int i = 0; i < (STACKED ? 8 : 16); ++i) {
          float lo = accl[n][i];
          if constexpr (STACKED) lo += fmaf(accl[n][i + 8], 1.f / kLoScale, acc[n][i + 8]);
          acc[n][i] = fmaf(lo, 1.f / kLoScale, acc[n][i]);
          a = fmaf(0.f, acc[n][i], a);
          big = fmaxf(big, fabsf(acc[n][i]));
          small = fminf(small, fabsf(acc[n][i]));
        }
      big = max_xor32(big);
      // Whether the parts kept what fp32 keeps: the sum of 2^4 or more; it and
      // every channel finite; the query's largest channel so large that N terms
      // rounded at 2^-36 beside values below 2^15 stay below 2^-20 of it (a
      // wave of sharp rows beside values 2^16 and more times theirs fails
      // this); and, in a row with an element below 2^-14, every channel above
      // 2^-14 of the sum.
      const bool zeros = __builtin_amdgcn_readfirstlane(vmax[par]) == 0u;
      const bool wide = __builtin_amdgcn_readfirstlane(tiny[par]) != 0u;
      const float least = zeros ? 0.f : 0.5f * __builtin_amdgcn_sqrtf(static_cast<float>(N));
      const bool fine = (l >= 16.f) & (fmaf(0.f, l, a) == 0.f) & (big >= least) & (small >= (wide ? l * 0x1p-14f : 0.f));
      int el = lane;
      asm volatile("" : "+v"(el));
      const int ecol = el & 31, ehalf = el >> 5;
      float* const lse_row = lse == nullptr ? nullptr : lse + uniform_offset(static_cast<size_t>(b) * 2 * N);
      const uint64_t bad = __ballot(!fine);
      const uint32_t rerun = static_cast<uint32_t>(bad) | static_cast<uint32_t>(bad >> 32);
      if (q0 + ecol < N && (rerun >> ecol & 1u) == 0u) {
        // log2 of the sum by exponent and mantissa: the logarithm's own error
        // is then at the last place of 1, not of log2 l (10 and more)
        if (lse_row != nullptr && ehalf == 0)
          lse_row[q0 + ecol] = (off + static_cast<float>(__builtin_amdgcn_frexp_expf(l))) +
                              log2f(__builtin_amdgcn_frexp_mantf(l));
        // 1 / vs is a power of two
        const float inv = __builtin_amdgcn_rcpf(l) * __uint_as_float((254u << 23) - __float_as_uint(vs));
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
          for (int i = 0; i < (STACKED ? 8 : 16); i += 4) {
            float w[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) w[r] = acc[n][i + r] * inv;
            st_f32<4>(O + boff + static_cast<size_t>(q0 + ecol) * D + 32 * n + 2 * i + 4 * ehalf, w);
          }
      }
      if (rerun != 0u) {
#pragma unroll 1
        for (int t = 0; t < 2; ++t)
          if (q0 + 16 * t < N && (rerun >> 16 * t & 0xffffu) != 0u)
            dense_online_global<D>(Q + boff, Kx + boff, V + boff, O + boff, lse_row, N, q0 + 16 * t,
                                   el, scale * kLog2e, rerun >> 16 * t);
      }
    }
  }
}

template <int D, int U>
static hipError_t launch_dense_split_u(const DenseArgs& a, int nw, int n_qblk) {
  using DS = DenseSplit<D>;
  // equal chunks of what the threads can hold, at most KC keys
  int kc = std::min(DS::KC, U * 64 * nw / DS::VPR / 32 * 32);
  if (kc < 32) return hipErrorInvalidValue;  // fewer threads than a 32-key block takes
  const int nch = (a.N + kc - 1) / kc;
  kc = std::min(kc, ((a.N + nch - 1) / nch + 31) / 32 * 32);
  const int nblocks = a.B * n_qblk;
  // workgroups stay for as many items as it takes: sixteen waves per CU
  const int grid = std::min(nblocks, kCUs * (16 / nw));
  hipLaunchKernelGGL((dense_split_kernel<D, U>), dim3(grid), dim3(64 * nw), DS::lds_bytes(kc),
                     static_cast<hipStream_t>(a.stream), static_cast<const float*>(a.q),
                     static_cast<const float*>(a.k), static_cast<const float*>(a.v),
                     static_cast<float*>(a.out), a.stats, a.N, n_qblk, kc, a.scale, nblocks);
  return hipGetLastError();
}

template <int D>
static hipError_t launch_dense_split(const DenseArgs& a) {
  const int waves = (a.N + 31) / 32;
  int nw = 8;
  while (nw > 4 && a.B * ((waves + nw - 1) / nw) < 2 * kCUs) nw /= 2;  // more CUs at work
  const int n_qblk = (waves + nw - 1) / nw;
  nw = (waves + n_qblk - 1) / n_qblk;
  // d = 64: two vectors a thread of fewer than four waves are less than a 32-key
  // block. Rows of three waves have a fourth that only stages (B=400 N=96: 15.8
  // -> 14.2 us against four vectors a thread of three), rows of one or two take
  // four vectors (B=1024 N=40: 14.5 against 19.1 with idle waves).
  if constexpr (D == 64) {
    if (nw < 3) return launch_dense_split_u<D, 4>(a, nw, n_qblk);
    nw = std::max(nw, 4);
  }
  return nw == 8 ? launch_dense_split_u<D, 1>(a, nw, n_qblk) : launch_dense_split_u<D, 2>(a, nw, n_qblk);
}

hipError_t run_dense_split(const DenseArgs& a) {
  switch (a.d) {
    case 16: return launch_dense_split<16>(a);
    case 32: return launch_dense_split<32>(a);
    case 64: return launch_dense_split<64>(a);
  }
  return hipErrorInvalidValue;
}

}  // namespace tarmac
