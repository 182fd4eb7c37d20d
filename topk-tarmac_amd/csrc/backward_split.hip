// Dense backward in fp32 on bf16 matrix instructions (d = 16, 32, 64): the two
// passes of backward.hip with every operand in three bf16 parts.
//
// Why: the seven products of the two passes are what the fp32 MFMA kernels
// spend their time on (at d = 16, N = 256: 100 of 175 us, and nothing runs
// beside an fp32 MFMA). Six bf16 products of parts take 6/16 of the time, with
// the VALU at work beside them; parts keep 24 bits and fp32's exponent range,
// so gradients of any scale need no normalisation. dS and P are split as they
// come out of the exponent; K, V, Q and dO when staged. The transposed operands
// (K^T, Q^T, dO^T) are read from the same staged rows by the transposing LDS
// read, where the fp32 kernels keep a second, transposed copy.
//
//   pass 1, a wave per 32 queries (lane: query l % 32), keys streamed:
//     S^T = K q, dP^T = V g, dS^T = 2^(S - lse) (dP - D), dQ^T += K^T dS^T.
//   pass 2, a wave per 32 keys (lane: key l % 32), queries streamed: the same
//     tiles with rows and columns exchanged (lse and D come from LDS);
//     dV^T += dO^T P, dK^T += Q^T dS.
//
// A column with an output that is not finite, or nonzero and below 2^-80 (parts
// of its terms may have left their range), runs again on fp32 MFMA from global
// memory (B=1024 N=256, every column: 424, 789, 1516 us at d = 16, 32, 64; keys
// that no one attends to have such gradients where q is 32 times N(0, 1): 145 us
// at d = 16). Both passes scale the queries and keep the products' order, so
// they form the bits of the forward's scores and their rounding drops out of
// s - lse: with pass 2 scaling its keys, dk and dv were 1.4 to 1.6 times as far
// off as dq with q 16 times N(0, 1) (now 1.0 and 0.9). One barrier a chunk: the
// next chunk is loaded into registers while the current one is computed on, then
// split into the other LDS buffer.
//
// Measured, both passes, against the fp32 MFMA kernels (us): B=1024 N=256 d=16
// 174 -> 120, d=32 298 -> 194, d=64 741 -> 387; B=256 N=512 d=16 165 -> 109;
// B=300 N=200 d=64 230 -> 113. Per 32 x 32 tile the passes take 20 and 28 MFMA
// of 33 cycles at d = 16 and 72 and 96 at d = 64, 190 and 300 VALU at d = 16. Bound
// by issue at d = 16 (traced 51.1 us, VALU 27.1 and MFMA 20.8; pass 2 73.1, 41.0
// and 28.5), above that (d = 64: 173, 36.1 and 76.1; 219, 47.5 and 102) also by LDS
// latency at two waves a SIMD. Error against 64 bits at d = 16, N = 256: dq, dk,
// dv 3.3, 3.3, 3.2e-7 (fp32 MFMA 4.7, 4.4, 4.1e-7); N = 512 3.5, 3.4, 3.3e-7 (5.7,
// 5.2, 5.1e-7); d = 64, N = 256 4.1, 4.1, 4.0e-7 (5.2, 5.2, 4.9e-7).
//
// Registers: at d = 64 pass 2 keeps 96 for its columns' parts and 64 for two
// accumulators of the 256 that two waves a SIMD leave, and uses no scratch (pass 1
// at d = 16 has one register there, read back once a chunk). What else would live
// across the loops is kept out of it: row offsets are scalars (uniform_offset),
// and lane addresses outside the loops come from opaque copies of the lane number
// (with them in registers it spilled 20 to 68, and both passes took B=300 N=200
// d=64 133 us).
#include <algorithm>

#include "parts.hpp"
#include "tarmac_internal.hpp"

namespace tarmac {

namespace {

template <int D>
struct BwdSplit {
  static constexpr int NB = D > 32 ? D / 32 : 1;  // 32-row blocks of a gradient's transpose
  static constexpr int LD = 3 * D + 8;            // halves per staged row: hi, mid, lo, zeros
  static constexpr int VPR = D / 4;
  static constexpr int KC = 2048 / D;             // most rows per chunk
  static constexpr size_t lds_bytes(int kc) {     // two buffers of two matrices and two scalars a row
    return static_cast<size_t>(kc) * 2 * (2 * LD * 2 + 8);
  }
};

// Half tile t (elements 8 t ..) of w in parts.
__device__ __forceinline__ void split_half(const f32x16& w, int t, bf16x8& hi, bf16x8& mid, bf16x8& lo) {
  uint32_t h[4], m[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) split3_dot(w[8 * t + 2 * i], w[8 * t + 2 * i + 1], h[i], m[i], l[i]);
  hi = __builtin_bit_cast(bf16x8, h);
  mid = __builtin_bit_cast(bf16x8, m);
  lo = __builtin_bit_cast(bf16x8, l);
}

// acc += X^T W over the 32 staged rows at X (the lane's piece) and a tile w: six
// products of parts. d = 16: the 32 operand rows hold two parts, hi over mid for
// three products and lo over zeros for one; the caller adds the halves. A bf16
// MFMA cuts what it adds at the accumulator's last place, so at d <= 32 a tile's
// products go from the smallest up into a sum of their own, which is added to
// acc with rounding (error of dv at d = 16, N = 256: 4.8e-7 without that, 4.1e-7
// on fp32 MFMA); d = 64 has no registers for it and keeps its accuracy without.
template <int D>
__device__ __forceinline__ void mma_parts(f32x16 (&acc)[BwdSplit<D>::NB], const bf16* X, const bf16* Xlo,
                                          const f32x16& w) {
  constexpr int LD = BwdSplit<D>::LD;
  auto t = [](const bf16* p) { return __builtin_bit_cast(bf16x8, load_t<LD>(p)); };
  if constexpr (D <= 32) {
    f32x16 sum = {};
    bf16x8 hi[2], top[2];  // top: hi rows (d = 16: hi over mid)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      bf16x8 mid, lo;
      split_half(w, i, hi[i], mid, lo);
      top[i] = t(X + 16 * i * LD);
      if constexpr (D == 16) {
        sum = mfma_bf16_32(t(Xlo + 16 * i * LD), hi[i], sum);
        sum = mfma_bf16_32(top[i], lo, sum);
        sum = mfma_bf16_32(top[i], mid, sum);
      } else {
        const bf16x8 m = t(X + D + 16 * i * LD), l = t(X + 2 * D + 16 * i * LD);
        sum = mfma_bf16_32(l, hi[i], sum);
        sum = mfma_bf16_32(top[i], lo, sum);
        sum = mfma_bf16_32(m, mid, sum);
        sum = mfma_bf16_32(m, hi[i], sum);
        sum = mfma_bf16_32(top[i], mid, sum);
      }
    }
    sum = mfma_bf16_32(top[0], hi[0], sum);
    sum = mfma_bf16_32(top[1], hi[1], sum);
    acc[0] += sum;
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      bf16x8 hi, mid, lo;
      split_half(w, i, hi, mid, lo);
      const bf16* Xi = X + 16 * i * LD;
#pragma unroll
      for (int n = 0; n < BwdSplit<D>::NB; ++n) {
        const bf16x8 h = t(Xi + 32 * n), m = t(Xi + D + 32 * n), l = t(Xi + 2 * D + 32 * n);
        acc[n] = mfma_bf16_32(l, hi, acc[n]);
        acc[n] = mfma_bf16_32(h, lo, acc[n]);
        acc[n] = mfma_bf16_32(m, mid, acc[n]);
        acc[n] = mfma_bf16_32(m, hi, acc[n]);
        acc[n] = mfma_bf16_32(h, mid, acc[n]);
        acc[n] = mfma_bf16_32(h, hi, acc[n]);
      }
    }
  }
}

// The channels of a gradient row that this lane holds, after the halves of a
// stacked accumulator are added: element i is channel 32 n + tile_row(i) + 4 half.
template <int D>
__device__ __forceinline__ void fold_halves(f32x16 (&acc)[BwdSplit<D>::NB]) {
  if constexpr (D == 16)
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[0][i] += acc[0][i + 8];
}
constexpr int grad_elems(int D) { return D == 16 ? 8 : 16; }

// Whether a lane's part of a result stands: every element finite, and zero or
// of 2^-80 or more. Parts keep a value to 2^-134, so an element loses bits of
// fp32's 24 only below 2^-110 times the sum of the magnitudes beside its small
// factors: 2^30, for instance 1024 rows of values up to 2^20.
constexpr uint32_t kGradTiny = 0x17800000u;  // 2^-80
template <int D>
__device__ __forceinline__ bool grad_stands(const f32x16 (&acc)[BwdSplit<D>::NB]) {
  float nan = 0.f;
  uint32_t low = 0xffffffffu;  // bits of the smallest nonzero magnitude, less one
#pragma unroll
  for (int n = 0; n < BwdSplit<D>::NB; ++n)
#pragma unroll
    for (int i = 0; i < grad_elems(D); ++i) {
      low = min(low, (__float_as_uint(acc[n][i]) & 0x7fffffffu) - 1u);
      nan = fmaf(0.f, acc[n][i], nan);
    }
  return (nan == 0.f) & (low >= kGradTiny - 1u);
}

template <int D>
__device__ __forceinline__ void store_grad(float* row, const f32x16 (&acc)[BwdSplit<D>::NB], int half,
                                           float scale) {
#pragma unroll
  for (int n = 0; n < BwdSplit<D>::NB; ++n)
#pragma unroll
    for (int i = 0; i < grad_elems(D); i += 4) {
      float w[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) w[r] = acc[n][i + r] * scale;
      st_f32<4>(row + 32 * n + 2 * i + 4 * half, w);
    }
}

// The rerun of 16 columns on fp32 MFMA from global memory; those whose bit of
// want is set are stored. Columns are queries
// (PASS2 false: row matrices A = K, B = V; out_a = dQ) or keys (true: A = Q, B =
// dO; out_a = dK, out_b = dV). lse, Dq: per query of the batch row.
template <int D, bool PASS2>
__device__ __forceinline__ void bwd_rerun(const float* __restrict__ colA, const float* __restrict__ colB,
                                          const float* __restrict__ A, const float* __restrict__ Bm,
                                          float lse1, float d1, const float* lse, const float* Dq,
                                          float* __restrict__ out_a, float* __restrict__ out_b, int N,
                                          int x0, int lane, float scale, uint32_t want) {
  using F = Frag<float, D>;
  constexpr int NH = D / 16;
  const int col = lane & 15, grp = lane >> 4, xi = min(x0 + col, N - 1);
  F fa, fb;
  fa.load_q(colA + static_cast<size_t>(xi) * D, grp, PASS2 ? 1.f : scale * kLog2eF);
  fb.load_q(colB + static_cast<size_t>(xi) * D, grp, 1.f);
  f32x4 ga[NH], gb[NH];
#pragma unroll
  for (int h = 0; h < NH; ++h) ga[h] = gb[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int r0 = 0; r0 < N; r0 += 16) {
    const size_t row = static_cast<size_t>(min(r0 + col, N - 1)) * D;
    typename F::KF ka = F::load_k(A + row, grp);
    const typename F::KF kb = F::load_k(Bm + row, grp);
    if constexpr (PASS2)
#pragma unroll
      for (int i = 0; i < F::NI; ++i) ka.v[i] *= scale * kLog2eF;
    f32x4 s = {0.f, 0.f, 0.f, 0.f}, dp = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < F::NI; ++i) {
      s = fa.step(ka, i, s);
      dp = fb.step(kb, i, dp);
    }
    f32x4 p, ds;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int y = r0 + 4 * grp + r, yi = min(y, N - 1);
      const bool in = y < N && y != x0 + col;
      p[r] = in ? fast_exp2(s[r] - (PASS2 ? lse[yi] : lse1)) : 0.f;
      ds[r] = in ? p[r] * (dp[r] - (PASS2 ? Dq[yi] : d1)) : 0.f;
    }
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int y = r0 + 4 * grp + u;
        const float a = y < N ? A[static_cast<size_t>(y) * D + 16 * h + col] : 0.f;
        ga[h] = mfma_f32_16x16x4(a, ds[u], ga[h]);
        if constexpr (PASS2) {
          const float g = y < N ? Bm[static_cast<size_t>(y) * D + 16 * h + col] : 0.f;
          gb[h] = mfma_f32_16x16x4(g, p[u], gb[h]);
        }
      }
  }
  if (x0 + col >= N || (want >> col & 1u) == 0u) return;
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    float w[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) w[r] = ga[h][r] * scale;
    st_f32<4>(out_a + static_cast<size_t>(xi) * D + 16 * h + 4 * grp, w);
    if constexpr (PASS2) {
#pragma unroll
      for (int r = 0; r < 4; ++r) w[r] = gb[h][r];
      st_f32<4>(out_b + static_cast<size_t>(xi) * D + 16 * h + 4 * grp, w);
    }
  }
}

// Both passes. Columns x (a wave's 32) against streamed rows y. PASS2 false:
// colA = Q, colB = dO, A = K, B = V, out_a = dQ; plane 1 of stats is written.
// PASS2 true: colA = K, colB = V, A = Q, B = dO, out_a = dK, out_b = dV.
// U: 16-byte vectors of A, and of B, per thread and chunk.
template <int D, int U, bool PASS2>
__global__ void __launch_bounds__(512) 
    __attribute__((amdgpu_waves_per_eu(D == 16 && !PASS2 && U == 1 ? 4 : 2)))
dense_bwd_split_kernel(const float* __restrict__ colA, const float* __restrict__ colB,
                       const float* __restrict__ A, const float* __restrict__ Bm,
                       const float* __restrict__ O, float* __restrict__ stats,
                       float* __restrict__ out_a, float* __restrict__ out_b, int N, int n_blk, int kc,
                       float scale, int nblocks) {
  using BS = BwdSplit<D>;
  constexpr int NB = BS::NB, LD = BS::LD, VPR = BS::VPR;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  bf16* const lds = reinterpret_cast<bf16*>(smem_raw);
  float* const sc = reinterpret_cast<float*>(lds + static_cast<size_t>(kc) * 4 * LD);  // PASS2: -lse, -D

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = blockDim.x >> 6, bd = blockDim.x;
  const int col = lane & 31, half = lane >> 5, self = col - 4 * half;
  const int row_off = col * LD + 8 * half;
  // this lane's piece of the transposing reads; d = 16: lanes 16-31 and 48-63
  // take the mid part's columns, or the row's zero padding beside lo
  const int piece = (4 * half + ((lane & 15) >> 2)) * LD, upper = (lane >> 4) & 1;
  const int t_off = piece + upper * 16 + 4 * (lane & 3);  // 16 = D: mid; else the block's next columns
  const int tlo_off = piece + (upper ? 3 * D : 2 * D + 4 * (lane & 3));

  // queries are scaled, in either pass, as in the forward: S - lse is then a
  // difference of like roundings (see tile_dot)
  const float c = uniform_value(scale * kLog2eF);
  f32x4 xa[U], xb[U];
  float xs = 0.f, xd = 0.f;
  auto load_chunk = [&](int b, int c0) {
    // uniform bases, so a thread's address is a 32-bit offset
    const size_t base = uniform_offset((static_cast<size_t>(b) * N + c0) * D);
    const char* const Ab = reinterpret_cast<const char*>(A + base);
    const char* const Bb = reinterpret_cast<const char*>(Bm + base);
    const int rows = min(kc, N - c0), avail = rows * VPR;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int v = threadIdx.x + u * bd;
      xa[u] = xb[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (v < avail) {
        xa[u] = *reinterpret_cast<const f32x4*>(Ab + static_cast<uint32_t>(v) * 16u);
        xb[u] = *reinterpret_cast<const f32x4*>(Bb + static_cast<uint32_t>(v) * 16u);
      }
    }
    if constexpr (PASS2) {  // a chunk has at most as many rows as threads
      const float* const lse = stats + uniform_offset(static_cast<size_t>(b) * 2 * N + c0);
      const float* const dsum = lse + N;
      xs = INFINITY;  // rows past the end: p = 0
      xd = 0.f;
      if (static_cast<int>(threadIdx.x) < rows) {
        xs = lse[threadIdx.x];
        xd = dsum[threadIdx.x];
      }
    }
  };
  const int grid = gridDim.x;
  int blk = __builtin_amdgcn_readfirstlane(xcd_logical_block(blockIdx.x, grid));
  if (blk >= nblocks) return;
  load_chunk(blk / n_blk, 0);
  if constexpr (D == 16)  // the zero padding of every row of both buffers
    for (int r = threadIdx.x; r < 4 * kc; r += bd)
      *reinterpret_cast<uint2*>(lds + static_cast<size_t>(r) * LD + 3 * D) = make_uint2(0u, 0u);
  int buf = 0;
  for (; blk < nblocks; blk = __builtin_amdgcn_readfirstlane(blk + grid)) {
    const int b = __builtin_amdgcn_readfirstlane(blk / n_blk), xblk = blk - b * n_blk;
    const int x0 = __builtin_amdgcn_readfirstlane((xblk * nw + wave) * 32);
    const size_t boff = uniform_offset(static_cast<size_t>(b) * N * D);
    float* const st = stats + uniform_offset(static_cast<size_t>(b) * 2 * N);
    // opaque copies of the lane number, here and after the loops: addresses
    // formed from them are not kept in registers across the loops
    int pl = lane;
    asm volatile("" : "+v"(pl));
    const int xi = min(x0 + (pl & 31), N - 1);
    RowParts<D> pa, pb;
    pa.load(colA + boff + static_cast<size_t>(xi) * D, pl >> 5, PASS2 ? 1.f : c);
    pb.load(colB + boff + static_cast<size_t>(xi) * D, pl >> 5, 1.f);
    float nl = 0.f, nd = 0.f;  // pass 1: -lse and -D of the lane's query
    if constexpr (!PASS2) {
      float dd = 0.f;
#pragma unroll
      for (int g = 0; g < D / 16; ++g) {
        float o[8], d[8];
        ld_f32<8>(o, O + boff + static_cast<size_t>(xi) * D + 16 * g + 8 * (pl >> 5));
        ld_f32<8>(d, colB + boff + static_cast<size_t>(xi) * D + 16 * g + 8 * (pl >> 5));
#pragma unroll
        for (int e = 0; e < 8; ++e) dd = fmaf(d[e], o[e], dd);
      }
      dd = add_xor32(dd);
      nd = -dd;
      nl = -st[xi];
      if (pl < 32 && x0 + pl < N) st[N + xi] = dd;
    }
    f32x16 ga[NB], gb[PASS2 ? NB : 1];
#pragma unroll
    for (int n = 0; n < NB; ++n) ga[n] = f32x16{};
    if constexpr (PASS2)
#pragma unroll
      for (int n = 0; n < NB; ++n) gb[n] = f32x16{};
    for (int c0 = 0; c0 < N; c0 += kc, buf = __builtin_amdgcn_readfirstlane(buf ^ 1)) {
      const int cn = min(kc, N - c0), kend = c0 + cn;
      bf16* const As = lds + static_cast<size_t>(buf) * 2 * kc * LD;
      bf16* const Bs = As + static_cast<size_t>(kc) * LD;
      float* const Ls = sc + buf * 2 * kc;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int v = threadIdx.x + u * bd, row = v / VPR, cv = v - row * VPR;
        if (row < kc) {
          store_parts3<D>(As + row * LD + 4 * cv, PASS2 ? xa[u] * c : xa[u]);
          store_parts3<D>(Bs + row * LD + 4 * cv, xb[u]);
        }
      }
      if constexpr (PASS2)
        if (static_cast<int>(threadIdx.x) < kc) {
          Ls[threadIdx.x] = -xs;
          Ls[kc + threadIdx.x] = -xd;
        }
      if (kend < N) load_chunk(b, kend);
      else if (blk + grid < nblocks) load_chunk(__builtin_amdgcn_readfirstlane((blk + grid) / n_blk), 0);
      lds_barrier();
      if (x0 < N) {
        for (int yb = 0; yb < cn; yb += 32) {
          // the products of each tile before the next tile's scores: P, then
          // dS, is all that is live between them (d = 16 then fits four waves
          // a SIMD; the barriers keep the scheduler from overlapping the two)
          f32x16 p = tile_dot<D, PASS2>(pa, As + yb * LD + row_off, f32x16{});
          if constexpr (PASS2) {
#pragma unroll
            for (int i = 0; i < 16; i += 4) {
              const f32x4 a = *reinterpret_cast<const f32x4*>(Ls + yb + tile_row(i) + 4 * half);
#pragma unroll
              for (int r = 0; r < 4; ++r) p[i + r] += a[r];
            }
          } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) p[i] += nl;
          }
          const int yabs = c0 + yb;
          if (yabs == x0) {  // the diagonal tile
#pragma unroll
            for (int i = 0; i < 16; ++i)
              if (tile_row(i) == self) p[i] = -INFINITY;
          }
          if (!PASS2 && yabs + 32 > kend) {  // pass 2: rows past the end have lse = inf
#pragma unroll
            for (int i = 0; i < 16; ++i)
              if (tile_row(i) >= kend - yabs - 4 * half) p[i] = -INFINITY;
          }
#pragma unroll
          for (int i = 0; i < 16; ++i) p[i] = fast_exp2(p[i]);
          if constexpr (PASS2) mma_parts<D>(gb, Bs + yb * LD + t_off, Bs + yb * LD + tlo_off, p);
          __builtin_amdgcn_sched_barrier(0);
          f32x16 dp = tile_dot<D, PASS2>(pb, Bs + yb * LD + row_off, f32x16{});
#pragma unroll
          for (int i = 0; i < 16; i += 4) {
            f32x4 d = {nd, nd, nd, nd};
            if constexpr (PASS2) d = *reinterpret_cast<const f32x4*>(Ls + kc + yb + tile_row(i) + 4 * half);
#pragma unroll
            for (int r = 0; r < 4; ++r) dp[i + r] = p[i + r] * (dp[i + r] + d[r]);
          }
          mma_parts<D>(ga, As + yb * LD + t_off, As + yb * LD + tlo_off, dp);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if (x0 < N) {
      fold_halves<D>(ga);
      bool stands = grad_stands<D>(ga);
      if constexpr (PASS2) {
        fold_halves<D>(gb);
        stands &= grad_stands<D>(gb);
      }
      const uint64_t bad = __ballot(!stands);
      const uint32_t again = static_cast<uint32_t>(bad) | static_cast<uint32_t>(bad >> 32);
      int el = lane;
      asm volatile("" : "+v"(el));
      const int ecol = el & 31, exi = min(x0 + ecol, N - 1);
      if (x0 + ecol < N && (again >> ecol & 1u) == 0u) {
        store_grad<D>(out_a + boff + static_cast<size_t>(exi) * D, ga, el >> 5, PASS2 ? uniform_value(scale / c) : scale);
        if constexpr (PASS2) store_grad<D>(out_b + boff + static_cast<size_t>(exi) * D, gb, el >> 5, 1.f);
      }
      if (again != 0u) {
#pragma unroll 1
        for (int t = 0; t < 2; ++t)
          if (x0 + 16 * t < N && (again >> 16 * t & 0xffffu) != 0u)
            bwd_rerun<D, PASS2>(colA + boff, colB + boff, A + boff, Bm + boff, -__shfl(nl, 16 * t + (el & 15)),
                                -__shfl(nd, 16 * t + (el & 15)), st, st + N, out_a + boff,
                                PASS2 ? out_b + boff : nullptr, N, x0 + 16 * t, el, scale, again >> 16 * t);
      }
    }
  }
}

template <int D, int U, bool PASS2>
hipError_t launch_pass(const DenseBwdArgs& a, int nw, int n_blk) {
  using BS = BwdSplit<D>;
  int kc = std::min(BS::KC, U * 64 * nw / BS::VPR / 32 * 32);
  if (kc < 32) return hipErrorInvalidValue;  // fewer threads than a 32-row block takes
  const int nch = (a.N + kc - 1) / kc;
  kc = std::min(kc, ((a.N + nch - 1) / nch + 31) / 32 * 32);
  const int nblocks = a.B * n_blk;
  const int grid = std::min(nblocks, kCUs * (16 / nw));  // workgroups stay for as many items as it takes
  hipStream_t st = static_cast<hipStream_t>(a.stream);
  if constexpr (PASS2)
    hipLaunchKernelGGL((dense_bwd_split_kernel<D, U, true>), dim3(grid), dim3(64 * nw), BS::lds_bytes(kc), st,
                       a.k, a.v, a.q, a.dout, nullptr, a.stats, a.dk, a.dv, a.N, n_blk, kc, a.scale, nblocks);
  else
    hipLaunchKernelGGL((dense_bwd_split_kernel<D, U, false>), dim3(grid), dim3(64 * nw), BS::lds_bytes(kc), st,
                       a.q, a.dout, a.k, a.v, a.out, a.stats, a.dq, nullptr, a.N, n_blk, kc, a.scale, nblocks);
  return hipGetLastError();
}

template <int D, bool PASS2>
hipError_t launch_pass_d(const DenseBwdArgs& a) {
  const int waves = (a.N + 31) / 32;
  // pass 2 at d = 16: workgroups of four waves divide rows of a few hundred
  // keys more evenly (B=256 N=384: 87.9 -> 81.9 us for both passes; N=256: no
  // change)
  int nw = D == 16 && PASS2 ? 4 : 8;
  while (nw > 4 && a.B * ((waves + nw - 1) / nw) < 2 * kCUs) nw /= 2;  // more CUs at work
  const int n_blk = (waves + nw - 1) / nw;
  nw = (waves + n_blk - 1) / n_blk;
  // d = 64: two vectors a thread of fewer than four waves are less than a 32-row
  // block, so rows of three waves have a fourth that only stages (four vectors
  // a thread instead spilled 35 registers in pass 2)
  if (D == 64) nw = std::max(nw, 4);
  if (nw == 8 || (D == 16 && PASS2 && nw == 4)) return launch_pass<D, 1, PASS2>(a, nw, n_blk);
  return launch_pass<D, 2, PASS2>(a, nw, n_blk);
}

}  // namespace

hipError_t run_dense_bwd_split(const DenseBwdArgs& a, bool pass2) {
  switch (a.d) {
    case 16: return pass2 ? launch_pass_d<16, true>(a) : launch_pass_d<16, false>(a);
    case 32: return pass2 ? launch_pass_d<32, true>(a) : launch_pass_d<32, false>(a);
    case 64: return pass2 ? launch_pass_d<64, true>(a) : launch_pass_d<64, false>(a);
  }
  return hipErrorInvalidValue;
}

}  // namespace tarmac
