"""The accumulation bound the exact bf16 / split-bf16 top-k proofs rest on.

The packed and filter top-k kernels score on bf16 MFMA (exact products, fp32
accumulation) and prove their retained set against an error bound
E = eps(d) |q| max_j |k_j| (``packed_eps`` / ``filter_eps``: 2^-18 at d <= 32,
2^-17 at d = 64). E must cover, relative to sum_c |q_c k_c| <= |q| |k_j|:

* the MFMA's accumulation error, measured here on this device
  (``tarmac_mfma_bf16_probe``) against exact float64 sums, on random,
  same-sign, mixed-magnitude, cancelling and one-dominant-product operands,
  chained over one to four 16x16x32 instructions (bf16 scores at d = 32, 64,
  128) and one to six 32x32x16 instructions (the 32 x 32 split kernel chains
  six), and over the split-bf16 chains of 16 x 16 tiles in their own order and
  magnitudes (3, 6 and 12 instructions at d = 16, 32, 64), relative to
  sum_c |q_c k_c|: the bound asserted is 2^-20.25 (the worst case seen is about
  2^-20.4, one dominant product among small ones);
* the canonical fmaf chain's error, at most d 2^-24 (one rounding per step);
* for split-bf16 scores, the dropped products (mid.lo, lo.mid, lo.lo, each
  at most 2^-24 of |q_c k_c|).

The margins (eps over the sum) are asserted too, and the top-k kernels are
run on inputs built like the worst accumulation case (one dominant
coordinate, the ranking decided by small products) with indices required
bit-exact against the canonical C oracle.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import tarmac_oracle as O

pytestmark = pytest.mark.gpu

MFMA_ACC_BOUND = 2.0 ** -20.25  # relative to the sum of |products|
EPS = {16: 2.0 ** -18, 32: 2.0 ** -18, 64: 2.0 ** -17, 128: 2.0 ** -16}  # packed_eps / filter_eps


def _bf16_bits(x):
    u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7FFF + ((u >> 16) & 1)) >> 16
    return u.astype(np.uint16)


def _bits_f64(b):
    return (b.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


def _mfma_chain(Am, Bm, shape=16):
    """shape 16: Am [T, chain, 16, 32], Bm [T, chain, 32, 16]; shape 32:
    Am [T, chain, 32, 16], Bm [T, chain, 16, 32] (float32, rounded to bf16):
    the chained MFMA result [T, M, M]."""
    from tarmac import _lib
    T, chain = Am.shape[:2]
    M = Am.shape[2]  # 16 or 32 rows (= columns) of the result
    Ab, Bb = _bf16_bits(Am), _bf16_bits(Bm)
    la = np.zeros((T, chain, 64, 8), np.uint16)
    lb = np.zeros((T, chain, 64, 8), np.uint16)
    for lane in range(64):
        i, g = lane % M, lane // M
        la[:, :, lane, :] = Ab[:, :, i, 8 * g:8 * g + 8]
        lb[:, :, lane, :] = Bb[:, :, 8 * g:8 * g + 8, i]
    da = torch.from_numpy(la.view(np.int16)).cuda()
    db = torch.from_numpy(lb.view(np.int16)).cuda()
    per = 4 if shape == 16 else 16
    out = torch.zeros(T, 64, per, device="cuda")
    rc = _lib.LIB.tarmac_mfma_bf16_probe(da.data_ptr(), db.data_ptr(), out.data_ptr(), T, chain,
                                         shape, None)
    _lib.check(rc)
    torch.cuda.synchronize()
    o = out.cpu().numpy()
    got = np.zeros((T, M, M))
    for lane in range(64):
        j, g = lane % M, lane // M
        for r in range(per):
            row = 4 * g + r if shape == 16 else 8 * (r // 4) + 4 * g + r % 4
            got[:, row, j] = o[:, lane, r]
    return got


def _mfma_rel_error(Am, Bm, shape=16):
    """Max over outputs of |MFMA - exact| / sum |products| (operands as
    _mfma_chain)."""
    got = _mfma_chain(Am, Bm, shape)
    Af, Bf = _bits_f64(_bf16_bits(Am)), _bits_f64(_bf16_bits(Bm))
    exact = np.einsum("tcik,tckj->tij", Af, Bf)
    mag = np.einsum("tcik,tckj->tij", np.abs(Af), np.abs(Bf))
    return float((np.abs(got - exact) / np.maximum(mag, 1e-300)).max())


PATTERNS = {
    "normal": lambda g, s: g.standard_normal(s),
    "same_sign": lambda g, s: 1.0 + g.random(s),
    "mixed_magnitude": lambda g, s: g.standard_normal(s) * 2.0 ** g.integers(-20, 20, s),
    "one_dominant": lambda g, s: np.where(g.random(s) < 0.03, 2.0 ** 12, 1.0 + g.random(s)),
    "cancelling": lambda g, s: np.where(g.random(s) < 0.5, 1.0, -1.0) * (1.0 + 2.0 ** -7 * g.integers(0, 128, s)),
}


@pytest.mark.parametrize("shape,chain", [(16, 1), (16, 2), (16, 3), (16, 4), (32, 1), (32, 2),
                                         (32, 6)])
@pytest.mark.parametrize("pattern", list(PATTERNS))
def test_mfma_accumulation_error_within_bound(pattern, shape, chain):
    g = np.random.default_rng(10 * list(PATTERNS).index(pattern) + chain + shape)
    T = 1024 if shape == 16 else 256
    rows, inner = (16, 32) if shape == 16 else (32, 16)
    Am = PATTERNS[pattern](g, (T, chain, rows, inner)).astype(np.float32)
    Bm = PATTERNS[pattern](g, (T, chain, inner, rows)).astype(np.float32)
    err = _mfma_rel_error(Am, Bm, shape)
    assert err <= MFMA_ACC_BOUND, f"MFMA accumulation error {err:.3e} above the bound"


def test_proof_margins_cover_the_error_sources():
    """eps(d) against the sum of the sources it must cover, with margin."""
    for d, eps in EPS.items():
        canonical = d * 2.0 ** -24
        assert canonical + MFMA_ACC_BOUND <= eps / 1.25, d
    # split-bf16 scores (fp32 inputs): products whose magnitudes sum to at most
    # 1 + 2^-7 times sum |q_c k_c|, and three dropped products of at most 2^-24
    # each
    for d in (16, 32, 64):
        split = d * 2.0 ** -24 + MFMA_ACC_BOUND * (1 + 2.0 ** -7) + 3 * 2.0 ** -24
        assert split <= EPS[d] / 1.25, d


def _parts(x):
    """x = hi + mid + lo, each a bf16 value (float32 arrays)."""
    x = x.astype(np.float32)
    hi = _bits_f64(_bf16_bits(x)).astype(np.float32)
    mid = _bits_f64(_bf16_bits(x - hi)).astype(np.float32)
    return {"h": hi, "m": mid, "l": _bits_f64(_bf16_bits(x - hi - mid)).astype(np.float32)}


def _split_chain(q, k):
    """The A (key) and B (query) operands of a split score's chain on 16 x 16
    tiles, in the kernels' order; q, k: [T, 16, d]."""
    d, Q, K = q.shape[-1], _parts(q), _parts(k)
    pair = lambda x, a, b: np.concatenate([x[a], x[b]], -1)
    if d == 16:  # two 16-wide products side by side in one 32-wide step
        steps = [(pair(K, "h", "m"), pair(Q, "h", "h")), (pair(K, "h", "m"), pair(Q, "m", "m")),
                 (pair(K, "l", "h"), pair(Q, "h", "l"))]
    else:
        halves = range(0, d, 32)
        steps = [(K[a][..., h:h + 32], Q[b][..., h:h + 32])
                 for a, b in ("mm", "lh", "hl", "mh", "hm", "hh") for h in halves]
    A = np.stack([a for a, _ in steps], 1)
    B = np.stack([b.transpose(0, 2, 1) for _, b in steps], 1)
    return A, B


# q and k of one dominant product (1) among products of 2^-2e to 2^(2 - 2e)
SPLIT_PATTERNS = {"normal": None, "same_sign": None, "mixed_magnitude": None,
                  **{f"dominant_{e}": e for e in (2, 5, 6, 7, 8, 9, 10, 11, 12)}}


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("pattern", list(SPLIT_PATTERNS))
def test_split_chain_error_within_bound(pattern, d):
    g = np.random.default_rng(100 + list(SPLIT_PATTERNS).index(pattern))
    e, shape = SPLIT_PATTERNS[pattern], (256, 16, d)
    if e is None:
        q, k = PATTERNS[pattern](g, shape), PATTERNS[pattern](g, shape)
    else:
        q, k = ((1.0 + g.random(shape)) * 2.0 ** -e for _ in range(2))
        q[..., 0] = k[..., 0] = 1.0
    q, k = q.astype(np.float32), k.astype(np.float32)
    A, B = _split_chain(q, k)
    Af, Bf = A.astype(np.float64), B.astype(np.float64)
    six = np.einsum("tcik,tckj->tij", Af, Bf)
    mag = np.einsum("tic,tjc->tij", np.abs(k.astype(np.float64)), np.abs(q.astype(np.float64)))
    err = float((np.abs(_mfma_chain(A, B, 16) - six) / mag).max())
    assert err <= MFMA_ACC_BOUND, f"split chain error {err:.3e} (2^{np.log2(err):.2f}) above the bound"


@pytest.mark.parametrize("mode", [1, 4, 5], ids=["auto", "split16", "split32"])
@pytest.mark.parametrize("d", [16, 32, 64, 128])
@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
def test_topk_exact_on_one_dominant_coordinate(d, dtype, mode):
    """Every score carries one dominant product (q_0 k_0 = 4096) and the
    ranking is decided by the small ones: the accumulation pattern with the
    largest MFMA error. Retained indices bit-exact against the canonical
    oracle (bf16: on the bf16 inputs). fp32 at d = 16, 32, 64 runs the
    split-bf16 pass on 16 x 16 tiles (mode 4), d = 16 also the 32 x 32 kernel
    (mode 5; bf16: its single-product form); where a mode does not serve a
    width or dtype it runs the packed pass."""
    from tarmac import _lib
    from tarmac.kernels import topk_attention
    B, N = 8, 256
    g = np.random.default_rng(d)
    q = g.standard_normal((B, N, d)).astype(np.float32) / 8
    k = g.standard_normal((B, N, d)).astype(np.float32) / 8
    v = g.standard_normal((B, N, d)).astype(np.float32)
    q[..., 0] = 64.0
    k[..., 0] = 64.0
    if dtype == "bf16":
        q, k, v = (O.bf16_round(x) for x in (q, k, v))
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float32
    qd, kd, vd = (torch.from_numpy(x).cuda().to(tdt) for x in (q, k, v))
    prev = _lib.LIB.tarmac_set_topk_filter(mode)
    try:
        for kk in (1, 2, 4):
            out, idx = topk_attention(qd, kd, vd, kk, return_indices=True)
            torch.cuda.synchronize()
            _, idx_c = O.canon_topk(q, k, v, kk)
            assert np.array_equal(idx.cpu().numpy(), idx_c), f"k={kk}: indices differ from the oracle"
    finally:
        _lib.LIB.tarmac_set_topk_filter(prev)
