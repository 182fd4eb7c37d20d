"""fp32 top-k at d = 32 and 64 on split-bf16 scores with two query tiles per
wave: the kernels that long rows of large batches take. Retained indices
bit-exact against the canonical oracle, in its order; outputs within 1e-5 of
the largest entry (normwise), the bar of the other fp32 top-k tests.
"""

from __future__ import annotations

import contextlib

import numpy as np
import pytest
import torch

import tarmac_oracle as O
from conftest import qkv

pytestmark = pytest.mark.gpu

AUTO, SPLIT = 1, 4
MODES = pytest.mark.parametrize("mode", [AUTO, SPLIT], ids=["auto", "split"])


@contextlib.contextmanager
def kernel(mode, tiles=2):
    from tarmac import _lib
    prev = _lib.LIB.tarmac_set_topk_filter(mode), _lib.LIB.tarmac_set_query_tiles(tiles)
    try:
        yield
    finally:
        _lib.LIB.tarmac_set_topk_filter(prev[0])
        _lib.LIB.tarmac_set_query_tiles(prev[1])


def check(q, k, v, kk, chunk=None):
    from tarmac.kernels import topk_attention
    out, idx = topk_attention(*(torch.from_numpy(x).cuda() for x in (q, k, v)), kk,
                              return_indices=True, key_chunk=chunk)
    out_c, idx_c = O.canon_topk(q, k, v, kk)
    assert np.array_equal(idx.cpu().numpy(), idx_c), "retained indices differ from the oracle"
    assert np.abs(out.cpu().numpy() - out_c).max() <= 1e-5 * np.abs(out_c).max()


@MODES
@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("N,chunk", [(512, None), (577, None), (577, 128), (1024, None), (1500, None)])
@pytest.mark.parametrize("kk", [1, 2, 3, 4, 5, 8])
def test_parity(N, chunk, d, kk, mode):
    """Resident and streamed rows (a 400-byte split row at d = 64 always
    streams), one packing segment and several (N > 1024)."""
    with kernel(mode):
        check(*qkv(N + 3 * d + kk, 2, N, d), kk, chunk)


@MODES
@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("N,chunk", [(512, None), (1024, 128), (1500, None)])
@pytest.mark.parametrize("kk", [1, 2, 3, 4, 8])
def test_ties(N, chunk, d, kk, mode):
    """Duplicated keys, zero and repeated queries: the proof fails and the
    per-query exact pass decides."""
    q, k, v = qkv(N + d, 2, N, d)
    k[:, 1::2] = k[:, 0::2]
    q[:, :6] = 0.0
    q[:, 6:12] = q[:, 6:7]
    with kernel(mode):
        check(q, k, v, kk, chunk)


@MODES
@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("N,kk,chunk", [(512, 2, None), (700, 8, None), (1024, 4, None), (1500, 3, 128)])
def test_near_ties(N, kk, chunk, d, mode):
    """Clusters of keys whose scores agree to about 1e-6."""
    q, k, v = qkv(17 + N + d, 2, N, d)
    rng = np.random.default_rng(N)
    for c0 in range(0, N - 40, 97):
        k[:, c0 + 1:c0 + 40] = k[:, c0:c0 + 1] * 3.0 + 1e-6 * rng.standard_normal((2, 39, d)).astype(np.float32)
    with kernel(mode):
        check(q, k, v, kk, chunk)


@MODES
@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("kk", [1, 4])
def test_one_dominant_coordinate(d, kk, mode):
    """The accumulation pattern with the largest error of a split score."""
    q, k, v = qkv(5 + d, 2, 1024, d)
    q, k = q / 8, k / 8
    q[..., 0] = k[..., 0] = 64.0
    with kernel(mode):
        check(q, k, v, kk)


@MODES
@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("N", [512, 519, 1024, 1300])
@pytest.mark.parametrize("kk", [1, 2, 3, 4, 8])
def test_tiles_of_unproven_queries(N, d, kk, mode):
    """Queries whose keys all tie: a batch row of them, and one with 1, 2, 3 and
    16 of them to a tile of 16 and in the last tile."""
    q, k, v = qkv(3 * N + d, 2, N, d)
    rng = np.random.default_rng(N)
    q[0], k[0] = (np.eye(d, dtype=np.float32)[rng.integers(0, d, N)] for _ in range(2))
    for at, n in ((5, 1), (16, 2), (45, 3), (64, 16), (N - 3, 3)):
        q[1, at:at + n] = 0.0
    with kernel(mode):
        check(q, k, v, kk)


@pytest.mark.parametrize("B,N,d,kk", [(256, 512, 32, 2), (256, 512, 32, 5), (256, 512, 32, 8),
                                      (256, 1024, 32, 7), (128, 512, 64, 4), (64, 1024, 64, 2),
                                      (1024, 512, 64, 3), (1024, 704, 64, 3)])
def test_batches_past_the_line(B, N, d, kk):
    """Nothing forced: the batch itself takes two query tiles per wave, on each
    side of the lines between the kernels. Sampled rows."""
    from tarmac.kernels import topk_attention
    g = torch.Generator().manual_seed(B + N + d + kk)
    q, k, v = (torch.randn(B, N, d, generator=g) for _ in range(3))
    out, idx = topk_attention(q.cuda(), k.cuda(), v.cuda(), kk, return_indices=True)
    rows = [0, 1, B // 2, B - 1]
    out_c, idx_c = O.canon_topk(*(x[rows].numpy() for x in (q, k, v)), kk)
    assert np.array_equal(idx[rows].cpu().numpy(), idx_c)
    assert np.abs(out[rows].cpu().numpy() - out_c).max() <= 1e-5 * np.abs(out_c).max()
