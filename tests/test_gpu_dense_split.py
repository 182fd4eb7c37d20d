"""Dense fp32 attention on split operands (``csrc/dense_split.hip``) against
float64: sizes around its tiles and chunks, and the rows that leave its fast
path (a late large score, values too far apart for two parts, values that are
not finite).

Tolerance: the split kernel keeps q and k to 2^-24 and v and the weights to
2^-22 of each value; the exponent's rounding, |c s| 2^-24 for scores up to
about 2^5, is the largest term: 2^-19 of a weight, 4e-6 normwise with the sum
of the others.
"""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

RTOL = 4e-6


def batch(N, least=3):
    """The smallest batch of N agents that takes the split kernel."""
    return max(least, -(-1024 // -(-N // 32)))


def heads(B, N, d, seed=0):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(B, N, d, generator=g).cuda() for _ in range(3)]


def exact(q, k, v):
    q, k, v = q.double(), k.double(), v.double()
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) / q.shape[-1] ** 0.5
    s.diagonal(dim1=1, dim2=2).fill_(float("-inf"))
    return torch.matmul(torch.softmax(s, -1), v), torch.logsumexp(s, -1)


def check(out, ref):
    """Every output row against its own largest entry."""
    err = (out.double() - ref).abs().amax(-1) / ref.abs().amax(-1)
    assert float(err.max()) <= RTOL * 4, float(err.max())
    assert float((out.double() - ref).norm() / ref.norm()) <= RTOL


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("N", [33, 65, 95, 96, 97, 127, 129, 160, 255, 256, 257, 289, 513, 1000])
def test_sizes(N, d):
    from tarmac.kernels import dense_attention_forward_stats
    q, k, v = heads(batch(N), N, d, seed=N + d)
    out, stats = dense_attention_forward_stats(q, k, v)
    ref, lse = exact(q, k, v)
    check(out, ref)
    got = stats[:, 0].double() * np.log(2.0)
    assert float((got - lse).abs().max()) <= 2e-5


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("N", [17, 24, 32, 33, 64, 96])
def test_chunk_below_the_row(N, d):
    """A caller's chunk is kept at every batch: the kernel that stages it gives
    a row the same bits at B = 1024, past the line of the split kernel, as at
    B = 2."""
    from tarmac.kernels import fused_dense_attention
    q, k, v = heads(1024, N, d, seed=N + d)
    ref = exact(q, k, v)[0]
    for chunk in (16, 32):
        out = fused_dense_attention(q, k, v, block_kn=chunk)
        check(out, ref)
        if chunk < N:
            assert torch.equal(out[:2], fused_dense_attention(q[:2], k[:2], v[:2], block_kn=chunk))


@pytest.mark.parametrize("d", [16, 32, 64])
def test_more_items_than_workgroups(d):
    """Workgroups that take several rows in turn, with V scales that differ."""
    from tarmac.kernels import fused_dense_attention
    q, k, v = heads(1100, 70, d)
    v *= torch.exp2(torch.arange(1100, device="cuda").remainder(41) - 20.0).view(-1, 1, 1)
    check(fused_dense_attention(q, k, v), exact(q, k, v)[0])


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("N", [100, 256, 1000])
def test_logsumexp_is_not_one_sided(N, d):
    """The mean error over all rows, which the backward would carry into every
    gradient. An fp32 logsumexp of 2^2 to 2^3 rounds at 2^-23 of it without a
    sign: its mean over B N rows is far below 1e-7, the bound here; sums of
    2^10 rounded down at their own last place gave 3.4e-7."""
    from tarmac.kernels import dense_attention_forward_stats
    q, k, v = heads(batch(N), N, d, seed=N)
    _, stats = dense_attention_forward_stats(q, k, v)
    err = stats[:, 0].double() * np.log(2.0) - exact(q, k, v)[1]
    assert abs(float(err.mean())) <= 1e-7


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("log2_gap", [8, 14, 40, 90, 120, 200])
def test_late_large_scores(d, log2_gap):
    """A key beyond the first tile scores up to 2^gap times the others: the
    offset is raised, or the row runs again, in steps along the row."""
    from tarmac.kernels import fused_dense_attention
    q, k, v = heads(batch(300), 300, d, seed=log2_gap)
    c = np.log2(np.e) / d ** 0.5
    for at, part in ((70, 0.3), (140, 0.6), (290, 1.0)):
        k[1, at] = q[1, 17] / q[1, 17].norm() ** 2 * (part * log2_gap / c)
    check(fused_dense_attention(q, k, v), exact(q, k, v)[0])


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("log2_gap", [120.0, 121.5, 122.2, 122.5, 122.9, 123.5])
def test_terms_whose_sum_overflows(d, log2_gap):
    """Two keys of one tile whose terms beside the row's first keys (2^5 there)
    are near fp32's limit: each still finite, their sum not, from 122 up; from
    123 each overflows."""
    from tarmac.kernels import dense_attention_forward_stats
    q, k, v = heads(batch(200), 200, d)
    c = np.log2(np.e) / d ** 0.5
    q[1], k[1, :, 0] = 0.0, 0.0
    q[1, 17, 0] = 1.0
    k[1, 70:72, 0] = log2_gap / c
    out, stats = dense_attention_forward_stats(q, k, v)
    ref, lse = exact(q, k, v)
    check(out, ref)
    assert float((stats[:, 0].double() * np.log(2.0) - lse).abs().max()) <= 2e-5


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("N", [33, 256, 1000])
@pytest.mark.parametrize("scale", [32, 64, 256])
def test_sharp_scores(N, d, scale):
    """Scores so far apart that a tile's terms overflow beside the offset of
    those before it. The scores' rounding, 2^-24 of the largest |c s| and as
    much again from the chain, is what a weight is off by."""
    from tarmac.kernels import fused_dense_attention
    q, k, v = heads(batch(N), N, d, seed=N + scale)
    q *= scale
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) * (np.log2(np.e) / d ** 0.5)
    out, ref = fused_dense_attention(q, k, v), exact(q, k, v)[0]
    err = (out.double() - ref).abs().amax(-1) / ref.abs().amax(-1)
    assert float(err.max()) <= 2.0 ** -23 * float(s.abs().max())
    assert float((out.double() - ref).norm() / ref.norm()) <= 2.0 ** -25 * float(s.abs().max())


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("scale", [1e-30, 1e-12, 1e12, 1e30])
def test_value_scales(d, scale):
    from tarmac.kernels import fused_dense_attention
    q, k, v = heads(batch(200), 200, d)
    v = v * scale
    check(fused_dense_attention(q, k, v), exact(q, k, v)[0])


@pytest.mark.parametrize("d", [16, 32, 64])
def test_values_far_apart(d):
    """One agent's value row is 1e25 times the others' and no one attends to
    it; another batch row grows along its keys from chunk to chunk."""
    from tarmac.kernels import fused_dense_attention
    q, k, v = heads(batch(400), 400, d)
    q[0, :, 0], k[0, :, 0] = 40.0, 1.0
    k[0, 150] = 0.0
    k[0, 150, 0] = -40.0 * d ** 0.5
    v[0, 150] = 1e25
    v[1] *= torch.exp2(torch.arange(400, device="cuda") / 25.0).view(-1, 1)
    q[2, 5] = 0.0  # a query of equal scores
    ref = exact(q, k, v)[0]
    out = fused_dense_attention(q, k, v)
    check(out[0, torch.arange(400) != 150][None], ref[0, torch.arange(400) != 150][None])
    check(out[1:], ref[1:])


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("log2_value", [6, 10, 14, 18])
@pytest.mark.parametrize("log2_weight", [-9, -15, -20])
def test_small_weights_of_large_values(d, log2_value, log2_weight):
    """Each query attends to one agent; the others weigh 2^-9 to 2^-20 of it
    and their values are 2^6 to 2^18 times as large, so the output is the sum
    of small weights and has to keep their relative precision."""
    from tarmac.kernels import fused_dense_attention
    N = 256
    q, k, v = heads(batch(N), N, d, seed=log2_value)
    gap = -log2_weight * np.log(2.0) * d ** 0.5
    q[1], k[1] = q[1] * 0.01, k[1] * 0.01
    q[1, :, 0], k[1, :, 0] = 1.0, -gap
    k[1, 77, 0] = 0.0  # the agent attended to
    v[1] *= 2.0 ** log2_value
    v[1, 77] *= 2.0 ** -log2_value
    check(fused_dense_attention(q, k, v), exact(q, k, v)[0])


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("N", [128, 256, 1000])
def test_channels_of_small_weights(N, d):
    """One-hot values: an output channel is the sum of the weights of the agents
    it stands for, from 1 down to 2^-20 of the row's largest, and is held to its
    own size (RTOL: the exponent's rounding, |c s| up to 20 here)."""
    from tarmac.kernels import fused_dense_attention
    q, k, v = heads(batch(N), N, d, seed=N)
    channel = torch.arange(N, device="cuda") % d
    q[1], k[1] = q[1] * 0.01, k[1] * 0.01
    q[1, :, 0] = 1.0
    k[1, :, 0] = channel * (-20.0 / (d - 1) * np.log(2.0) * d ** 0.5)
    v[1] = torch.nn.functional.one_hot(channel, d).float()
    out, ref = fused_dense_attention(q, k, v), exact(q, k, v)[0]
    check(out, ref)
    assert float(((out[1].double() - ref[1]).abs() / ref[1]).max()) <= RTOL


def test_not_finite_stays_in_its_row():
    from tarmac.kernels import fused_dense_attention
    q, k, v = heads(batch(130), 130, 16)
    v[1, 3, 2] = float("inf")
    k[2, 7, 1] = float("nan")
    out = fused_dense_attention(q, k, v)
    ref = exact(q, k, v)[0]
    check(out[3:], ref[3:])
    check(out[:1], ref[:1])
    keep = torch.arange(16) != 2
    check(out[1][:, keep][None], ref[1][:, keep][None])
    assert not bool(torch.isfinite(out[1, 4:, 2]).any())
    others = torch.arange(130) != 7
    assert bool(torch.isnan(out[2, others]).all())
