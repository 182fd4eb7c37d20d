"""Dense backward on split operands (``csrc/backward_split.hip``) against
float64 autograd: sizes around its tiles, chunks and launch shapes, gradients
of any scale, and inputs that are not finite.

Tolerance: 1e-5 of the largest entry, the bar of the fp32 gradient tests.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-5


def batch(N, least=3):
    """The smallest batch of N agents that takes the split kernels."""
    return max(least, -(-1024 // -(-N // 32)))


def case(B, N, d, seed=0):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(B, N, d, generator=g).cuda() for _ in range(4)]


def exact(q, k, v, dout):
    a = [t.double().requires_grad_(True) for t in (q, k, v)]
    s = torch.matmul(a[0], a[1].transpose(1, 2).contiguous()) / q.shape[-1] ** 0.5
    eye = torch.eye(q.shape[1], dtype=torch.bool, device=q.device)
    out = torch.matmul(torch.softmax(s.masked_fill(eye, float("-inf")), -1), a[2])
    return torch.autograd.grad(out, a, dout.double())


def grads(q, k, v, dout, with_stats=True):
    from tarmac.kernels import dense_attention_backward, dense_attention_forward_stats
    out, stats = dense_attention_forward_stats(q, k, v)
    return dense_attention_backward(q, k, v, out, dout, stats if with_stats else None)


def check(got, ref):
    for g, r in zip(got, ref):
        assert float((g.double() - r).abs().max() / r.abs().max()) <= TOL
        assert float((g.double() - r).norm() / r.norm()) <= 2e-6


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("N", [33, 65, 96, 97, 128, 129, 160, 255, 256, 257, 300, 513])
def test_sizes(N, d):
    x = case(batch(N), N, d, seed=N + d)
    check(grads(*x), exact(*x))


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("N,N1_error", [(100, 3.0e-7), (256, 4.1e-7)])
def test_no_further_from_float64_than_fp32_mfma(N, N1_error, d):
    """N(0, 1) inputs: the normwise error of each gradient against that of the
    fp32 MFMA kernels at d = 16 (the smallest of dq, dk, dv; d = 64 has four
    times the products a score and 1.2 times the error)."""
    x = case(batch(N), N, d, seed=1)
    for g, r in zip(grads(*x), exact(*x)):
        assert float((g.double() - r).norm() / r.norm()) <= N1_error * (1.2 if d == 64 else 1.0)


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("N", [100, 256, 1000])
@pytest.mark.parametrize("scale", [16, 64])
def test_sharp_scores(N, d, scale):
    """Scores of 2^7 and more, where a weight 2^(s - lse) is off by what s is
    rounded differently from the forward's. Both passes form the forward's bits,
    so dk and dv are no further off than dq (apart: 1.4 to 1.6 times); keys that
    no one attends to, whose gradients run again, leave the others as they are."""
    q, k, v, dout = case(batch(N), N, d, seed=7)
    q *= scale
    err = [float((g.double() - r).norm() / r.norm())
           for g, r in zip(grads(q, k, v, dout), exact(q, k, v, dout))]
    assert max(err[1:]) <= 1.2 * err[0], err


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("N", [100, 256, 1000])
def test_scores_rising_along_the_row(N, d):
    """Every tile of 32 keys overflows beside the one before it (30 / sqrt(d) nats
    a key): the forward's logsumexp still comes from the scores that pass 1 forms,
    so dq, differences of weights next to 1, is as near as on the small-batch
    kernels (apart: 60 to 200 times as far)."""
    q, k, v, dout = case(batch(N), N, d, seed=7)
    k[..., 0] = torch.arange(N, device="cuda") * 30.0
    q[..., 0] = 1.0
    n = 2  # rows for which B ceil(N / 32) is below the split kernels' line
    small = [t[:n].contiguous() for t in (q, k, v, dout)]
    ref = exact(*small)[0]
    here, there = grads(q, k, v, dout)[0][:n], grads(*small)[0]
    assert float((here.double() - ref).norm()) <= 1.5 * float((there.double() - ref).norm())


@pytest.mark.parametrize("d", [16, 32, 64])
def test_launch_shapes(d):
    """Eight-wave workgroups over full rows, more items than workgroups, and
    the logsumexp formed by the backward itself."""
    x = case(520 if d == 16 else 300, 256, d)
    ref = exact(*x)
    check(grads(*x), ref)
    check(grads(*x, with_stats=False), ref)
    x = case(1100, 70, d)
    check(grads(*x), exact(*x))


@pytest.mark.parametrize("d", [16, 32, 64])
def test_one_vector_a_thread(d):
    """Workgroups of eight waves (from 512 rows on): one vector a thread."""
    x = case(520, 250, d)
    check(grads(*x), exact(*x))


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("scale", [1e-33, 1e-20, 1e20])
def test_gradient_scales(d, scale):
    q, k, v, dout = case(batch(150), 150, d)
    check(grads(q, k, v, dout * scale), exact(q, k, v, dout * scale))


@pytest.mark.parametrize("d", [16, 32, 64])
@pytest.mark.parametrize("scale", [1e-33, 1e-34])
def test_small_gradients_beside_ordinary_ones(d, scale):
    """Every other query's output gradient, and one of its channels for the
    others, is far below its neighbours': each row of dq and each channel of dv
    is held against its own size."""
    q, k, v, dout = case(batch(150), 150, d)
    dout[:, ::2] *= scale
    dout[:, :, 5] = dout[:, :1, 5]
    dq, dk, dv = grads(q, k, v, dout)
    ref = exact(q, k, v, dout)
    check([dq[:, ::2], dq[:, 1::2]], [ref[0][:, ::2], ref[0][:, 1::2]])
    check([dv[:, :, 5:6], dv[:, :, :5]], [ref[2][:, :, 5:6], ref[2][:, :, :5]])


@pytest.mark.parametrize("d", [16, 64])
def test_zero_and_not_finite_rows(d):
    q, k, v, dout = case(batch(100), 100, d)
    dout[0] = 0.0
    dout[1, 5, 3] = float("inf")
    dq, dk, dv = grads(q, k, v, dout)
    for g in (dq, dk, dv):
        assert bool((g[0] == 0).all())
    ref = exact(q, k, v, dout)
    check([g[2:] for g in (dq, dk, dv)], [r[2:] for r in ref])
    # the other queries of that row, and the other channels of its dv
    others = torch.arange(100) != 5
    check([dq[1:2, others]], [ref[0][1:2, others]])
    keep = torch.arange(d) != 3
    check([dv[1:2, :, keep]], [ref[2][1:2, :, keep]])
