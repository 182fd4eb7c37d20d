"""Dense attention with the self-diagonal masked, as one HIP kernel.

Drop-in for ``src/kernels/fused_dense_attention.py:106-152``
(``fused_dense_attention``). The kernel is flash-style (online softmax over key
blocks staged in LDS, MFMA for both contractions), so no score matrix reaches
HBM. It is also the function of the composed dense paths
``scripts/bench_attention_core.py:74-82`` and ``src/agents/mappo.py:174-190``.
"""

from __future__ import annotations

import torch

from .. import _launch, _lib


@_launch.half_on_f32
def fused_dense_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                          block_m: int | None = None,
                          block_kn: int | None = None,
                          num_warps: int | None = None,
                          num_stages: int | None = None,
                          precision: str = "ieee") -> torch.Tensor:
    """Streaming dense self-attention with the diagonal masked. q, k, v: [B, N, d].

    ``precision="ieee"`` is the only fp32 mode (gfx950 has no TF32 path). It
    runs on fp32 MFMA, or, at d = 16, 32 and 64 on batches of
    ``B * ceil(N / 32) >= 1024``, on 16-bit MFMA with every operand split into
    parts (scores: three bf16 parts, 24 bits; weights and values: two fp16
    parts, 22 bits; sums in fp32), no further from float64 than fp32 MFMA; rows
    that parts would not hold run on fp32 MFMA. ``block_kn`` sets the keys
    staged per LDS pass (rounded up to 16); below N it selects the fp32 MFMA
    kernel. ``block_m``, ``num_warps`` and ``num_stages`` are Triton tiling
    knobs of the reference and are accepted for signature compatibility only.
    """
    if precision != "ieee":
        raise ValueError(f"precision={precision!r}: gfx950 has no TF32 mode; use 'ieee'")
    q, k, v = _launch.core(q, k, v)
    B, N, d = q.shape
    out = torch.empty_like(q)
    chunk = 0 if block_kn is None else -(-int(block_kn) // 16) * 16
    if B == 0:  # an empty batch: nothing to launch
        return out
    with _launch.on_device_of(q):
        _lib.check(_lib.LIB.tarmac_dense_fwd(
            _launch.ptr(q), _launch.ptr(k), _launch.ptr(v), _launch.ptr(out),
            B, N, d, _launch.dtype_code(q), chunk, _launch.stream(q)))
    return out
