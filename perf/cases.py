"""What the performance of this framework is measured on: the calls that a user
of it makes, through the public entry points of :mod:`tarmac`.

Seven kinds of call, over the sizes of the configurations, tests and benchmark
of this repository (batches of 32 to 4096 rows, 6 to 1024 agents, head widths
16 to 64, fp32 and bf16):

``topk``      exact top-k attention, the framework's main call
``stream``    the same with keys streamed through LDS
``dense``     dense attention, which top-k is compared with
``zorder``    Z-order selection and attention in one call
``prescore``  a positional selector, then attention over its sets
``grad``      one training pass of a core: forward, then its backward
``module``    one training pass of ``AttentionComm``, projections included

Everything a call returns is compared. Retained sets are exact by contract
(the order of the canonical fp32 score, ties to the lower agent index), so
index outputs may not differ at all; ``exact`` forms the sets from that order
and everything after them in 64 bits.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "topk-tarmac_amd"))

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
IN_DIM = 64  # the module benchmark's observation encoding


def listed():
    return [
        # the smallest call: the six-agent particle environment's episodes
        {"name": "topk_n6", "kind": "topk", "B": 256, "N": 6, "d": 16, "k": 2, "dtype": "f32",
         "idx": False},
        # the headline call: 256 agents, two peers each, indices wanted
        {"name": "topk_n256", "kind": "topk", "B": 1024, "N": 256, "d": 16, "k": 2, "dtype": "f32",
         "idx": True},
        # the largest call: half precision, wide heads, the largest batch
        {"name": "topk_bf16_n512_d64", "kind": "topk", "B": 4096, "N": 512, "d": 64, "k": 4,
         "dtype": "bf16", "idx": False},
        # no size a multiple of anything: a batch that a variable agent count gives
        {"name": "topk_ragged", "kind": "topk", "B": 77, "N": 333, "d": 32, "k": 3, "dtype": "f32",
         "idx": True},
        # many agents, keys streamed through LDS
        {"name": "stream_n1024", "kind": "stream", "B": 256, "N": 1024, "d": 16, "k": 2,
         "dtype": "f32", "block_n": 0},
        # dense attention at the headline shape
        {"name": "dense_n256", "kind": "dense", "B": 1024, "N": 256, "d": 16, "dtype": "f32"},
        # dense attention in half precision at a large batch
        {"name": "dense_bf16_d32", "kind": "dense", "B": 4096, "N": 256, "d": 32, "dtype": "bf16"},
        # agents attend to their neighbours along the Z-order curve
        {"name": "zorder_n512", "kind": "zorder", "B": 1024, "N": 512, "d": 16, "k": 2,
         "dtype": "f32"},
        # the nearest peers of a spatial grid, then attention over them
        {"name": "prescore_grid", "kind": "prescore", "B": 256, "N": 512, "d": 16, "k": 16,
         "selector": "grid_knn"},
        # training through the dense core at the headline shape
        {"name": "grad_dense_n256", "kind": "grad", "core": "dense", "B": 1024, "N": 256, "d": 16,
         "k": 0},
        # training through the top-k core as the module benchmark sets it: a quarter of the peers
        {"name": "grad_topk_k95", "kind": "grad", "core": "topk", "B": 256, "N": 384, "d": 16,
         "k": 95},
        # a training pass of the communication block, projections included
        {"name": "module_n96_k23", "kind": "module", "mode": "topk_gather", "B": 256, "N": 96,
         "d": 16, "k": 23},
    ]


# -- drawn cases ---------------------------------------------------------------

#: Scores times head width that a drawn case of each kind may ask for: what
#: keeps it under the largest listed case's time (the fp32 matrix rate is a
#: sixteenth of the bf16 one; a training pass forms about seven products).
MOST = {"f32": 1.2e10, "bf16": 6.8e10, "grad": 4e9}


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["topk", "topk", "topk", "stream", "dense", "dense", "zorder", "prescore",
                       "grad", "grad", "module"])
    c = {"kind": kind, "B": _log_int(rng, 32, 4096), "N": _log_int(rng, 6, 1024),
         "d": rng.choice([16, 16, 32, 64])}
    if kind == "topk":
        c.update(k=rng.choice([1, 2, 2, 3, 4, 8]), dtype=rng.choice(["f32", "bf16"]),
                 idx=rng.random() < 0.5)
        c["k"] = min(c["k"], c["N"] - 1)
    elif kind == "stream":
        c.update(B=_log_int(rng, 32, 512), N=rng.randint(512, 1024), d=16,
                 k=rng.choice([1, 2, 4]), dtype=rng.choice(["f32", "bf16"]),
                 block_n=rng.choice([0, 0, 64, 128, 256]))
    elif kind == "dense":
        c.update(dtype=rng.choice(["f32", "bf16"]))
    elif kind == "zorder":
        c.update(B=_log_int(rng, 32, 2048), k=rng.choice([1, 2, 3, 4, 8]), dtype="f32")
        c["k"] = min(c["k"], c["N"] - 1)
    elif kind == "prescore":
        c.update(B=_log_int(rng, 32, 512), N=_log_int(rng, 64, 512), d=16,
                 k=rng.choice([2, 4, 8, 16]),
                 selector=rng.choice(["radius_knn", "grid_knn", "morton_window"]))
    elif kind == "grad":
        core = rng.choice(["dense", "topk"])
        c.update(core=core, B=_log_int(rng, 32, 1024), N=_log_int(rng, 6, 512), k=0)
        if core == "topk":
            c["k"] = min(rng.choice([1, 2, 4, max(1, (c["N"] - 1) // 4)]), c["N"] - 1)
    else:
        c.update(mode=rng.choice(["dense", "topk_gather"]), B=_log_int(rng, 32, 512),
                 N=_log_int(rng, 6, 384), d=16, k=2)
        c["k"] = min(rng.choice([2, max(1, (c["N"] - 1) // 4)]), c["N"] - 1)
    most = MOST["grad" if kind in ("grad", "module") else c.get("dtype", "f32")]
    c["B"] = max(32, min(c["B"], int(most / (c["N"] ** 2 * c["d"]))))
    return c


# -- inputs and calls ----------------------------------------------------------

def _inputs(case, seed):
    """q, k, v (and what else the kind takes) from the seed: N(0, 1) heads, as
    projected observations are, and positions uniform in the unit square."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    B, N, d = case["B"], case["N"], case["d"]
    dtype = DTYPES[case.get("dtype", "f32")]

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device=dev).to(dtype)

    if case["kind"] == "module":
        return {"x": normal(B, N, IN_DIM), "dout": normal(B, N, d)}
    s = {"q": normal(B, N, d), "k": normal(B, N, d), "v": normal(B, N, d)}
    if case["kind"] in ("zorder", "prescore"):
        s["pos"] = torch.rand(B, N, 2, generator=gen, device=dev)
    if case["kind"] == "grad":
        s["dout"] = normal(B, N, d)
    return s


def _module(case, seed):
    from tarmac.agents.mappo import AttentionComm, MAPPOConfig

    with torch.random.fork_rng(devices=[]):
        torch.manual_seed(int(seed))
        m = AttentionComm(MAPPOConfig(obs_dim=IN_DIM, n_actions=5, n_agents=case["N"],
                                      use_comm=True, msg_dim=case["d"], attn_mode=case["mode"],
                                      topk=case["k"]), IN_DIM)
    m.collect_info = False  # the diagnostics synchronise; training loops switch them off
    return m.to("cuda")


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = dict(case)
    if case["kind"] == "module":
        s["module"] = _module(case, seed)
        s["x"].requires_grad_(True)
    return s


def _module_grads(m, x, dout):
    msg, _ = m(x)
    params = [p for n, p in m.named_parameters() if not n.startswith("k_gate")]
    grads = torch.autograd.grad(msg, [x, *params], dout)
    return {"msg": msg.detach(), "grads": list(grads)}


def run(s):
    from tarmac import kernels as K

    c = s["case"]
    kind = c["kind"]
    if kind == "module":
        return _module_grads(s["module"], s["x"], s["dout"])
    q, k, v = s["q"], s["k"], s["v"]
    if kind == "topk":
        if c["idx"]:
            out, idx = K.topk_attention(q, k, v, c["k"], return_indices=True)
            return {"out": out, "idx": idx}
        return {"out": K.fused_topk_attention(q, k, v, c["k"])}
    if kind == "stream":
        out, idx = K.streaming_topk_attention(q, k, v, c["k"], block_n=c["block_n"] or None,
                                              return_indices=True)
        return {"out": out, "idx": idx}
    if kind == "dense":
        return {"out": K.fused_dense_attention(q, k, v)}
    if kind == "zorder":
        out, idx = K.zorder_attention(q, k, v, s["pos"], c["k"], bits=16, return_indices=True)
        return {"out": out, "idx": idx}
    if kind == "prescore":
        idx = K.SELECTORS[c["selector"]](s["pos"], c["k"])
        return {"out": K.fused_prescore_attention(q, k, v, idx), "idx": idx}
    if c["core"] == "dense":
        out, stats = K.dense_attention_forward_stats(q, k, v)
        dq, dk, dv = K.dense_attention_backward(q, k, v, out, s["dout"], stats)
        return {"out": out, "dq": dq, "dk": dk, "dv": dv}
    out, idx = K.topk_attention(q, k, v, c["k"], return_indices=True)
    dq, dk, dv = K.fixedset_attention_backward(q, k, v, idx, s["dout"])
    return {"out": out, "idx": idx, "dq": dq, "dk": dk, "dv": dv}


# -- work and tolerance --------------------------------------------------------

def work(case):
    """Each input read once and each output written once; the products the
    function is defined by (selection compares count nothing)."""
    B, N, d, kind = case["B"], case["N"], case["d"], case["kind"]
    k = case.get("k", 0)
    rows = B * N
    size = 2 if case.get("dtype") == "bf16" else 4
    heads = 4 * rows * d * size                       # q, k, v in, the message out
    scores = 2 * rows * N * d
    if kind == "topk":
        return {"bytes": heads + (4 * rows * k if case["idx"] else 0),
                "flops": scores + 2 * rows * k * d}
    if kind == "stream":
        return {"bytes": heads + 4 * rows * k, "flops": scores + 2 * rows * k * d}
    if kind == "dense":
        return {"bytes": heads, "flops": 2 * scores}
    if kind == "zorder":
        return {"bytes": heads + 8 * rows + 4 * rows * k, "flops": 4 * rows * k * d}
    if kind == "prescore":                            # the set goes out and is part of the answer
        return {"bytes": heads + 8 * rows + 8 * rows * k, "flops": 4 * rows * k * d}
    dense = kind == "grad" and case["core"] == "dense" or kind == "module" and case["mode"] == "dense"
    core = 2 * scores + 5 * scores if dense else scores + 2 * rows * k * d + 10 * rows * k * d
    if kind == "grad":                                # q, k, v, dout in; out, dq, dk, dv out
        return {"bytes": 8 * rows * d * size + (0 if dense else 4 * rows * k), "flops": core}
    proj = 3 * 2 * rows * (IN_DIM * 3 * d + d * d)    # forward, input and weight gradients
    return {"bytes": 4 * rows * (2 * IN_DIM + 2 * d), "flops": core + proj}


def tolerance(case):
    """Outputs in fp32: sums over up to 1024 terms in another order. bf16
    outputs: one rounding of the result (and of the dense weights)."""
    if case.get("dtype") == "bf16":
        return {"rel": 1e-2, "max": 5e-2}
    if case["kind"] == "module":
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 5e-6, "max": 1e-4}


# -- the same in 64 bits -------------------------------------------------------

def _canonical_scores(q, k):
    """The scores that rank peers: one fp32 fused multiply-add chain over the
    elements in the order c = kk * (d / 4) + t (t outer, kk inner), times
    fp32(1 / sqrt(d)). A product of two fp32 values is exact in 64 bits, so
    each step rounds once to fp32."""
    d = q.shape[-1]
    acc = torch.zeros(q.shape[0], q.shape[1], k.shape[1], device=q.device)
    q, k = q.double(), k.double()
    for t in range(d // 4):
        for kk in range(4):
            c = kk * (d // 4) + t
            acc = torch.addcmul(acc.double(), q[:, :, None, c], k[:, None, :, c]).float()
    return acc * torch.tensor(1.0 / math.sqrt(d), device=q.device)


def _rows(B, N, width=1):
    """Batch slices of at most about 2^27 scores."""
    step = max(1, (1 << 27) // (N * N * width))
    return [slice(b, min(B, b + step)) for b in range(0, B, step)]


def _topk_sets(q, k, kk):
    """The retained sets, best first."""
    B, N, _ = q.shape
    sets = []
    for r in _rows(B, N, 2):
        s = _canonical_scores(q[r].float(), k[r].float())
        s.diagonal(dim1=1, dim2=2).fill_(float("-inf"))
        if kk <= 8:  # first maximum each time: ties to the lower index
            got = []
            for _ in range(kk):
                best = s.amax(-1, keepdim=True)
                at = torch.where(s == best, torch.arange(N, device=q.device), N).amin(-1, keepdim=True)
                got.append(at)
                s.scatter_(-1, at, float("-inf"))
            sets.append(torch.cat(got, -1))
        else:
            sets.append(torch.sort(s, dim=-1, descending=True, stable=True).indices[..., :kk])
    return torch.cat(sets)


def _set_attention(q, k, v, idx):
    """Attention over the peer sets idx, differentiable, in q's precision."""
    B, N, d = q.shape
    kk = idx.shape[-1]
    flat = idx.reshape(B, N * kk, 1).expand(B, N * kk, d)
    kg = torch.gather(k, 1, flat).view(B, N, kk, d)
    vg = torch.gather(v, 1, flat).view(B, N, kk, d)
    w = torch.softmax((q.unsqueeze(2) * kg).sum(-1) / math.sqrt(d), -1)
    return (w.unsqueeze(-1) * vg).sum(2)


def _dense_attention(q, k, v):
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[-1])
    eye = torch.eye(q.shape[1], dtype=torch.bool, device=q.device)
    return torch.matmul(torch.softmax(s.masked_fill(eye, float("-inf")), -1), v)


def _attention(q, k, v, idx):
    return _dense_attention(q, k, v) if idx is None else _set_attention(q, k, v, idx)


def _in_slices(q, k, v, idx, dout=None):
    """Attention (and, given dout, its gradients) in 64 bits, in batch slices."""
    B, N, d = q.shape
    outs = []
    for r in _rows(B, N, 2 if idx is None else 1 + 4 * idx.shape[-1] * d // N):
        a = [t[r].double().requires_grad_(dout is not None) for t in (q, k, v)]
        out = _attention(*a, None if idx is None else idx[r])
        grads = () if dout is None else torch.autograd.grad(out, a, dout[r].double())
        outs.append((out.detach(), *grads))
    return [torch.cat(t) for t in zip(*outs)]


def _morton_sets(pos, k, bits):
    """The k curve neighbours of each agent: quantisation in fp32 as the
    selector defines it, then whole numbers."""
    B, N, _ = pos.shape
    lo, hi = pos.amin(1, keepdim=True), pos.amax(1, keepdim=True)
    cell = ((pos - lo) / (hi - lo).clamp_min(1e-6) * (2 ** bits - 1)).long().clamp(0, 2 ** bits - 1)
    code = torch.zeros(B, N, dtype=torch.int64, device=pos.device)
    for b in range(bits):
        for axis in (0, 1):
            code |= ((cell[..., axis] >> b) & 1) << (2 * b + axis)
    order = torch.sort(code, dim=-1, stable=True).indices
    rank = torch.empty_like(order).scatter_(1, order, torch.arange(N, device=pos.device).expand(B, N))
    up = (k + 1) // 2
    steps = torch.tensor(list(range(1, up + 1)) + list(range(-1, -(k - up) - 1, -1)), device=pos.device)
    at = (rank.unsqueeze(-1) + steps) % N
    return torch.gather(order, 1, at.reshape(B, N * k)).view(B, N, k)


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "module":
        return _exact_module(case, seed, s["x"], s["dout"])
    q, k, v = s["q"], s["k"], s["v"]
    if kind == "dense":
        return {"out": _in_slices(q, k, v, None)[0]}
    if kind in ("topk", "stream"):
        return {"out": _in_slices(q, k, v, _topk_sets(q, k, case["k"]))[0], "idx": None}
    if kind == "zorder":
        return {"out": _in_slices(q, k, v, _morton_sets(s["pos"], case["k"], 16))[0], "idx": None}
    if kind == "prescore":
        if case["selector"] == "morton_window":
            idx = _morton_sets(s["pos"], case["k"], 10)
        elif case["selector"] == "radius_knn":
            p = s["pos"]
            dist = (p[:, :, None] - p[:, None]).square()
            dist = dist[..., 0] + dist[..., 1]
            dist.diagonal(dim1=1, dim2=2).fill_(float("inf"))
            idx = torch.sort(dist, dim=-1, stable=True).indices[..., :case["k"]]
        else:  # the grid's capacity cut is a definition, not arithmetic
            return None
        return {"out": _in_slices(q, k, v, idx)[0], "idx": None}
    idx = None if case["core"] == "dense" else _topk_sets(q, k, case["k"])
    out, dq, dk, dv = _in_slices(q, k, v, idx, s["dout"])
    got = {"out": out, "dq": dq, "dk": dk, "dv": dv}
    return got if idx is None else {**got, "idx": None}


def _exact_module(case, seed, x, dout):
    """The block in 64 bits. Its sets are those of the fp32 heads it ranks."""
    m = _module(case, seed)
    d = case["d"]
    idx = None
    if case["mode"] != "dense":
        with torch.no_grad():
            q, k, _ = m.qkv(x).split(d, -1)
        idx = _topk_sets(q.contiguous(), k.contiguous(), case["k"])
    params = [p.detach().double().requires_grad_(True) for n, p in m.named_parameters()
              if not n.startswith("k_gate")]
    wq, bq, wp, bp = params
    x = x.detach().double().requires_grad_(True)
    q, k, v = torch.nn.functional.linear(x, wq, bq).split(d, -1)
    msg = torch.nn.functional.linear(torch.nn.functional.gelu(_attention(q, k, v, idx)), wp, bp)
    grads = torch.autograd.grad(msg, [x, *params], dout.double())
    return {"msg": msg.detach(), "grads": list(grads)}
