"""The calls whose speed matters to a user of this repository, over their range of sizes.

Every case is one pass through the public entry points of ``ringmaster_amd`` as a training
program makes it: attention blocks and rings forward and backward, the ring's explicit step
(block, merge, backward with the global out / lse), the zigzag shard, the linear scan and the
Mamba2 context-parallel pieces. ``listed()`` names twelve of them, ``draw`` gives more of the
same ranges, ``exact`` is what a pass should return, in 64 bits and plain torch.
"""

from __future__ import annotations

import math

import torch

BF16, F16 = "bf16", "f16"
_DT = {BF16: torch.bfloat16, F16: torch.float16}


def listed():
    return [
        # The smallest call: a short block of a GQA model, where launches and host time count.
        dict(name="block_small", kind="block", b=2, sq=321, sk=321, hq=8, hkv=2, d=64, causal=True,
             dtype=BF16, window=0, dropout=0.0),
        # One rank's diagonal block at a 4k context, 32 query heads on 8 KV heads.
        dict(name="block_4k", kind="block", b=1, sq=4096, sk=4096, hq=32, hkv=8, d=128, causal=True,
             dtype=BF16, window=0, dropout=0.0),
        # fp16, a head dim below the kernel's, a sliding window, dropout, ragged length.
        dict(name="block_options", kind="block", b=2, sq=3001, sk=3001, hq=16, hkv=4, d=96,
             causal=True, dtype=F16, window=1023, dropout=0.1),
        # One explicit ring step at 16k per rank (non-causal, GQA 4:1): the block forward, its
        # merge into the running pair of a prior step, the backward with the global out / lse.
        dict(name="step_16k", kind="step", b=1, sq=16384, sk=16384, hq=32, hkv=8, d=128, dtype=BF16),
        # Two ranks at a 4k sequence, 8 heads of 64: a small zigzag ring, forward and backward.
        dict(name="ring_4k", kind="ring", layout="zigzag", P=2, b=1, L=2048, hq=8, hkv=8, d=64,
             dtype=BF16, docs=0),
        # The headline: 8 ranks at 16k each, 16 heads of 128, zigzag, forward and backward.
        dict(name="ring_128k", kind="ring", layout="zigzag", P=8, b=1, L=16384, hq=16, hkv=16,
             d=128, dtype=BF16, docs=0),
        # Packed documents (lognormal lengths) over 4 ranks and 64k tokens.
        dict(name="ring_packed", kind="ring", layout="zigzag", P=4, b=1, L=16384, hq=32, hkv=8,
             d=128, dtype=BF16, docs=2048),
        # The data path in front of the headline ring: q, k, v to their ranks, out back.
        dict(name="shard_128k", kind="shard", P=8, b=1, S=131072, row=2048, dtype=BF16, tensors=3),
        # State passing over 256 chunk states of 64 heads x 64 x 128 (one decay per head).
        dict(name="scan_states", kind="scan", b=1, L=256, d=524288, G=64, world=8),
        # Mamba2 layer, 8 ranks of 8192 tokens, 64 heads of 64, d_state 128: chunk decay,
        # entering states and the output / state correction, forward and backward.
        dict(name="mamba_cp", kind="mamba_cp", P=8, b=1, T=8192, H=64, D=64, G=1, N=128),
        # The same layer's shard states, forward and backward.
        dict(name="mamba_state", kind="mamba_state", P=8, b=1, T=8192, H=64, D=64, G=1, N=128),
        # The same layer's convolution over x, B and C channels, with its halos.
        dict(name="mamba_conv", kind="conv", P=8, b=1, C=4352, L=8192, W=4, act="silu", docs=0),
    ]


# ------------------------------------------------------------------------------- draws
def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block"] * 4 + ["ring"] * 4 + ["step", "shard", "scan", "mamba_cp",
                                                      "mamba_state", "conv"])
    if kind == "block":
        # lengths of short batches up to 8k, square or the halves a zigzag step attends
        sq = _log(rng, 64, 8192)
        sk = rng.choice([sq, sq, sq, max(1, sq // 2), 2 * sq])
        hq = rng.choice([4, 8, 16, 32])
        d = rng.choice([64, 64, 96, 128, 128, 128, 192, 256])
        causal = rng.random() < 0.6 and sk >= sq
        return dict(kind=kind, b=rng.choice([1, 1, 2]), sq=sq, sk=sk, hq=hq,
                    hkv=max(1, hq // rng.choice([1, 2, 4, 8])), d=d, causal=causal,
                    dtype=rng.choice([BF16, BF16, F16]),
                    window=_log(rng, 64, 4096) if causal and rng.random() < 0.3 else 0,
                    dropout=0.1 if rng.random() < 0.2 else 0.0)
    if kind == "step":
        sq = _log(rng, 512, 16384)
        hq = rng.choice([8, 16, 32])
        return dict(kind=kind, b=1, sq=sq, sk=rng.choice([sq, max(1, sq // 2)]), hq=hq,
                    hkv=max(1, hq // rng.choice([1, 4])), d=128, dtype=BF16)
    if kind == "ring":
        hq = rng.choice([4, 8, 16, 32])
        layout = rng.choice(["zigzag", "zigzag", "zigzag", "contiguous", "distflash", "allgather"])
        docs = _log(rng, 128, 2048) if layout != "allgather" and rng.random() < 0.4 else 0
        return dict(kind=kind, layout=layout, P=rng.choice([2, 4, 8]), b=rng.choice([1, 1, 2]),
                    L=2 * _log(rng, 64, 2048), hq=hq, hkv=max(1, hq // rng.choice([1, 2, 4])),
                    d=rng.choice([64, 128, 128, 256]), dtype=rng.choice([BF16, BF16, F16]), docs=docs)
    if kind == "shard":
        row = rng.choice([0, 2048, 4096, 1024 + 8 * rng.randint(0, 64)])
        return dict(kind=kind, P=rng.choice([2, 4, 8]), b=rng.choice([1, 2]),
                    S=_log(rng, 1000, 131072), row=row, dtype=BF16, tensors=rng.choice([1, 3]))
    if kind == "scan":
        if rng.random() < 0.5:  # chunk states: few steps, many channels
            n = 2 * 64 * 128
            H = rng.choice([8, 16, 32, 64])
            return dict(kind=kind, b=1, L=8 * _log(rng, 2, 32), d=H * n // 2, G=H,
                        world=rng.choice([1, 2, 8]))
        d = rng.choice([64, 128, 256, 512, 1024, 4096])  # token-level recurrences
        return dict(kind=kind, b=rng.choice([1, 2]), L=8 * _log(rng, 64, 8192), d=d,
                    G=rng.choice([d, max(1, d // 64)]), world=rng.choice([1, 2, 8]))
    if kind == "conv":
        return dict(kind=kind, P=rng.choice([2, 4, 8]), b=rng.choice([1, 2]),
                    C=rng.choice([768, 1792, 2304, 4352]), L=8 * _log(rng, 16, 1024), W=4,
                    act=rng.choice(["silu", "silu", ""]), docs=rng.choice([0, 0, 300]))
    H = rng.choice([8, 16, 24, 32, 64])
    return dict(kind=kind, P=rng.choice([2, 4, 8]), b=rng.choice([1, 2]), T=_log(rng, 128, 4096),
                H=H, D=rng.choice([64, 64, 128]), G=rng.choice([1, 1, 2]), N=rng.choice([64, 128]))


# ------------------------------------------------------------------------------- inputs
class _Gen:
    """Seeded values on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, shape, dtype=torch.float32, scale=1.0):
        x = torch.empty(shape, dtype=dtype, device="cuda")
        flat = x.view(-1)
        step = 1 << 27  # a piece at a time, drawn in fp32
        for i in range(0, flat.numel(), step):
            n = min(step, flat.numel() - i)
            flat[i:i + n] = torch.randn(n, generator=self.g, device="cuda") * scale
        return x

    def uniform(self, shape, lo, hi):
        return torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo


def _doc_lens(total, median, seed):
    """Lognormal document lengths (sigma 1, at least median / 16, at most 8 medians) that
    cover ``total``; the last one is cut to the remainder."""
    g = torch.Generator().manual_seed(seed)
    lens, acc = [], 0
    while acc < total:
        z = torch.randn(1, generator=g).item()
        n = int(min(max(round(median * math.exp(z)), max(1, median // 16)), 8 * median))
        n = min(n, total - acc)
        lens.append(n)
        acc += n
    return lens


def _ring_docs(case, seed):
    """Documents of the packed ring: every row its own over contiguous shards, the rows of
    the other layouts share them. A list of rows of lengths (None: not packed)."""
    if not case["docs"]:
        return None
    S = case["P"] * case["L"]
    rows = case["b"] if case["layout"] == "contiguous" else 1
    return [_doc_lens(S, case["docs"], 1000 * seed + i) for i in range(rows)]


def _cu(rows):
    """cu_seqlens over the concatenated rows (zero-length documents nowhere)."""
    lens = [n for row in rows for n in row]
    return torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32, device="cuda")


def _mamba_steps(g, H):
    """A and dt_bias of a Mamba2 layer: A = -exp(U(log 1, log 16)), softplus(dt_bias)
    log-uniform in [1e-3, 1e-1]."""
    A = -torch.exp(g.uniform((H,), 0.0, math.log(16.0)))
    dt = torch.exp(g.uniform((H,), math.log(1e-3), math.log(1e-1)))
    return A, torch.log(torch.expm1(dt))


def prepare(case, seed):
    g = _Gen(seed)
    st = {"case": case}
    kind = case["kind"]
    if kind in ("block", "step"):
        dt = _DT[case["dtype"]]
        b, sq, sk, hq, hkv, d = (case[x] for x in ("b", "sq", "sk", "hq", "hkv", "d"))
        st["q"] = g.normal((b, sq, hq, d), dt)
        st["k"], st["v"] = g.normal((b, sk, hkv, d), dt), g.normal((b, sk, hkv, d), dt)
        st["dout"] = g.normal((b, sq, hq, d), dt)
        st["seed"] = 7919 * seed + 1
        if kind == "step":
            # what a prior step over as many keys leaves: an average of about sk / e values
            st["prior_out"] = g.normal((b, sq, hq, d), dt, scale=math.sqrt(math.e / sk))
            st["prior_lse"] = math.log(sk) + 0.5 + g.normal((b, hq, sq), scale=0.05)
        else:
            for x in "qkv":
                st[x].requires_grad_(True)
    elif kind == "ring":
        dt = _DT[case["dtype"]]
        P, b, L, hq, hkv, d = (case[x] for x in ("P", "b", "L", "hq", "hkv", "d"))
        st["q"] = g.normal((P, b, hq, L, d), dt).requires_grad_(True)
        st["k"] = g.normal((P, b, hkv, L, d), dt).requires_grad_(True)
        st["v"] = g.normal((P, b, hkv, L, d), dt).requires_grad_(True)
        st["dout"] = g.normal((P, b, L, hq, d), dt)
        rows = _ring_docs(case, seed)
        st["cu"] = None if rows is None else _cu(rows)
    elif kind == "shard":
        P, b, S, row = case["P"], case["b"], case["S"], case["row"]
        if row == 0:  # token ids
            st["x"] = [torch.randint(0, 1 << 17, (b, S), generator=g.g, device="cuda")
                       for _ in range(case["tensors"])]
            st["back"] = torch.randint(0, 1 << 17, (P, b, 2 * -(-S // (2 * P))), generator=g.g,
                                       device="cuda")
        else:
            st["x"] = [g.normal((b, S, row), _DT[case["dtype"]]) for _ in range(case["tensors"])]
            st["back"] = g.normal((P, b, 2 * -(-S // (2 * P)), row), _DT[case["dtype"]])
    elif kind == "scan":
        b, L, d, G = case["b"], case["L"], case["d"], case["G"]
        # decays of a gated recurrence: sigmoid of N(2, 1.5)
        st["a"] = torch.sigmoid(g.normal((b, L, G)) * 1.5 + 2.0).requires_grad_(True)
        st["x"] = g.normal((b, L, d)).requires_grad_(True)
        st["dh"] = g.normal((b, L, d))
    elif kind == "conv":
        P, b, C, L, W = (case[x] for x in ("P", "b", "C", "L", "W"))
        st["x"] = g.normal((P, b, C, L), torch.bfloat16).requires_grad_(True)
        st["w"] = g.normal((C, W), torch.bfloat16, scale=1 / math.sqrt(W)).requires_grad_(True)
        st["bias"] = g.normal((C,), torch.bfloat16, scale=0.1).requires_grad_(True)
        st["dy"] = g.normal((P, b, C, L), torch.bfloat16)
        st["cu"] = _cu([_doc_lens(P * L, case["docs"], seed)]) if case["docs"] else None
    else:
        P, b, T, H, D, G, N = (case[x] for x in ("P", "b", "T", "H", "D", "G", "N"))
        A, bias = _mamba_steps(g, H)
        st["A"], st["dt_bias"] = A.requires_grad_(True), bias.requires_grad_(True)
        st["dt"] = g.normal((P, b, T, H), torch.bfloat16).requires_grad_(True)
        st["bc"] = g.normal((P, b, T, G, N), torch.bfloat16).requires_grad_(True)
        st["x"] = g.normal((P, b, T, H, D), torch.bfloat16).requires_grad_(True)
        if kind == "mamba_cp":
            st["state"] = g.normal((P, b, H, D, N)).requires_grad_(True)
            st["dy"] = g.normal((P, b, T, H, D), torch.bfloat16)
        st["dstate"] = g.normal((P, b, H, D, N))
    return st


# ------------------------------------------------------------------------------- passes
def _ring_call(case):
    from ringmaster_amd import ring

    if case["layout"] == "zigzag":
        return lambda q, k, v, cu: ring.zigzag_ring_attention(q, k, v, cu_seqlens=cu)
    if case["layout"] == "distflash":
        return lambda q, k, v, cu: ring.distflash_attention(q, k, v, scaling=None, cu_seqlens=cu)
    if case["layout"] == "contiguous" and case["docs"]:
        return lambda q, k, v, cu: ring.varlen_ring_attention(q, k, v, scaling=None, cu_seqlens=cu)
    method = "allgather" if case["layout"] == "allgather" else "alltoall"
    return lambda q, k, v, cu: ring.ring_attention(q, k, v, causal=True, rotate_method=method)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "block":
        from ringmaster_amd.ring import PROVIDERS

        q, k, v = state["q"], state["k"], state["v"]
        window = (case["window"], 0) if case["window"] else None
        out, lse = PROVIDERS["mi355x_hip"](q, k, v, causal=case["causal"], scaling=None,
                                           dropout=case["dropout"], window=window,
                                           dropout_seed=state["seed"] if case["dropout"] else None)
        dq, dk, dv = torch.autograd.grad(out, (q, k, v), state["dout"])
        return {"out": out.detach(), "lse": lse.detach(), "dq": dq, "dk": dk, "dv": dv}
    if kind == "step":
        from ringmaster_amd.ring import flash_ops, update_out_and_lse

        fwd, bwd = flash_ops()
        q, k, v = state["q"], state["k"], state["v"]
        scale = case["d"] ** -0.5
        out, lse = update_out_and_lse(None, None, state["prior_out"], state["prior_lse"])
        bo, bl, _, _ = fwd(q, k, v, 0.0, scale, False)
        out, lse = update_out_and_lse(out, lse, bo, bl)
        o16 = out.to(q.dtype)
        glse = lse.squeeze(-1).transpose(1, 2).contiguous()
        dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        bwd(state["dout"], q, k, v, o16, glse, dq, dk, dv, 0.0, scale, False)
        return {"out": out, "lse": lse, "dq": dq, "dk": dk, "dv": dv}
    if kind == "ring":
        q, k, v = state["q"], state["k"], state["v"]
        out = _ring_call(case)(q, k, v, state["cu"])
        dq, dk, dv = torch.autograd.grad(out, (q, k, v), state["dout"])
        return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv}
    if kind == "shard":
        from ringmaster_amd.shard import zigzag_shard, zigzag_unshard

        return [*(zigzag_shard(x, case["P"]) for x in state["x"]),
                zigzag_unshard(state["back"], case["S"])]
    if kind == "scan":
        from ringmaster_amd.strategies.state_passing import cp_linear_scan

        h = cp_linear_scan(state["a"], state["x"], world=case["world"])
        da, db = torch.autograd.grad(h, (state["a"], state["x"]), state["dh"])
        return {"h": h.detach(), "da": da, "db": db}
    if kind == "conv":
        from ringmaster_amd.strategies.mamba import causal_conv1d_cp

        args = (state["x"], state["w"], state["bias"])
        y = causal_conv1d_cp(*args, activation=case["act"] or None, cu_seqlens=state["cu"])
        dx, dw, db = torch.autograd.grad(y, args, state["dy"])
        return {"y": y.detach(), "dx": dx, "dw": dw, "db": db}
    if kind == "mamba_cp":
        from ringmaster_amd.strategies.mamba import mamba2_cp_apply

        args = (state["x"], state["state"], state["dt"], state["A"], state["bc"])
        y, h = mamba2_cp_apply(*args, dt_bias=state["dt_bias"], dt_softplus=True)
        grads = torch.autograd.grad((y, h), (*args, state["dt_bias"]), (state["dy"], state["dstate"]))
        return {"y": y.detach(), "h": h.detach(), **dict(zip(
            ("dx", "dstate", "ddt", "dA", "dC", "dbias"), grads))}
    from ringmaster_amd.strategies.mamba import mamba2_chunk_state

    args = (state["x"], state["dt"], state["A"], state["bc"])
    s = mamba2_chunk_state(*args, dt_bias=state["dt_bias"], dt_softplus=True)
    grads = torch.autograd.grad(s, (*args, state["dt_bias"]), state["dstate"])
    return {"state": s.detach(), **dict(zip(("dx", "ddt", "dA", "dB", "dbias"), grads))}


# ------------------------------------------------------------------------------- work
def _band_pairs(sq, sk, causal, window):
    """(query, key) pairs of a bottom-right aligned block."""
    if not causal:
        return sq * sk
    off, tot = sk - sq, 0
    for i in range(sq):
        hi = min(sk, i + off + 1)
        lo = max(0, i + off - window) if window else 0
        tot += max(0, hi - lo)
    return tot


def _ring_pairs(case):
    S = case["P"] * case["L"]
    if not case["docs"]:
        return case["b"] * S * (S + 1) // 2
    rows = _ring_docs(case, 0)  # the documents of one seed: their mean differs little
    return case["b"] * sum(n * (n + 1) // 2 for row in rows for n in row) // len(rows)


def work(case):
    kind = case["kind"]
    if kind in ("block", "step"):
        pairs = case["b"] * _band_pairs(case["sq"], case["sk"], case.get("causal", False),
                                        case.get("window", 0))
        nq = case["b"] * case["sq"] * case["hq"]
        nk = case["b"] * case["sk"] * case["hkv"]
        # q, dout in, out, dq out; k, v in, dk, dv out; lse (and a step's prior pair and fp32 out)
        nbytes = 2 * case["d"] * 4 * (nq + nk) + 4 * nq
        if kind == "step":
            nbytes += nq * (2 * case["d"] + 2 * case["d"] + 4)
        return {"bytes": nbytes, "flops": 14 * case["d"] * case["hq"] * pairs}
    if kind == "ring":
        n = case["P"] * case["b"] * case["L"] * (case["hq"] + case["hkv"])
        return {"bytes": 2 * case["d"] * 4 * n, "flops": 14 * case["d"] * case["hq"] * _ring_pairs(case)}
    if kind == "shard":
        rb = 8 if case["row"] == 0 else 2 * case["row"]
        local = 2 * -(-case["S"] // (2 * case["P"]))
        full = case["b"] * case["P"] * local * rb
        part = case["b"] * case["S"] * rb
        return {"bytes": case["tensors"] * (part + full) + 2 * part, "flops": 0}
    if kind == "scan":
        n, na = case["b"] * case["L"] * case["d"], case["b"] * case["L"] * case["G"]
        return {"bytes": 4 * (5 * n + 3 * na), "flops": 7 * n}
    if kind == "conv":
        n = case["P"] * case["b"] * case["C"] * case["L"]
        return {"bytes": 2 * 5 * n, "flops": 2 * 4 * case["W"] * n}
    rows, T, H, D, G, N = case["P"] * case["b"], case["T"], case["H"], case["D"], case["G"], case["N"]
    tok, st = rows * T, rows * H * D * N * 4
    small = tok * (3 * 2 * H + 3 * 2 * G * N)  # dt twice and its gradient; B or C twice, its gradient
    if kind == "mamba_cp":
        # x, dy in, y, dx out; states in, out, their gradients in and out
        return {"bytes": 2 * 4 * tok * H * D + 4 * st + small, "flops": 2 * 4 * tok * H * D * N}
    return {"bytes": 2 * 3 * tok * H * D + 2 * st + small, "flops": 2 * 3 * tok * H * D * N}


def tolerance(case):
    # About four times the largest error of any output against 64 bits, over the listed and
    # some dozens of drawn cases: attention 2.5e-3 in bf16 and 3.3e-4 in fp16 (their 2^-9 and
    # 2^-12 roundings of P, dS and the results), the convolution 1.7e-3 and the Mamba2 pieces
    # 2.9e-3 (bf16 results and operands), the fp32 scan 1.2e-7 (to 1e-5: other orders of sums).
    kind = case["kind"]
    if kind == "shard":
        return "exact"
    if kind == "scan":
        return {"rel": 1e-5}
    if kind == "conv":
        return {"rel": 7e-3}
    if case.get("dtype") == F16:
        return {"rel": 1.3e-3}
    return {"rel": 1e-2 if "dtype" in case else 1.2e-2}


# ------------------------------------------------------------------------------- 64 bits
def _f64(x):
    return x.detach().double()


def _mix32(h):
    """The 32-bit finalizer of MurmurHash3 on int64 tensors holding 32-bit values."""
    m = 0xFFFFFFFF
    h = h ^ (h >> 16)
    h = (h * 0x85EBCA6B) & m
    h = h ^ (h >> 13)
    h = (h * 0xC2B2AE35) & m
    return h ^ (h >> 16)


def _keep(seed, p, bh, q0, q1, sk):
    """The dropout mask of queries [q0, q1) of (batch, head) index ``bh``: the hash that the C
    header specifies (RMX_DROPOUT)."""
    m = 0xFFFFFFFF
    one = lambda x: torch.tensor(x & m, dtype=torch.int64, device="cuda")  # noqa: E731
    mix = _mix32(one(seed) ^ _mix32(one(seed >> 32) ^ one(bh * 0x9E3779B9)))
    q = (torch.arange(q0, q1, device="cuda") * 0x85EBCA77) & m
    k = (torch.arange(sk, device="cuda") * 0xC2B2AE3D) & m
    thr = math.floor(torch.tensor(p, dtype=torch.float32).double().item() * 4294967296.0)
    return _mix32(mix ^ q[:, None] ^ k[None, :]) >= thr


def _attend(q, k, v, do, scale, causal, window=0, drop=None, prior=None):
    """One head in 64 bits, q [sq, d], k/v [sk, d], bottom-right aligned: (out, lse, dq, dk, dv).
    ``drop`` is None or (seed, p, batch-head index); ``prior`` an (out, lse) merged in first
    (the gradients then use the merged pair). Query rows are taken in pieces."""
    sq, sk = q.shape[0], k.shape[0]
    off = sk - sq
    out, lse, dq = torch.empty_like(q), q.new_empty(sq), torch.empty_like(q)
    dk, dv = torch.zeros_like(k), torch.zeros_like(v)
    step = max(256, min(sq, (1 << 26) // max(sk, 1)))
    for i in range(0, sq, step):
        j = min(sq, i + step)
        hi = min(sk, j + off) if causal else sk
        lo = max(0, i + off - window) if window else 0
        kk, vv = k[lo:hi], v[lo:hi]
        s = (q[i:j] @ kk.t()) * scale
        if causal:
            rows = torch.arange(i, j, device="cuda")[:, None] + off
            cols = torch.arange(lo, hi, device="cuda")[None, :]
            bad = cols > rows
            if window:
                bad |= rows - cols > window
            s.masked_fill_(bad, float("-inf"))
        bl = torch.logsumexp(s, 1)
        ls = bl if prior is None else torch.logaddexp(bl, prior[1][i:j])
        p = torch.exp_(s.sub_(ls[:, None]))
        if drop is not None:
            keep = _keep(drop[0], drop[1], drop[2], i, j, sk)[:, lo:hi]
            m = keep.double() / (1.0 - torch.tensor(drop[1], dtype=torch.float32).double().item())
        pm = p if drop is None else p * m
        o = pm @ vv
        if prior is not None:
            o = o + prior[0][i:j] * torch.exp(prior[1][i:j] - ls)[:, None]
        g = do[i:j]
        dv[lo:hi] += pm.t() @ g
        dp = g @ vv.t()
        if drop is not None:
            dp *= m
        ds = p * dp.sub_((g * o).sum(1, keepdim=True)) * scale
        dq[i:j] = ds @ kk
        dk[lo:hi] += ds.t() @ q[i:j]
        out[i:j], lse[i:j] = o, ls
    return out, lse, dq, dk, dv


def _exact_block(case, st):
    b, sq, hq, hkv, d = (case[x] for x in ("b", "sq", "hq", "hkv", "d"))
    step = case["kind"] == "step"
    out, dq = (torch.empty((b, sq, hq, d), dtype=torch.float64, device="cuda") for _ in range(2))
    lse = torch.empty((b, hq, sq), dtype=torch.float64, device="cuda")
    dk, dv = (torch.zeros((b, case["sk"], hkv, d), dtype=torch.float64, device="cuda") for _ in range(2))
    for i in range(b):
        for h in range(hq):
            kh = h // (hq // hkv)
            prior = (_f64(st["prior_out"][i, :, h]), _f64(st["prior_lse"][i, h])) if step else None
            drop = (st["seed"], case["dropout"], i * hq + h) if case.get("dropout") else None
            o, l, a, c, e = _attend(_f64(st["q"][i, :, h]), _f64(st["k"][i, :, kh]),
                                    _f64(st["v"][i, :, kh]), _f64(st["dout"][i, :, h]), d ** -0.5,
                                    case.get("causal", False), case.get("window", 0), drop, prior)
            out[i, :, h], lse[i, h], dq[i, :, h] = o, l, a
            dk[i, :, kh] += c
            dv[i, :, kh] += e
    if step:
        lse = lse.transpose(1, 2).unsqueeze(-1).contiguous()
    return {"out": out, "lse": lse, "dq": dq, "dk": dk, "dv": dv}


def _rank_rows(case):
    """Global token of every local row of every rank, [P, L]."""
    P, L = case["P"], case["L"]
    if case["layout"] != "zigzag":
        return torch.arange(P * L, device="cuda").view(P, L)
    c = torch.arange(P * L, device="cuda").view(2 * P, L // 2)
    return torch.cat([c[:P], c[P:].flip(0)], 1)


def _exact_ring(case, st, seed):
    P, b, L, hq, hkv, d = (case[x] for x in ("P", "b", "L", "hq", "hkv", "d"))
    if b * hq * _ring_pairs(case) / b * d > 4e12:
        return None
    rows, S = _rank_rows(case).reshape(-1), P * L
    docs = _ring_docs(case, seed) or [[S]]

    def put(shape_h):
        return torch.zeros((P, b, shape_h, L, d), dtype=torch.float64, device="cuda")

    res = {"out": torch.empty((P, b, L, hq, d), dtype=torch.float64, device="cuda"),
           "dq": put(hq), "dk": put(hkv), "dv": put(hkv)}
    for i in range(b):
        lens = docs[i if len(docs) > 1 else 0]
        for h in range(hq):
            kh = h // (hq // hkv)

            def seq(x):  # [P, L, d] -> the sequence in order
                y = torch.empty((S, d), dtype=torch.float64, device="cuda")
                y[rows] = _f64(x).reshape(S, d)
                return y

            q, k, v = seq(st["q"][:, i, h]), seq(st["k"][:, i, kh]), seq(st["v"][:, i, kh])
            g = seq(st["dout"][:, i, :, h])
            parts, t = [], 0
            for n in lens:
                sl = slice(t, t + n)
                parts.append(_attend(q[sl], k[sl], v[sl], g[sl], d ** -0.5, True))
                t += n
            o, a, c, e = (torch.cat([p[x] for p in parts])[rows].view(P, L, d) for x in (0, 2, 3, 4))
            res["out"][:, i, :, h], res["dq"][:, i, h] = o, a
            res["dk"][:, i, kh] += c
            res["dv"][:, i, kh] += e
    return res


def _doubling_scan(a, b):
    """h_t = a_t h_{t-1} + b_t over dim 1 by doubling, in place of copies of a and b."""
    a, b = a.clone(), b.clone()
    s = 1
    while s < b.shape[1]:
        b[:, s:] = b[:, s:] + a[:, s:] * b[:, :-s]
        a[:, s:] = a[:, s:] * a[:, :-s]
        s *= 2
    return b


def _exact_scan(case, st):
    b, L, d, G = case["b"], case["L"], case["d"], case["G"]
    a = _f64(st["a"])
    h, da, db = (torch.empty((b, L, n), dtype=torch.float64, device="cuda") for n in (d, G, d))
    per = d // G
    step = max(1, (1 << 26) // (b * L * per))  # decay groups at a time
    for i in range(0, G, step):
        j = min(G, i + step)
        c = slice(i * per, j * per)
        ae = a[:, :, i:j].repeat_interleave(per, 2)
        hh = _doubling_scan(ae, _f64(st["x"][:, :, c]))
        # g_t = dh_t + a_{t+1} g_{t+1}: the same scan from the end
        an = torch.cat([ae[:, 1:], torch.zeros_like(ae[:, :1])], 1)
        gg = _doubling_scan(an.flip(1), _f64(st["dh"][:, :, c]).flip(1)).flip(1)
        prev = torch.cat([torch.zeros_like(hh[:, :1]), hh[:, :-1]], 1)
        h[:, :, c], db[:, :, c] = hh, gg
        da[:, :, i:j] = (gg * prev).view(b, L, j - i, per).sum(3)
    return {"h": h, "da": da, "db": db}


def _exact_conv(case, st, seed):
    P, b, C, L, W = (case[x] for x in ("P", "b", "C", "L", "W"))
    S = P * L
    w, bias = _f64(st["w"]).requires_grad_(True), _f64(st["bias"]).requires_grad_(True)
    doc = torch.zeros(S, dtype=torch.int64, device="cuda")
    if case["docs"]:
        lens = torch.tensor(_doc_lens(S, case["docs"], seed), device="cuda")
        doc = torch.repeat_interleave(torch.arange(lens.numel(), device="cuda"), lens)
    y, dx = (torch.empty((P, b, C, L), dtype=torch.float64, device="cuda") for _ in range(2))
    dw, db = torch.zeros_like(w), torch.zeros_like(bias)
    step = max(1, (1 << 26) // (S * b))
    for i in range(0, C, step):
        c = slice(i, min(C, i + step))
        n = c.stop - c.start
        x = _f64(st["x"][:, :, c]).permute(1, 2, 0, 3).reshape(b, n, S).requires_grad_(True)
        wc, bc = w[c].detach().requires_grad_(True), bias[c].detach().requires_grad_(True)
        z = bc[None, :, None].expand(b, n, S)
        for j in range(W):
            s = W - 1 - j  # tap j reads the token s before
            xs = x if s == 0 else torch.nn.functional.pad(x, (s, 0))[..., :S]
            same = torch.nn.functional.pad(doc, (s, 0), value=-1)[:S] == doc
            z = z + wc[None, :, j, None] * (xs * same)
        out = torch.nn.functional.silu(z) if case["act"] else z
        g = _f64(st["dy"][:, :, c]).permute(1, 2, 0, 3).reshape(b, n, S)
        gx, gw, gb = torch.autograd.grad(out, (x, wc, bc), g)
        y[:, :, c] = out.detach().view(b, n, P, L).permute(2, 0, 1, 3)
        dx[:, :, c] = gx.view(b, n, P, L).permute(2, 0, 1, 3)
        dw[c], db[c] = gw, gb
    return {"y": y, "dx": dx, "dw": dw.detach(), "db": db.detach()}


def _dt_eff(dt, bias):
    return torch.nn.functional.softplus(dt + bias)


def _exact_mamba_cp(case, st):
    P, b, T, H, D, G, N = (case[x] for x in ("P", "b", "T", "H", "D", "G", "N"))
    state, dt, A, C, bias = (_f64(st[x]).requires_grad_(True)
                             for x in ("state", "dt", "A", "bc", "dt_bias"))
    cum = torch.cumsum(_dt_eff(dt, bias) * A, 2)  # [P, b, T, H]
    decay = torch.exp(cum[:, :, -1])
    h_in = [torch.zeros_like(state[0])]
    for r in range(P - 1):
        h_in.append(h_in[-1] * decay[r][..., None, None] + state[r])
    h_in = torch.stack(h_in)
    hf = state + decay[..., None, None] * h_in
    y = torch.empty((P, b, T, H, D), dtype=torch.float64, device="cuda")
    # y's gradient by head, so that the products stay small: one graph over the head sums
    leaf = [x.detach().requires_grad_(True) for x in (cum, C, h_in)]
    for r in range(P):
        for i in range(b):
            for h in range(H):
                e = torch.exp(leaf[0][r, i, :, h])[:, None]
                yy = (leaf[1][r, i, :, h // (H // G)] @ leaf[2][r, i, h].t()) * e
                y[r, i, :, h] = _f64(st["x"][r, i, :, h]) + yy.detach()
                yy.backward(_f64(st["dy"][r, i, :, h]))
    grads = torch.autograd.grad((hf, cum, h_in), (state, dt, A, bias),
                                (_f64(st["dstate"]), leaf[0].grad, leaf[2].grad))
    return {"y": y, "h": hf.detach(), "dx": _f64(st["dy"]), "dstate": grads[0], "ddt": grads[1],
            "dA": grads[2], "dC": leaf[1].grad, "dbias": grads[3]}


def _exact_mamba_state(case, st):
    P, b, T, H, D, G, N = (case[x] for x in ("P", "b", "T", "H", "D", "G", "N"))
    dt, A, bias = (_f64(st[x]).requires_grad_(True) for x in ("dt", "A", "dt_bias"))
    e = _dt_eff(dt, bias)
    cum = torch.cumsum(e * A, 2)
    w = torch.exp(cum[:, :, -1:] - cum) * e  # [P, b, T, H]
    wl = w.detach()
    out, dx = torch.empty((P, b, H, D, N), dtype=torch.float64, device="cuda"), torch.empty(
        (P, b, T, H, D), dtype=torch.float64, device="cuda")
    dB = torch.zeros((P, b, T, G, N), dtype=torch.float64, device="cuda")
    gw = torch.empty_like(wl)
    for r in range(P):
        for i in range(b):
            for h in range(H):
                x, B = _f64(st["x"][r, i, :, h]), _f64(st["bc"][r, i, :, h // (H // G)])
                g, ww = _f64(st["dstate"][r, i, h]), wl[r, i, :, h][:, None]
                out[r, i, h] = (x * ww).t() @ B
                u = B @ g.t()  # [T, D]
                dx[r, i, :, h] = ww * u
                gw[r, i, :, h] = (x * u).sum(1)
                dB[r, i, :, h // (H // G)] += (x * ww) @ g
    gdt, gA, gb = torch.autograd.grad(w, (dt, A, bias), gw)
    return {"state": out, "dx": dx, "ddt": gdt, "dA": gA, "dB": dB, "dbias": gb}


def exact(case, seed):
    st = prepare(case, seed)
    kind = case["kind"]
    if kind in ("block", "step"):
        return _exact_block(case, st)
    if kind == "ring":
        return _exact_ring(case, st, seed)
    if kind == "scan":
        return _exact_scan(case, st)
    if kind == "conv":
        return _exact_conv(case, st, seed)
    if kind == "mamba_cp":
        return _exact_mamba_cp(case, st)
    if kind == "mamba_state":
        return _exact_mamba_state(case, st)
    return None
