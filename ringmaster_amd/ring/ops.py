"""Tensor-level wrappers of the batched block-attention kernels.

A *job* is one block problem of the C ABI: ``q[sq]`` attends ``k/v[sk]`` with
tensors given as ``[batch, seq, heads, dim]`` views (any strides on the first
three axes, contiguous ``dim``), lse-like tensors as ``[batch, heads, seq]``
views with a contiguous ``seq`` axis. All jobs of one call share the layout
(strides) of each tensor kind, as the per-rank views of one stacked tensor do,
and are launched together (up to 16 per kernel launch).
"""

from __future__ import annotations

import collections
import ctypes
import dataclasses
import threading

import torch

from ringmaster_amd import abi


@dataclasses.dataclass
class FwdJob:
    q: torch.Tensor
    k: torch.Tensor
    v: torch.Tensor
    mode: int = abi.FWD_WRITE
    out: torch.Tensor | None = None
    lse: torch.Tensor | None = None
    acc_out: torch.Tensor | None = None
    acc_lse: torch.Tensor | None = None
    # document-mask metadata: [sq] / [sk], or [batch, sq] / [batch, sk] per batch row
    q_gidx: torch.Tensor | None = None
    k_gidx: torch.Tensor | None = None
    q_doc: torch.Tensor | None = None
    k_doc: torch.Tensor | None = None
    window: int | None = None  # bound on pos_q - pos_k (global indices with document masks)
    drop_q0: int = 0  # dropout coordinates of the first query / key
    drop_k0: int = 0
    right: int = 0  # causal masks: bound on pos_k - pos_q (0: causal attention)


@dataclasses.dataclass
class BwdJob:
    q: torch.Tensor
    k: torch.Tensor
    v: torch.Tensor
    dout: torch.Tensor
    lse: torch.Tensor
    delta: torch.Tensor
    dq_mode: int
    dkv_mode: int
    nlse: torch.Tensor | None = None
    dq_acc: torch.Tensor | None = None
    dq: torch.Tensor | None = None
    dk_acc: torch.Tensor | None = None
    dv_acc: torch.Tensor | None = None
    dk: torch.Tensor | None = None
    dv: torch.Tensor | None = None
    q_gidx: torch.Tensor | None = None
    k_gidx: torch.Tensor | None = None
    q_doc: torch.Tensor | None = None
    k_doc: torch.Tensor | None = None
    window: int | None = None
    drop_q0: int = 0
    drop_k0: int = 0
    right: int = 0


def _i32_field(v, what):
    v = int(v)
    if not -(1 << 31) <= v < (1 << 31):
        raise ValueError(f"{what} {v} outside int32")
    return v


def _set_problem_extras(p, job):
    if job.window is not None:
        p.has_window, p.window_left = 1, _i32_field(job.window, "window bound")
    p.drop_q0 = _i32_field(job.drop_q0, "dropout query offset")
    p.drop_k0 = _i32_field(job.drop_k0, "dropout key offset")
    p.window_right = _i32_field(job.right, "right window bound")


def _set_dropout(lay, dropout):
    """``dropout``: None or (p, seed), seed a 64-bit integer."""
    if dropout is None or not dropout[0]:
        return
    p, seed = float(dropout[0]), int(dropout[1]) & ((1 << 64) - 1)
    lay.dropout_p = p
    lay.drop_seed_lo, lay.drop_seed_hi = seed & 0xFFFFFFFF, seed >> 32


_H = None  # the call's 16-bit element type (bf16 or fp16), the dtype of q

_ROLES = {
    # role -> (layout field prefix, number of strides, dtype)
    "q": ("q", 3, _H),
    "k": ("k", 3, _H),
    "v": ("v", 3, _H),
    "out": ("o", 3, _H),
    "dout": ("o", 3, _H),
    "dq": ("o", 3, _H),
    "acc_out": ("a", 3, torch.float32),
    "dq_acc": ("a", 3, torch.float32),
    "lse": ("l", 2, torch.float32),
    "acc_lse": ("l", 2, torch.float32),
    "delta": ("l", 2, torch.float32),
    "nlse": ("l", 2, torch.float32),
    "dk": ("dk", 3, _H),
    "dv": ("dk", 3, _H),
    "dk_acc": ("ka", 3, torch.float32),
    "dv_acc": ("ka", 3, torch.float32),
}

_DTYPES = {torch.bfloat16: abi.DTYPE_BF16, torch.float16: abi.DTYPE_F16}


def _fill_layout(jobs, batch, hq, hkv, head_dim, scale, mask, half=None) -> abi.AttnLayout:
    """The call's layout; ``half`` (default: the first job's q dtype) is the 16-bit type
    of q/k/v/out/dout and the 16-bit gradients."""
    half = half if half is not None else jobs[0].q.dtype
    if half not in _DTYPES:
        raise NotImplementedError(f"attention computes in bf16 or fp16 (got {half})")
    lay = abi.AttnLayout()
    lay.batch, lay.hq, lay.hkv, lay.head_dim = batch, hq, hkv, head_dim
    lay.scale = float(scale)
    lay.mask = mask
    lay.dtype = _DTYPES[half]
    seen: dict[str, tuple] = {}
    for job in jobs:
        for role, (prefix, n, dtype) in _ROLES.items():
            t = getattr(job, role, None)
            if t is None:
                continue
            dtype = half if dtype is _H else dtype
            if t.dtype != dtype:
                raise ValueError(f"{role} must be {dtype} (got {t.dtype})")
            abi.require_device(t)
            if n == 3:
                if t.dim() != 4 or t.stride(3) != 1:
                    raise ValueError(f"{role} must be [batch, seq, heads, dim] with contiguous dim")
                st = (t.stride(0), t.stride(1), t.stride(2))
            else:
                if t.dim() != 3 or (t.shape[2] > 1 and t.stride(2) != 1):
                    raise ValueError(f"{role} must be [batch, heads, seq] with contiguous seq")
                st = (t.stride(0), t.stride(1))
            if prefix in seen and seen[prefix] != st:
                raise ValueError(f"all {prefix}-kind tensors of one call must share strides "
                                 f"({seen[prefix]} vs {st} for {role})")
            seen[prefix] = st
    for prefix, st in seen.items():
        names = ("_sb", "_ss", "_sh") if len(st) == 3 else ("_sb", "_sh")
        for nm, s in zip(names, st):
            setattr(lay, prefix + nm, int(s))
    return lay


def _check_shapes(q, k, v, batch, hq, hkv, d):
    if q.shape[0] != batch or q.shape[2] != hq or q.shape[3] != d:
        raise ValueError(f"q shape {tuple(q.shape)} does not match the call layout")
    if k.shape[0] != batch or k.shape[2] != hkv or k.shape[3] != d or v.shape != k.shape:
        raise ValueError(f"k/v shapes {tuple(k.shape)}/{tuple(v.shape)} do not match")


def _int32(t):
    if t is None:
        return None
    if t.dtype != torch.int32 or t.stride(-1) != 1:
        raise ValueError("index tensors must be int32 with a contiguous last axis")
    abi.require_device(t)
    return t.data_ptr()


_META = ("q_gidx", "k_gidx", "q_doc", "k_doc")


def _set_meta_stride(lay, jobs, batch):
    """Document-mask metadata is [n] (every batch row shares it) or [batch, n] (per row,
    ring/loop.py:178): the layout's m_sb is the row stride, which all of a call's
    per-row arrays must share."""
    strides = set()
    for j in jobs:
        for name in _META:
            t = getattr(j, name)
            if t is None:
                continue
            if t.dim() == 1 or (t.dim() == 2 and t.shape[0] == 1):
                strides.add(0)
            elif t.dim() == 2 and t.shape[0] == batch:
                strides.add(t.stride(0))
            else:
                raise ValueError(f"{name} must be [n] or [batch, n] (got {tuple(t.shape)})")
    if len(strides) > 1:
        raise ValueError("the document metadata of one call must share its row stride")
    lay.m_sb = int(strides.pop()) if strides else 0


def _pack_fwd(jobs, scale, mask, dropout):
    """The (layout, problem array) of one rmx_attn_fwd call."""
    q0, k0 = jobs[0].q, jobs[0].k
    batch, hq, d, hkv = q0.shape[0], q0.shape[2], q0.shape[3], k0.shape[2]
    for j in jobs:
        _check_shapes(j.q, j.k, j.v, batch, hq, hkv, d)
    lay = _fill_layout(jobs, batch, hq, hkv, d, scale, mask)
    _set_dropout(lay, dropout)
    _set_meta_stride(lay, jobs, batch)
    arr = (abi.FwdProblem * len(jobs))()
    for i, j in enumerate(jobs):
        p = arr[i]
        p.q, p.k, p.v = j.q.data_ptr(), j.k.data_ptr(), j.v.data_ptr()
        p.out, p.lse = abi.ptr(j.out), abi.ptr(j.lse)
        p.acc_out, p.acc_lse = abi.ptr(j.acc_out), abi.ptr(j.acc_lse)
        p.q_gidx, p.k_gidx = _int32(j.q_gidx), _int32(j.k_gidx)
        p.q_doc, p.k_doc = _int32(j.q_doc), _int32(j.k_doc)
        p.sq, p.sk, p.mode = j.q.shape[1], j.k.shape[1], j.mode
        _set_problem_extras(p, j)
    return lay, arr


def attn_fwd(jobs: list[FwdJob], *, scale: float, mask: int, dropout=None) -> None:
    """Launch the batched block forward (rmx_attn_fwd) for ``jobs``; ``dropout`` is None or
    (p, seed)."""
    if not jobs:
        return
    lay, arr = _pack_fwd(jobs, scale, mask, dropout)
    abi.check(abi.lib().rmx_attn_fwd(ctypes.byref(lay), arr, len(jobs), abi.stream_of(jobs[0].q)))


def attn_bwd_delta(out: torch.Tensor, dout: torch.Tensor, delta: torch.Tensor, hkv: int,
                   lse: torch.Tensor | None = None, nlse: torch.Tensor | None = None) -> None:
    """delta[b, h, s] = sum_d dout * out (fp32). dout: [b, s, h, d] bf16 or fp16; out: the same
    type with the strides of dout, or the fp32 final out (any strides with a contiguous dim). With ``nlse``
    (and the global ``lse``), also nlse = -lse * log2(e), which the dK/dV kernel reads; lse,
    delta and nlse must share their strides."""
    batch, sq, hq, d = dout.shape
    if out.shape != dout.shape:
        raise ValueError("out and dout must share their shape")
    f32 = out.dtype == torch.float32
    if not f32 and (out.stride() != dout.stride() or out.dtype != dout.dtype):
        raise ValueError("a 16-bit out must share dout's type and strides")
    if (nlse is None) != (lse is None):
        raise ValueError("lse and nlse go together")
    if nlse is not None and (lse.shape != delta.shape or nlse.shape != delta.shape):
        raise ValueError("lse, delta and nlse must share their shape")

    def layout():
        job = FwdJob(q=dout, k=dout[:, :0, :hkv], v=dout[:, :0, :hkv], out=dout, lse=delta,
                     acc_out=out if f32 else None)
        jobs = [job]
        if nlse is not None:
            jobs += [FwdJob(q=dout, k=job.k, v=job.v, lse=lse), FwdJob(q=dout, k=job.k, v=job.v, lse=nlse)]
        return _fill_layout(jobs, batch, hq, hkv, d, 1.0, abi.MASK_FULL)

    lay = plan(("delta", hkv, signature(out, dout, delta, lse, nlse)), layout)
    abi.check(abi.lib().rmx_attn_bwd_delta(ctypes.byref(lay), out.data_ptr(), int(f32),
                                           dout.data_ptr(), delta.data_ptr(), abi.ptr(lse),
                                           abi.ptr(nlse), sq, abi.stream_of(dout)))


def _pack_bwd(jobs, scale, mask, dropout):
    """The (layout, problem array) of one rmx_attn_bwd call."""
    q0, k0 = jobs[0].q, jobs[0].k
    batch, hq, d, hkv = q0.shape[0], q0.shape[2], q0.shape[3], k0.shape[2]
    for j in jobs:
        _check_shapes(j.q, j.k, j.v, batch, hq, hkv, d)
    lay = _fill_layout(jobs, batch, hq, hkv, d, scale, mask)
    _set_dropout(lay, dropout)
    _set_meta_stride(lay, jobs, batch)
    arr = (abi.BwdProblem * len(jobs))()
    for i, j in enumerate(jobs):
        p = arr[i]
        p.q, p.k, p.v, p.dout = j.q.data_ptr(), j.k.data_ptr(), j.v.data_ptr(), j.dout.data_ptr()
        p.lse, p.delta, p.nlse = j.lse.data_ptr(), j.delta.data_ptr(), abi.ptr(j.nlse)
        p.dq_acc, p.dq = abi.ptr(j.dq_acc), abi.ptr(j.dq)
        p.dk_acc, p.dv_acc = abi.ptr(j.dk_acc), abi.ptr(j.dv_acc)
        p.dk, p.dv = abi.ptr(j.dk), abi.ptr(j.dv)
        p.q_gidx, p.k_gidx = _int32(j.q_gidx), _int32(j.k_gidx)
        p.q_doc, p.k_doc = _int32(j.q_doc), _int32(j.k_doc)
        p.sq, p.sk = j.q.shape[1], j.k.shape[1]
        p.dq_mode, p.dkv_mode = j.dq_mode, j.dkv_mode
        _set_problem_extras(p, j)
    return lay, arr


def attn_bwd(jobs: list[BwdJob], *, scale: float, mask: int, dropout=None) -> None:
    """Launch the batched block backward (rmx_attn_bwd) for ``jobs``; ``dropout`` must be the
    forward's (p, seed) and each job the forward's dropout offsets."""
    if not jobs:
        return
    lay, arr = _pack_bwd(jobs, scale, mask, dropout)
    lib = abi.lib()
    # partial dK/dV sums of calls with few or uneven key blocks (0 bytes: none)
    nbytes = lib.rmx_attn_bwd_workspace(ctypes.byref(lay), arr, len(jobs))
    _launch_bwd(lib, lay, arr, len(jobs), nbytes, jobs[0].q)


def _launch_bwd(lib, lay, problems, n, nbytes, like):
    ws = torch.empty(nbytes, dtype=torch.uint8, device=like.device) if nbytes else None
    abi.check(lib.rmx_attn_bwd_ws(ctypes.byref(lay), problems, n, abi.ptr(ws), nbytes,
                                  abi.stream_of(like)))


def cast_half(tensors, dtype):
    """Contiguous fp32 tensors (element counts multiples of 8) as bf16 or fp16, one launch."""
    outs = [torch.empty(t.shape, dtype=dtype, device=t.device) for t in tensors]
    n = len(tensors)
    abi.check(abi.lib().rmx_cast_half(
        (ctypes.c_void_p * n)(*(t.data_ptr() for t in tensors)),
        (ctypes.c_void_p * n)(*(t.data_ptr() for t in outs)),
        (ctypes.c_int64 * n)(*(t.numel() for t in tensors)), n, _DTYPES[dtype],
        abi.stream_of(tensors[0])))
    return outs


# ---------------------------------------------------------------- launch plans
# Building a call's jobs (views, checks, strides) takes 20-40 us of host time per job, more
# than a small ring step's kernels. A plan keeps what those jobs come to for one signature of
# shapes, strides, types and options: the layouts, and the problem tables with every pointer as
# an offset from its base tensor. A later call of the same signature adds its own base
# addresses to a copy of the table. Plans hold no address and no tensor of a call, are immutable
# and at most PLANS_MAX of them are kept.
PLANS_MAX = 256
_plans: collections.OrderedDict = collections.OrderedDict()
_plans_lock = threading.Lock()


def signature(*tensors):
    """What a plan depends on of its base tensors."""
    return tuple(None if t is None else (t.shape, t.stride(), t.dtype, t.device) for t in tensors)


class _NoSpan:
    def __call__(self, name):
        return self

    def __enter__(self):
        return None

    def __exit__(self, *exc):
        return False


NO_SPAN = _NoSpan()


class LaunchPlan:
    """The calls ``steps`` = [(jobs, scale, mask)] over views of ``bases`` (problem field ->
    base tensor). ``drop_p``: the dropout probability of every step (its seed comes with each
    run)."""

    def __init__(self, steps, bases, drop_p=0.0):
        steps = [s for s in steps if s[0]]
        self.bwd = bool(steps) and isinstance(steps[0][0][0], BwdJob)
        self.struct = abi.BwdProblem if self.bwd else abi.FwdProblem
        pack = _pack_bwd if self.bwd else _pack_fwd
        drop = (drop_p, 0) if drop_p else None
        self.drop = bool(drop_p)
        self.steps, parts, lo = [], [], 0  # (layout, first row, rows, workspace bytes)
        for jobs, scale, mask in steps:
            lay, arr = pack(jobs, scale, mask, drop)
            nbytes = (abi.lib().rmx_attn_bwd_workspace(ctypes.byref(lay), arr, len(jobs))
                      if self.bwd else 0)
            self.steps.append((lay, lo, len(jobs), nbytes))
            parts.append(bytes(arr))
            lo += len(jobs)
        # [problem, 8-byte word of the struct], on the host
        self.words = ctypes.sizeof(self.struct) // 8
        self.table = (torch.frombuffer(bytearray(b"".join(parts)), dtype=torch.int64)
                      .view(lo, self.words) if parts else None)
        self.fields = []  # (word, name)
        for name, base in bases.items():
            if self.table is None or base is None:
                continue
            word = getattr(self.struct, name).offset // 8
            col = self.table[:, word]
            if not col.any():
                continue
            if not col.all():
                raise AssertionError(f"{name} is set in some problems only")
            col -= base.data_ptr()
            self.fields.append((word, name))

    def bind(self, bases):
        """The problem tables at the addresses of ``bases``."""
        at = [0] * self.words
        for word, name in self.fields:
            at[word] = bases[name].data_ptr()
        return self.table + torch.tensor(at, dtype=torch.int64, device="cpu")

    def _layout(self, lay, seed):
        if not self.drop:
            return lay
        lay = abi.AttnLayout.from_buffer_copy(lay)
        lay.drop_seed_lo, lay.drop_seed_hi = seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF
        return lay

    def problems(self, table, lo):
        """The rows of a bound table from ``lo`` on (which the caller keeps alive)."""
        return ctypes.byref(self.struct.from_address(table.data_ptr() + 8 * self.words * lo))

    def _set(self, table, field, value):
        """A copy of a bound table with an int32 field of every problem set."""
        table = table.clone()
        table.view(torch.int32)[:, getattr(self.struct, field).offset // 4] = value
        return table

    def run_fwd(self, bases, seed, like, span):
        """Launch the forward steps; ``span()`` brackets each (timing)."""
        if self.table is None:
            return
        t, lib, stream = self.bind(bases), abi.lib(), abi.stream_of(like)
        for lay, lo, n, _ in self.steps:
            with span("attn_fwd"):
                abi.check(lib.rmx_attn_fwd(ctypes.byref(self._layout(lay, seed)),
                                           self.problems(t, lo), n, stream))

    def run_bwd(self, bases, seed, like, span=None):
        """Launch the backward steps: dK/dV then dQ of each, in one call, or in one call each
        bracketed by ``span``."""
        if self.table is None:
            return
        t, lib = self.bind(bases), abi.lib()
        if span is None:
            for lay, lo, n, nbytes in self.steps:
                _launch_bwd(lib, self._layout(lay, seed), self.problems(t, lo), n, nbytes, like)
            return
        tk, tq = (self._set(t, f, abi.GRAD_NONE) for f in ("dq_mode", "dkv_mode"))
        for lay, lo, n, nbytes in self.steps:
            lay = self._layout(lay, seed)
            with span("attn_bwd_dkdv"):
                _launch_bwd(lib, lay, self.problems(tk, lo), n, nbytes, like)
            with span("attn_bwd_dq"):
                _launch_bwd(lib, lay, self.problems(tq, lo), n, 0, like)


def plan(key, build):
    """The kept plan of ``key``, built (``build()``) on first use."""
    with _plans_lock:
        p = _plans.get(key)
        if p is not None:
            _plans.move_to_end(key)
            return p
    p = build()
    with _plans_lock:
        _plans[key] = p
        while len(_plans) > PLANS_MAX:
            _plans.popitem(last=False)
    return p
