"""Launch plans (ops.LaunchPlan): the kept tables against the calls they replace, on the CPU
(the jobs' tensors stay on the host: nothing is launched)."""
import ctypes

import numpy as np
import pytest
import torch

from ringmaster_amd import abi
from ringmaster_amd.ring import ops, zigzag


@pytest.fixture(autouse=True)
def _host(monkeypatch):
    monkeypatch.setattr(abi, "require_device", lambda *t: None)


def _table_dtype(struct):
    kinds = {ctypes.c_void_p: "u8", ctypes.c_int32: "i4"}
    return np.dtype({"names": [n for n, _ in struct._fields_],
                     "formats": [kinds[t] for _, t in struct._fields_],
                     "offsets": [getattr(struct, n).offset for n, _ in struct._fields_],
                     "itemsize": ctypes.sizeof(struct)})


def _recorded(monkeypatch, fn):
    """The (layout bytes, problem bytes) of every call ``fn`` makes, with no library."""
    calls = []

    def rows(arr, n):
        return ctypes.string_at(ctypes.addressof(arr._obj), n * ctypes.sizeof(arr._obj))

    class Lib:
        def rmx_attn_fwd(self, lay, arr, n, stream):
            calls.append(("fwd", bytes(lay._obj), rows(arr, n), n))
            return 0

        def rmx_attn_bwd_workspace(self, lay, arr, n):
            return 0

        def rmx_attn_bwd_ws(self, lay, arr, n, ws, nbytes, stream):
            calls.append(("bwd", bytes(lay._obj), rows(arr, n), n))
            return 0

        def rmx_attn_bwd_delta(self, *a):
            return 0

    monkeypatch.setattr(abi, "lib", Lib)
    monkeypatch.setattr(abi, "stream_of", lambda t: None)
    fn()
    return list(calls)


def _bound(monkeypatch, fn):
    """The calls of ``fn`` as (kind, layout bytes, problem table, bases): ``bases`` are the tensors
    the call's plan was bound to, which stay alive with the result, so that no later call's
    tensors can take their addresses."""
    bound = []
    bind = ops.LaunchPlan.bind

    def recording(self, bases):
        bound.extend([{k: t for k, t in bases.items() if t is not None}] * len(self.steps))
        return bind(self, bases)

    with monkeypatch.context() as m:
        m.setattr(ops.LaunchPlan, "bind", recording)
        calls = _recorded(m, fn)
    assert len(bound) == len(calls)
    return [(kind, lay, np.frombuffer(rows, dtype=_table_dtype(
        abi.FwdProblem if kind == "fwd" else abi.BwdProblem)), bases)
        for (kind, lay, rows, _), bases in zip(calls, bound)]


def _check_moved(built, kept, first, layouts_equal=True):
    """Call by call, the kept plan's tables equal the built one's, every pointer at the same
    offset of its own call's base tensor and inside it; ``first``: the calls the plans were built
    by, whose addresses must not appear."""
    assert len(built) == len(kept) == len(first)
    for (ka, la, ta, ba), (kc, lc, tc, bc), (_, _, _, bf) in zip(built, kept, first):
        assert ka == kc and (not layouts_equal or la == lc) and len(ta) == len(tc)
        for f in ta.dtype.names:
            if ta.dtype[f] == np.int32:
                assert (ta[f] == tc[f]).all(), f
            elif f not in ba:
                assert not ta[f].any() and not tc[f].any(), f
            else:
                t = bc[f]
                span = (1 + sum((n - 1) * st for n, st in zip(t.shape, t.stride()))) * t.element_size()
                at = tc[f].astype(np.int64) - t.data_ptr()
                assert (at == ta[f].astype(np.int64) - ba[f].data_ptr()).all(), f
                assert ((at >= 0) & (at < span)).all(), f
                assert t.data_ptr() != bf[f].data_ptr(), f"{f}: the check needs another address"


@pytest.mark.parametrize("layout,causal,docs,window", [
    ("zigzag", True, False, None), ("contiguous", True, False, None),
    ("contiguous", False, True, None), ("distflash", True, True, None),
    ("contiguous", True, False, [100] * 4), ("zigzag", True, True, [64] * 4)])
@pytest.mark.parametrize("strided", [False, True])
def test_ring_plans_follow_their_base_tensors(monkeypatch, layout, causal, docs, window, strided):
    """A plan built on one set of tensors and run on another equals the plan built on that
    other one: every pointer moves with its base, everything else is the signature's."""
    P, b, hq, hkv, L, d = 4, 2, 4, 2, 24, 64

    def inputs(seed):
        g = torch.Generator().manual_seed(seed)
        mk = lambda h: torch.randn(P, b, h, L, 2 * d if strided else d,  # noqa: E731
                                   generator=g).to(torch.bfloat16)[..., :d]
        q, k, v = mk(hq), mk(hkv), mk(hkv)
        doc = torch.arange(P * L, dtype=torch.int32) // 30 if docs else None
        return q, k, v, torch.randn(P, b, L, hq, d).to(torch.bfloat16), doc

    def passes(t):
        q, k, v, do, doc = t
        zigzag._ROWS_CACHE.clear()  # (the global indices are kept and would be the same tensor)
        out, lse, o32 = zigzag.ring_forward(q, k, v, 0.125, doc, layout=layout, causal=causal,
                                            window=window)
        zigzag.ring_backward(do, q, k, v, o32, lse, 0.125, doc, layout=layout, causal=causal,
                             window=window)

    first, second = inputs(1), inputs(2)
    ops._plans.clear()
    built = _bound(monkeypatch, lambda: passes(second))
    ops._plans.clear()
    before = _bound(monkeypatch, lambda: passes(first))
    n_plans = len(ops._plans)
    kept = _bound(monkeypatch, lambda: passes(second))
    assert len(ops._plans) == n_plans, "the second pass built plans of its own"
    _check_moved(built, kept, before)
    for (_, _, ta, _), (_, _, tc, _) in zip(built, kept):
        for f in ("q", "k", "v", "dout"):
            if f in ta.dtype.names:
                assert (ta[f] == tc[f]).all(), f
    ops._plans.clear()


def test_kept_ring_plans_refuse_what_building_refused(monkeypatch):
    """The global lse is no part of the backward plan's key: one of another layout is refused
    with the plan in place as without it."""
    q = torch.randn(2, 1, 2, 16, 64).to(torch.bfloat16)
    do = torch.randn(2, 1, 16, 2, 64).to(torch.bfloat16)
    out, lse = torch.zeros(2, 1, 16, 2, 64), torch.zeros(2, 1, 2, 16)

    def passes(stat):
        return _recorded(monkeypatch, lambda: zigzag.ring_backward(do, q, q, q, out, stat, 0.125))

    swapped = lse.transpose(2, 3).contiguous()
    ops._plans.clear()
    with pytest.raises(ValueError):
        passes(swapped)
    ops._plans.clear()
    assert passes(lse)
    with pytest.raises(ValueError):
        passes(swapped)
    ops._plans.clear()


def test_ring_plans_of_some_ranks(monkeypatch):
    """``only_ranks`` is part of a plan's key: two subsets keep two plans, each its own blocks."""
    mk = lambda seed: torch.randn(4, 1, 2, 16, 64, generator=torch.Generator().manual_seed(  # noqa: E731
        seed)).to(torch.bfloat16)
    first, second = mk(1), mk(2)

    def passes(q, ranks):
        out, lse, o32 = zigzag.ring_forward(q, q, q, 0.125, only_ranks=ranks)
        zigzag.ring_backward(out, q, q, q, o32, lse, 0.125, only_ranks=ranks)

    built = {}
    for ranks in ({0}, {1, 3}):
        ops._plans.clear()
        built[frozenset(ranks)] = _bound(monkeypatch, lambda: passes(second, ranks))
    ops._plans.clear()
    before = {frozenset(r): _bound(monkeypatch, lambda: passes(first, r)) for r in ({0}, {1, 3})}
    n_plans = len(ops._plans)
    for ranks, ref in built.items():
        _check_moved(ref, _bound(monkeypatch, lambda: passes(second, set(ranks))), before[ranks])
    assert len(ops._plans) == n_plans
    ops._plans.clear()


@pytest.mark.parametrize("keep_f32", [False, True])
def test_block_plans_follow_their_tensors_and_the_seed(monkeypatch, keep_f32):
    """A block's forward and backward plans: pointers move with their tensors, and the dropout
    seed, which is no part of the signature, with the call."""
    from ringmaster_amd.ring.kernels import block_backward, block_forward

    def inputs(seed):
        g = torch.Generator().manual_seed(seed)
        mk = lambda h: torch.randn(2, 24, h, 64, generator=g).to(torch.bfloat16)  # noqa: E731
        return mk(4), mk(2), mk(2), mk(4)

    def passes(t, seed):
        q, k, v, do = t
        out, lse, *o32 = block_forward(q, k, v, 0.125, True, keep_f32=keep_f32, dropout=(0.25, seed))
        block_backward(do, q, k, v, out, lse, 0.125, True, out_f32=o32[0] if o32 else None,
                       dropout=(0.25, seed))

    first, second = inputs(1), inputs(2)
    ops._plans.clear()
    built = _bound(monkeypatch, lambda: passes(second, (7 << 32) + 5))
    ops._plans.clear()
    before = _bound(monkeypatch, lambda: passes(first, 3))
    n_plans = len(ops._plans)
    kept = _bound(monkeypatch, lambda: passes(second, (7 << 32) + 5))
    assert len(ops._plans) == n_plans
    _check_moved(built, kept, before)
    seeds = lambda calls: {(lay.drop_seed_lo, lay.drop_seed_hi) for lay in (  # noqa: E731
        abi.AttnLayout.from_buffer_copy(c[1]) for c in calls)}
    assert seeds(kept) == {(5, 7)} and seeds(before) == {(3, 0)}
    ops._plans.clear()


@pytest.mark.parametrize("f32", [False, True])
def test_delta_plans_hold_no_address(monkeypatch, f32):
    """The delta pass keeps a layout only; its addresses are the call's."""
    seen = []

    class Lib:
        def rmx_attn_bwd_delta(self, lay, out, is_f32, dout, delta, lse, nlse, sq, stream):
            seen.append((bytes(lay._obj), out, is_f32, dout, delta, lse, nlse, sq))
            return 0

    monkeypatch.setattr(abi, "lib", Lib)
    monkeypatch.setattr(abi, "stream_of", lambda t: None)
    ops._plans.clear()
    held = []
    for _ in range(2):
        dout = torch.zeros(2, 24, 4, 64, dtype=torch.bfloat16)
        out = torch.zeros(2, 24, 4, 64, dtype=torch.float32 if f32 else torch.bfloat16)
        delta, lse, nlse = (torch.zeros(2, 4, 24) for _ in range(3))
        held.append((out, dout, delta, lse, nlse))
        ops.attn_bwd_delta(out, dout, delta, 2, lse=lse, nlse=nlse)
        o, g, d, l, n = (t.data_ptr() for t in held[-1])
        assert seen[-1][1:] == (o, int(f32), g, d, l, n, 24)
    assert len(ops._plans) == 1 and seen[0][0] == seen[1][0]
    ops._plans.clear()


def test_ring_plans_take_the_scale_by_value(monkeypatch):
    """A scale given as a tensor that the program changes in place: the second pass takes its
    new value, and no plan keeps the tensor."""
    q = torch.randn(2, 1, 2, 16, 64).to(torch.bfloat16)
    scale = torch.tensor(0.125)
    ops._plans.clear()

    def scales():
        calls = _recorded(monkeypatch, lambda: zigzag.ring_forward(q, q, q, scale))
        return {abi.AttnLayout.from_buffer_copy(c[1]).scale for c in calls}

    assert scales() == {0.125}
    scale.mul_(2)
    assert scales() == {0.25}
    ops._plans.clear()


def test_block_plans_take_scale_and_window_by_value(monkeypatch):
    """The same of a block's scale and window bound, forward and backward."""
    from ringmaster_amd.ring.kernels import block_backward, block_forward

    q = torch.randn(1, 16, 2, 64).to(torch.bfloat16)
    scale, window = torch.tensor(0.125), torch.tensor(5)
    ops._plans.clear()

    def seen():
        def passes():
            out, lse = block_forward(q, q, q, scale, True, window=window)
            block_backward(q, q, q, q, out, lse, scale, True, window=window)

        return {(abi.AttnLayout.from_buffer_copy(c[1]).scale,
                 (abi.FwdProblem if c[0] == "fwd" else abi.BwdProblem).from_buffer_copy(c[2]).window_left)
                for c in _recorded(monkeypatch, passes)}

    assert seen() == {(0.125, 5)}
    scale.mul_(2)
    window.add_(4)
    assert seen() == {(0.25, 9)}
    ops._plans.clear()


def test_plans_keep_the_workspace_of_their_shapes():
    """The first call of a signature may be refused for an address (here tensors two bytes past
    alignment); the plan that stays is the one an aligned first call leaves."""
    def step_bytes(off):
        mk = lambda h: torch.zeros(512 * h * 64 + 8, dtype=torch.bfloat16)[  # noqa: E731
            off:off + 512 * h * 64].view(1, 512, h, 64)
        stat = torch.zeros(1, 8, 512)
        bases = dict(q=mk(8), k=mk(2), v=mk(2), dout=mk(8), lse=stat, delta=stat, nlse=stat,
                     dq=mk(8), dk=mk(2), dv=mk(2))
        job = ops.BwdJob(dq_mode=abi.GRAD_WRITE_BF16, dkv_mode=abi.GRAD_WRITE_BF16, **bases)
        return ops.LaunchPlan([([job], 0.125, abi.MASK_CAUSAL)], bases).steps[0][3]

    assert step_bytes(1) == step_bytes(0) > 0


@pytest.mark.parametrize("timed", [False, True])
def test_one_call_or_one_per_gradient(monkeypatch, timed):
    """Without a timer a step's dK/dV and dQ are one call, with one two calls of a gradient each,
    which differ from it in the other gradient's mode alone."""
    q = torch.randn(2, 1, 2, 16, 64).to(torch.bfloat16)
    do, out = torch.randn(2, 1, 16, 2, 64).to(torch.bfloat16), torch.zeros(2, 1, 16, 2, 64)
    lse = torch.zeros(2, 1, 2, 16)
    spans = []

    class Span:
        def __call__(self, name):
            spans.append(name)
            return self

        def __enter__(self):
            pass

        def __exit__(self, *exc):
            return False

    ops._plans.clear()
    calls = _recorded(monkeypatch, lambda: zigzag.ring_backward(
        do, q, q, q, out, lse, 0.125, timer=Span() if timed else None))
    tables = [np.frombuffer(rows, dtype=_table_dtype(abi.BwdProblem)) for _, _, rows, _ in calls]
    modes = [(set(t["dq_mode"].tolist()), set(t["dkv_mode"].tolist())) for t in tables]
    w, a, n = {abi.GRAD_WRITE_F32}, {abi.GRAD_ACC_F32}, {abi.GRAD_NONE}
    if timed:
        assert modes == [(n, w), (w, n), (n, a), (a, n)]
        assert spans == ["attn_bwd_delta"] + ["attn_bwd_dkdv", "attn_bwd_dq"] * 2
        assert all(t["dk_acc"].all() and t["dq_acc"].all() for t in tables)
    else:
        assert modes == [(w, w), (a, a)]
    ops._plans.clear()


def test_plans_are_bounded():
    ops._plans.clear()
    for i in range(ops.PLANS_MAX + 9):
        ops.plan(("bound", i), lambda: i)
    assert len(ops._plans) == ops.PLANS_MAX and ("bound", 0) not in ops._plans
    ops._plans.clear()
