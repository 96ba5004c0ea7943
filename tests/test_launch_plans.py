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
        out, lse, o32 = zigzag.ring_forward(q, k, v, 0.125, doc, layout=layout, causal=causal,
                                            window=window)
        zigzag.ring_backward(do, q, k, v, o32, lse, 0.125, doc, layout=layout, causal=causal,
                             window=window)

    first, second = inputs(1), inputs(2)
    ops._plans.clear()
    built = _recorded(monkeypatch, lambda: passes(second))
    ops._plans.clear()
    passes(first)
    n_plans = len(ops._plans)
    kept = _recorded(monkeypatch, lambda: passes(second))
    assert len(ops._plans) == n_plans, "the second pass built plans of its own"
    assert [c[:2] + c[3:] for c in built] == [c[:2] + c[3:] for c in kept]
    for a, c in zip(built, kept):
        st = abi.FwdProblem if a[0] == "fwd" else abi.BwdProblem
        ta, tc = (np.frombuffer(x[2], dtype=ops._table_dtype(st)) for x in (a, c))
        for f in ta.dtype.names:
            if f in ("q", "k", "v", "dout") or ta.dtype[f] == np.int32:
                assert (ta[f] == tc[f]).all(), f
            else:  # allocated per call: null together
                assert ((ta[f] == 0) == (tc[f] == 0)).all(), f


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


def test_plans_are_bounded():
    ops._plans.clear()
    for i in range(ops.PLANS_MAX + 9):
        ops.plan(("bound", i), lambda: i)
    assert len(ops._plans) == ops.PLANS_MAX and ("bound", 0) not in ops._plans
    ops._plans.clear()
