"""dK/dV with split key blocks (rmx_attn_bwd_ws) against the whole ones (rmx_attn_bwd)."""
import ctypes

import pytest
import torch

from tests.gpu_util import bf16_pair, rel_l2

pytestmark = pytest.mark.gpu

# b, sq, sk, hq, hkv, d, mask, extras; each is a shape the rule splits
CASES = [
    (1, 512, 512, 8, 2, 128, "causal", {}),
    (2, 200, 333, 8, 1, 64, "full", {}),
    (1, 700, 300, 4, 1, 96, "full", {}),                       # sq > sk, padded head dim
    (1, 300, 700, 8, 2, 128, "causal", dict(window=90)),
    (1, 257, 257, 8, 2, 256, "causal", {}),
    (2, 320, 129, 8, 2, 200, "full", dict(drop=(0.3, 5))),
    (1, 640, 640, 8, 1, 64, "doc", {}),
    (1, 600, 600, 16, 1, 128, "causal", dict(drop=(0.1, 9), f16=True)),
]


@pytest.mark.parametrize("b,sq,sk,hq,hkv,d,kind,x", CASES)
@pytest.mark.parametrize("off", [0, 1])
def test_split_equals_whole(b, sq, sk, hq, hkv, d, kind, x, off):
    """Two problems of one call (the second with half the keys), every mode; ``off`` = 1 puts
    the outputs one element past vector alignment. The splits only change the order of fp32
    sums (rel-L2 a few 2^-24, held to 1e-6); 16-bit results may differ by one rounding of it."""
    from ringmaster_amd import abi
    from ringmaster_amd.ring import ops
    from ringmaster_amd.ring.kernels import block_forward

    print(f"case split b={b} {sq}x{sk} h={hq}/{hkv} d={d} {kind} {x} off={off}", flush=True)
    h16 = torch.float16 if x.get("f16") else torch.bfloat16
    q, k, v, do = (bf16_pair((b, n, h, d), s)[1].to(h16)
                   for n, h, s in ((sq, hq, 1), (sk, hkv, 2), (sk, hkv, 3), (sq, hq, 4)))
    sc, drop = d ** -0.5, x.get("drop")
    mask = {"causal": abi.MASK_CAUSAL, "doc": abi.MASK_DOC}.get(kind, abi.MASK_FULL)
    _, lse, out32 = block_forward(q, k, v, sc, kind == "causal", keep_f32=True, dropout=drop,
                                  window=x.get("window"))
    delta = torch.empty((b, hq, sq), device="cuda")
    nlse = torch.empty_like(delta)
    ops.attn_bwd_delta(out32, do, delta, hkv, lse=lse, nlse=nlse)
    meta = [{}, {}]
    sk2 = sk // 2
    if kind == "doc":
        ar = torch.arange(sq, dtype=torch.int32, device="cuda")
        meta = [dict(q_gidx=ar, k_gidx=ar[:n], q_doc=ar // 250, k_doc=ar[:n] // 250)
                for n in (sk, sk2)]

    lib = abi.lib()

    def run(mode, split):
        acc = [torch.empty(b * sk * hkv * d + 8, device="cuda") for _ in range(4)]
        half = [torch.zeros(b * sk * hkv * d + 8, dtype=h16, device="cuda") for _ in range(4)]
        for i, t in enumerate(acc):
            t[:] = torch.linspace(-1, 1 + i, t.numel(), device="cuda")
        jobs, outs = [], []
        for i, n in enumerate((sk, sk2)):
            view = lambda t: t[off:off + b * sk * hkv * d].view(b, sk, hkv, d)[:, :n]  # noqa: E731
            g = dict(dk_acc=view(acc[2 * i]), dv_acc=view(acc[2 * i + 1]),
                     dk=view(half[2 * i]), dv=view(half[2 * i + 1]))
            jobs.append(ops.BwdJob(q=q, k=k[:, :n], v=v[:, :n], dout=do, lse=lse, delta=delta,
                                   nlse=nlse, dq_mode=abi.GRAD_NONE, dkv_mode=mode,
                                   window=x.get("window"), **g, **meta[i]))
            outs += [g["dk"], g["dv"]] if mode in (abi.GRAD_WRITE_BF16, abi.GRAD_ACC_FINAL) \
                else [g["dk_acc"], g["dv_acc"]]
        seen = []
        real = lib.rmx_attn_bwd_workspace

        class Spy:
            def __getattr__(self, name):
                if name == "rmx_attn_bwd_workspace":
                    def size(*a):
                        n = real(*a)
                        seen.append(n)
                        return n if split else 0
                    return size
                return getattr(lib, name)

        keep, abi.lib = abi.lib, lambda: Spy()
        try:
            ops.attn_bwd(jobs, scale=sc, mask=mask, dropout=drop)
        finally:
            abi.lib = keep
        torch.cuda.synchronize()
        assert seen[0] > 0, "the rule does not split this shape"
        return [o.float().clone() for o in outs]

    for mode in (abi.GRAD_WRITE_F32, abi.GRAD_ACC_F32, abi.GRAD_WRITE_BF16, abi.GRAD_ACC_FINAL):
        whole, split = run(mode, False), run(mode, True)
        bar = 1e-6 if mode in (abi.GRAD_WRITE_F32, abi.GRAD_ACC_F32) else 1e-3
        for a, c in zip(whole, split):
            assert a.abs().sum() > 0 and rel_l2(c.cpu(), a.cpu()) < bar


@pytest.mark.parametrize("d,docs", [(64, 40), (128, 40), (128, 300), (256, 40), (128, 5000)])
@pytest.mark.parametrize("layout,causal", [("zigzag", True), ("contiguous", False)])
def test_packed_ring_split_equals_whole(monkeypatch, d, docs, layout, causal):
    """A packed ring backward whose steps the rule splits: most key blocks past the first step have
    no query of their documents (all of them at 40 tokens), which the splits leave as the
    unsplit kernel does, whatever the workspace holds."""
    from ringmaster_amd import abi
    from ringmaster_amd.ring import ops, zigzag

    print(f"case packed split d={d} docs={docs} {layout} causal={causal}", flush=True)
    P, L, hq, hkv = 4, 640, 8, 2
    mk = lambda h, s: bf16_pair((P, 1, h, L, d), s)[1]  # noqa: E731
    q, k, v, do = mk(hq, 1), mk(hkv, 2), mk(hkv, 3), mk(hq, 4).transpose(2, 3).contiguous()
    doc = torch.arange(P * L, dtype=torch.int32, device="cuda") // docs
    kw = dict(layout=layout, causal=causal)
    out, lse, o32 = zigzag.ring_forward(q, k, v, d ** -0.5, doc, **kw)
    lib, sizes = abi.lib(), []

    class Lib:
        split = True

        def __getattr__(self, name):
            return getattr(lib, name)

        def rmx_attn_bwd_workspace(self, *a):
            sizes.append(lib.rmx_attn_bwd_workspace(*a) if self.split else 0)
            return sizes[-1]

    one = Lib()
    monkeypatch.setattr(abi, "lib", lambda: one)
    real = torch.empty

    def filled(*a, **kw):  # workspaces hold NaN: nothing unwritten may reach a gradient
        t = real(*a, **kw)
        return t.fill_(255) if t.dtype == torch.uint8 else t

    def grads(split):
        ops._plans.clear()
        one.split = split
        for _ in range(2):  # the second pass runs from the plans that the first one left
            r = [g.clone() for g in zigzag.ring_backward(do, q, k, v, o32, lse, d ** -0.5, doc, **kw)]
        ops._plans.clear()
        return r

    whole = grads(False)
    sizes.clear()
    monkeypatch.setattr(torch, "empty", filled)
    split = grads(True)
    assert max(sizes) > 0, "the rule does not split this ring"
    assert torch.equal(whole[0], split[0])
    for a, c in zip(whole[1:], split[1:]):
        assert rel_l2(c.cpu(), a.cpu()) < 1e-6


@pytest.mark.parametrize("d", [64, 128, 256])
def test_empty_document_blocks_touch_no_memory(d):
    """A split launch of pairs of different documents, accumulating: neither the accumulators
    (-0.0 would turn to 0.0) nor the workspace's partial rows are written."""
    from ringmaster_amd import abi
    from ringmaster_amd.ring import ops

    print(f"case empty documents d={d}", flush=True)
    n, hq, hkv = 512, 8, 2
    q, k, v, do = (bf16_pair((1, n, h, d), s)[1] for h, s in ((hq, 1), (hkv, 2), (hkv, 3), (hq, 4)))
    stat = torch.zeros((1, hq, n), device="cuda")
    ar = torch.arange(n, dtype=torch.int32, device="cuda")
    acc = [torch.full((1, n, hkv, d), -0.0, device="cuda") for _ in range(2)]
    job = ops.BwdJob(q=q, k=k, v=v, dout=do, lse=stat, delta=stat, nlse=stat, dq_mode=abi.GRAD_NONE,
                     dkv_mode=abi.GRAD_ACC_F32, dk_acc=acc[0], dv_acc=acc[1], q_gidx=ar + n,
                     k_gidx=ar, q_doc=ar // 100 + 50, k_doc=ar // 100)
    lay, arr = ops._pack_bwd([job], d ** -0.5, abi.MASK_DOC, None)
    lib = abi.lib()
    need = lib.rmx_attn_bwd_workspace(ctypes.byref(lay), arr, 1)
    assert need > 0, "the rule does not split this shape"
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device="cuda")
    abi.check(lib.rmx_attn_bwd_ws(ctypes.byref(lay), arr, 1, ws.data_ptr(), need, abi.stream_of(q)))
    assert all(torch.signbit(a).all() and (a == 0).all() for a in acc)
    assert (ws[:need - 4 * hkv * (n // 128)] == 0xFF).all()


@pytest.mark.parametrize("kind", ["causal", "doc"])
def test_workspace_contract(kind):
    """A workspace below the queried size is not touched and the call runs unsplit, one of that
    size is not written past its end, a misaligned one is refused; problems of different
    lengths keep to their own rows."""
    from ringmaster_amd import abi
    from ringmaster_amd.ring import ops
    from ringmaster_amd.ring.kernels import block_forward

    print(f"case workspace contract {kind}", flush=True)
    b, sq, hq, hkv, d = 1, 700, 8, 2, 128
    q, k, v, do = (bf16_pair((b, sq, h, d), s)[1] for h, s in ((hq, 1), (hkv, 2), (hkv, 3), (hq, 4)))
    _, lse, out32 = block_forward(q, k, v, d ** -0.5, True, keep_f32=True)
    delta = torch.empty((b, hq, sq), device="cuda")
    nlse = torch.empty_like(delta)
    ops.attn_bwd_delta(out32, do, delta, hkv, lse=lse, nlse=nlse)
    ar = torch.arange(sq, dtype=torch.int32, device="cuda")
    jobs, outs = [], []
    for n in (129, 700, 33):
        dk, dv = (torch.empty((b, n, hkv, d), device="cuda") for _ in range(2))
        meta = dict(q_gidx=ar, k_gidx=ar[:n], q_doc=ar // 250, k_doc=ar[:n] // 250) \
            if kind == "doc" else {}
        jobs.append(ops.BwdJob(q=q, k=k[:, :n], v=v[:, :n], dout=do, lse=lse, delta=delta,
                               nlse=nlse, dq_mode=abi.GRAD_NONE, dkv_mode=abi.GRAD_WRITE_F32,
                               dk_acc=dk, dv_acc=dv, **meta))
        outs += [dk, dv]
    # one call has one set of strides: give every problem the longest one's buffers
    big = [torch.empty((b, 700, hkv, d), device="cuda") for _ in outs]
    for i, j in enumerate(jobs):
        n = j.k.shape[1]
        j.dk_acc, j.dv_acc = big[2 * i][:, :n], big[2 * i + 1][:, :n]
    mask = abi.MASK_DOC if kind == "doc" else abi.MASK_CAUSAL
    lay, arr = ops._pack_bwd(jobs, d ** -0.5, mask, None)
    lib = abi.lib()
    need = lib.rmx_attn_bwd_workspace(ctypes.byref(lay), arr, len(jobs))
    assert need > 16
    ws = torch.full((need + 4096,), 0xFF, dtype=torch.uint8, device="cuda")

    def call(ptr, nbytes):
        for t in big:
            t.fill_(7.0)
        rc = lib.rmx_attn_bwd_ws(ctypes.byref(lay), arr, len(jobs), ptr, nbytes, abi.stream_of(q))
        torch.cuda.synchronize()
        return rc, [t.clone() for t in big]

    _, whole = call(None, 0)
    rc, small = call(ws.data_ptr(), need - 1)
    assert rc == abi.RMX_OK and (ws == 0xFF).all()
    assert all(torch.equal(a, c) for a, c in zip(whole, small))
    assert call(ws.data_ptr() + 4, need)[0] == abi.RMX_EINVAL
    rc, split = call(ws.data_ptr(), need)
    assert rc == abi.RMX_OK and (ws[need:] == 0xFF).all() and not (ws[:need] == 0xFF).all()
    for i, (a, c) in enumerate(zip(whole, split)):
        n = jobs[i // 2].k.shape[1]
        assert (c[:, n:] == 7.0).all() and rel_l2(c[:, :n].cpu(), a[:, :n].cpu()) < 1e-6


def test_refused_arguments_and_small_workspaces():
    """The workspace query of a refused call is 0 and the call itself still refuses."""
    from ringmaster_amd import abi

    lib = abi.lib()
    lay = abi.AttnLayout()
    lay.batch, lay.hq, lay.hkv, lay.head_dim, lay.scale = 1, 3, 2, 64, 1.0
    arr = (abi.BwdProblem * 1)()
    assert lib.rmx_attn_bwd_workspace(ctypes.byref(lay), arr, 1) == 0
    assert lib.rmx_attn_bwd_ws(ctypes.byref(lay), arr, 1, None, 0, None) == abi.RMX_EINVAL
