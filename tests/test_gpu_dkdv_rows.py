"""The row-staged dK/dV epilogues of the kernels (whole key blocks)."""
import pytest
import torch

from tests.gpu_util import bf16_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["full", "causal", "doc", "dropout"])
@pytest.mark.parametrize("d", [40, 64, 96, 128, 200, 256])
def test_dkdv_unaligned_and_padded_buffers(monkeypatch, d, kind):
    """Every gradient mode, into caller buffers below vector alignment (one element past an
    aligned base; rows padded past the head dim), equals aligned contiguous buffers bit for
    bit, and the padding keeps its sentinel. Key counts leave the last key block, and the last
    wave's rows, partly past the end. No workspace:
    a split call would store from the fold."""
    from ringmaster_amd import abi
    from ringmaster_amd.ring import ops
    from ringmaster_amd.ring.kernels import block_forward

    b, sq, sk, hq, hkv = 2, 140, 277, 4, 2
    print(f"case dkdv rows d={d} {kind}", flush=True)
    lib = abi.lib()

    class Whole:
        def __getattr__(self, name):
            return getattr(lib, name)

        def rmx_attn_bwd_workspace(self, *a):
            return 0

    whole = Whole()
    monkeypatch.setattr(abi, "lib", lambda: whole)
    q, k, v, do = (bf16_pair((b, n, h, d), s)[1]
                   for n, h, s in ((sq, hq, 21), (sk, hkv, 22), (sk, hkv, 23), (sq, hq, 24)))
    sc = d ** -0.5
    drop = (0.2, 77) if kind == "dropout" else None
    causal = kind == "causal"
    mask = {"causal": abi.MASK_CAUSAL, "doc": abi.MASK_DOC}.get(kind, abi.MASK_FULL)
    out, lse, out32 = block_forward(q, k, v, sc, causal, keep_f32=True, dropout=drop)
    delta = torch.empty((b, hq, sq), device="cuda")
    nlse = torch.empty_like(delta)
    ops.attn_bwd_delta(out32, do, delta, hkv, lse=lse, nlse=nlse)
    meta = {}
    if kind == "doc":
        ar = lambda n: torch.arange(n, dtype=torch.int32, device="cuda")  # noqa: E731
        meta = dict(q_gidx=ar(sq) + 100, k_gidx=ar(sk), q_doc=(ar(sq) + 100) // 90, k_doc=ar(sk) // 90)
    pad = d + 8

    def run(mode, aligned):
        f32 = mode != abi.GRAD_WRITE_BF16
        h16 = mode in (abi.GRAD_WRITE_BF16, abi.GRAD_ACC_FINAL)
        n, off = b * sk * hkv * pad, 0 if aligned else 1
        mk = lambda dt, s: torch.full((n + 8,), 3.0, dtype=dt, device="cuda")[  # noqa: E731
            off:off + n].view(b, sk, hkv, pad)
        acc = [mk(torch.float32, s) for s in (1, 2)]
        half = [mk(torch.bfloat16, s) for s in (1, 2)]
        if mode in (abi.GRAD_ACC_F32, abi.GRAD_ACC_FINAL):
            for i, t in enumerate(acc):
                t[..., :d] = torch.linspace(-2 + i, 2, t[..., :d].numel(),
                                            device="cuda").view(b, sk, hkv, d)
        kw = {}
        if f32:
            kw.update(dk_acc=acc[0][..., :d], dv_acc=acc[1][..., :d])
        if h16:
            kw.update(dk=half[0][..., :d], dv=half[1][..., :d])
        ops.attn_bwd([ops.BwdJob(q=q, k=k, v=v, dout=do, lse=lse, delta=delta, nlse=nlse,
                                 dq_mode=abi.GRAD_NONE, dkv_mode=mode, **kw, **meta)],
                     scale=sc, mask=mask, dropout=drop)
        torch.cuda.synchronize()
        res = half if h16 else acc
        for t in acc + half:
            assert (t[..., d:] == 3.0).all()
        return [t[..., :d].clone() for t in res]

    for mode in (abi.GRAD_WRITE_F32, abi.GRAD_ACC_F32, abi.GRAD_WRITE_BF16, abi.GRAD_ACC_FINAL):
        a, u = run(mode, True), run(mode, False)
        for x, y in zip(a, u):
            assert torch.equal(x, y), mode
            assert x.float().abs().sum() > 0
