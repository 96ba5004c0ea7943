"""Forward and dQ on either side of the 4-wave / 8-wave line (256 workgroups of 128 queries)."""
import pytest
import torch

from tests.gpu_util import bf16_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["full", "causal", "doc", "window", "dropout"])
@pytest.mark.parametrize("sq,sk,d", [(129, 200, 128), (256, 65, 64), (383, 383, 96), (1, 300, 64)])
def test_small_and_large_launches_agree(sq, sk, d, kind):
    """A wave's 32 queries see the same tiles whatever the workgroup holds, so the same rows
    come out bit for bit from a small launch (4 waves) and as two of the rows of a batch large
    enough for 8 waves."""
    from ringmaster_amd import abi
    from ringmaster_amd.ring import ops

    hq, hkv = 4, 2
    big = 256 // (hq * ((sq + 127) // 128)) + 2  # batch rows that pass the line
    print(f"case half sq={sq} sk={sk} d={d} {kind} batch={big}", flush=True)
    q, k, v, do = (bf16_pair((2, n, h, d), s)[1]
                   for n, h, s in ((sq, hq, 1), (sk, hkv, 2), (sk, hkv, 3), (sq, hq, 4)))
    mask = {"causal": abi.MASK_CAUSAL, "window": abi.MASK_CAUSAL,
            "doc": abi.MASK_DOC}.get(kind, abi.MASK_FULL)
    drop = (0.3, 11) if kind == "dropout" else None
    meta = {}
    if kind == "doc":
        ar = lambda n: torch.arange(n, dtype=torch.int32, device="cuda")  # noqa: E731
        meta = dict(q_gidx=ar(sq) + 70, k_gidx=ar(sk), q_doc=(ar(sq) + 70) // 90, k_doc=ar(sk) // 90)
    win = 50 if kind == "window" else None

    def run(rep):
        # rows 0 and 1 first (the dropout mask is of the batch row), then copies
        qq, kk, vv, dd = (torch.cat([t] + [t[:1]] * (rep - 2)) if rep > 2 else t
                          for t in (q, k, v, do))
        b = qq.shape[0]
        out = torch.empty_like(qq)
        lse = torch.empty((b, hq, sq), device="cuda")
        acc = torch.empty(qq.shape, device="cuda")
        ops.attn_fwd([ops.FwdJob(q=qq, k=kk, v=vv, mode=abi.FWD_WRITE, out=out, lse=lse,
                                 acc_out=acc, window=win, **meta)],
                     scale=d ** -0.5, mask=mask, dropout=drop)
        delta, nlse = torch.empty_like(lse), torch.empty_like(lse)
        ops.attn_bwd_delta(acc, dd, delta, hkv, lse=lse, nlse=nlse)
        dq = torch.empty(qq.shape, device="cuda")
        ops.attn_bwd([ops.BwdJob(q=qq, k=kk, v=vv, dout=dd, lse=lse, delta=delta, nlse=nlse,
                                 dq_mode=abi.GRAD_WRITE_F32, dkv_mode=abi.GRAD_NONE, dq_acc=dq,
                                 window=win, **meta)], scale=d ** -0.5, mask=mask, dropout=drop)
        torch.cuda.synchronize()
        return out[:2], lse[:2], acc[:2], dq[:2]

    for a, c in zip(run(2), run(big)):
        assert torch.equal(a, c)
        assert a.float().isfinite().all() or kind in ("doc", "causal", "window")
