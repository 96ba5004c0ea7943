"""The chunked dt cumsum (rmx_mamba2_dt_cumsum and its two backwards) at the edges of its
chunks: 512 / HT runs of 16 tokens, HT = 8, 16, 32 or 64 heads per workgroup."""
import pytest
import torch

from tests.gpu_util import seeded

pytestmark = pytest.mark.gpu

# chunk tokens: H <= 8: 1024, <= 16: 512, <= 32: 256, else 128
CASES = [(1, 1, 1), (2, 1024, 8), (1, 1025, 3), (2, 513, 16), (1, 255, 24), (2, 769, 32),
         (1, 128, 64), (2, 129, 64), (3, 2000, 65), (1, 17, 130)]


@pytest.mark.parametrize("softplus,f32", [(True, False), (True, True), (False, True)])
@pytest.mark.parametrize("rows,T,H", CASES)
def test_dt_cumsum_chunks(rows, T, H, softplus, f32):
    """Values within 8 fp32 roundings of the largest prefix (chunk, run and token sums of one
    sign), gradients within the same of their absolute sums, against fp64."""
    from ringmaster_amd import abi

    print(f"case dt rows={rows} T={T} H={H} softplus={softplus} f32={f32}", flush=True)
    raw = seeded((rows, T, H), 1)
    # without softplus the step itself is given, and steps are positive
    dt = (raw if softplus else 0.1 * raw.abs()).to(torch.float32 if f32 else torch.bfloat16)
    bias = seeded((H,), 2) - 2.0 if softplus else None
    A = -torch.exp(seeded((H,), 3))
    g_cum, g_e, g_dec = seeded((rows, T, H), 4), seeded((rows, T, H), 5), seeded((rows, H), 6)

    def ref(closed):
        d, a = dt.double().requires_grad_(True), A.double().requires_grad_(True)
        b = bias.double().requires_grad_(True) if softplus else None
        e = torch.nn.functional.softplus(d + b) if softplus else d * 1.0
        cum = torch.cumsum(e * a, 1)
        g = g_cum.double()
        loss = (e * g_e.double()).sum()
        if closed:
            loss = loss + ((cum - cum[:, -1:]) * g)[:, :-1].sum()
        else:
            loss = loss + (cum * g).sum() + (torch.exp(cum[:, -1]) * g_dec.double()).sum()
        leaves = [d, a] + ([b] if softplus else [])
        return e, cum, torch.autograd.grad(loss, leaves)

    dev = lambda x: None if x is None else x.cuda()  # noqa: E731
    dd, bd, Ad, gc, ge, gd = (dev(x) for x in (dt, bias, A, g_cum, g_e, g_dec))
    cum, e, decay = (torch.empty(s, device="cuda") for s in ((rows, T, H), (rows, T, H), (rows, H)))
    lib, s = abi.lib(), abi.stream_of(dd)
    abi.check(lib.rmx_mamba2_dt_cumsum(dd.data_ptr(), int(f32), abi.ptr(bd), Ad.data_ptr(),
                                       int(softplus), cum.data_ptr(), e.data_ptr(),
                                       decay.data_ptr(), rows, T, H, s))
    e_r, cum_r, _ = ref(False)
    eps = 2.0 ** -23
    scale = (e_r * A.double()).abs().sum(1, keepdim=True).detach()
    assert ((cum.cpu() - cum_r).abs() <= 8 * eps * scale + 1e-30).all()
    assert ((e.cpu() - e_r).abs() <= 8 * eps * e_r.abs() + 1e-30).all()
    # exp turns the absolute error of cum_A into a relative one
    dec_r = torch.exp(cum_r[:, -1]).detach()
    dec_err = (16 * eps * (1 + scale[:, 0])) * dec_r + 1e-37
    assert ((decay.cpu() - dec_r).abs() <= dec_err).all()

    for closed in (False, True):
        g_dt = torch.empty_like(cum)
        g_A, g_b = torch.zeros(H, device="cuda"), torch.zeros(H, device="cuda")
        head = (dd.data_ptr(), int(f32), abi.ptr(bd), Ad.data_ptr(), int(softplus))
        tail = (g_dt.data_ptr(), g_A.data_ptr(), g_b.data_ptr() if softplus else None, rows, T, H, s)
        if closed:
            abi.check(lib.rmx_mamba2_dt_cumsum_state_bwd(*head, gc.data_ptr(), ge.data_ptr(), *tail))
        else:
            abi.check(lib.rmx_mamba2_dt_cumsum_bwd(*head, gc.data_ptr(), ge.data_ptr(),
                                                   gd.data_ptr(), decay.data_ptr(), *tail))
        _, _, grads = ref(closed)
        # the summands a suffix sum can hold (the decay's own error with them), times |A|, plus
        # the direct gradient
        g_abs = g_cum.double().abs().sum(1, keepdim=True) + (
            (dec_r + dec_err / eps) * g_dec.double()).abs()[:, None]
        bar = 32 * eps * (A.double().abs() * g_abs + g_e.double().abs())
        assert ((g_dt.cpu() - grads[0]).abs() <= bar).all()
        bar_A = 32 * eps * (g_abs * e_r.detach().abs()).sum((0, 1))
        assert ((g_A.cpu() - grads[1]).abs() <= bar_A).all()
        if softplus:
            assert ((g_b.cpu() - grads[2]).abs() <= bar.sum((0, 1))).all()


@pytest.mark.parametrize("rows,T,H", [(1, 4096, 8), (1, 1025, 3), (2, 2000, 16), (1, 300, 24),
                                      (5, 400, 64), (3, 2000, 65), (1, 8192, 64)])
@pytest.mark.parametrize("state", [False, True])
def test_parameter_gradients_repeat(rows, T, H, state):
    """dA and d(bias) of several chunks: with the workspace they repeat bit for bit, without it
    for one or two rows; both forms within 32 roundings of their absolute sums of each other; a
    workspace below the queried size is left alone."""
    from ringmaster_amd import abi

    print(f"case dt repeat rows={rows} T={T} H={H} state={state}", flush=True)
    lib = abi.lib()
    dt, bias, A = seeded((rows, T, H), 1).cuda(), (seeded((H,), 2) - 2).cuda(), -torch.exp(
        seeded((H,), 3)).cuda()
    g_cum, g_e = seeded((rows, T, H), 4).cuda(), seeded((rows, T, H), 5).cuda()
    need = lib.rmx_mamba2_dt_cumsum_bwd_workspace(rows, T, H)
    assert need > 0

    def call(ws_bytes, ws):
        g_dt, g_A, g_b = torch.empty_like(dt), torch.zeros_like(A), torch.zeros_like(A)
        abi.check(lib.rmx_mamba2_dt_cumsum_bwd_ws(
            dt.data_ptr(), 1, bias.data_ptr(), A.data_ptr(), 1, g_cum.data_ptr(), g_e.data_ptr(),
            None, None, g_dt.data_ptr(), g_A.data_ptr(), g_b.data_ptr(), rows, T, H, int(state),
            abi.ptr(ws), ws_bytes, abi.stream_of(dt)))
        return g_dt, g_A, g_b

    ws = torch.full((need + 64,), 0x5A, dtype=torch.uint8, device="cuda")
    plain, again = call(need - 4, ws), [call(need - 4, ws) for _ in range(4)]
    assert (ws == 0x5A).all(), "a workspace below the queried size was written"
    if rows <= 2:
        assert all(torch.equal(x, y) for other in again for x, y in zip(plain, other))
    first, again = call(need, ws), [call(need, ws) for _ in range(4)]
    assert (ws[need:] == 0x5A).all(), "written past the workspace"
    assert all(torch.equal(x, y) for other in again for x, y in zip(first, other))
    # R e and g_dt summed in absolute value bound every partial sum of either order
    e = torch.nn.functional.softplus(dt.double() + bias)
    g_abs = g_cum.double().abs().sum(1, keepdim=True)
    bar_A = 32 * 2.0 ** -23 * (g_abs * e).sum((0, 1))
    bar_b = 32 * 2.0 ** -23 * (A.double().abs() * g_abs + g_e.double().abs()).sum((0, 1))
    assert ((first[1] - plain[1]).abs() <= bar_A).all()
    assert ((first[2] - plain[2]).abs() <= bar_b).all()


def test_one_row_calls_repeat():
    """The public calls on one row (what a rank of a real run has): dA and d(bias) repeat."""
    from ringmaster_amd.strategies.mamba import mamba2_chunk_decay, mamba2_chunk_state

    T, H = 4096, 24
    dt = seeded((1, T, H), 1).to(torch.bfloat16).cuda().requires_grad_(True)
    A = (-torch.exp(seeded((H,), 2))).cuda().requires_grad_(True)
    bias = (seeded((H,), 3) - 4).cuda().requires_grad_(True)
    x = seeded((1, T, H, 64), 4).to(torch.bfloat16).cuda()
    B = seeded((1, T, 1, 64), 5).to(torch.bfloat16).cuda()
    g_cum, g_st = seeded((1, T, H), 6).cuda(), seeded((1, H, 64, 64), 7).cuda()

    def grads():
        cum, _ = mamba2_chunk_decay(dt, A, bias, True)
        st = mamba2_chunk_state(x, dt, A, B, dt_bias=bias, dt_softplus=True)
        return (*torch.autograd.grad(cum, (dt, A, bias), g_cum),
                *torch.autograd.grad(st, (dt, A, bias), g_st))

    first = grads()
    for _ in range(8):
        assert all(torch.equal(a, b) for a, b in zip(first, grads()))


@pytest.mark.parametrize("lo,hi,bar", [(-8, -4, 3.75e-8), (-2, -1, 3.75e-8), (-0.5, 0, 3.45e-8),
                                       (0, 0.5, 2.96e-8), (1, 4, 2.66e-8)])
def test_softplus_is_as_exact_as_the_library(lo, hi, bar):
    """The effective step's rms error against fp64 stays within that of log1pf(expf(x)) over the
    same x (3.63, 3.61, 3.35, 2.87 and 2.58e-8, 3% of room)."""
    from ringmaster_amd import abi

    rows, T, H = 16, 1024, 64
    dt = (torch.rand((rows, T, H), generator=torch.Generator().manual_seed(5)) * (hi - lo) + lo).cuda()
    cum, e = torch.empty_like(dt), torch.empty_like(dt)
    decay, A, bias = (torch.zeros(s, device="cuda") for s in ((rows, H), (H,), (H,)))
    abi.check(abi.lib().rmx_mamba2_dt_cumsum(
        dt.data_ptr(), 1, bias.data_ptr(), A.data_ptr(), 1, cum.data_ptr(), e.data_ptr(),
        decay.data_ptr(), rows, T, H, abi.stream_of(dt)))
    ref = torch.log1p(torch.exp(dt.double()))
    rms = ((e - ref) / ref).pow(2).mean().sqrt().item()
    print(f"case softplus [{lo}, {hi}): rms {rms:.3e}", flush=True)
    assert rms < bar


@pytest.mark.parametrize("lo,hi,bar", [(-8, -4, 5.0e-8), (-2, -1, 4.45e-8), (-0.5, 0, 3.4e-8),
                                       (0.5, 1, 3.3e-8), (2, 4, 2.2e-8), (4, 10, 1.8e-8)])
def test_softplus_gradient_is_as_exact_as_the_library(lo, hi, bar):
    """The step's derivative (dL/de = 1, no other gradient) stays within the rms error of
    expf(x) / (expf(x) + 1) over the same range: 4.99, 4.45, 3.38, 3.27, 2.18 and 1.75e-8."""
    from ringmaster_amd import abi

    rows, T, H = 16, 1024, 64
    dt = (torch.rand((rows, T, H), generator=torch.Generator().manual_seed(5)) * (hi - lo) + lo).cuda()
    A, bias, g_A, g_b = (torch.zeros(H, device="cuda") for _ in range(4))
    g_e, g_dt = torch.ones_like(dt), torch.empty_like(dt)
    abi.check(abi.lib().rmx_mamba2_dt_cumsum_bwd(
        dt.data_ptr(), 1, bias.data_ptr(), A.data_ptr(), 1, None, g_e.data_ptr(), None, None,
        g_dt.data_ptr(), g_A.data_ptr(), g_b.data_ptr(), rows, T, H, abi.stream_of(dt)))
    ref = torch.sigmoid(dt.double())
    rms = ((g_dt - ref) / ref).pow(2).mean().sqrt().item()
    print(f"case softplus gradient [{lo}, {hi}): rms {rms:.3e}", flush=True)
    assert rms < bar
