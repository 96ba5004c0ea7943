"""rmx_cast_half against torch's cast, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sizes", [(8,), (2048, 2056, 8), (16, 0, 4096, 8 * 70001)])
def test_cast_half_equals_torch(sizes, dtype):
    from ringmaster_amd.ring import ops

    print(f"case cast {sizes} {dtype}", flush=True)
    g = torch.Generator().manual_seed(3)
    ts = [torch.randn(n, generator=g) * 10.0 ** torch.randint(-42, 6, (n,), generator=g) for n in sizes]
    edge = torch.tensor([0.0, -0.0, float("inf"), -float("inf"), 1.00390625, 1.01171875, 65520.0, 3.4e38])
    ts = [torch.cat([edge, t[8:]]) if t.numel() else t for t in ts]
    dev = [t.cuda() for t in ts]
    for got, t in zip(ops.cast_half(dev, dtype), dev):
        assert got.dtype == dtype and torch.equal(got.view(torch.int16), t.to(dtype).view(torch.int16))
    nan = torch.full((8,), float("nan"), device="cuda")
    assert ops.cast_half([nan], dtype)[0].isnan().all()
