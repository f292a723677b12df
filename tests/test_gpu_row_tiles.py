"""Calls whose plan moved from 256- to 128-row tiles (one partial round, m above 256):
against float64 on the dequantized weights at row counts around the tiles, split and
unsplit, with the bound of bf16 operands (1.7e-3 on average for the weights, 2.4e-3 with x
rounded too, 2.9e-3 with a bf16 y; 4e-3 asserted)."""
import pytest

torch = pytest.importorskip("torch")

from mold_amd import Device, GgmlDType, Linear, QTensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,n,k", [("Q4_K", 12288, 3072), ("Q6_K", 5120, 5120), ("Q8_0", 4096, 10240), ("Q4_K", 9216, 3072)])
def test_one_partial_round(t, n, k):
    dev = Device(0)
    g = torch.Generator(device="cuda").manual_seed(n + k)
    qt = QTensor.quantize(dev, torch.randn((n, k), device="cuda", generator=g) * 0.02, GgmlDType[t])
    lin, w = Linear(qt, torch.randn(n, device="cuda", generator=g) * 0.02), qt.dequantize().double()
    for m in (257, 300, 384, 385, 512, 640):
        x = torch.randn((m, k), device="cuda", generator=g)
        ref = x.double() @ w.t() + lin.bias.double()
        for y in (lin.forward(x), lin.forward(x.bfloat16(), out_dtype=torch.bfloat16)):
            assert ((y.double() - ref).norm() / ref.norm()).item() < 4e-3, m
        assert torch.equal(lin.forward(x), lin.forward(x))
