"""The few-rows GEMM (9 <= m <= 96): row tiles of 32 / 64 / 96, K in chunks of 512 or 256
columns split over workgroups, two K halves per workgroup, f32 x rounded on its way into
LDS.  Against float64 on the dequantized weights; the bound is that of the operands'
roundings to bf16 (2^-9 relative each at most, 1.7e-3 on average each for the weight and
the f32 x: 2.4e-3 together, 2.9e-3 with a bf16 y); 4e-3 is asserted."""
import pytest

torch = pytest.importorskip("torch")

from mold_amd import ACT_GELU_TANH, Device, GgmlDType, Linear, QTensor

pytestmark = pytest.mark.gpu
BLOCK32 = ["Q4_0", "Q4_1", "Q5_0", "Q5_1", "Q8_0"]
TYPES = BLOCK32 + ["Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K"]
BOUND = 4e-3


@pytest.fixture(scope="module")
def dev():
    return Device(0)


def _weight(dev, t, n, k, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + 31 * n + k)
    qt = QTensor.quantize(dev, torch.randn((n, k), device="cuda", generator=g) * 0.02, GgmlDType[t])
    lin = Linear(qt, torch.randn(n, device="cuda", generator=g) * 0.02)
    return lin, qt.dequantize().double().cpu(), lin.bias.double().cpu(), g


def _err(y, ref):
    return ((y.double().cpu() - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("n,k", [(65, 256), (33, 768), (300, 512), (130, 1280), (4100, 2304), (128, 8448)])
def test_tiles_and_chunks(dev, t, n, k):
    """One chunk, an odd number of units (half a last chunk), one chunk a part, several, and n off the tile."""
    lin, w, b, g = _weight(dev, t, n, k)
    for m in (9, 31, 32, 33, 64, 65, 96):
        x = torch.randn((m, k), device="cuda", generator=g)
        ref = x.double().cpu() @ w.t() + b
        y = lin.forward(x)
        assert _err(y, ref) < BOUND, (t, m)
        assert torch.equal(y, lin.forward(x))
        assert torch.equal(y, lin.forward(x.bfloat16(), out_dtype=torch.float32)), (t, m)   # the same rounding of x
        assert _err(lin.forward(x, out_dtype=torch.bfloat16), ref) < BOUND


@pytest.mark.parametrize("m", [9, 40, 96])
def test_k_of_half_a_unit_pair(dev, m):
    """Q8_0 units of 128: K of 3 and 9 of them, so a chunk ends in the middle of a wave's share."""
    for k in (128, 384, 1152):
        lin, w, b, g = _weight(dev, "Q8_0", 200, k, seed=2)
        x = torch.randn((m, k), device="cuda", generator=g)
        assert _err(lin.forward(x), x.double().cpu() @ w.t() + b) < BOUND


@pytest.mark.parametrize("m", [9, 50, 77, 96])
def test_epilogues_strides_and_unsplit(dev, m):
    lin, w, b, g = _weight(dev, "Q4_K", 1000, 3072, seed=3)
    wide = torch.randn((m, 3072 + 40), device="cuda", generator=g)
    x = wide[:, 8:3080]                                     # strided rows, 16-byte aligned
    odd = torch.zeros((m, 3072 + 5), device="cuda")
    odd[:, 3:3075] = x                                      # not aligned: the staged path
    ref = x.double().cpu() @ w.t() + b
    y = lin.forward(x)
    assert _err(y, ref) < BOUND and _err(lin.forward(odd[:, 3:3075]), ref) < BOUND
    act = lin.forward(x, act=ACT_GELU_TANH, act_from=333)
    gelu = ref.clone()
    gelu[:, 333:] = torch.nn.functional.gelu(ref[:, 333:], approximate="tanh")
    assert _err(act, gelu) < BOUND and torch.equal(act[:, :333], y[:, :333])
    gate = torch.randn(1000, device="cuda", generator=g)
    buf = torch.randn((m, 1024), device="cuda", generator=g)
    res = buf[:, :1000]
    want = res.double().cpu() + gate.double().cpu() * ref
    tail = buf[:, 1000:].clone()
    lin.gated_add(x, gate, res)
    assert _err(res, want) < BOUND and torch.equal(buf[:, 1000:], tail)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    dev.set_stream_tail_split(s, False)
    with torch.cuda.stream(s):
        whole = lin.forward(x)                              # K in one part
    s.synchronize()
    dev.set_stream_tail_split(s, True)
    assert _err(whole, ref) < BOUND


@pytest.mark.parametrize("k", [256, 3072])
def test_whole_and_ragged_blocks_of_rows(dev, k):
    """Whole 32-row blocks and the last one, columns with and without GELU in one wave, the residual's rows, in one part of K."""
    lin, w, b, g = _weight(dev, "Q4_K", 333, k, seed=7)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    dev.set_stream_tail_split(s, False)
    gate = torch.randn(333, device="cuda", generator=g)
    with torch.cuda.stream(s):
        for m in (1, 3, 8, 9, 31, 32, 33, 60, 63, 64):
            x = torch.randn((m, k), device="cuda", generator=g).bfloat16()
            ref = x.double().cpu() @ w.t() + b
            gelu = ref.clone()
            gelu[:, 77:] = torch.nn.functional.gelu(ref[:, 77:], approximate="tanh")
            buf = torch.full((m + 2, 400), 5.0, device="cuda")
            res, full = buf[1:m + 1, 30:363], torch.full((m + 2, 333), 3.0, device="cuda")
            r0 = torch.randn((m, 333), device="cuda", generator=g)
            res.copy_(r0)
            lin.gated_add(x, gate, res)
            s.synchronize()
            assert _err(res, r0.double().cpu() + gate.double().cpu() * ref) < BOUND, m
            res.fill_(5.0)
            assert bool((buf == 5.0).all()), m
            if m > 8:                                           # up to 8 rows are the GEMV's
                for dt in (torch.float32, torch.bfloat16):
                    out = full.to(dt)
                    lin.matmul.forward(x, bias=lin.bias, act=ACT_GELU_TANH, act_from=77, out=out[1:m + 1])
                    s.synchronize()
                    assert _err(out[1:m + 1], gelu) < BOUND and bool((out[0] == 3).all()) and bool((out[m + 1] == 3).all()), m
    dev.set_stream_tail_split(s, True)


def test_y_over_f32_x(dev):
    """y written over f32 x: x is read whole before any of y is written."""
    lin, w, b, g = _weight(dev, "Q8_0", 512, 512, seed=4)
    x = torch.randn((48, 512), device="cuda", generator=g)
    ref = x.double().cpu() @ w.t() + b
    lin.matmul.forward(x, bias=lin.bias, out=x)
    assert _err(x, ref) < BOUND


def test_captured_after_reserving_the_stated_workspace(dev):
    lin, w, b, g = _weight(dev, "Q6_K", 4096, 4096, seed=5)
    x = torch.randn((77, 4096), device="cuda", generator=g)
    y = torch.empty((77, 4096), device="cuda")
    s = torch.cuda.Stream()
    dev.reserve_stream_scratch(lin.matmul.workspace_bytes(77), s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        lin.matmul.forward(x, bias=lin.bias, out=y)
    for i in range(3):
        x.copy_(torch.randn((77, 4096), device="cuda", generator=g))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, lin.forward(x)), i


def test_far_apart_rows_fit_the_stated_workspace(dev):
    """f32 rows that lie too far apart for the kernel's 31-bit offsets, in a stream with exactly workspace_bytes."""
    lin, w, b, g = _weight(dev, "Q8_0", 6144, 512, seed=6)
    m, ldx = 64, 1 << 23
    x = torch.empty(((m - 1) * ldx + 512,), device="cuda").as_strided((m, 512), (ldx, 1))
    x.copy_(torch.randn((m, 512), device="cuda", generator=g))
    y = torch.empty((m, 6144), device="cuda")
    s = torch.cuda.Stream()
    dev.reserve_stream_scratch(lin.matmul.workspace_bytes(m), s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        lin.matmul.forward(x, bias=lin.bias, out=y)
    for i in range(2):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert _err(y, x.double().cpu() @ w.t() + b) < BOUND
        assert torch.equal(y, lin.forward(x.contiguous())), i
