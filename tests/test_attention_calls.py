"""The calls around the attention kernel, on the CPU: a stand-in for mq_attention_bf16
that works on host memory a head and 32 query rows at a time, each read and written
before the next, so that a destination over its own inputs shows in the values."""
import contextlib
import ctypes
import math
import types

import pytest

torch = pytest.importorskip("torch")

from mold_amd import flux as F
from mold_amd import fused as FU

H, L, HD = 2, 96, 128


def _at(ptr, n, dtype=torch.bfloat16, ctype=ctypes.c_uint16):
    return torch.frombuffer((ctype * n).from_address(ptr), dtype=dtype)


class _Lib:
    """Records each call's out, ldo, lse and guard, and computes it (no masked keys)."""

    def __init__(self):
        self.calls = []
        self.fill_lse = torch.full((H,), 50.0)     # each head's log-sum-exp

    def mq_attention_scratch_size(self, *a):
        return 0

    def mq_attention_bf16(self, q, k, v, batch, heads, l, hd, valid, drop, out, sb, ldo, lse, guard, *_):
        batch, heads, l, valid, sb, ldo = map(int, (batch, heads, l, valid, sb, ldo))     # a trace's sizes are tensors
        self.calls.append(types.SimpleNamespace(out=out, ldo=ldo, lse=lse, guard=guard))
        assert hd == HD and ldo >= heads * HD
        if lse:
            _at(lse, heads * valid, torch.float32, ctypes.c_float).view(heads, valid).copy_(
                self.fill_lse[:, None].expand(heads, valid))
        for b in range(batch):
            for h in range(heads):
                qh, kh, vh = (_at(p + 2 * HD * l * (b * heads + h), l * HD).view(l, HD) for p in (q, k, v))
                for r in range(0, valid, 32):
                    n = min(32, valid - r)
                    s = qh[r:r + n].float() @ kh[:valid].float().t() / math.sqrt(HD)
                    o = _at(out + 2 * (b * sb + r * ldo), (n - 1) * ldo + heads * HD)
                    o.as_strided((n, HD), (ldo, 1), h * HD).copy_(torch.softmax(s, -1) @ vh[:valid].float())
        return 0


def _efficient(q, k, v, bias, want_lse):
    s = q.float() @ k.float().transpose(-1, -2) / math.sqrt(HD)
    return (torch.softmax(s, -1) @ v.float()).to(q.dtype), torch.logsumexp(s, -1)


@pytest.fixture
def lib(monkeypatch):
    fake = _Lib()
    monkeypatch.setattr(FU._lib, "load", lambda *a: fake)
    monkeypatch.setattr(FU, "_stream_ptr", lambda *a: 0)
    monkeypatch.setattr(FU, "takes_attention", lambda q, k, v: not FU.recorded(q, k, v))
    monkeypatch.setattr(torch.cuda, "device", lambda d: contextlib.nullcontext())
    monkeypatch.setattr(F, "ATTENTION_BACKEND", {"name": None})
    monkeypatch.setattr(torch.ops.aten, "_scaled_dot_product_efficient_attention", _efficient)    # not on the CPU
    return fake


def _qkv():
    """q, k, v [H, L, 128], the three in one buffer."""
    g = torch.Generator().manual_seed(3)
    return torch.randn((3, H, L, HD), generator=g).to(torch.bfloat16)


def test_out_on_another_device(lib):
    """Unpadded: filled through a copy.  Padded: refused.  Its address never reaches the kernel."""
    q, k, v = _qkv()
    out = torch.empty((L, H * HD), dtype=torch.bfloat16, device="meta")
    assert F.attention_bf16(q, k, v, out=out) is out
    with pytest.raises(ValueError):
        F.attention_bf16(q, k, v, valid=L - 3, out=out[:L - 3])
    assert len(lib.calls) == 1 and lib.calls[0].out


def _reference(q, k, v, valid=L):
    s = q[:, :valid].float() @ k[:, :valid].float().transpose(1, 2) / math.sqrt(HD)
    return (torch.softmax(s, -1) @ v[:, :valid].float()).transpose(0, 1).reshape(valid, H * HD)


@pytest.mark.parametrize("over", ["q", "k", "v", "q and k"])
@pytest.mark.parametrize("padded", [False, True])
def test_out_over_its_inputs(lib, over, padded):
    """q, k and v are read whole before out changes; a recomputed head (the scores of head 1 are all
    below -10 over the padding's 0) reads them too."""
    qkv = _qkv()
    valid = L - 5 if padded else L
    if padded:
        qkv[1, 1] = -qkv[0, 1, :1] * 4
        qkv[0, 1] = qkv[0, 1, :1]
        qkv[1:, :, valid:] = 0
    q, k, v = qkv
    ref = _reference(q, k, v, valid)
    at = {"q": 0, "k": 1, "v": 2, "q and k": 0.5}[over]
    flat = qkv.view(-1)
    out = flat[int(at * q.numel()):][:valid * H * HD].view(valid, H * HD)
    if padded:
        lib.fill_lse = torch.tensor([50.0, -50.0])
    assert F.attention_bf16(q, k, v, valid=valid, out=out) is out
    assert ((out.float() - ref).norm() / ref.norm()).item() < 6e-3     # two roundings to bf16
    assert all(c.out != out.data_ptr() for c in lib.calls)


def test_a_separate_out_is_written_directly(lib):
    q, k, v = _qkv()
    wide = torch.full((L, H * HD + 16), 3.0, dtype=torch.bfloat16)
    out = wide[:, 8:8 + H * HD]
    assert F.attention_bf16(q, k, v, out=out) is out and lib.calls[0].out == out.data_ptr()
    ref = _reference(q, k, v)
    assert ((out.float() - ref).norm() / ref.norm()).item() < 6e-3
    assert bool((wide[:, :8] == 3.0).all()) and bool((wide[:, 8 + H * HD:] == 3.0).all())


@pytest.mark.parametrize("at", [-1, 0, 3])
def test_c_entry_refuses_out_over_its_inputs(at):
    """Addresses only: the refusal comes before any launch."""
    from mold_amd import _lib
    base, size = 1 << 20, 64 * HD * 2
    ins = [base, base + 4 * size, base + 8 * size]
    for i in range(3):
        args = list(ins)
        out = args[i] + at * size // 4
        rc = _lib.load().mq_attention_bf16(*args, 1, 1, 64, HD, 64, None, out, 0, HD, None, None, None, 0, None)
        assert rc == -1 and b"lies over" in _lib.load().mq_last_error()


@pytest.mark.parametrize("guard", [torch.zeros((), dtype=torch.bfloat16), torch.zeros((), dtype=torch.float64), torch.zeros(2),
                                   torch.zeros((), device="meta")], ids=["bf16", "f64", "two", "elsewhere"])
def test_a_guard_the_kernel_cannot_raise(lib, guard):
    """Refused where the call is padded or batched, not looked at in an unpadded single one."""
    q, k, v = _qkv()
    for call in (lambda: F.attention_bf16(q, k, v, valid=L - 1, guard=guard),
                 lambda: F.attention_bf16_batch(q[None], k[None], v[None], L - 1, guard, [None]),
                 lambda: F.attention_bf16_batch(q[None], k[None], v[None], L, guard, [None])):
        with pytest.raises(ValueError):
            call()
    assert not lib.calls
    assert F.attention_bf16(q, k, v, guard=guard).shape == (L, H * HD) and lib.calls[0].guard is None
    one = torch.zeros((1, 1))
    F.attention_bf16(q, k, v, valid=L - 1, guard=one)
    assert lib.calls[1].guard == one.data_ptr()


def test_an_lse_or_out_the_kernel_cannot_write(lib):
    q, k, v = _qkv()
    for lse in (torch.empty((1, H, L), dtype=torch.bfloat16), torch.empty((1, H, L - 1)), torch.empty((1, H, 2 * L))[:, :, ::2],
                torch.empty((1, H, L), device="meta")):
        with pytest.raises(ValueError):
            FU.attention(q, k, v, L, lse=lse)
    for out in (torch.empty((L, H * HD)), torch.empty((L - 1, H * HD), dtype=torch.bfloat16),
                torch.empty((H * HD, L), dtype=torch.bfloat16).t()):
        with pytest.raises(ValueError):
            FU.attention(q, k, v, L, out=out)
    assert not lib.calls


def test_a_traced_call_replays(lib):
    """torch.jit.trace: the kernel's call would leave only the allocation of its result in the graph."""
    q, k, v = _qkv()
    traced = torch.jit.trace(lambda a, b, c: F.attention_bf16(a, b, c), (q, k, v), check_trace=False)
    assert not lib.calls
    x, y, z = (t.flip(1).contiguous() for t in (q, k, v))
    ref = _reference(x, y, z)
    assert ((traced(x, y, z).float() - ref).norm() / ref.norm()).item() < 6e-3


def test_a_function_mode_sees_the_operations(lib):
    """A mode that records functions gets PyTorch's; the one that torch.device(..) pushes records nothing."""
    from torch.overrides import TorchFunctionMode

    class Names(TorchFunctionMode):
        seen = []

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.seen.append(getattr(func, "__name__", str(func)))
            return func(*args, **(kwargs or {}))
    q, k, v = _qkv()
    with Names():
        F.attention_bf16(q, k, v)
    assert not lib.calls and "softmax" in Names.seen
    with torch.device("cpu"):
        F.attention_bf16(q, k, v)
    assert len(lib.calls) == 1
    with Names(), torch.device("cpu"):
        F.attention_bf16(q, k, v)
    with Names(), torch._C.DisableTorchFunction():
        F.attention_bf16(q, k, v)
    assert len(lib.calls) == 2


def test_one_row_of_out_may_have_any_stride(lib):
    """A dimension of one has any stride; the library takes ldo >= H * 128."""
    q, k, v = (t[:, :1].contiguous() for t in _qkv())
    ref = v.transpose(0, 1).reshape(1, H * HD)
    for stride in (0, 1, 8, H * HD + 4):
        out = torch.empty(2 * H * HD, dtype=torch.bfloat16).as_strided((1, H * HD), (stride, 1))
        assert F.attention_bf16(q, k, v, out=out) is out and torch.equal(out, ref)
    one = torch.empty((1, H * HD), dtype=torch.bfloat16).as_strided((1, 1, H * HD), (3, 5, 1))
    assert torch.equal(FU.attention(q[None], k[None], v[None], 1, out=one)[0], ref)
    assert [c.ldo for c in lib.calls] == [H * HD] * 5


@pytest.mark.parametrize("valid", [L, L - 3])
def test_autograd_sees_out_change(lib, valid):
    """out is written in place: a graph that saved its old values must not go on with the new ones, and an
    out that requires gradients is recorded (or, a leaf, refused)."""
    q, k, v = _qkv()
    q, k, v = q, *(torch.cat([t[:, :valid], 0 * t[:, valid:]], 1) for t in (k, v))
    out = torch.randn((valid, H * HD)).to(torch.bfloat16)
    x = torch.ones_like(out, requires_grad=True)
    y = (out * x).sum()
    F.attention_bf16(q, k, v, valid=valid, out=out)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward()
    leaf = torch.zeros_like(out, requires_grad=True)
    with pytest.raises(RuntimeError):
        F.attention_bf16(q, k, v, valid=valid, out=leaf)
    assert not leaf.detach().any()
    with torch.no_grad():
        F.attention_bf16(q, k, v, valid=valid, out=leaf)
    assert torch.equal(leaf, out)


def test_pytorchs_backend_does_not_decide_for_the_kernel(lib):
    """A call of another head size that found no fused kernel leaves calls of 128 where they were."""
    q, k, v = _qkv()
    F.ATTENTION_BACKEND["name"] = "chunked"
    F.attention_bf16(q, k, v)
    F.attention_bf16_batch(q[None], k[None], v[None], L, torch.zeros(()), [None])
    assert len(lib.calls) == 2 and F.ATTENTION_BACKEND["name"] == "chunked"


def test_sizes_the_entry_refuses_stay_with_pytorch():
    assert FU.takes_shape((24, 4608, 128)) and FU.takes_shape((2, 24, 4608, 128)) and FU.takes_shape((1 << 20, 1, 128))
    assert FU.takes_shape((2, 1 << 19, 1, 128)) and FU.takes_shape((1, 1 << 23, 128))
    for shape in ((1 + (1 << 20), 1, 128), (2, 1 + (1 << 19), 1, 128), (1, 1 + (1 << 23), 128), (0, 4, 128), (4, 0, 128),
                  (0, 4, 4, 128), (4, 4, 64), (4, 128), (1, 1, 4, 4, 128)):
        assert not FU.takes_shape(shape), shape


@pytest.mark.parametrize("batch,heads", [(1 << 62, 4), (1 << 21, 1), (1, (1 << 20) + 1), ((1 << 20) // 3 + 1, 3)])
def test_c_entry_refuses_more_heads_than_it_counts(batch, heads):
    """Also where batch * heads does not fit 64 bits (addresses only: refused before any launch)."""
    from mold_amd import _lib
    rc = _lib.load().mq_attention_bf16(4096, 4096, 4096, batch, heads, 64, HD, 64, None, 1 << 40, 0, heads * HD, None, None, None, 0,
                                       None)
    assert rc == -1 and b"2^20 heads" in _lib.load().mq_last_error()
