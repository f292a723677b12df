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

    def mq_attention_scratch_size(self, *a):
        return 0

    def mq_attention_bf16(self, q, k, v, batch, heads, l, hd, valid, drop, out, sb, ldo, lse, guard, *_):
        self.calls.append(types.SimpleNamespace(out=out, ldo=ldo, lse=lse, guard=guard))
        assert hd == HD and ldo >= heads * HD
        for b in range(batch):
            for h in range(heads):
                qh, kh, vh = (_at(p + 2 * HD * l * (b * heads + h), l * HD).view(l, HD) for p in (q, k, v))
                for r in range(0, valid, 32):
                    n = min(32, valid - r)
                    s = qh[r:r + n].float() @ kh[:valid].float().t() / math.sqrt(HD)
                    o = _at(out + 2 * (b * sb + r * ldo), (n - 1) * ldo + heads * HD)
                    o.as_strided((n, HD), (ldo, 1), h * HD).copy_(torch.softmax(s, -1) @ vh[:valid].float())
        return 0


@pytest.fixture
def lib(monkeypatch):
    fake = _Lib()
    monkeypatch.setattr(FU._lib, "load", lambda *a: fake)
    monkeypatch.setattr(FU, "_stream_ptr", lambda *a: 0)
    monkeypatch.setattr(FU, "takes_attention", lambda q, k, v: True)
    monkeypatch.setattr(torch.cuda, "device", lambda d: contextlib.nullcontext())
    monkeypatch.setattr(F, "ATTENTION_BACKEND", {"name": None})
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
