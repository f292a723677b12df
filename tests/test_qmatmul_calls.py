"""The arguments QMatMul.forward hands to mq_qmatmul, on the CPU with a recording stand-in
for the library."""
import types

import pytest

torch = pytest.importorskip("torch")

from mold_amd import QMatMul
from mold_amd import quantized as QZ

N, K = 64, 256


@pytest.fixture
def calls(monkeypatch):
    seen = []
    lib = types.SimpleNamespace(mq_qmatmul=lambda dev, w, x, xt, m, ldx, y, yt, ldy, *a: seen.append((x, m, ldx, ldy)) or 0)
    monkeypatch.setattr(QZ._lib, "load", lambda *a: lib)
    monkeypatch.setattr(QZ, "_stream_ptr", lambda *a: 0)
    return seen


def _matmul():
    return QMatMul(types.SimpleNamespace(shape=(N, K), device=types.SimpleNamespace(handle=1), handle=2))


@pytest.mark.parametrize("x", [torch.ones(K, 1).t(), torch.ones(K).expand(1, K), torch.ones(2 * K + 3)[1:].as_strided((1, K), (0, 1)),
                               torch.ones(1, K + 3)[:, :K], torch.ones(K), torch.ones(1, 1, K)],
                         ids=["column", "expanded", "stride 0", "wide", "vector", "leading one"])
def test_one_row_has_row_stride_k(calls, x):
    """A dimension of one has any stride; the library takes ldx >= k."""
    assert _matmul().forward(x).shape == (*x.shape[:-1], N)
    assert calls == [(x.data_ptr(), 1, K, N)]


def test_rows_keep_their_stride(calls):
    x = torch.ones(3, K + 8)[:, 8:]
    _matmul().forward(x)
    assert calls == [(x.data_ptr(), 3, K + 8, N)]
