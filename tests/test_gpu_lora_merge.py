"""The one-pass LoRA merge of k-quants against the separate calls (dequantize, apply per
patch, quantize), byte for byte: ranks around the 32-rank chunks, patches that overlap, end
inside a workgroup's rows or cover none of them, and rows past the last full tile."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mold_amd import Device, GgmlDType, MoldqError, QTensor, _lib
from mold_amd import lora as L

pytestmark = pytest.mark.gpu
TYPES = ["Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K"]


@pytest.fixture(scope="module")
def dev():
    return Device(0)


def _chain(qt, patches):
    t = qt.dequantize()
    for off, b, a, s in patches:
        L.lora_apply(t[off:off + b.shape[0]], b, a, s)
    return QTensor.quantize(qt.device, t, qt.dtype()).data()


def _merge(qt, patches):
    arr = (_lib.LoraPatchC * max(1, len(patches)))(*[
        _lib.LoraPatchC(b.data_ptr(), a.data_ptr(), b.stride(0), a.stride(0), off, b.shape[0], a.shape[0], s)
        for off, b, a, s in patches])
    h = ctypes.c_void_p()
    _lib.check(_lib.load().mq_lora_merge(qt.device.handle, qt.handle, arr, len(patches),
                                         torch.cuda.current_stream().cuda_stream, ctypes.byref(h)))
    return QTensor(qt.device, h).data()


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("n,k", [(1, 256), (17, 768), (64, 512), (131, 1024)])
def test_equals_the_separate_calls(dev, t, n, k):
    g = torch.Generator(device="cuda").manual_seed(n)
    rn = lambda *s: torch.randn(s, device="cuda", generator=g)
    qt = QTensor.quantize(dev, rn(n, k) * 0.02, GgmlDType[t])
    cases = [[]]
    for rank in (1, 31, 32, 33, 70):
        cases.append([(0, rn(n, rank) * 0.02, rn(rank, k) * 0.05, 0.8)])
    lo, hi = n // 3, n - n // 4
    wide = rn(12, k + 9) * 0.05
    cases.append([(lo, rn(hi - lo, 8) * 0.1, rn(8, k), 0.3), (0, rn(max(1, n // 2), 40) * 0.1, rn(40, k) * 0.2, -1.5),
                  (n - 1, rn(1, 3), rn(3, k), 0.01), (0, rn(n, 12) * 0.05, wide[:, 4:4 + k], 2.0)])
    for patches in cases:
        keep = [(o, b, a, s) for o, b, a, s in patches]
        assert np.array_equal(_merge(qt, keep), _chain(qt, [(o, b, a.contiguous(), s) for o, b, a, s in keep])), len(patches)


def test_patch_qtensor_takes_it_and_falls_back(dev):
    """k-quants in one pass; more patches than it holds, and 32-element types, by the separate calls."""
    g = torch.Generator(device="cuda").manual_seed(1)
    rn = lambda *s: torch.randn(s, device="cuda", generator=g)
    for t, count in (("Q4_K", 3), ("Q4_K", 9), ("Q8_0", 2)):
        qt = QTensor.quantize(dev, rn(96, 256) * 0.02, GgmlDType[t])
        fs = [(rn(96, 4) * 0.1, rn(4, 256) * 0.1) for _ in range(count)]
        out, applied = L.patch_qtensor(qt, [L.LoraPatch(a, b, 0.5, L.LoraTarget("w")) for b, a in fs])
        assert applied == count and np.array_equal(out.data(), _chain(qt, [(0, b, a, 0.5) for b, a in fs])), (t, count)


@pytest.mark.parametrize("t,rank,one", [("Q4_K", 32, True), ("Q4_K", 240, True), ("Q4_K", 241, False), ("Q3_K", 97, False),
                                         ("Q6_K", 512, False), ("Q2_K", 160, True), ("Q5_K", 300, False)])
def test_high_ranks_take_the_separate_calls(dev, t, rank, one, monkeypatch):
    """Where they are faster; the blocks are the same."""
    g = torch.Generator(device="cuda").manual_seed(rank)
    rn = lambda *s: torch.randn(s, device="cuda", generator=g)
    qt = QTensor.quantize(dev, rn(131, 512) * 0.02, GgmlDType[t])
    b, a = rn(131, rank) * 0.02, rn(rank, 512) * 0.05
    merges, lib = [], _lib.load()
    real = lib.mq_lora_merge
    monkeypatch.setattr(lib, "mq_lora_merge", lambda *args: merges.append(1) or real(*args))
    out, _ = L.patch_qtensor(qt, [L.LoraPatch(a, b, 0.5, L.LoraTarget("w"))])
    assert len(merges) == one
    assert np.array_equal(out.data(), _chain(qt, [(0, b, a, 0.5)])) and np.array_equal(out.data(), _merge(qt, [(0, b, a, 0.5)]))


def test_refuses(dev):
    g = torch.Generator(device="cuda").manual_seed(1)
    rn = lambda *s: torch.randn(s, device="cuda", generator=g)
    qt = QTensor.quantize(dev, rn(32, 256), GgmlDType.Q4_K)
    ok = (0, rn(32, 4), rn(4, 256), 1.0)
    for bad in ([(1, rn(32, 4), rn(4, 256), 1.0)], [(-1, rn(4, 4), rn(4, 256), 1.0)], [(0, rn(32, 4), rn(4, 128), 1.0)], [ok] * 9):
        with pytest.raises(MoldqError):
            _merge(qt, bad)
    with pytest.raises(MoldqError):
        _merge(QTensor.quantize(dev, rn(32, 256), GgmlDType.Q8_0), [ok])
