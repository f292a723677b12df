"""The k-quant quantizers against the reference quantizers, byte for byte (the arithmetic is
fixed, so there is no tolerance): row counts around the 64-row tiles and the 16 / 32 rows
of a workgroup, sources that are strided or not 16-byte aligned, and sub-blocks whose
quantized scale is zero inside a block that is not (they keep the search's quants)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from mold_amd import Device, GgmlDType, QTensor
from oracle import oracle as O

pytestmark = pytest.mark.gpu
TYPES = ["Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K"]


@pytest.fixture(scope="module")
def dev():
    return Device(0)


def _same(dev, t, x, src=None):
    qt = QTensor.quantize(dev, torch.from_numpy(x).cuda() if src is None else src, GgmlDType[t])
    assert np.array_equal(qt.data(), O.quantize(getattr(O, t), x).reshape(-1)), t


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 63, 64, 65, 129])
def test_row_counts(dev, t, n):
    x = (np.random.default_rng(n).standard_normal((n, 512)) * 0.02).astype(np.float32)
    _same(dev, t, x)
    wide = torch.zeros((n, 512 + 5), device="cuda")
    wide[:, 3:515] = torch.from_numpy(x).cuda()
    _same(dev, t, x, wide[:, 3:515])


@pytest.mark.parametrize("t", TYPES)
def test_uneven_blocks(dev, t):
    rng = np.random.default_rng(5)
    rows = []
    for spread in (1e-7, 1e-5, 1e-3, 1.0):     # sub-blocks of 16 and 32 far below, equal to zero, or spread inside
        for w in (16, 32):
            x = rng.standard_normal((8, 256 // w, w)) * np.where(rng.random((8, 256 // w, 1)) < 0.5, spread, 1.0)
            x[rng.random((8, 256 // w)) < 0.2] = 0.0
            rows.append(x.reshape(8, 256))
    rows.append(5 + 1e-3 * rng.standard_normal((8, 256)))        # one sign, far from zero
    rows.append(-5 + 1e-3 * rng.standard_normal((8, 256)))
    rows.append(np.exp(6 * rng.standard_normal((8, 256))))
    rows.append(np.round(3 * rng.standard_normal((8, 256))))     # ties
    rows.append(1e-38 * rng.standard_normal((8, 256)))           # denormal sums: 1 / range overflows
    rows.append(1e30 * rng.standard_normal((8, 256)))
    _same(dev, t, np.concatenate(rows).astype(np.float32))
