"""mq_attention_bf16 against float64 attention: the edges of its key blocks (64, two per
loop turn, V in a ring of three) and query tiles (128 / 256 rows), masked key ranges,
strided outputs, and the calls that stay with PyTorch's attention.

The bound on the relative error is that of the roundings: the probabilities and the
output to bf16, 2^-9 / sqrt(3) * sqrt(2) relative on average = 1.6e-3 each at most
(uniform mantissas: 1.66e-3), so 2.4e-3 together; 3e-3 is asserted."""
import math

import pytest

torch = pytest.importorskip("torch")

from mold_amd import MoldqError, _lib
from mold_amd import fused as FU
from mold_amd.flux import PAD_MIN_SHARE, attention_bf16, attention_bf16_batch
from tests.test_build_checks import HIPCC, _asm, _functions, _m0_outside_asm

gpu = pytest.mark.gpu


def _inputs(b, h, l, valid, sharp=1.0, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + 7919 * valid)
    q, k, v = (torch.randn((b, h, l, 128), device="cuda", generator=g) for _ in range(3))
    q = q * sharp
    k[:, :, valid:] = 0
    v[:, :, valid:] = 0
    return [t.to(torch.bfloat16) for t in (q, k, v)]


def _ref(q, k, v, valid, drop=None):
    """[H, L, 128] -> ([valid, H * 128], scores) in float64 on the host over the kept keys."""
    keep = [i for i in range(valid) if drop is None or not drop[0] <= i < drop[1]]
    qf, kf, vf = (t.double().cpu() for t in (q[:, :valid], k[:, keep], v[:, keep]))
    s = qf @ kf.transpose(1, 2).contiguous() / math.sqrt(128)
    o = torch.softmax(s, dim=-1) @ vf
    return o.transpose(0, 1).reshape(valid, -1), s


def _err(out, ref):
    return ((out.double().cpu() - ref).norm() / ref.norm()).item()


@gpu
@pytest.mark.parametrize("valid", [1, 2, 31, 33, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 320, 511, 577])
@pytest.mark.parametrize("heads", [1, 3])
def test_block_and_tile_edges(valid, heads):
    q, k, v = _inputs(1, heads, valid, valid)
    assert FU.takes_attention(q[0], k[0], v[0])
    out = attention_bf16(q[0], k[0], v[0])
    ref, _ = _ref(q[0], k[0], v[0], valid)
    assert out.shape == (valid, heads * 128) and _err(out, ref) < 3e-3
    assert torch.equal(out, attention_bf16(q[0], k[0], v[0]))


@gpu
@pytest.mark.parametrize("heads,valid", [(40, 1664), (140, 512), (24, 2816)])
def test_eight_wave_tiles_match_four_wave_tiles(heads, valid, monkeypatch):
    """Enough tiles for the 8-wave variant: without scratch each head equals the same head alone (4 waves)
    bit for bit."""
    monkeypatch.setattr(_lib.load(), "mq_attention_scratch_size", lambda *a: 0)
    q, k, v = _inputs(1, heads, valid, valid)
    out = attention_bf16(q[0], k[0], v[0])
    for i in (0, heads // 2, heads - 1):
        one = attention_bf16(q[0, i:i + 1], k[0, i:i + 1], v[0, i:i + 1])
        assert torch.equal(out[:, 128 * i:128 * i + 128], one)
    ref, _ = _ref(q[0, :1], k[0, :1], v[0, :1], valid)
    assert _err(out[:, :128], ref) < 3e-3


@gpu
@pytest.mark.parametrize("heads,valid,drop", [
    (1, 2048, None), (1, 2049, (64, 1985)), (3, 2111, (0, 2110)), (2, 2560, (1, 2560)), (2, 4097, (100, 300)),
    (12, 2816, None), (12, 3000, (1000, 1001))])
def test_split_tiles(heads, valid, drop):
    """Tiles whose keys are shared between workgroups: all of them (few heads) or those after whole rounds (12 heads x 2
    elements), shares left empty by a masked range, remainders of rows and keys, the log-sum-exp and the guard."""
    assert _lib.load().mq_attention_scratch_size(2, heads, valid) > 0
    l = -(-valid // 256) * 256
    q, k, v = _inputs(2, heads, l, valid, seed=13)
    if drop is not None:
        k[1, :, drop[0]:drop[1]] = 0
        v[1, :, drop[0]:drop[1]] = 0
    guard, lse = torch.zeros((), device="cuda"), torch.empty((2, heads, valid), device="cuda")
    out = FU.attention(q, k, v, valid, drops=[None, drop], guard=guard, lse=lse)
    assert torch.equal(out, FU.attention(q, k, v, valid, drops=[None, drop]))
    share, hs = 0.0, sorted({0, heads - 1})
    for b, d in ((0, None), (1, drop)):
        n = l - valid + (0 if d is None else d[1] - d[0])
        for h in hs:
            ref, s = _ref(q[b, h:h + 1], k[b, h:h + 1], v[b, h:h + 1], valid, d)
            assert _err(out[b, :, 128 * h:128 * h + 128], ref) < 3e-3, (b, h)
            z = n + torch.exp(s[0]).sum(-1)
            assert (lse[b, h].double().cpu() - z.log()).abs().max() < 1e-4, (b, h)
            share = max(share, float((n / z).max()))
    assert float(guard) >= share * (1 - 1e-4) and (len(hs) < heads or abs(float(guard) - share) <= 1e-4 * share)


@gpu
@pytest.mark.parametrize("valid,drop", [(130, (0, 1)), (130, (1, 65)), (300, (64, 128)), (300, (10, 299)), (300, (0, 299)),
                                        (300, (100, 300)), (65, (1, 65))])
def test_masked_key_range(valid, drop):
    q, k, v = _inputs(2, 2, 320, valid, seed=3)
    k[1, :, drop[0]:drop[1]] = 0
    v[1, :, drop[0]:drop[1]] = 0
    guard = torch.zeros((), device="cuda")
    out = attention_bf16_batch(q, k, v, valid, guard, [None, drop])
    share = 0.0
    for b, d in ((0, None), (1, drop)):
        ref, s = _ref(q[b], k[b], v[b], valid, d)
        assert _err(out[b], ref) < 3e-3, b
        n = 320 - valid + (0 if d is None else d[1] - d[0])
        share = max(share, float((n / (n + torch.exp(s).sum(-1))).max()))
    # one f32 exponential and logarithm of scores up to ~6 from bf16 products summed in f32
    assert abs(float(guard) - share) < 1e-4 * share
    guard.fill_(2.0)
    attention_bf16_batch(q, k, v, valid, guard, [None, drop])
    assert float(guard) == 2.0


@gpu
@pytest.mark.parametrize("sharp", [0.0, 30.0])
def test_flat_and_one_hot_rows(sharp):
    """Equal scores (a mean of v), and scores of up to a few hundred (one key takes nearly all)."""
    q, k, v = _inputs(1, 2, 200, 200, sharp=sharp, seed=5)
    ref, _ = _ref(q[0], k[0], v[0], 200)
    assert _err(attention_bf16(q[0], k[0], v[0]), ref) < 3e-3


@gpu
def test_non_finite_rows_stay_in_their_rows():
    q, k, v = _inputs(1, 1, 192, 192, seed=9)
    clean = attention_bf16(q[0], k[0], v[0])
    q[0, 0, 5, 3] = float("nan")
    q[0, 0, 70, 3] = float("inf")
    out = attention_bf16(q[0], k[0], v[0])
    assert not torch.isfinite(out[5].float()).any() and torch.isnan(out[70].float()).any()
    keep = [i for i in range(192) if i not in (5, 70)]
    assert torch.equal(out[keep], clean[keep])


@gpu
def test_lse_and_strided_out():
    valid, l, h = 150, 256, 2
    q, k, v = _inputs(2, h, l, valid, seed=11)
    lse = torch.empty((2, h, valid), device="cuda")
    buf = torch.full((2, valid, h * 128 + 64), 3.0, dtype=torch.bfloat16, device="cuda")
    out = FU.attention(q, k, v, valid, out=buf[:, :, 24:24 + h * 128], lse=lse)
    assert torch.equal(out, FU.attention(q, k, v, valid))
    assert bool((buf[:, :, :24] == 3.0).all()) and bool((buf[:, :, 24 + h * 128:] == 3.0).all())
    odd = torch.full((2, valid, h * 128 + 3), 3.0, dtype=torch.bfloat16, device="cuda")   # rows not 16-byte aligned
    assert torch.equal(FU.attention(q, k, v, valid, out=odd[:, :, 1:1 + h * 128]), out)
    assert bool((odd[:, :, 0] == 3.0).all()) and bool((odd[:, :, 1 + h * 128:] == 3.0).all())
    for b in range(2):
        _, s = _ref(q[b], k[b], v[b], valid)
        want = torch.log(torch.exp(s).sum(-1) + (l - valid))
        assert (lse[b].double().cpu() - want).abs().max() < 1e-4


@gpu
def test_out_on_the_host():
    """Filled by a copy where nothing is padded, refused where something is."""
    q, k, v = (t[0] for t in _inputs(1, 2, 96, 96, seed=17))
    host = torch.empty((96, 256), dtype=torch.bfloat16)
    assert attention_bf16(q, k, v, out=host) is host
    assert torch.equal(host, attention_bf16(q, k, v).cpu())
    for guard in (None, torch.zeros((), device="cuda")):
        with pytest.raises(ValueError):
            attention_bf16(q, k, v, valid=90, guard=guard, out=host[:90])


@gpu
def test_other_calls_keep_pytorch_attention():
    """Inputs that autograd records, other head sizes and non-contiguous or mixed inputs do not take the kernel and still work."""
    q, k, v = (t[0] for t in _inputs(1, 2, 64, 64, seed=13))
    out = attention_bf16(q, k, v)
    leaf = q.clone().requires_grad_(True)
    assert not FU.takes_attention(leaf, k, v)
    got = attention_bf16(leaf, k, v)
    assert got.requires_grad and _err(got.detach(), out.double().cpu()) < 5e-3
    with torch.no_grad():
        assert FU.takes_attention(leaf, k, v) and torch.equal(attention_bf16(leaf, k, v), out)
    assert not FU.takes_attention(q.transpose(0, 1).contiguous().transpose(0, 1), k, v)
    assert torch.equal(attention_bf16(q.float(), k.transpose(0, 1).contiguous().transpose(0, 1), v), out)   # made bf16, contiguous
    small = [t[:, :, :64].contiguous() for t in (q, k, v)]
    assert not FU.takes_attention(*small) and attention_bf16(*small).shape == (64, 128)


@gpu
@pytest.mark.parametrize("name,args", [
    ("test_padded_attention_matches_reference", (295, 512)), ("test_padded_attention_matches_reference", (1000, 1024)),
    ("test_padded_attention_matches_reference", (512, 512)), ("test_batched_padded_attention_with_dropped_keys", ()),
    ("test_padded_attention_ill_conditioned_rows_recomputed", ()), ("test_padded_attention_guard_and_step_rerun", ())])
def test_pytorch_route_of_padded_calls(name, args, monkeypatch):
    """The zero-key correction, the recompute and the masked keys of calls the kernel does not take."""
    from tests import test_gpu_glue
    monkeypatch.setattr(FU, "takes_attention", lambda q, k, v: False)
    monkeypatch.setattr(FU, "attention", None)
    getattr(test_gpu_glue, name)(*args)


def test_argument_checks():
    from mold_amd import _lib
    lib = _lib.load()

    def call(hd=128, batch=1, heads=1, l=64, valid=64, drop=None, ldo=128, q=4096, scratch=None):
        return lib.mq_attention_bf16(q, 4096, 4096, batch, heads, l, hd, valid, drop, 4096, 0, ldo, None, None, scratch, 0, None)
    import ctypes
    rng = lambda *a: (ctypes.c_int64 * len(a))(*a)
    bad = [dict(hd=64), dict(valid=65), dict(heads=0), dict(ldo=120), dict(ldo=132), dict(q=4100), dict(q=0), dict(batch=-1),
           dict(drop=rng(0, 64)), dict(drop=rng(5, 3)), dict(drop=rng(-1, 3)), dict(drop=rng(1, 65)), dict(l=1 << 24), dict(scratch=4100)]
    for kw in bad:
        assert call(**kw) == -1, kw
        with pytest.raises(MoldqError):
            _lib.check(call(**kw))
    assert call(batch=0) == 0 and call(valid=0) == 0
    assert 0 < PAD_MIN_SHARE < 1


@pytest.mark.skipif(HIPCC is None, reason="hipcc not available")
def test_kernel_leaves_m0_alone_and_does_not_spill(tmp_path):
    funcs = {k: v for k, v in _functions(_asm(tmp_path, "mq_attn.hip")).items() if "attention_kernel" in k}
    assert len(funcs) == 3
    for name, (lines, meta) in funcs.items():
        assert not _m0_outside_asm(lines), name
        assert meta.get("ScratchSize", 0) == 0, (name, meta)
