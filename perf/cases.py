"""The workloads this framework is timed on: quantized linears from the smallest
GEMV to the largest projection, the attention and weight passes around them, and
whole FLUX / Qwen-Image forwards.

Weights are GGUF blocks made here field by field (`_Blocks`), so that their values
are also known in float64 without any code of the package: `prepare` uploads the
blocks, `exact` multiplies the values.  Everything is made on the GPU from the seed.
Shapes are those of the repository's own configurations (FLUX.1-dev, Qwen-Image,
the T5-XXL encoder, decode linears) or generic.
"""
import functools
import math
import zlib

import torch

import mold_amd
from mold_amd import ACT_GELU_TANH, ACT_NONE, GgmlDType, Linear, QMatMul, QTensor
from mold_amd import flux as F
from mold_amd import lora as L
from mold_amd import qwen_image as Q

# block type -> (elements, bytes)
TYPES = {"Q4_0": (32, 18), "Q4_1": (32, 20), "Q5_0": (32, 22), "Q5_1": (32, 24), "Q8_0": (32, 34),
         "Q2_K": (256, 84), "Q3_K": (256, 110), "Q4_K": (256, 144), "Q5_K": (256, 176), "Q6_K": (256, 210)}
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "bf16": 2}


@functools.lru_cache(maxsize=None)
def _device():
    """The context a program keeps for the life of the process."""
    return mold_amd.Device(0)


def _gen(seed, name):
    return torch.Generator(device="cuda").manual_seed(zlib.crc32(f"{seed}/{name}".encode()))


def _randn(seed, name, *shape):
    return torch.randn(shape, device="cuda", generator=_gen(seed, name))


# ------------------------------------------------------------------ weights

class _Blocks:
    """A random GGUF weight [n, k] with entries near N(0, 0.02^2): its fields (f16 block
    scales, sub-block scales and quants), the packed blocks and the float64 values."""

    def __init__(self, seed, name, qtype, n, k):
        self.qtype, self.n, self.k = qtype, n, k
        g = _gen(seed, name)
        bs = TYPES[qtype][0]
        self.nb = n * k // bs
        self.kquant = bs == 256
        bits = {"Q4_0": 4, "Q4_1": 4, "Q5_0": 5, "Q5_1": 5, "Q8_0": 8, "Q2_K": 2, "Q3_K": 3, "Q4_K": 4, "Q5_K": 5,
                "Q6_K": 6}[qtype]
        top = 2 ** bits - 1
        self.zero = {"Q4_0": 8, "Q5_0": 16, "Q8_0": 128, "Q3_K": 4, "Q6_K": 32}.get(qtype, 0)   # the quant of weight 0
        mid, sd = self.zero or top / 2, 0.9 if bits == 2 else top / 5.2
        q = torch.randn((self.nb, bs), device="cuda", generator=g).mul_(sd).add_(mid).round_().clamp_(0, top)
        self.q = q.to(torch.uint8)
        jitter = torch.rand((self.nb, 1), device="cuda", generator=g) * 0.4 + 0.8

        def ints(lo, hi, sub):
            return torch.randint(lo, hi, (self.nb, sub), device="cuda", generator=g)
        self.sc = self.mn = None
        if qtype in ("Q4_K", "Q5_K"):
            self.sc = ints(24, 64, 8)
            self.mn = (self.sc + ints(-3, 4, 8)).clamp(0, 63)
            mean_sc = 43.5
        elif qtype == "Q2_K":
            self.sc = ints(7, 16, 16)
            self.mn = (self.sc + ints(-1, 2, 16)).clamp(0, 15)
            mean_sc = 11.0
        elif qtype == "Q3_K":
            self.sc = ints(0, 2, 16) * 64 - 32 + ints(-8, 8, 16)      # signs both ways, |scale| 24 .. 40
            self.sc = self.sc.clamp(-32, 31)
            mean_sc = 29.0
        elif qtype == "Q6_K":
            self.sc = (ints(0, 2, 16) * 2 - 1) * ints(60, 128, 16)
            mean_sc = 94.0
        else:
            mean_sc = 1.0
        self.d = (0.02 / (sd * mean_sc) * jitter).half()
        if qtype in ("Q4_K", "Q5_K", "Q2_K"):
            self.m = (self.d.float() * mid).half()                 # dmin: the mean of d * sc * q is taken out
        elif qtype in ("Q4_1", "Q5_1"):
            self.m = (-self.d.float() * mid * jitter).half()
        else:
            self.m = None

    def values(self):
        """The weight in float64, [n, k]."""
        q, d = self.q.double(), self.d.double()
        if not self.kquant:
            w = (q - self.zero) * d
            if self.m is not None:
                w += self.m.double()
            return w.reshape(self.n, self.k)
        sub = self.sc.shape[1]
        w = (q - self.zero).reshape(self.nb, sub, 256 // sub) * (d * self.sc.double())[..., None]
        if self.m is not None:
            w -= (self.m.double() * self.mn.double())[..., None]
        return w.reshape(self.n, self.k)

    def packed(self):
        """The GGUF blocks, uint8 [nb, bytes per block]."""
        q, t, nb = self.q, self.qtype, self.nb
        u8 = torch.uint8

        def halves(*hs):
            return [torch.cat(hs, dim=1).contiguous().view(u8)]

        def nibbles(v, width):      # groups of 2 * width: low half in the low nibbles, high half in the high ones
            v = v.reshape(nb, -1, 2, width)
            return (v[:, :, 0] | (v[:, :, 1] << 4)).reshape(nb, -1)
        if t == "Q8_0":
            return torch.cat(halves(self.d) + [q ^ 0x80], dim=1)
        if t in ("Q4_0", "Q4_1"):
            return torch.cat(halves(*([self.d] if self.m is None else [self.d, self.m])) + [nibbles(q, 16)], dim=1)
        if t in ("Q5_0", "Q5_1"):
            w = torch.arange(8, device="cuda", dtype=torch.int32)
            qh = ((q >> 4).reshape(nb, 4, 8).int() << w).sum(-1).to(u8)
            return torch.cat(halves(*([self.d] if self.m is None else [self.d, self.m])) + [qh, nibbles(q & 15, 16)], dim=1)
        if t in ("Q4_K", "Q5_K"):
            s, m = self.sc.to(u8), self.mn.to(u8)
            sb = torch.cat([s[:, :4] | (s[:, 4:] >> 4 << 6), m[:, :4] | (m[:, 4:] >> 4 << 6),
                            (s[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)], dim=1)
            out = halves(self.d, self.m) + [sb]
            if t == "Q5_K":
                w = torch.arange(8, device="cuda", dtype=torch.int32)[:, None]
                out.append(((q >> 4).reshape(nb, 8, 32).int() << w).sum(1).to(u8))
            return torch.cat(out + [nibbles(q & 15, 32)], dim=1)
        # the 2-bit planes: byte 32 H + l holds elements 128 H + 32 p + l at bits 2 p
        w = 2 * torch.arange(4, device="cuda", dtype=torch.int32)[:, None]

        def planes2(v):
            return (v.reshape(nb, 2, 4, 32).int() << w).sum(2).to(u8).reshape(nb, 64)
        if t == "Q2_K":
            return torch.cat([(self.sc | (self.mn << 4)).to(u8), planes2(q)] + halves(self.d, self.m), dim=1)
        if t == "Q3_K":
            w8 = torch.arange(8, device="cuda", dtype=torch.int32)[:, None]
            hm = ((q >> 2).reshape(nb, 8, 32).int() << w8).sum(1).to(u8)
            s = (self.sc + 32).to(u8)
            lo = (s[:, :8] & 15) | ((s[:, 8:] & 15) << 4)
            hi = (s >> 4).reshape(nb, 4, 4)
            hi = hi[:, 0] | (hi[:, 1] << 2) | (hi[:, 2] << 4) | (hi[:, 3] << 6)
            return torch.cat([hm, planes2(q & 3), lo, hi] + halves(self.d), dim=1)
        # Q6_K: ql[64 H + 32 (p & 1) + l] nibble p / 2, qh[32 H + l] bits 2 p
        lo = (q & 15).reshape(nb, 2, 2, 64)
        return torch.cat([(lo[:, :, 0] | (lo[:, :, 1] << 4)).reshape(nb, 128), planes2(q >> 4),
                          self.sc.to(torch.int8).view(u8)] + halves(self.d), dim=1)

    def upload(self):
        return QTensor.from_device_blocks(_device(), GgmlDType[self.qtype], (self.n, self.k), self.packed().contiguous())


def _wbytes(qtype, n, k):
    bs, ts = TYPES[qtype]
    return n * k // bs * ts


def _bias(seed, name, n):
    return _randn(seed, name + ".bias", n) * 0.02


def _gelu64(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


# ------------------------------------------------------------------ linears

def _x(case, seed, name, m, k):
    return _randn(seed, name, m, k).to(DTYPES[case["x"]])


def _prepare_linear(case, seed):
    n, k = case["n"], case["k"]
    lin = Linear(_Blocks(seed, "w", case["type"], n, k).upload(), _bias(seed, "w", n))
    return dict(case=case, lin=lin, x=_x(case, seed, "x", case["m"], k))


def _run_linear(s):
    c = s["case"]
    return s["lin"].forward(s["x"], act=ACT_GELU_TANH if c["gelu_from"] >= 0 else ACT_NONE, out_dtype=DTYPES[c["y"]],
                            act_from=max(0, c["gelu_from"]))


def _exact_linear(case, seed):
    w = _Blocks(seed, "w", case["type"], case["n"], case["k"]).values()
    y = _x(case, seed, "x", case["m"], case["k"]).double() @ w.t() + _bias(seed, "w", case["n"]).double()
    if case["gelu_from"] >= 0:
        y[:, case["gelu_from"]:] = _gelu64(y[:, case["gelu_from"]:])
    return y


def _work_linear(case):
    m, n, k = case["m"], case["n"], case["k"]
    return {"bytes": _wbytes(case["type"], n, k) + m * k * SIZE[case["x"]] + m * n * SIZE[case["y"]] + 4 * n,
            "flops": 2 * m * n * k}


def _prepare_mlp(case, seed):
    h, f = case["hidden"], case["mlp"]
    fc1 = Linear(_Blocks(seed, "fc1", case["type"], f, h).upload(), _bias(seed, "fc1", f))
    fc2 = Linear(_Blocks(seed, "fc2", case["type"], h, f).upload(), _bias(seed, "fc2", h))
    return dict(fc1=fc1, fc2=fc2, x=_x(case, seed, "x", case["m"], h))


def _run_mlp(s):
    h = s["fc1"].forward(s["x"], act=ACT_GELU_TANH, out_dtype=torch.bfloat16)
    return s["fc2"].forward(h, out_dtype=torch.float32)


def _exact_mlp(case, seed):
    h, f = case["hidden"], case["mlp"]
    x = _x(case, seed, "x", case["m"], h).double()
    y = _gelu64(x @ _Blocks(seed, "fc1", case["type"], f, h).values().t() + _bias(seed, "fc1", f).double())
    return y @ _Blocks(seed, "fc2", case["type"], h, f).values().t() + _bias(seed, "fc2", h).double()


def _work_mlp(case):
    m, h, f = case["m"], case["hidden"], case["mlp"]
    return {"bytes": 2 * _wbytes(case["type"], h, f) + m * h * (SIZE[case["x"]] + 4) + 4 * (h + f), "flops": 4 * m * h * f}


# ------------------------------------------------------------------ attention

def _qkv(case, seed):
    """Joint q, k, v buffers as the blocks make them: RmsNormed q and k rows, zero rows past `valid`."""
    h, valid = case["heads"], case["valid"]
    q, k, v = (_randn(seed, nm, h, F.padded_len(valid), 128) for nm in "qkv")
    q, k = (t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + 1e-6) for t in (q, k))
    q = q * case["sharp"]
    for t in (k, v):
        t[:, valid:] = 0
    return [t.to(torch.bfloat16) for t in (q, k, v)]


def _prepare_attention(case, seed):
    return dict(qkv=_qkv(case, seed), valid=case["valid"], guard=torch.zeros((), device="cuda"))


def _run_attention(s):
    return F.attention_bf16(*s["qkv"], valid=s["valid"], guard=s["guard"])


def _attention64(q, k, v):
    """[H, L, 128] -> [L, H * 128] in float64, in chunks of rows."""
    h, l, d = q.shape
    out = torch.empty((l, h, d), dtype=torch.float64, device=q.device)
    for i in range(h):
        kt, vi = k[i].double().t().contiguous(), v[i].double()
        for r in range(0, l, 4096):
            out[r:r + 4096, i] = torch.softmax(q[i, r:r + 4096].double() @ kt / math.sqrt(d), dim=-1) @ vi
    return out.reshape(l, h * d)


def _exact_attention(case, seed):
    return _attention64(*(t[:, :case["valid"]] for t in _qkv(case, seed)))


def _work_attention(case):
    h, l = case["heads"], case["valid"]
    return {"bytes": 4 * h * l * 128 * 2, "flops": 4 * h * l * l * 128}


# ------------------------------------------------------------------ weight passes

def _prepare_dequantize(case, seed):
    return dict(qt=_Blocks(seed, "w", case["type"], case["n"], case["k"]).upload(), dtype=DTYPES[case["y"]])


def _run_dequantize(s):
    return s["qt"].dequantize(s["dtype"])


def _exact_dequantize(case, seed):
    return _Blocks(seed, "w", case["type"], case["n"], case["k"]).values()


def _work_dequantize(case):
    n, k = case["n"], case["k"]
    return {"bytes": _wbytes(case["type"], n, k) + n * k * SIZE[case["y"]], "flops": 2 * n * k}


def _lora_slices(case):
    """(rows, component) of the patches: q, k, v and the rest for a fused linear1, else one for the whole tensor."""
    n, k = case["n"], case["k"]
    return [(k, 0), (k, 1), (k, 2), (n - 3 * k, 3)] if n > 4 * k else [(n, None)]


def _prepare_lora(case, seed):
    patches = []
    for rows, comp in _lora_slices(case):
        target = L.LoraTarget("w") if comp is None else L.LoraTarget("w", comp, 0)
        patches.append(L.LoraPatch(_randn(seed, f"a{comp}", case["rank"], case["k"]) * 0.05,
                                   _randn(seed, f"b{comp}", rows, case["rank"]) * 0.02, 0.8, target))
    return dict(qt=_Blocks(seed, "w", case["type"], case["n"], case["k"]).upload(), patches=patches)


def _run_lora(s):
    qt, _ = L.patch_qtensor(s["qt"], s["patches"])
    return qt.dequantize()          # the merged weight's values: its blocks stay on the device


def _work_lora(case):
    n, k, r = case["n"], case["k"], case["rank"]
    return {"bytes": 2 * _wbytes(case["type"], n, k) + 4 * n * k + 4 * r * (n + k * len(_lora_slices(case))),
            "flops": 2 * n * k * r}


# ------------------------------------------------------------------ whole forwards

def _rms64(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()


def _ln64(x):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), eps=1e-6)


def _rope64(x, ang):
    """[H, L, 128] rotated in (even, odd) pairs by ang [L, 64]."""
    c, s = torch.cos(ang), torch.sin(ang)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((c * a - s * b, s * a + c * b), dim=-1).reshape(x.shape)


def _freqs(n, theta=10000.0):
    return theta ** (-torch.arange(0, n, 2, dtype=torch.float64, device="cuda") / n)


def _heads64(y, heads, qw, kw, ang):
    y = y.reshape(y.shape[0], 3, heads, 128).permute(1, 2, 0, 3)
    return _rope64(_rms64(y[0], qw), ang), _rope64(_rms64(y[1], kw), ang), y[2]


class _Params64:
    """A model's linears and norms in float64, made from the same seed as `_params`."""

    def __init__(self, seed, shapes, types, dense):
        self.seed, self.shapes, self.types, self.dense = seed, shapes, types, _dense(seed, dense)

    def __call__(self, name, x):
        n, k = self.shapes[name][:2]
        return x.double() @ _Blocks(self.seed, name, self.types[name], n, k).values().t() + _bias(self.seed, name, n).double()


def _dense(seed, shapes):
    out = {}
    for name, shape in shapes.items():
        t = _randn(seed, name, *shape) * 0.02
        if name != "img_in.bias":
            t = (t if name == "img_in.weight" else t + 1).to(torch.bfloat16)
        out[name] = t
    return out


def _params(cls, cfg, seed, shapes, types, dense):
    lin = {nm: Linear(_Blocks(seed, nm, types[nm], s[0], s[1]).upload(), _bias(seed, nm, s[0])) for nm, s in shapes.items()}
    return cls(cfg, lin, _dense(seed, dense))


def _flux_cfg(case):
    cfg = F.FluxConfig(depth=case["double"], depth_single_blocks=case["single"])
    shapes = F.linear_shapes(cfg)
    return cfg, shapes, dict.fromkeys(shapes, case["type"])


def _prepare_flux(case, seed):
    cfg, shapes, types = _flux_cfg(case)
    step = F.FluxStep(_params(F.FluxParams, cfg, seed, shapes, types, F.dense_shapes(cfg)))
    return dict(step=step, inputs=F.make_inputs(cfg, case["height"], case["width"], case["txt"], seed=seed))


def _run_step(s):
    return s["step"].forward(**s["inputs"])


def _exact_flux(case, seed):
    cfg, shapes, types = _flux_cfg(case)
    p = _Params64(seed, shapes, types, F.dense_shapes(cfg))
    i = F.make_inputs(cfg, case["height"], case["width"], case["txt"], seed=seed)
    silu, D = torch.nn.functional.silu, p.dense

    def embed(prefix, x):
        return p(prefix + ".out_layer", silu(p(prefix + ".in_layer", x)))

    def time(t):
        a = t.double()[:, None] * 1000 * torch.exp(-math.log(10000.0) * torch.arange(128, device="cuda").double() / 128)
        return torch.cat([a.cos(), a.sin()], -1)
    ids = torch.cat([i["txt_ids"], i["img_ids"]]).double()
    ang = torch.cat([ids[:, a:a + 1] * _freqs(d) for a, d in enumerate(cfg.axes_dim)], -1)
    vec = embed("time_in", time(i["t"])) + embed("guidance_in", time(i["guidance"])) + embed("vector_in", i["y"])
    img = i["img"].double() @ D["img_in.weight"].double().t() + D["img_in.bias"].double()
    txt = p("txt_in", i["txt"])
    lt, h, sv = txt.shape[0], cfg.hidden_size, silu(vec)
    for b in range(cfg.depth):
        n = f"double_blocks.{b}."
        mods = {st: p(n + st + "_mod.lin", sv).chunk(6, -1) for st in ("txt", "img")}
        xs, parts = {"txt": txt, "img": img}, {}
        for st in ("txt", "img"):
            m = mods[st]
            y = p(n + st + "_attn.qkv", _ln64(xs[st]) * (1 + m[1]) + m[0])
            parts[st] = _heads64(y, cfg.num_heads, D[n + st + "_attn.norm.query_norm.scale"],
                                 D[n + st + "_attn.norm.key_norm.scale"], ang[:lt] if st == "txt" else ang[lt:])
        a = _attention64(*(torch.cat(z, 1) for z in zip(parts["txt"], parts["img"])))
        for st, at in (("txt", a[:lt]), ("img", a[lt:])):
            m = mods[st]
            x = xs[st] + m[2] * p(n + st + "_attn.proj", at)
            xs[st] = x + m[5] * p(n + st + "_mlp.2", _gelu64(p(n + st + "_mlp.0", _ln64(x) * (1 + m[4]) + m[3])))
        txt, img = xs["txt"], xs["img"]
    x = torch.cat([txt, img])
    for b in range(cfg.depth_single_blocks):
        n = f"single_blocks.{b}."
        m = p(n + "modulation.lin", sv).chunk(3, -1)
        y = p(n + "linear1", _ln64(x) * (1 + m[1]) + m[0])
        a = _attention64(*_heads64(y[:, :3 * h], cfg.num_heads, D[n + "norm.query_norm.scale"],
                                   D[n + "norm.key_norm.scale"], ang))
        x = x + m[2] * p(n + "linear2", torch.cat([a, _gelu64(y[:, 3 * h:])], -1))
    m = p("final_layer.adaLN_modulation.1", sv).chunk(2, -1)
    return p("final_layer.linear", _ln64(x[lt:]) * (1 + m[1]) + m[0])


def _flux_len(case):
    return (case["height"] // 16) * (case["width"] // 16), case["txt"]


def _work_flux(case):
    cfg, shapes, types = _flux_cfg(case)
    li, lt = _flux_len(case)
    lin, attn = F.step_flop(cfg, li, lt)
    return {"bytes": sum(_wbytes(types[nm], s[0], s[1]) for nm, s in shapes.items()) + li * 64 * 8 + lt * 4096 * 4,
            "flops": lin + attn}


def _qwen_cfg(case):
    cfg = Q.QwenConfig(num_layers=case["layers"])
    shapes = Q.linear_shapes(cfg)
    return cfg, shapes, {nm: cfg.qtype(s[2]).name for nm, s in shapes.items()}


def _qwen_inputs(case, cfg, seed):
    i = Q.make_inputs(cfg, case["height"], case["width"], case["txt"], seed=seed)
    if not case["cfg_valid"]:
        return i
    # guidance: the prompt and a shorter, padded and masked, negative prompt on the same latents
    other = _randn(seed, "uncond", case["txt"], cfg.joint_attention_dim)
    return dict(img=torch.stack([i["img"]] * 2), txt=torch.stack([i["txt"], other]), t=i["t"].repeat(2), grid=i["grid"],
                txt_valid=[case["txt"], case["cfg_valid"]])


def _prepare_qwen(case, seed):
    cfg, shapes, types = _qwen_cfg(case)
    step = Q.QwenImageStep(_params(Q.QwenParams, cfg, seed, shapes, types, Q.dense_shapes(cfg)))
    return dict(step=step, inputs=_qwen_inputs(case, cfg, seed), batched=bool(case["cfg_valid"]))


def _run_qwen(s):
    return s["step"].forward_batched(**s["inputs"]) if s["batched"] else s["step"].forward(**s["inputs"])


def _exact_qwen(case, seed):
    cfg, shapes, types = _qwen_cfg(case)
    p = _Params64(seed, shapes, types, Q.dense_shapes(cfg))
    i = _qwen_inputs(case, cfg, seed)
    if not case["cfg_valid"]:
        return _qwen64(cfg, p, i["img"], i["txt"], i["t"], i["grid"], case["txt"])
    return torch.stack([_qwen64(cfg, p, i["img"][b], i["txt"][b], i["t"][b:b + 1], i["grid"], i["txt_valid"][b])
                        for b in range(2)])


def _qwen64(cfg, p, img, txt, t, grid, valid):
    silu, D, (gh, gw) = torch.nn.functional.silu, p.dense, grid
    lt, (fd, hd, wd) = txt.shape[0], cfg.axes_dims_rope

    def pos(n):
        return torch.cat([torch.arange(-(n - n // 2), 0), torch.arange(0, n // 2)]).double().cuda()
    ang = torch.cat([torch.zeros((gh, gw, fd // 2), dtype=torch.float64, device="cuda"),
                     (pos(gh)[:, None] * _freqs(hd))[:, None].expand(gh, gw, hd // 2),
                     (pos(gw)[:, None] * _freqs(wd))[None].expand(gh, gw, wd // 2)], -1).reshape(gh * gw, 64)
    tp = max(gh // 2, gw // 2) + torch.arange(lt, device="cuda").double()[:, None]
    angs = {"txt": torch.cat([tp * _freqs(d) for d in (fd, hd, wd)], -1), "img": ang}
    a = t.double()[:, None] * torch.exp(-math.log(10000.0) * torch.arange(128, device="cuda").double() / 128)
    e = "time_text_embed.timestep_embedder.linear_"
    sv = silu(p(e + "2", silu(p(e + "1", torch.cat([a.cos(), a.sin()], -1)))))
    xs = {"img": img.double() @ D["img_in.weight"].double().t() + D["img_in.bias"].double(),
          "txt": p("txt_in", _rms64(txt.double(), D["txt_norm.weight"]))}
    names = {"img": ("attn.to_qkv", "attn.norm_", "attn.to_out.0"),
             "txt": ("attn.add_qkv_proj", "attn.norm_added_", "attn.to_add_out")}
    for b in range(cfg.num_layers):
        n = f"transformer_blocks.{b}."
        mods = {st: p(f"{n}{st}_mod.1", sv).chunk(6, -1) for st in xs}
        parts = {}
        for st, (qkv, norm, _) in names.items():
            y = p(n + qkv, _ln64(xs[st]) * (1 + mods[st][1]) + mods[st][0])
            parts[st] = _heads64(y, cfg.num_attention_heads, D[n + norm + "q.weight"], D[n + norm + "k.weight"], angs[st])
        q, k, v = (torch.cat(z, 1) for z in zip(parts["txt"], parts["img"]))
        keep = torch.cat([torch.arange(valid), torch.arange(lt, q.shape[1])]).cuda()   # masked text keys are left out
        att = _attention64(q, k[:, keep], v[:, keep])
        for st, (_, _, out) in names.items():
            m = mods[st]
            x = xs[st] + m[2] * p(n + out, att[:lt] if st == "txt" else att[lt:])
            xs[st] = x + m[5] * p(f"{n}{st}_mlp.net.2", _gelu64(p(f"{n}{st}_mlp.net.0.proj", _ln64(x) * (1 + m[4]) + m[3])))
    scale, shift = p("norm_out.linear", sv).chunk(2, -1)
    return p("proj_out", _ln64(xs["img"]) * (1 + scale) + shift)


def _work_qwen(case):
    cfg, shapes, types = _qwen_cfg(case)
    b = 2 if case["cfg_valid"] else 1
    li, lt = _flux_len(case)
    lin, attn = Q.step_flop(cfg, li, lt)
    return {"bytes": sum(_wbytes(types[nm], s[0], s[1]) for nm, s in shapes.items()) + b * (li * 64 * 8 + lt * 3584 * 4),
            "flops": b * (lin + attn)}


# ------------------------------------------------------------------ the interface

_KINDS = {"linear": (_prepare_linear, _run_linear, _exact_linear, _work_linear),
          "mlp": (_prepare_mlp, _run_mlp, _exact_mlp, _work_mlp),
          "attention": (_prepare_attention, _run_attention, _exact_attention, _work_attention),
          "dequantize": (_prepare_dequantize, _run_dequantize, _exact_dequantize, _work_dequantize),
          "lora": (_prepare_lora, _run_lora, None, _work_lora),
          "flux": (_prepare_flux, _run_step, _exact_flux, _work_flux),
          "qwen": (_prepare_qwen, _run_qwen, _exact_qwen, _work_qwen)}


def _linear(m, n, k, qtype, x, y, gelu_from=-1):
    """gelu_from: first output column that goes through GELU, -1 for none."""
    return dict(kind="linear", m=m, n=n, k=k, type=qtype, x=x, y=y, gelu_from=gelu_from)


def listed():
    return [
        # one adaLN modulation of a FLUX single block: batch 1, f32 in and out, latency-bound
        dict(_linear(1, 9216, 3072, "Q4_K", "f32", "f32"), name="modulation_gemv"),
        # a token of an LLM decode (up projection), the weight read once
        dict(_linear(1, 10240, 4096, "Q6_K", "f32", "f32"), name="decode_gemv"),
        # a few sequences decoded together
        dict(_linear(4, 4096, 4096, "Q8_0", "f32", "f32"), name="decode_batch4"),
        # a short prompt through a T5-XXL encoder linear: 77 rows, f32 activations
        dict(_linear(77, 4096, 4096, "Q8_0", "f32", "f32"), name="prompt77_linear"),
        # FLUX's text stream (512 tokens), MLP up projection with GELU, bf16 between the linears
        dict(_linear(512, 12288, 3072, "Q4_K", "bf16", "bf16", 0), name="text_mlp_up"),
        # FLUX single block linear1 at 1024 x 1024: [q | k | v | gelu(mlp)], the largest projection
        dict(_linear(4608, 21504, 3072, "Q4_K", "bf16", "bf16", 9216), name="linear1_1024px"),
        # Qwen-Image's image MLP at 1328 x 1328 (a ragged row count) in its 2-bit type
        dict(kind="mlp", m=6889, hidden=3072, mlp=12288, type="Q2_K", x="bf16", name="qwen_mlp"),
        # the joint attention of that model: 256 text and 6889 image tokens, padded buffers
        dict(kind="attention", heads=24, valid=7145, sharp=1.0, name="joint_attention"),
        # a weight to dense bf16 (a caller with its own dense matmul)
        dict(kind="dequantize", n=18432, k=3072, type="Q4_K", y="bf16", name="dequantize"),
        # an adapter merged into a FLUX linear1: dequantize, four patches, quantize again
        dict(kind="lora", n=21504, k=3072, type="Q4_K", rank=32, name="lora_merge"),
        # FLUX.1-dev forward, 1024 x 1024, two double and four single blocks of its 19 and 38
        dict(kind="flux", double=2, single=4, height=1024, width=1024, txt=512, type="Q4_K", name="flux_forward"),
        # Qwen-Image guidance forward (prompt and padded negative prompt in one batch), two of its 60 blocks
        dict(kind="qwen", layers=2, height=1328, width=1328, txt=256, cfg_valid=77, name="qwen_cfg_forward"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "linear", "linear", "linear", "mlp", "attention", "attention", "dequantize", "lora",
                       "flux", "qwen"])
    qtype = rng.choice(sorted(TYPES))
    f = lambda: rng.choice(["f32", "bf16"])
    if kind == "gemv":        # batch 1 .. 8 (modulations, decode)
        k = 256 * _log(rng, 4, 48) if rng.random() < 0.9 else 128 * (2 * rng.randrange(4, 40) + 1)
        if k % 256:
            qtype = rng.choice(["Q4_0", "Q4_1", "Q5_0", "Q5_1", "Q8_0"])
        return _linear(rng.randint(1, 8), _log(rng, 256, 20000), k, qtype, f(), f())
    if kind == "linear":      # prompts, text streams and images
        k, n, m = 256 * _log(rng, 3, 60), _log(rng, 512, 21504), _log(rng, 9, 7000)
        return _linear(m, n, k, qtype, f(), f(), rng.choice([-1, -1, 0, n // 3]))
    if kind == "mlp":
        h = 256 * rng.randint(4, 16)
        return dict(kind="mlp", m=_log(rng, 16, 7000), hidden=h, mlp=4 * h if h <= 3072 else 10240, type=qtype, x=f())
    if kind == "attention":   # joint lengths of 256 .. 1536 pixel images with their prompts
        return dict(kind="attention", heads=rng.choice([2, 8, 16, 24, 24, 32]), valid=_log(rng, 300, 9000),
                    sharp=round(rng.uniform(0.7, 3.0), 2))
    if kind == "dequantize":
        return dict(kind=kind, n=_log(rng, 256, 21504), k=256 * _log(rng, 1, 60), type=qtype, y=f())
    if kind == "lora":
        k = 256 * rng.randint(2, 12)
        n = rng.choice([k, 3 * k, 4 * k, 7 * k])
        return dict(kind=kind, n=n, k=k, type=qtype, rank=rng.choice([4, 8, 16, 32, 64, rng.randint(3, 96)]))
    side = lambda: 16 * rng.randint(16, 64)
    if kind == "flux":
        return dict(kind=kind, double=rng.randint(1, 2), single=rng.randint(1, 3), height=side(), width=side(),
                    txt=rng.choice([77, 256, 512]), type=rng.choice(["Q4_K", "Q4_1", "Q8_0", "Q6_K", "Q5_K"]))
    txt = rng.randint(24, 256)
    return dict(kind=kind, layers=1, height=side(), width=side(), txt=txt,
                cfg_valid=rng.choice([0, rng.randint(1, txt)]))


def prepare(case, seed):
    return dict(_KINDS[case["kind"]][0](case, seed), kind=case["kind"])


def run(state):
    return _KINDS[state["kind"]][1](state)


def exact(case, seed):
    fn = _KINDS[case["kind"]][2]
    return None if fn is None else fn(case, seed)


def work(case):
    return _KINDS[case["kind"]][3](case)


def tolerance(case):
    kind = case["kind"]
    if kind in ("dequantize", "lora"):
        return "exact"                        # the GGUF formulas and quantizers fix every bit
    if kind == "linear" and case["m"] <= 8:
        # exact weights and f32 sums; a Q4_K weight takes x rounded to 8 bits (Q8_K: 7e-3 from float64)
        rel = 2e-2 if case["type"] == "Q4_K" else 1e-5
        return {"rel": rel if case["y"] == "f32" else max(rel, 1e-2)}
    # bf16 operands, f32 sums: 1.7e-3 .. 3e-3 from float64 for one layer; whole forwards that
    # round elsewhere differ from each other by 5e-3 (FLUX) and 2e-3 (Qwen-Image)
    return {"rel": 2e-2 if kind == "flux" else 1e-2}
