"""Timed cases: the work that a user of this framework has it do, through its public entry points.

Every case is one stage of image restoration as a model on the `hip` backend runs it: calls of the
operator dispatch (`Ops`), of the NAFNet harness or of the metrics object. The kinds are

  chain       two pointwise GEMMs (gate, then scale + residual), as two calls or one
  nafblock    one NAFNet block in the reference model's calls (LN / gate / map prologues, depthwise
              conv, TLC local mean, residual GEMMs)
  nafnet      a whole NAFNet forward, captured once per image size and replayed (the worker's way)
  restormer   one Restormer block: channel attention (MDTA) and the gated feed-forward (GDFN)
  fftformer   one FFTformer block: patch correlation (FSAS) and the frequency feed-forward (DFFN)
  patch       the standalone 8x8 patch frequency filter
  rrdb        one RRDBNet dense block on channel slices, then a nearest-x2 up conv
  scan        EVSSM's selective scan
  metrics     PSNR + SSIM of an 8-bit image pair

The path is forward only: the framework restores images, it has no training direction.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from clarus_amd import spatial_torch  # noqa: F401  (registers "torch" for the non-GEMM ops)
from clarus_amd.dispatch import Ops
from clarus_amd.metrics import make_metrics
from clarus_amd.nafnet import NAFNet

DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
LEAKY = 0.2


def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _ops(dtype):
    return Ops(["hip", "torch"], dtype, _device(), log=lambda *a: None)


# ------------------------------------------------------------------------------- the cases
def listed():
    return [
        # a thumbnail or tile through the fp32 pointwise chain: launches and latency
        {"name": "chain_f32_64x64_c32", "kind": "chain", "dtype": "fp32", "n": 1, "h": 64, "w": 64, "c": 32,
         "one_call": False},
        # the block that 28 of the 36 blocks of NAFNet-w64 are, at its 720p size (fp32 residual stream)
        {"name": "nafblock_c512_90x160", "kind": "nafblock", "n": 1, "h": 90, "w": 160, "c": 512, "window": 48},
        # a block at an early level on a batch of two odd-sized images
        {"name": "nafblock_c128_2x173x251", "kind": "nafblock", "n": 2, "h": 173, "w": 251, "c": 128, "window": 192},
        # deblurring one 720p frame with NAFNet-GoPro-w64: the headline call
        {"name": "nafnet_w64_720x1280", "kind": "nafnet", "width": 64, "n": 1, "h": 720, "w": 1280, "fused": True},
        # a small photo of odd size through the width-32 network in the reference block's calls
        {"name": "nafnet_w32_251x333", "kind": "nafnet", "width": 32, "n": 1, "h": 251, "w": 333, "fused": False},
        # Restormer's first level on a 720p frame
        {"name": "restormer_bf16_l0_720x1280", "kind": "restormer", "dtype": "bf16", "n": 1, "h": 720, "w": 1280,
         "level": 0},
        # its deepest level in fp32
        {"name": "restormer_f32_l3_90x160", "kind": "restormer", "dtype": "fp32", "n": 1, "h": 90, "w": 160,
         "level": 3},
        # FFTformer's first level on a 720p frame
        {"name": "fftformer_bf16_l0_720x1280", "kind": "fftformer", "dtype": "bf16", "n": 1, "h": 720, "w": 1280,
         "level": 0},
        # the fp32 frequency filter by itself, at the second level
        {"name": "patch_f32_c96_360x640", "kind": "patch", "dtype": "fp32", "n": 1, "h": 360, "w": 640, "c": 96},
        # a Real-ESRGAN dense block and up conv on a 256 x 384 image
        {"name": "rrdb_bf16_256x384", "kind": "rrdb", "n": 1, "h": 256, "w": 384},
        # EVSSM level 0: eight 384 x 384 crops of a 720p frame
        {"name": "scan_8x384x384_d96", "kind": "scan", "dtype": "bf16", "n": 8, "h": 384, "w": 384, "d": 96, "r": 3},
        # scoring a restored 720p frame
        {"name": "metrics_720x1280", "kind": "metrics", "h": 720, "w": 1280},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _image(rng, pixels, lo=24):
    """(h, w) of log-uniform area up to `pixels`, aspect 0.4 to 2.5, any parity."""
    area = math.exp(rng.uniform(math.log(lo * lo * 2), math.log(pixels)))
    aspect = math.exp(rng.uniform(math.log(0.4), math.log(2.5)))
    h = max(lo, int(math.sqrt(area * aspect)))
    return h, max(lo, int(min(area, pixels) / h))


def draw(rng):
    kind = rng.choice(["chain", "nafblock", "nafblock", "nafnet", "restormer", "restormer", "fftformer", "patch",
                       "rrdb", "scan", "metrics"])
    if kind == "chain":
        c = rng.choice([32, 64, 128])
        h, w = _image(rng, 921600 * 32 // c)
        return {"kind": kind, "dtype": rng.choice(["fp32", "bf16"]), "n": 1, "h": h, "w": w, "c": c,
                "one_call": rng.random() < 0.5}
    if kind == "nafblock":
        level = rng.randrange(5)
        c = rng.choice([32, 64]) << level
        n = rng.choice([1, 1, 2, 4])
        h, w = _image(rng, 921600 // n >> (2 * level), 16)
        return {"kind": kind, "n": n, "h": h, "w": w, "c": c, "window": 384 >> level}
    if kind == "nafnet":
        h, w = _image(rng, 500000, 48)
        return {"kind": kind, "width": rng.choice([32, 64]), "n": 1, "h": h, "w": w, "fused": rng.random() < 0.5}
    if kind in ("restormer", "fftformer"):
        level = rng.randrange(4 if kind == "restormer" else 3)
        n = rng.choice([1, 1, 2])
        dtype = rng.choice(["bf16", "fp32"])
        h, w = _image(rng, (921600 if dtype == "bf16" else 460800) // n >> (2 * level))
        if kind == "fftformer":  # the model pads its input, so every level sees whole patches
            h, w = -(-h // 8) * 8, -(-w // 8) * 8
        return {"kind": kind, "dtype": dtype, "n": n, "h": h, "w": w, "level": level}
    if kind == "patch":
        level = rng.randrange(3)
        h, w = _image(rng, 921600 >> (2 * level))
        return {"kind": kind, "dtype": rng.choice(["fp32", "bf16"]), "n": 1, "h": h, "w": w, "c": 48 << level}
    if kind == "rrdb":
        h, w = _image(rng, 98304)
        return {"kind": kind, "n": rng.choice([1, 1, 2]), "h": h, "w": w}
    if kind == "scan":
        level = rng.randrange(3)
        side = _log_int(rng, 24, 384 >> level)
        return {"kind": kind, "dtype": rng.choice(["bf16", "fp32"]), "n": rng.choice([1, 2, 8]), "h": side,
                "w": side + rng.randrange(-3, 1), "d": 96 << level, "r": 3 << level}
    h, w = _image(rng, 921600)
    return {"kind": kind, "h": h, "w": w}


# ------------------------------------------------------------------------------- inputs
class _Rand:
    """Seeded tensors on the device."""

    def __init__(self, seed):
        self.dev = _device()
        self.g = torch.Generator(device=self.dev).manual_seed(seed)

    def normal(self, *shape, scale=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.g, device=self.dev) * scale).to(dtype)

    def uniform(self, *shape, lo=0.0, hi=1.0, dtype=torch.float32):
        return (torch.rand(*shape, generator=self.g, device=self.dev) * (hi - lo) + lo).to(dtype)

    def weight(self, k, n, dtype):
        """[K, N] pointwise weight, nn.Conv2d's default bound 1 / sqrt(K)."""
        b = 1.0 / math.sqrt(k)
        return self.uniform(k, n, lo=-b, hi=b, dtype=dtype)

    def bias(self, n):
        return self.uniform(n, lo=-0.1, hi=0.1)

    def taps(self, c):
        return self.uniform(c, 1, 3, 3, lo=-1 / 3, hi=1 / 3)


def _residual_dtype(c):
    """NAFNet's residual stream is fp32 from level 3 on (width 64: c >= 512)."""
    return torch.float32 if c >= 512 else torch.bfloat16


def _inputs(case, seed):
    """The case's tensors by name: activations and weights as the model holds them."""
    r = _Rand(seed)
    kind = case["kind"]
    dt = DTYPES[case.get("dtype", "bf16")]
    if kind == "metrics":
        h, w = case["h"], case["w"]
        gt = r.uniform(h, w, 3, lo=0, hi=256).to(torch.uint8)
        pred = (gt.float() * 0.9 + 12 + 6 * r.normal(h, w, 3)).round().clamp(0, 255).to(torch.uint8)
        return dict(pred=pred, gt=gt)
    n, h, w = case["n"], case["h"], case["w"]
    if kind == "chain":
        c = case["c"]
        return dict(x=r.normal(n, h, w, c, dtype=dt), w1=r.weight(c, 2 * c, dt), b1=r.bias(2 * c),
                    w2=r.weight(c, c, dt), b2=r.bias(c), beta=r.normal(c, scale=0.1))
    if kind == "nafblock":
        c = case["c"]
        return dict(x=r.normal(n, h, w, c, dtype=_residual_dtype(c)),
                    w1=r.weight(c, 2 * c, dt), b1=r.bias(2 * c), dw=r.taps(2 * c), dwb=r.bias(2 * c),
                    ws=r.weight(c, c, dt), bs=r.bias(c), w3=r.weight(c, c, dt), b3=r.bias(c),
                    beta=r.normal(c, scale=0.2), w4=r.weight(c, 2 * c, dt), b4=r.bias(2 * c),
                    w5=r.weight(c, c, dt), b5=r.bias(c), gamma=r.normal(c, scale=0.2))
    if kind == "nafnet":
        return dict(img=r.uniform(n, 3, h, w), sd=_nafnet_weights(r, case["width"]))
    if kind == "restormer":
        c, hd = 48 << case["level"], _restormer_hidden(case["level"])
        heads = 1 << case["level"]
        return dict(x=r.normal(n, h, w, c, dtype=dt), wq=r.weight(c, 3 * c, dt), bq=r.bias(3 * c),
                    dq=r.taps(3 * c), temp=r.uniform(heads, 1, 1, lo=0.5, hi=2.0), wp=r.weight(c, c, dt),
                    wi=r.weight(c, 2 * hd, dt), bi=r.bias(2 * hd), di=r.taps(2 * hd), wo=r.weight(hd, c, dt))
    if kind == "fftformer":
        c = 48 << case["level"]
        return dict(x=r.normal(n, h, w, c, dtype=dt), wh=r.weight(c, 6 * c, dt), bh=r.bias(6 * c), dh=r.taps(6 * c),
                    lnw=1 + r.normal(2 * c, scale=0.1), lnb=r.normal(2 * c, scale=0.1), wp=r.weight(2 * c, c, dt),
                    wi=r.weight(c, 6 * c, dt), bi=r.bias(6 * c), f=1 + r.normal(6 * c, 8, 5, scale=0.3),
                    di=r.taps(6 * c), wo=r.weight(3 * c, c, dt))
    if kind == "patch":
        c = case["c"]
        return dict(x=r.normal(n, h, w, c, dtype=dt), f=r.normal(c, 8, 5))
    if kind == "rrdb":
        def conv(cout, cin):
            return r.normal(cout, cin, 3, 3, scale=0.1 * math.sqrt(2.0 / (9 * cin)), dtype=dt)
        t = dict(x=r.normal(n, h, w, 64, dtype=dt))
        for i in range(4):
            t[f"w{i}"], t[f"b{i}"] = conv(32, 64 + 32 * i), r.bias(32)
        t["w4"], t["b4"] = conv(64, 192), r.bias(64)
        t["wu"], t["bu"] = conv(64, 64), r.bias(64)
        return t
    if kind == "scan":
        d, rk = case["d"], case["r"]
        return dict(u=r.normal(n, h, w, d, dtype=dt), dbl=r.normal(n, h, w, rk + 16), dtw=r.normal(d, rk, scale=0.5),
                    dtb=r.normal(d) - 2, A=-r.uniform(d, 8, lo=0.5, hi=4.5), D=r.normal(d))
    raise ValueError(kind)


def _restormer_hidden(level):
    """int(2.66 c) gated channels, padded to a multiple of 16 as the model pads its weights."""
    return -(-int((48 << level) * 2.66) // 16) * 16


ENC, MID, DEC = [1, 1, 1, 28], 1, [1, 1, 1, 1]
TLC = 256


def _nafnet_blocks(width):
    """(state-dict prefix, channels) of every block, in the order of the forward."""
    out, c = [], width
    for i, k in enumerate(ENC):
        out += [(f"encoders.{i}.{j}", c) for j in range(k)]
        c *= 2
    out += [(f"middle_blks.{j}", c) for j in range(MID)]
    for i, k in enumerate(DEC):
        c //= 2
        out += [(f"decoders.{i}.{j}", c) for j in range(k)]
    return out


def _nafnet_weights(r, width):
    """Random weights in the upstream state-dict layout (default conv bounds, random beta / gamma)."""
    sd = {}

    def conv(name, cout, cin, k, scale=1.0, fan=None):
        b = scale / math.sqrt(fan or cin * k * k)
        sd[f"{name}.weight"] = r.uniform(cout, cin, k, k, lo=-b, hi=b)
        sd[f"{name}.bias"] = r.uniform(cout, lo=-b, hi=b)
    conv("intro", width, 3, 3)
    conv("ending", 3, width, 3, scale=0.1)
    for p, c in _nafnet_blocks(width):
        conv(f"{p}.conv1", 2 * c, c, 1)
        conv(f"{p}.conv2", 2 * c, 1, 3)
        for name in ("conv3", "sca.1", "conv5"):
            conv(f"{p}.{name}", c, c, 1)
        conv(f"{p}.conv4", 2 * c, c, 1)
        for name in ("norm1", "norm2"):
            sd[f"{p}.{name}.weight"] = 1 + r.normal(c, scale=0.1)
            sd[f"{p}.{name}.bias"] = r.normal(c, scale=0.1)
        sd[f"{p}.beta"] = r.normal(1, c, 1, 1, scale=0.2)
        sd[f"{p}.gamma"] = r.normal(1, c, 1, 1, scale=0.2)
    c = width
    for i in range(len(ENC)):
        conv(f"downs.{i}", 2 * c, c, 2)
        c *= 2
    for i in range(len(DEC)):
        conv(f"ups.{i}.0", 2 * c, c, 1)
        c //= 2
    return sd


def prepare(case, seed):
    kind = case["kind"]
    t = _inputs(case, seed)
    st = {"case": dict(case)}
    if kind == "metrics":
        m = make_metrics(_device(), "hip")
        st.update(t, m=m, res=torch.zeros(2, dtype=torch.float64, device=_device()),
                  scratch=m.scratch(case["h"], case["w"]))
    elif kind == "nafnet":
        model = NAFNet(_ops(torch.bfloat16), width=case["width"], enc=ENC, mid=MID, dec=DEC, tlc=(TLC, TLC),
                       state_dict=t["sd"], fused_pairs=case["fused"])
        stream = torch.cuda.Stream(_device())
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            model.forward(t["img"])
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            y = model.forward(t["img"])
        st.update(model=model, img=t["img"], graph=graph, y=y)
    else:
        st.update(t, ops=_ops(DTYPES[case.get("dtype", "bf16")]))
    if kind == "rrdb":  # the dense block's feature buffer and its output, kept by the model
        n, h, w, _ = t["x"].shape
        st["buf"] = t["x"].new_empty(n, h, w, 192)
        st["buf"][..., :64] = t["x"]
        st["out"] = t["x"].new_empty(n, h, w, 64)
    return st


# ------------------------------------------------------------------------------- one pass
def run(state):
    return _RUN[state["case"]["kind"]](state)


def _run_chain(s):
    o = s["ops"]
    if s["case"]["one_call"]:
        return o.linear_gate_linear(s["x"], s["w1"], s["b1"], s["w2"], s["b2"], scale=s["beta"])
    u = o.linear(s["x"], s["w1"], s["b1"], gate=True)
    return o.linear(u, s["w2"], s["b2"], scale=s["beta"], residual=s["x"])


def _run_nafblock(s):
    o, x = s["ops"], s["x"]
    rdt = x.dtype
    k = s["case"]["window"]
    t = o.linear(x, s["w1"], s["b1"], ln=True)
    t = o.dwconv(t, s["dw"], s["dwb"], gate=True)
    sca = o.linear(o.boxmean(t, (k, k)), s["ws"], s["bs"])
    y = o.linear(t, s["w3"], s["b3"], scale=s["beta"], residual=x, mul=sca, out_dtype=rdt)
    u = o.linear(y, s["w4"], s["b4"], ln=True, gate=True)
    return o.linear(u, s["w5"], s["b5"], scale=s["gamma"], residual=y, out_dtype=rdt)


def _run_nafnet(s):
    s["graph"].replay()
    return s["y"]


def _run_restormer(s):
    o, x = s["ops"], s["x"]
    n, _, _, c = x.shape
    heads = 1 << s["case"]["level"]
    qkv = o.dwconv(o.linear(x, s["wq"], s["bq"], ln=True, ln_eps=1e-5), s["dq"], None)
    a = o.channel_attention(qkv, heads, s["temp"])
    # attn . V and the projection as one matrix per image
    mix = torch.matmul(a.transpose(-1, -2).contiguous(), s["wp"].float().view(1, heads, c // heads, c))
    y = o.linear_per_image(qkv[..., 2 * c:], mix.reshape(n, c, c).to(x.dtype), residual=x)
    u = o.dwconv(o.linear(y, s["wi"], s["bi"], ln=True, ln_eps=1e-5), s["di"], None, gate="gelu")
    return o.linear(u, s["wo"], residual=y)


def _run_fftformer(s):
    o, x = s["ops"], s["x"]
    c = x.shape[-1]
    hid = o.dwconv(o.linear(x, s["wh"], s["bh"], ln=True, ln_eps=1e-5), s["dh"], None)
    corr = o.patch_corr(hid, 2 * c)
    y = o.ln_mul_linear(corr, s["lnw"], s["lnb"], hid[..., 4 * c:], s["wp"], residual=x)
    u = o.linear_patch_filter(y, s["wi"], s["bi"], s["f"], ln=True, ln_eps=1e-5)
    return o.linear(o.dwconv(u, s["di"], None, gate="gelu"), s["wo"], residual=y)


def _run_patch(s):
    return s["ops"].patch_filter(s["x"], s["f"])


def _run_rrdb(s):
    o, buf = s["ops"], s["buf"]
    for i in range(4):
        cin = 64 + 32 * i
        o.conv3x3(buf[..., :cin], s[f"w{i}"], s[f"b{i}"], act="lrelu", out=buf[..., cin:cin + 32])
    y = o.conv3x3(buf, s["w4"], s["b4"], out_scale=0.2, residual=buf[..., :64], out=s["out"])
    return y, o.conv3x3(y, s["wu"], s["bu"], act="lrelu", up2=True)


def _run_scan(s):
    return s["ops"].selective_scan(s["u"], s["dbl"], s["dtw"], s["dtb"], s["A"], s["D"])


def _run_metrics(s):
    s["m"].compute(s["pred"], s["gt"], s["res"], s["scratch"])
    return s["res"]


_RUN = {"chain": _run_chain, "nafblock": _run_nafblock, "nafnet": _run_nafnet, "restormer": _run_restormer,
        "fftformer": _run_fftformer, "patch": _run_patch, "rrdb": _run_rrdb, "scan": _run_scan,
        "metrics": _run_metrics}


# ------------------------------------------------------------------------------- work
def _gemm(m, k, n, e_in, e_out, e_w, res=0, flops_n=None):
    """Bytes and flops of one pointwise GEMM call: rows in, rows out, weights, a residual of `res` bytes
    per element. flops_n: weight columns (2n with a gate)."""
    fn = flops_n or n
    return m * (k * e_in + n * e_out + n * res) + k * fn * e_w, 2.0 * m * k * fn


def _naf_work(m, c, mmap, fused):
    """One NAFNet block: its calls' inputs, outputs and weights. fused: pairs of calls handed over as
    one (their intermediate needs no memory)."""
    e = 4 if c >= 512 else 2
    parts = [_gemm(m, c, 2 * c, e, 2, 2), (m * 3 * c * 2, m * (2 * c * 18 + c)),
             (m * c * 2 + mmap * c * 2, m * c * 4.0), _gemm(mmap, c, c, 2, 2, 2),
             _gemm(m, c, c, 2, e, 2, res=e), _gemm(m, c, c, e, 2, 2, flops_n=2 * c), _gemm(m, c, c, 2, e, 2, res=e)]
    b, f = map(sum, zip(*parts))
    b += mmap * c * 2  # the map, read by the GEMM that multiplies by it
    if fused:
        b -= m * c * (2 * e if c != 512 else e)
    return b, f


def work(case):
    kind = case["kind"]
    if kind == "metrics":
        px = case["h"] * case["w"] * 3
        return {"bytes": 2.0 * px, "flops": px * (11 * 30 + 11 * 10 + 20 + 3.0)}
    n, h, w = case["n"], case["h"], case["w"]
    m = n * h * w
    e = 4 if case.get("dtype", "bf16") == "fp32" else 2
    if kind == "chain":
        c = case["c"]
        parts = [_gemm(m, c, c, e, e, e, flops_n=2 * c), _gemm(m, c, c, e, e, e, res=e)]
        if case["one_call"]:
            parts.append((-3.0 * m * c * e, 0))  # u stays inside, x is read once
    elif kind == "nafblock":
        k1, k2 = min(case["window"], h), min(case["window"], w)
        parts = [_naf_work(m, case["c"], n * (h - k1 + 1) * (w - k2 + 1), False)]
    elif kind == "nafnet":
        width = case["width"]
        hp, wp = -(-h // 16) * 16, -(-w // 16) * 16
        parts = [(n * hp * wp * (12.0 + 2 * width), 2.0 * 27 * n * hp * wp * width),
                 (n * hp * wp * (24.0 + 2 * width), 2.0 * 27 * n * hp * wp * width)]
        for _, c in _nafnet_blocks(width):
            lvl = int(math.log2(c // width))
            hl, wl, k = hp >> lvl, wp >> lvl, 384 >> lvl
            parts.append(_naf_work(n * hl * wl, c, n * (hl - min(k, hl) + 1) * (wl - min(k, wl) + 1), case["fused"]))
        for i in range(4):
            c, q = width << i, n * (hp >> i + 1) * (wp >> i + 1)
            parts.append(_gemm(q, 4 * c, 2 * c, 2, 2, 2))          # down
            parts.append(_gemm(q, 2 * c, 4 * c, 2, 2, 2, res=2))   # up
    elif kind == "restormer":
        c, hd, ch = 48 << case["level"], _restormer_hidden(case["level"]), 48
        parts = [_gemm(m, c, 3 * c, e, e, e), (m * 6 * c * e, m * 3 * c * 18.0),
                 (m * 2 * c * e, m * c * (2 * ch + 4.0)), _gemm(m, c, c, e, e, e, res=e),
                 _gemm(m, c, 2 * hd, e, e, e), (m * 3 * hd * e, m * hd * 46.0), _gemm(m, hd, c, e, e, e, res=e)]
    elif kind == "fftformer":
        c = 48 << case["level"]
        dft = 20720.0 / 64  # dense forward (64 -> 80), filter and inverse (80 -> 64) per pixel and channel
        parts = [_gemm(m, c, 6 * c, e, e, e), (m * 12 * c * e, m * 6 * c * 18.0),
                 (m * 2 * c * (2 * e + 4), m * 2 * c * dft * 1.5),
                 (m * (2 * c * (4 + e) + 2 * c * e), 2.0 * m * 2 * c * c),
                 _gemm(m, c, 6 * c, e, e, e), (0, m * 6 * c * dft), (m * 9 * c * e, m * 3 * c * 46.0),
                 _gemm(m, 3 * c, c, e, e, e, res=e)]
    elif kind == "patch":
        c = case["c"]
        parts = [(2.0 * m * c * e, m * c * 20720.0 / 64)]
    elif kind == "rrdb":
        parts = [(m * (cin + 32) * 2.0 + 18 * cin * 32, 18.0 * m * cin * 32) for cin in (64, 96, 128, 160)]
        parts += [(m * (192 + 64) * 2.0 + 18 * 192 * 64, 18.0 * m * 192 * 64),
                  (m * (64 + 256) * 2.0 + 18 * 64 * 64, 72.0 * m * 64 * 64)]
    else:
        d, r = case["d"], case["r"]
        parts = [(m * d * (e + 4.0) + m * (r + 16) * 4.0, m * d * (2.0 * r + 4 + 48 + 18))]
    b, f = map(sum, zip(*parts))
    return {"bytes": float(b), "flops": float(f)}


# ------------------------------------------------------------------------------- tolerance
def tolerance(case):
    """Relative error (2-norm) that another correct implementation may show: about four times the
    distance of the path from the 64-bit result."""
    kind, dtype = case["kind"], case.get("dtype", "bf16")
    if kind == "metrics":
        return {"rel": 1e-12}  # 64-bit sums of exact integers and Gaussian taps
    if kind == "nafnet":
        return {"rel": 9e-4}  # the image itself, added at the end, is most of the output
    if kind == "scan":
        return {"rel": 2e-6}
    if dtype == "fp32":  # products split over bf16 units carry 3.5e-6 through the patch transforms
        return {"rel": {"chain": 2e-6, "restormer": 4e-6, "fftformer": 1.5e-5, "patch": 1.5e-5}[kind]}
    if kind == "nafblock" and case["c"] >= 512:
        return {"rel": 6e-4}  # the fp32 residual stream dominates
    return {"rel": 1e-2}


# ------------------------------------------------------------------------------- 64-bit results
def exact(case, seed):
    t = {k: (v.double() if torch.is_tensor(v) and v.is_floating_point() else v)
         for k, v in _inputs(case, seed).items()}
    with torch.no_grad():
        return _EXACT[case["kind"]](case, t)


def _ln64(x, eps):
    x = x - x.mean(-1, keepdim=True)
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _shift(x, dy, dx):
    """x [N, H, W, C] moved so that position (y, x) holds (y + dy, x + dx), zeros outside."""
    n, h, w, c = x.shape
    p = F.pad(x, (0, 0, 1, 1, 1, 1))
    return p[:, 1 + dy:1 + dy + h, 1 + dx:1 + dx + w]


def _dw64(x, taps, b=None):
    y = sum(_shift(x, ky - 1, kx - 1) * taps[:, 0, ky, kx] for ky in range(3) for kx in range(3))
    return y if b is None else y + b


def _conv64(x, w, b):
    return sum(_shift(x, ky - 1, kx - 1) @ w[:, :, ky, kx].t() for ky in range(3) for kx in range(3)) + b


def _halves(y):
    c = y.shape[-1] // 2
    return y[..., :c], y[..., c:]


def _simple_gate(y):
    a, b = _halves(y)
    return a * b


def _gelu_gate(y):
    a, b = _halves(y)
    return F.gelu(a) * b


def _local_mean64(x, k):
    """Mean over the valid (k, k) windows (clipped to the image), replicated to the image's size."""
    n, h, w, c = x.shape
    k1, k2 = min(k, h), min(k, w)
    s = F.pad(x.cumsum(1).cumsum(2), (0, 0, 1, 0, 1, 0))
    m = (s[:, k1:, k2:] + s[:, :-k1, :-k2] - s[:, :-k1, k2:] - s[:, k1:, :-k2]) / (k1 * k2)
    oh, ow = h - k1 + 1, w - k2 + 1
    rows = (torch.arange(h, device=x.device) - (h - oh) // 2).clamp(0, oh - 1)
    cols = (torch.arange(w, device=x.device) - (w - ow) // 2).clamp(0, ow - 1)
    return m, rows, cols


def _exact_chain(case, t):
    u = _simple_gate(t["x"] @ t["w1"] + t["b1"])
    return t["x"] + (u @ t["w2"] + t["b2"]) * t["beta"]


def _block64(x, t, k):
    v = _simple_gate(_dw64(_ln64(x, 1e-6) @ t["w1"] + t["b1"], t["dw"], t["dwb"]))
    m, rows, cols = _local_mean64(v, k)
    s = m @ t["ws"] + t["bs"]
    y = x + ((v * s[:, rows][:, :, cols]) @ t["w3"] + t["b3"]) * t["beta"]
    u = _simple_gate(_ln64(y, 1e-6) @ t["w4"] + t["b4"])
    return y + (u @ t["w5"] + t["b5"]) * t["gamma"]


def _exact_nafblock(case, t):
    return _block64(t["x"], t, case["window"])


def _exact_nafnet(case, t):
    sd = {k: v.double() for k, v in t["sd"].items()}
    img = t["img"]
    h, w = img.shape[-2:]
    xp = F.pad(img, (0, -w % 16, 0, -h % 16)).permute(0, 2, 3, 1)

    def block(x, p, lvl):
        def kn(name):
            return sd[f"{p}.{name}.weight"].flatten(1).t()

        def folded(conv, norm):  # the LayerNorm's affine belongs to the conv after it
            wt = kn(conv)
            return wt * sd[f"{p}.{norm}.weight"][:, None], sd[f"{p}.{conv}.bias"] + sd[f"{p}.{norm}.bias"] @ wt
        b = {"dw": sd[f"{p}.conv2.weight"], "dwb": sd[f"{p}.conv2.bias"], "ws": kn("sca.1"),
             "bs": sd[f"{p}.sca.1.bias"], "w3": kn("conv3"), "b3": sd[f"{p}.conv3.bias"],
             "beta": sd[f"{p}.beta"].flatten(), "w5": kn("conv5"), "b5": sd[f"{p}.conv5.bias"],
             "gamma": sd[f"{p}.gamma"].flatten()}
        b["w1"], b["b1"] = folded("conv1", "norm1")
        b["w4"], b["b4"] = folded("conv4", "norm2")
        return _block64(x, b, 384 >> lvl)
    x = _conv64(xp, sd["intro.weight"], sd["intro.bias"])
    skips, lvl = [], 0
    for i, nb in enumerate(ENC):
        for j in range(nb):
            x = block(x, f"encoders.{i}.{j}", lvl)
        skips.append(x)
        n, hh, ww, c = x.shape
        x = x.reshape(n, hh // 2, 2, ww // 2, 2, c).permute(0, 1, 3, 5, 2, 4).reshape(n, hh // 2, ww // 2, 4 * c)
        x = x @ sd[f"downs.{i}.weight"].flatten(1).t() + sd[f"downs.{i}.bias"]
        lvl += 1
    for j in range(MID):
        x = block(x, f"middle_blks.{j}", lvl)
    for i, nb in enumerate(DEC):
        lvl -= 1
        y = x @ sd[f"ups.{i}.0.weight"].flatten(1).t()
        n, hh, ww, c4 = y.shape
        y = y.reshape(n, hh, ww, c4 // 4, 2, 2).permute(0, 1, 4, 2, 5, 3).reshape(n, 2 * hh, 2 * ww, c4 // 4)
        x = y + skips.pop()
        for j in range(nb):
            x = block(x, f"decoders.{i}.{j}", lvl)
    out = _conv64(x, sd["ending.weight"], sd["ending.bias"]) + xp
    return out.permute(0, 3, 1, 2)[:, :, :h, :w]


def _exact_restormer(case, t):
    x = t["x"]
    n, h, w, c = x.shape
    heads = 1 << case["level"]
    qkv = _dw64(_ln64(x, 1e-5) @ t["wq"] + t["bq"], t["dq"])
    q, k, v = (qkv[..., i * c:(i + 1) * c].reshape(n, h * w, heads, c // heads).permute(0, 2, 3, 1).contiguous()
               for i in range(3))
    q = q * q.square().sum(-1, keepdim=True).clamp_min(1e-24).rsqrt()
    k = k * k.square().sum(-1, keepdim=True).clamp_min(1e-24).rsqrt()
    a = torch.softmax((q @ k.transpose(-1, -2).contiguous()) * t["temp"], -1)
    o = (a @ v).permute(0, 3, 1, 2).reshape(n, h, w, c)
    y = x + o @ t["wp"]
    return y + _gelu_gate(_dw64(_ln64(y, 1e-5) @ t["wi"] + t["bi"], t["di"])) @ t["wo"]


def _patches(x):
    """[N, H, W, C] (whole patches) -> [N, H / 8, W / 8, C, 8, 8]."""
    n, h, w, c = x.shape
    return x.reshape(n, h // 8, 8, w // 8, 8, c).permute(0, 1, 3, 5, 2, 4)


def _unpatch(p):
    n, ph, pw, c = p.shape[:4]
    return p.permute(0, 1, 4, 2, 5, 3).reshape(n, 8 * ph, 8 * pw, c)


def _filter64(x, f):
    n, h, w, c = x.shape
    p = F.pad(x.permute(0, 3, 1, 2), (0, -w % 8, 0, -h % 8), mode="reflect").permute(0, 2, 3, 1)
    y = torch.fft.irfft2(torch.fft.rfft2(_patches(p).contiguous()) * f, s=(8, 8))
    return _unpatch(y)[:, :h, :w]


def _exact_fftformer(case, t):
    x = t["x"]
    c = x.shape[-1]
    hid = _dw64(_ln64(x, 1e-5) @ t["wh"] + t["bh"], t["dh"])
    q, k = (torch.fft.rfft2(_patches(hid[..., 2 * i * c:2 * (i + 1) * c]).contiguous()) for i in range(2))
    corr = _unpatch(torch.fft.irfft2(q * k, s=(8, 8)))
    del q, k
    y = x + ((_ln64(corr, 1e-5) * t["lnw"] + t["lnb"]) * hid[..., 4 * c:]) @ t["wp"]
    u = _filter64(_ln64(y, 1e-5) @ t["wi"] + t["bi"], t["f"])
    return y + _gelu_gate(_dw64(u, t["di"])) @ t["wo"]


def _exact_patch(case, t):
    return _filter64(t["x"], t["f"])


def _exact_rrdb(case, t):
    def lrelu(y):
        return F.leaky_relu(y, LEAKY)
    feats = t["x"]
    for i in range(4):
        feats = torch.cat([feats, lrelu(_conv64(feats, t[f"w{i}"], t[f"b{i}"]))], -1)
    y = _conv64(feats, t["w4"], t["b4"]) * 0.2 + t["x"]
    up = y.repeat_interleave(2, 1).repeat_interleave(2, 2)
    return y, lrelu(_conv64(up, t["wu"], t["bu"]))


def _exact_scan(case, t):
    """h[l] = exp(delta A) h[l - 1] + delta B u, y = C . h + D u: doubling inside blocks of 256 steps,
    then block after block."""
    n, hh, ww, d = t["u"].shape
    r, steps, blk = case["r"], hh * ww, 256
    out = []
    for i in range(n):
        u, dbl = t["u"][i].reshape(steps, d), t["dbl"][i].reshape(steps, -1)
        pad = -steps % blk
        delta = F.softplus(dbl[:, :r] @ t["dtw"].t() + t["dtb"])
        la = F.pad(delta, (0, 0, 0, pad)).view(-1, blk, d, 1) * t["A"]
        b = F.pad((delta * u)[..., None] * dbl[:, None, r:r + 8], (0, 0, 0, 0, 0, pad)).view(-1, blk, d, 8)
        s = 1
        while s < blk:
            b = torch.cat([b[:, :s], b[:, s:] + la[:, s:].exp() * b[:, :-s]], 1)
            la = torch.cat([la[:, :s], la[:, s:] + la[:, :-s]], 1)
            s *= 2
        start = torch.zeros(d, 8, device=u.device, dtype=u.dtype)
        starts = []
        for j in range(b.shape[0]):
            starts.append(start)
            start = la[j, -1].exp() * start + b[j, -1]
        hs = (b + la.exp() * torch.stack(starts)[:, None]).view(-1, d, 8)[:steps]
        out.append(((hs * dbl[:, None, r + 8:r + 16]).sum(-1) + t["D"] * u).view(hh, ww, d))
    return torch.stack(out)


def _exact_metrics(case, t):
    a, b = t["pred"].double(), t["gt"].double()
    peak = 1.0 if a.max() <= 1 else 255.0
    psnr = 20 * torch.log10(peak / (a - b).square().mean().sqrt())
    g = torch.tensor([math.exp(-((i - 5) ** 2) / 4.5) for i in range(11)], dtype=torch.float64)
    g = (g / g.sum()).tolist()

    def blur(x):
        for axis in range(3):
            size = x.shape[axis]
            idx = torch.arange(-5, size + 5, device=x.device).clamp(0, size - 1)
            p = x.index_select(axis, idx)
            x = sum(g[k] * p.narrow(axis, k, size) for k in range(11))
        return x
    c1, c2 = (0.01 * peak) ** 2, (0.03 * peak) ** 2
    ma, mb = blur(a), blur(b)
    saa, sbb, sab = blur(a * a) - ma * ma, blur(b * b) - mb * mb, blur(a * b) - ma * mb
    ssim = ((2 * ma * mb + c1) * (2 * sab + c2)) / ((ma * ma + mb * mb + c1) * (saa + sbb + c2))
    return torch.stack([psnr, ssim.mean()])


_EXACT = {"chain": _exact_chain, "nafblock": _exact_nafblock, "nafnet": _exact_nafnet,
          "restormer": _exact_restormer, "fftformer": _exact_fftformer, "patch": _exact_patch, "rrdb": _exact_rrdb,
          "scan": _exact_scan, "metrics": _exact_metrics}
