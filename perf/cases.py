"""Performance cases: the work that programs built on the library hand it.

Four models restore, upscale, inpaint and segment images of any size, and the
op interface offers the layers that they are made of.  Each case below is one
such call, with its inputs and outputs in device memory:

  esrgan    Real-ESRGAN x4: a whole image, or one tile of a photograph
  scunet    SCUNet denoising: a whole image
  lama      Big LaMa inpainting: an image and its mask
  birefnet  BiRefNet-lite segmentation: a square normalised image
  swin      a Swin transformer block on a token map
  spectral  the spectral branch of a fast Fourier convolution
  conv      a convolution of a map (NHWC as the models chain them, or NCHW)
  rows      a product over token rows (a projection or an MLP's layer)

prepare() holds what such a program keeps: the loaded weights, the input and
the output buffers.  Models that a service runs at one size over and over are
captured as a graph (`graph`); a one-off size is launched eagerly.
"""

import functools
import importlib
import math

import numpy as np
import torch
import torch.nn.functional as F

ien = importlib.import_module("image-engine-native_amd.ien")
synthetic = importlib.import_module("image-engine-native_amd.synthetic")

DEVICE = "cuda:0"


def listed():
    return [
        # A thumbnail or an icon: latency, one launch with a few tiles.
        dict(name="esrgan_64x48", kind="esrgan", height=48, width=64, graph=False),
        # The network's benchmark size.
        dict(name="esrgan_384x256", kind="esrgan", height=256, width=384, graph=False),
        # An inner tile of a photograph: 768 pixels with 34 of surroundings on each side.
        dict(name="esrgan_836x836", kind="esrgan", height=836, width=836, graph=False),
        # The network's benchmark size, served over and over.
        dict(name="scunet_768x512", kind="scunet", height=512, width=768, graph=True),
        # A photograph of an odd size in an editor: maps of 125 x 85 at an eighth, over the
        # fused spectral branch's 64.
        dict(name="lama_1000x680", kind="lama", height=680, width=1000, graph=False),
        # The network's benchmark size, served over and over.
        dict(name="birefnet_1024", kind="birefnet", side=1024, window=12, offsets=0.0, graph=True),
        # SCUNet's second level of a 768 x 512 image, the block's Swin half, shifted windows.
        dict(name="swin8_64_384x256", kind="swin", c=64, window=8, shift=4, height=256, width=384),
        # BiRefNet's third stage at 1024: windows of 12 that do not divide the map.
        dict(name="swin12_384_64x64", kind="swin", c=384, window=12, shift=6, height=64, width=64),
        # A global layer's spectral branch at LaMa's 512 x 512.
        dict(name="spectral_64x64", kind="spectral", height=64, width=64),
        # LaMa's local convolution on the ragged map of the editor's photograph.
        dict(name="conv3_512_128_125x85", kind="conv", layout="nhwc", size=3, step=1, pad="reflect",
             cin=512, cout=128, height=85, width=125, act="relu"),
        # A layer on channel planes, as the convolution sweep has it.
        dict(name="conv3_128_128_nchw", kind="conv", layout="nchw", size=3, step=1, pad="zero",
             cin=128, cout=128, height=128, width=192, act="none"),
        # The first layer of the third stage's MLP.
        dict(name="rows_4096_384_1536", kind="rows", rows=4096, k=384, n=1536, act="gelu"),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _sides(rng, low, high, area):
    """Two sides spread over their logarithm, their product at most `area`."""
    while True:
        h, w = _log_int(rng, low, high), _log_int(rng, low, high)
        if h * w <= area:
            return h, w


def draw(rng):
    kind = rng.choice(("esrgan", "esrgan", "scunet", "lama", "birefnet", "swin", "swin", "spectral",
                       "conv", "conv", "rows", "rows"))
    if kind == "esrgan":
        h, w = _sides(rng, 32, 836, 836 * 836 - 1)
        return dict(kind=kind, height=h, width=w, graph=False)
    if kind == "scunet":
        h, w = _sides(rng, 64, 768, 512 * 700)
        return dict(kind=kind, height=h, width=w, graph=rng.random() < 0.5)
    if kind == "lama":
        h, w = _sides(rng, 96, 1000, 660 * 1000)
        return dict(kind=kind, height=h, width=w, graph=rng.random() < 0.5)
    if kind == "birefnet":
        # Windows of 12 without deformable branches, or of 7 with them: the two networks the
        # weights files hold.
        window = rng.choice((7, 12))
        return dict(kind=kind, side=64 * rng.randint(4, 15), window=window,
                    offsets=0.0 if window == 12 else round(rng.uniform(0.01, 0.05), 4),
                    graph=rng.random() < 0.5)
    if kind == "swin":
        # Channels and the largest map side at the two networks' benchmark sizes.
        c, window, side = rng.choice(((32, 8, 512), (64, 8, 256), (128, 8, 128), (256, 8, 64),
                                      (96, 12, 256), (192, 12, 128), (384, 12, 64), (768, 12, 32),
                                      (96, 7, 256), (192, 7, 128), (384, 7, 64), (768, 7, 32)))
        return dict(kind=kind, c=c, window=window, shift=rng.choice((0, window // 2)),
                    height=rng.randint(side // 8, side), width=rng.randint(side // 8, side))
    if kind == "spectral":
        return dict(kind=kind, height=rng.randint(12, 64), width=rng.randint(12, 64))
    if kind == "conv":
        layout = rng.choice(("nhwc", "nhwc", "nchw"))
        while True:
            size = rng.choice((1, 3, 3, 3, 7))
            cin, cout = rng.choice((32, 64, 128, 256, 512)), rng.choice((32, 48, 64, 128, 256, 512))
            h, w = _sides(rng, 16, 512, 512 * 512)
            flops = 2.0 * h * w * size * size * cin * cout
            if 2e6 < flops < 1e11 and h * w * max(cin, cout) <= 1 << 26:
                break
        reflect = layout == "nhwc" and size > 1 and rng.random() < 0.4
        return dict(kind=kind, layout=layout, size=size,
                    step=2 if layout == "nhwc" and size == 3 and rng.random() < 0.25 else 1,
                    pad="reflect" if reflect else "zero", cin=cin, cout=cout, height=h, width=w,
                    act=rng.choice(("none", "relu")))
    k = rng.choice((64, 96, 128, 192, 256, 384, 512, 768))
    wide = rng.random() < 0.5
    act = rng.choice(("none", "gelu")) if wide else "none"
    n = k * rng.choice((3, 4)) if wide else k
    if not wide and rng.random() < 0.5:
        k *= 4
    return dict(kind="rows", rows=_log_int(rng, 64, 65536 * 96 // max(96, k)), k=k, n=n, act=act)


# ---- what a program holds -------------------------------------------------------

MODELS = {"esrgan": ien.MODEL_REALESRGAN, "scunet": ien.MODEL_SCUNET, "lama": ien.MODEL_LAMA,
          "birefnet": ien.MODEL_BIREFNET}
ACTS = {"none": ien.ACT_NONE, "relu": ien.ACT_RELU, "gelu": ien.ACT_GELU}
LOCAL, GLOBAL, SPECTRAL = synthetic.LAMA_LOCAL, synthetic.LAMA_GLOBAL, synthetic.LAMA_GLOBAL // 2


@functools.lru_cache(maxsize=None)
def _context():
    return ien.Context(0)


@functools.lru_cache(maxsize=8)
def _weights(kind, window, offsets):
    """A model's weights as its file holds them."""
    if kind == "esrgan":
        return synthetic.esrgan_tensors()
    if kind == "scunet":
        return synthetic.scunet_tensors(init="fan")
    if kind == "lama":
        return synthetic.lama_tensors()
    return synthetic.birefnet_tensors(window=window, init="fan", offsets=offsets)


def _model_weights(case):
    return _weights(case["kind"], case.get("window", 0), case.get("offsets", 0.0))


def _half(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).half()


def _inputs(case, seed):
    """The host arrays of a case: f32 images, f16 maps and f32 weights."""
    rng = np.random.default_rng([seed, 17])
    normal = lambda *s: rng.standard_normal(s, dtype=np.float32)  # noqa: E731
    kind = case["kind"]
    if kind in ("esrgan", "scunet"):
        return dict(image=rng.random((case["height"], case["width"], 3), dtype=np.float32))
    if kind == "lama":
        return dict(image=rng.random((case["height"], case["width"], 3), dtype=np.float32),
                    mask=synthetic.lama_mask(case["height"], case["width"], seed=seed))
    if kind == "birefnet":
        return dict(image=normal(case["side"], case["side"], 3))
    if kind == "swin":
        c, n, heads = case["c"], case["window"] ** 2, case["c"] // 32
        side = 2 * case["window"] - 1
        weights = dict(
            ln1_gamma=1 + 0.1 * normal(c), ln1_beta=0.1 * normal(c),
            qkv_w=normal(c, 3 * c) / math.sqrt(c), qkv_b=0.1 * normal(3 * c),
            position=synthetic.gathered_position_bias(normal(side * side, heads), case["window"], True),
            proj_w=normal(c, c) / math.sqrt(c), proj_b=0.1 * normal(c),
            ln2_gamma=1 + 0.1 * normal(c), ln2_beta=0.1 * normal(c),
            fc1_w=normal(c, 4 * c) / math.sqrt(c), fc1_b=0.1 * normal(4 * c),
            fc2_w=normal(4 * c, c) / math.sqrt(16 * c), fc2_b=0.1 * normal(c))
        assert weights["position"].shape == (heads, n, n)
        return dict(x=_half(normal(case["height"] * case["width"], c)), weights=weights)
    if kind == "spectral":
        h, w = case["height"], case["width"]
        return dict(x=_half(normal(h, w, GLOBAL)), cross=_half(normal(h, w, GLOBAL)),
                    w_in=normal(GLOBAL, SPECTRAL) * math.sqrt(2 / GLOBAL), b_in=0.02 * normal(SPECTRAL),
                    w_f=normal(2 * SPECTRAL, 2 * SPECTRAL) * math.sqrt(1 / SPECTRAL),
                    b_f=0.02 * normal(2 * SPECTRAL),
                    w_out=normal(SPECTRAL, GLOBAL) * math.sqrt(2 / SPECTRAL))
    if kind == "conv":
        k = case["size"] ** 2 * case["cin"]
        return dict(x=_half(normal(case["height"], case["width"], case["cin"])),
                    w=normal(k, case["cout"]) / math.sqrt(k), b=0.1 * normal(case["cout"]))
    return dict(x=_half(normal(case["rows"], case["k"])),
                w=normal(case["k"], case["n"]) / math.sqrt(case["k"]), b=0.1 * normal(case["n"]))


def _grid(case):
    """A convolution's output rows and columns."""
    return -(-case["height"] // case["step"]), -(-case["width"] // case["step"])


def prepare(case, seed):
    ctx = _context()
    got = _inputs(case, seed)
    kind = case["kind"]
    s = dict(case=case, ctx=ctx)
    half = lambda *shape: torch.empty(shape, dtype=torch.float16, device=DEVICE)  # noqa: E731
    if kind in MODELS:
        h, w = (case["side"],) * 2 if kind == "birefnet" else (case["height"], case["width"])
        s["model"] = ien.Model(ctx, MODELS[kind], tensors=_model_weights(case))
        s["model"].set_graph(case["graph"])
        s["height"], s["width"] = h, w
        s["image"] = torch.from_numpy(got["image"]).to(DEVICE)
        s["mask"] = torch.from_numpy(got["mask"]).to(DEVICE) if kind == "lama" else None
        shape = (h, w) if kind == "birefnet" else (4 * h, 4 * w, 3) if kind == "esrgan" else (h, w, 3)
        s["out"] = torch.empty(shape, dtype=torch.float32, device=DEVICE)
    elif kind == "swin":
        s["block"] = ien.Swin(ctx, case["c"], case["window"], case["shift"],
                              -math.inf if case["window"] == 8 else -100.0, got["weights"])
        s["x"] = got["x"].to(DEVICE)
        s["out"] = torch.empty_like(s["x"])
    elif kind == "spectral":
        h, w = case["height"], case["width"]
        s["plan"] = ien.Spectral(ctx, h, w)
        s["m_in"] = ien.Matrix(ctx, got["w_in"], got["b_in"])
        s["m_f"] = ien.Matrix(ctx, got["w_f"], got["b_f"])
        s["m_out"] = ien.Matrix(ctx, got["w_out"])
        s["x"], s["cross"] = got["x"].to(DEVICE), got["cross"].to(DEVICE)
        s["out"] = torch.empty_like(s["cross"])
        s["map"] = half(h, SPECTRAL, w)
        s["work"] = torch.empty(s["plan"].work_floats, dtype=torch.float32, device=DEVICE)
    elif kind == "conv":
        nchw = case["layout"] == "nchw"
        x = got["x"].permute(2, 0, 1).contiguous() if nchw else got["x"]
        s["x"] = x.to(DEVICE)
        s["m"] = ien.Matrix(ctx, got["w"], got["b"])
        s["layout"] = ien.NCHW if nchw else ien.NHWC
        s["input"] = ien.image_input(s["x"], case["height"], case["width"], case["cin"],
                                     layout=s["layout"], size=case["size"], step=case["step"],
                                     pad=ien.PAD_REFLECT if case["pad"] == "reflect" else ien.PAD_ZERO)
        oh, ow = _grid(case)
        s["rows"] = oh * ow
        s["stride"] = oh * ow if nchw else case["cout"]
        s["out"] = half(case["cout"], oh, ow) if nchw else half(oh, ow, case["cout"])
    else:
        s["x"] = got["x"].to(DEVICE)
        s["m"] = ien.Matrix(ctx, got["w"], got["b"])
        s["input"] = ien.rows_input(s["x"], case["k"])
        s["out"] = half(case["rows"], case["n"])
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind in MODELS:
        s["model"].run_device(s["image"], s["width"], s["height"], s["out"], s["mask"])
    elif kind == "swin":
        # The block works in place: the pass before it wrote the map.
        s["out"].copy_(s["x"])
        s["block"].run(s["out"], case["c"], case["height"], case["width"])
    elif kind == "spectral":
        # Accumulates onto what the cross convolution wrote.
        s["out"].copy_(s["cross"])
        s["plan"].run(s["x"], GLOBAL, s["m_in"], s["m_f"], s["m_out"], s["map"], s["work"], s["out"], GLOBAL)
    elif kind == "conv":
        ien.multiply_ex(ctx, s["input"], 0, s["rows"], s["m"], s["out"], s["stride"], layout=s["layout"],
                        act=ACTS[case["act"]])
    else:
        ien.multiply(ctx, s["input"], 0, case["rows"], s["m"], s["out"], case["n"], act=ACTS[case["act"]])
    return s["out"]


# ---- what a pass cannot do without ----------------------------------------------


def work(case):
    """Each input, weight (f16) and output moved once; the products' operations."""
    kind = case["kind"]
    if kind == "esrgan":
        px = case["height"] * case["width"]
        return dict(bytes=px * 51 * 4 + 2 * 1.213e6, flops=2.0 * px * (27 * 64 + 32 * 576 * 64 + 576 * 48))
    if kind == "scunet":
        px = (-(-case["height"] // 64) * 64) * (-(-case["width"] // 64) * 64)
        return dict(bytes=case["height"] * case["width"] * 6 * 4 + 2 * 18.29e6,
                    flops=944.9e9 * px / (512 * 768))
    if kind == "lama":
        px = (-(-case["height"] // 8) * 8) * (-(-case["width"] // 8) * 8)
        return dict(bytes=case["height"] * case["width"] * 7 * 4 + 2 * 50.94e6,
                    flops=439.8e9 * px / (512 * 512))
    if kind == "birefnet":
        return dict(bytes=case["side"] ** 2 * 4 * 4 + 2 * 44e6, flops=548.6e9 * case["side"] ** 2 / 1024 ** 2)
    if kind == "swin":
        c, tokens, n = case["c"], case["height"] * case["width"], case["window"] ** 2
        return dict(bytes=4.0 * tokens * c + 24 * c * c, flops=tokens * (24.0 * c * c + 4 * n * c))
    if kind == "spectral":
        h, w = case["height"], case["width"]
        px, half = h * w, h * (w // 2 + 1)
        products = px * (GLOBAL * SPECTRAL + SPECTRAL * GLOBAL) + half * 4 * SPECTRAL * SPECTRAL
        fft = 2 * 2.5 * px * math.log2(max(2, px)) * SPECTRAL
        return dict(bytes=6.0 * px * GLOBAL + 2 * (2 * GLOBAL * SPECTRAL + 4 * SPECTRAL ** 2),
                    flops=2.0 * products + fft)
    if kind == "conv":
        oh, ow = _grid(case)
        k = case["size"] ** 2 * case["cin"]
        return dict(bytes=2.0 * (case["height"] * case["width"] * case["cin"] + oh * ow * case["cout"]
                                 + k * case["cout"]),
                    flops=2.0 * oh * ow * k * case["cout"])
    return dict(bytes=2.0 * (case["rows"] * (case["k"] + case["n"]) + case["k"] * case["n"]),
                flops=2.0 * case["rows"] * case["k"] * case["n"])


# About four times the distance from exact() over these ranges: f16 maps and weights, sums in
# 32 bits (esrgan 1.6e-3, scunet 1.3e-3, lama 3.7e-4, birefnet 5.8e-4, swin 3.9e-4, spectral
# 4.6e-4, products 3.0e-4).
TOLERANCE = dict(esrgan=6e-3, scunet=5e-3, lama=1.5e-3, birefnet=2.5e-3, swin=1.6e-3, spectral=2e-3,
                 conv=1.2e-3, rows=1.2e-3)


def tolerance(case):
    return {"rel": TOLERANCE[case["kind"]]}


# ---- the same in 64 bits ----------------------------------------------------------


def _d(a):
    """A host array in 64 bits on the device."""
    t = a if isinstance(a, torch.Tensor) else torch.from_numpy(np.ascontiguousarray(a))
    return t.to(DEVICE).double()


def _conv(x, w, b, size, step=1, reflect=False):
    """x [H, W, C], w [(ky, kx, c), n]: the sum over taps of shifted products."""
    h, wd, c = x.shape
    p = size // 2
    if p:
        x = F.pad(x.permute(2, 0, 1)[None], (p,) * 4, mode="reflect" if reflect else "constant")
        x = x[0].permute(1, 2, 0)
    oh, ow = -(-h // step), -(-wd // step)
    out = x.new_zeros(oh * ow, w.shape[1])
    for t in range(size * size):
        ky, kx = divmod(t, size)
        part = x[ky:ky + step * (oh - 1) + 1:step, kx:kx + step * (ow - 1) + 1:step]
        out += part.reshape(-1, c) @ w[t * c:(t + 1) * c]
    if b is not None:
        out += b
    return out.reshape(oh, ow, -1)


def _norm(x, g, b):
    return F.layer_norm(x, (x.shape[-1],), g, b, eps=1e-5)


def _swin(x, t, window, shift, masked):
    """A Swin block on x [H, W, C], weights named as the library's."""
    h, w, c = x.shape
    heads, n = c // 32, window * window
    ph, pw = -(-h // window) * window, -(-w // window) * window
    y = F.pad(_norm(x, t["ln1_gamma"], t["ln1_beta"]), (0, 0, 0, pw - w, 0, ph - h))
    y = torch.roll(y, (-shift, -shift), (0, 1))

    def windows(z):
        z = z.reshape(ph // window, window, pw // window, window, -1)
        return z.permute(0, 2, 1, 3, 4).reshape(-1, n, z.shape[-1])

    q, k, v = (windows(y) @ t["qkv_w"] + t["qkv_b"]).split(c, dim=-1)
    cut = lambda z: z.reshape(-1, n, heads, 32).permute(0, 2, 1, 3).contiguous()  # noqa: E731
    scores = cut(q) @ cut(k).transpose(-1, -2).contiguous() / math.sqrt(32) + t["position"]
    if shift:
        # In a last window, tokens rolled in from the other edge are another region: the
        # last `shift` rows and columns of the padded map.
        rows = (torch.arange(ph, device=x.device) >= ph - shift).long()
        cols = (torch.arange(pw, device=x.device) >= pw - shift).long()
        region = windows((2 * rows[:, None] + cols[None, :])[..., None])[..., 0]
        apart = region[:, :, None] != region[:, None, :]
        scores = scores.masked_fill(apart[:, None], masked) if math.isinf(masked) else \
            scores + masked * apart[:, None]
    o = (scores.softmax(-1) @ cut(v)).permute(0, 2, 1, 3).reshape(-1, n, c) @ t["proj_w"] + t["proj_b"]
    o = o.reshape(ph // window, pw // window, window, window, c).permute(0, 2, 1, 3, 4).reshape(ph, pw, c)
    x = x + torch.roll(o, (shift, shift), (0, 1))[:h, :w]
    z = F.gelu(_norm(x, t["ln2_gamma"], t["ln2_beta"]) @ t["fc1_w"] + t["fc1_b"])
    return x + z @ t["fc2_w"] + t["fc2_b"]


def _spectral(x, cross, w_in, b_in, w_f, b_f, w_out):
    h, w, _ = x.shape
    s = torch.relu(x @ w_in + b_in)
    z = torch.fft.rfftn(s, dim=(0, 1), norm="ortho")
    z = torch.relu(torch.cat([z.real, z.imag], dim=-1) @ w_f + b_f)
    half = z.shape[-1] // 2
    back = torch.fft.irfftn(torch.complex(z[..., :half], z[..., half:]), s=(h, w), dim=(0, 1), norm="ortho")
    return torch.relu(cross + (s + back) @ w_out)


def _exact_esrgan(t, image):
    x = image
    for i in range(synthetic.ESRGAN_STEPS):
        x = _conv(x, t[f"body.{2 * i}.weight"], t[f"body.{2 * i}.bias"], 3)
        if i < synthetic.ESRGAN_STEPS - 1:
            x = torch.where(x >= 0, x, x * t[f"body.{2 * i + 1}.weight"])
    up = F.pixel_shuffle(x.permute(2, 0, 1)[None], 4)[0].permute(1, 2, 0)
    return up + image.repeat_interleave(4, 0).repeat_interleave(4, 1)


SCUNET_SWIN = dict(ln1_gamma="ln1.weight", ln1_beta="ln1.bias", qkv_w="msa.embedding_layer.weight",
                   qkv_b="msa.embedding_layer.bias", position="msa.position_bias",
                   proj_w="msa.linear.weight", proj_b="msa.linear.bias", ln2_gamma="ln2.weight",
                   ln2_beta="ln2.bias", fc1_w="mlp.0.weight", fc1_b="mlp.0.bias",
                   fc2_w="mlp.2.weight", fc2_b="mlp.2.bias")


def _scunet_block(x, t, p, shift):
    y = x @ t[f"{p}.conv1_1.weight"] + t[f"{p}.conv1_1.bias"]
    conv, tokens = y.chunk(2, dim=-1)
    r = torch.relu(_conv(conv, t[f"{p}.conv_block.0.weight"], None, 3))
    conv = conv + _conv(r, t[f"{p}.conv_block.2.weight"], None, 3)
    names = {k: t[f"{p}.trans_block.{v}"] for k, v in SCUNET_SWIN.items()}
    tokens = _swin(tokens, names, 8, shift, -math.inf)
    return x + torch.cat([conv, tokens], dim=-1) @ t[f"{p}.conv1_2.weight"] + t[f"{p}.conv1_2.bias"]


def _exact_scunet(t, image):
    h, w, _ = image.shape
    ph, pw = -(-h // 64) * 64, -(-w // 64) * 64
    x = F.pad(image.permute(2, 0, 1)[None], (0, pw - w, 0, ph - h), mode="replicate")[0].permute(1, 2, 0)
    x = head = _conv(x, t["m_head.0.weight"], None, 3)
    skips = []

    def blocks(x, name, first):
        for b in range(4):
            x = _scunet_block(x, t, f"{name}.{first + b}", 4 * (b % 2))
        return x

    for i in (1, 2, 3):
        x = blocks(x, f"m_down{i}", 0)
        x = torch.cat([x[0::2, 0::2], x[0::2, 1::2], x[1::2, 0::2], x[1::2, 1::2]], dim=-1)
        x = x @ t[f"m_down{i}.4.weight"]
        skips.append(x)
    x = blocks(x, "m_body", 0)
    for i in (3, 2, 1):
        x = (x + skips.pop()) @ t[f"m_up{i}.0.weight"]
        a, b, c = x.shape[0], x.shape[1], x.shape[2] // 4
        x = x.reshape(a, b, 2, 2, c).permute(0, 2, 1, 3, 4).reshape(2 * a, 2 * b, c)
        x = blocks(x, f"m_up{i}", 1)
    return _conv(x + head, t["m_tail.0.weight"], None, 3)[:h, :w]


def _exact_lama(t, image, mask):
    h, w = mask.shape
    ph, pw = -(-h // 8) * 8, -(-w // 8) * 8
    mirror = lambda n, p: torch.tensor([i if i < n else 2 * n - 1 - i for i in range(p)], device=DEVICE)  # noqa: E731
    image, mask = (z[mirror(h, ph)][:, mirror(w, pw)] for z in (image, mask))
    x = torch.cat([image * (1 - mask[..., None]), mask[..., None]], dim=-1)
    conv = lambda x, n, size, step=1: _conv(x, t[n + ".weight"], t[n + ".bias"], size, step, True)  # noqa: E731

    def ffc(x, n):
        local = torch.relu(conv(x, n + ".local", 3))
        spectral = _spectral(x[..., LOCAL:], conv(x[..., :LOCAL], n + ".cross", 3),
                             t[n + ".spectral_in.weight"], t[n + ".spectral_in.bias"],
                             t[n + ".fourier.weight"], t[n + ".fourier.bias"], t[n + ".spectral_out.weight"])
        return torch.cat([local, spectral], dim=-1)

    x = torch.relu(conv(x, "first", 7))
    for i in range(3):
        x = torch.relu(conv(x, f"down{i}", 3, 2))
    for b in range(synthetic.LAMA_BLOCKS):
        x = x + ffc(ffc(x, f"block{b}.ffc0"), f"block{b}.ffc1")
    for i in range(3):
        a, b, c = x.shape
        grown = F.pad(x, (0, 0, 0, 1, 0, 1))
        phases = []
        for p in range(4):
            m, cols = t[f"up{i}.phase{p}.weight"], []
            for dy in range(1 + p // 2):
                for dx in range(1 + p % 2):
                    cols.append(grown[dy:dy + a, dx:dx + b])
            phases.append(torch.cat(cols, dim=-1) @ m + t[f"up{i}.phase{p}.bias"])
        x = torch.relu(torch.stack(phases, 2).reshape(a, b, 2, 2, -1).permute(0, 2, 1, 3, 4)
                       .reshape(2 * a, 2 * b, -1))
    return torch.sigmoid(conv(x, "last", 7))[:h, :w]


BIREFNET_SWIN = dict(ln1_gamma="norm1.weight", ln1_beta="norm1.bias", qkv_w="qkv.weight", qkv_b="qkv.bias",
                     position="position_bias", proj_w="proj.weight", proj_b="proj.bias",
                     ln2_gamma="norm2.weight", ln2_beta="norm2.bias", fc1_w="fc1.weight", fc1_b="fc1.bias",
                     fc2_w="fc2.weight", fc2_b="fc2.bias")


def _resize(x, side):
    return F.interpolate(x.permute(2, 0, 1)[None], size=(side, side), mode="bilinear",
                         align_corners=True)[0].permute(1, 2, 0)


def _backbone(t, x, window):
    h, w, _ = x.shape
    x = x.reshape(h // 4, 4, w // 4, 4, 3).permute(0, 2, 1, 3, 4).reshape(h // 4, w // 4, 48)
    x = _norm(x @ t["patch_embed.weight"] + t["patch_embed.bias"], t["patch_embed.norm.weight"],
              t["patch_embed.norm.bias"])
    maps = []
    for s, (_, depth) in enumerate(synthetic.BIREFNET_STAGES):
        for b in range(depth):
            names = {k: t[f"stage{s}.block{b}.{v}"] for k, v in BIREFNET_SWIN.items()}
            x = _swin(x, names, window, window // 2 * (b % 2), -100.0)
        maps.append(_norm(x, t[f"stage{s}.norm.weight"], t[f"stage{s}.norm.bias"]))
        if s < 3:
            x = torch.cat([x[0::2, 0::2], x[1::2, 0::2], x[0::2, 1::2], x[1::2, 1::2]], dim=-1)
            x = _norm(x, t[f"stage{s}.merge.norm.weight"], t[f"stage{s}.merge.norm.bias"])
            x = x @ t[f"stage{s}.merge.weight"]
    return maps


def _aspp_branch(tm, t, p, size):
    h, w, c = tm.shape
    off = _conv(tm, t[p + ".offset.weight"], t[p + ".offset.bias"], size)
    taps = size * size
    ys, xs = (torch.arange(n, device=DEVICE, dtype=torch.float64) for n in (h, w))
    planes = tm.permute(2, 0, 1)[None].contiguous()
    out = tm.new_zeros(h, w, 256)
    for k in range(taps):
        py = ys[:, None] - size // 2 + k // size + off[..., 2 * k]
        px = xs[None, :] - size // 2 + k % size + off[..., 2 * k + 1]
        grid = torch.stack([(2 * px + 1) / w - 1, (2 * py + 1) / h - 1], dim=-1)[None]
        at = F.grid_sample(planes, grid, mode="bilinear", padding_mode="zeros", align_corners=False)[0]
        at = at.permute(1, 2, 0) * (2 * torch.sigmoid(off[..., 2 * taps + k]))[..., None]
        out += at @ t[p + ".weight"][k * c:(k + 1) * c]
    return torch.relu(out + t[p + ".bias"])


def _decoder_block(x, t, q, gate):
    tm = torch.relu(_conv(x, t[q + ".conv_in.weight"], t[q + ".conv_in.bias"], 3))
    pooled = torch.relu(tm.mean((0, 1)) @ t[q + ".aspp.pool.weight"] + t[q + ".aspp.pool.bias"])
    branches = [_aspp_branch(tm, t, f"{q}.aspp.branch{i}", k) for i, k in enumerate(synthetic.BIREFNET_ASPP_SIZES)]
    w1 = t[q + ".aspp.conv1.weight"]
    a = torch.relu(torch.cat(branches, -1) @ w1[:1024] + (t[q + ".aspp.conv1.bias"] + pooled @ w1[1024:]))
    out = _conv(a, t[q + ".conv_out.weight"], t[q + ".conv_out.bias"], 3)
    if gate:
        g = torch.relu(_conv(out, t[q + ".gdt.weight"], t[q + ".gdt.bias"], 3))
        out = out * torch.sigmoid(g @ t[q + ".gdt_attn.weight"] + t[q + ".gdt_attn.bias"])
    return out


def _exact_birefnet(t, image, window):
    side = image.shape[0]
    two = lambda x, p: _conv(_conv(x, t[p + ".conv1.weight"], t[p + ".conv1.bias"], 3),  # noqa: E731
                             t[p + ".conv_out.weight"], t[p + ".conv_out.bias"], 3)
    full, small = _backbone(t, image, window), _backbone(t, _resize(image, side // 2), window)
    levels = [torch.cat([f, _resize(s, f.shape[0])], -1) for f, s in zip(full, small)]
    x = torch.cat([_resize(v, side >> 5) for v in levels[:3]] + [levels[3]], -1)
    x = _decoder_block(x, t, "squeeze", False)
    for i in range(4):
        g = side >> (5 - i)
        if i:
            x = levels[3 - i] @ t[f"lateral{5 - i}.weight"] + t[f"lateral{5 - i}.bias"] + _resize(x, g)
        n = side // g
        patches = image.reshape(n, g, n, g, 3).permute(1, 3, 4, 0, 2).reshape(g, g, 3 * n * n)
        x = _decoder_block(torch.cat([x, two(patches, f"patches{5 - i}")], -1), t, f"block{4 - i}", i < 3)
    logits = _resize(x @ t["head.weight"] + t["head.bias"], side)
    return (logits + two(image, "patches1"))[..., 0]


def exact(case, seed):
    kind = case["kind"]
    got = _inputs(case, seed)
    if kind in MODELS:
        t = {k: _d(v) for k, v in _model_weights(case).items()}
        image = _d(got["image"])
        if kind == "lama":
            return _exact_lama(t, image, _d(got["mask"]))
        if kind == "birefnet":
            return _exact_birefnet(t, image, case["window"])
        return (_exact_esrgan if kind == "esrgan" else _exact_scunet)(t, image)
    if kind == "swin":
        t = {k: _d(v) for k, v in got["weights"].items()}
        x = _d(got["x"]).reshape(case["height"], case["width"], case["c"])
        masked = -math.inf if case["window"] == 8 else -100.0
        return _swin(x, t, case["window"], case["shift"], masked).reshape(-1, case["c"])
    if kind == "spectral":
        return _spectral(*(_d(got[k]) for k in ("x", "cross", "w_in", "b_in", "w_f", "b_f", "w_out")))
    act = {"none": lambda z: z, "relu": torch.relu, "gelu": F.gelu}[case["act"]]
    if kind == "conv":
        out = act(_conv(_d(got["x"]), _d(got["w"]), _d(got["b"]), case["size"], case["step"],
                        case["pad"] == "reflect"))
        return out.permute(2, 0, 1).contiguous() if case["layout"] == "nchw" else out
    return act(_d(got["x"]) @ _d(got["w"]) + _d(got["b"]))
