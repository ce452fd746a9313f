"""The work whose speed this package is judged by, through its public entry points.

``listed()`` holds the fixed cases, ``draw(rng)`` makes further ones of the same
ranges, and ``prepare`` / ``run`` / ``work`` / ``tolerance`` / ``exact`` say for a
case what a program holds beforehand, one pass, what the pass cannot do without,
how far another correct implementation may be off, and the result in 64 bits.

Sizes are those of SDXL (UNetConfig, VaeConfig): latents of 1024-pixel images
and of the other aspect ratios and smaller sizes the models accept, channels
320 / 640 / 1280, 77 text tokens, a conditional and an unconditional half
(B = 2) or one prediction (B = 1).  Layers get weights of unit gain, so that
every part of a sum counts in its result; the whole models get the package's
own random initialisation.
"""
import math

import torch
import torch.nn.functional as F

from dollama_amd import ops
from dollama_amd import unet as U
from dollama_amd import vae as V
from dollama_amd.flops import unet_step_flops

DEV = "cuda:0"
CTX, CROSS = 77, 2048
# the widths and blocks of the SDXL UNet with one transformer block per level,
# for a program that runs single resnet blocks
RESNET_CFG = U.UNetConfig(depth1=1, depth2=1)


def listed():
    return [
        # time and size embeddings of a guided step: the smallest launches of a
        # step, where latency is everything
        {"name": "embeddings_b2", "op": "embeddings", "B": 2},
        # a GroupNorm + SiLU over a skip concatenation of the up path, as a
        # layer of its own
        {"name": "group_norm_64x64_concat", "op": "group_norm", "B": 2, "H": 64, "W": 64, "Ca": 640, "Cb": 320,
         "f32": False},
        # attention output projection with bias and residual, 1024 tokens
        {"name": "linear_2048x1280x1280", "op": "linear", "M": 2048, "N": 1280, "K": 1280, "residual": True},
        # feed-forward (LayerNorm, GEGLU, projection, residual): the layer with
        # the most work of a step
        {"name": "feed_forward_1024", "op": "feed_forward", "B": 2, "S": 1024, "C": 1280},
        # self-attention layer at the level with the most tokens
        {"name": "self_attention_4096", "op": "self_attention", "B": 2, "S": 4096, "C": 640},
        # cross-attention layer at the deepest level of a 832 x 1216 image:
        # a token count that is no multiple of any tile
        {"name": "cross_attention_988", "op": "cross_attention", "B": 2, "S": 988, "C": 1280},
        # the drop-in attention call on [B, H, S, D] tensors
        {"name": "attention_bhsd_1024", "op": "attention_bhsd", "B": 2, "heads": 20, "Sq": 1024, "Sk": 1024, "D": 64},
        # a resnet's first 3x3 conv at full latent resolution, with the time bias
        {"name": "conv3x3_128x128x320", "op": "conv", "B": 2, "H": 128, "W": 128, "Cin": 320, "Cout": 320,
         "stride": 1, "up": False, "form": "tbias"},
        # the drop-in convolution call on NCHW tensors, an odd-sized downsampler
        {"name": "conv_nchw_stride2_104x152", "op": "conv_nchw", "B": 2, "H": 104, "W": 152, "Cin": 320,
         "Cout": 320, "k": 3, "stride": 2},
        # a whole resnet block of the up path over a concatenation (1x1 shortcut)
        {"name": "resnet_up_32x32", "op": "resnet", "B": 2, "H": 32, "W": 32, "block": "up_blocks.0.resnets.2",
         "Ca": 1280, "Cb": 640},
        # the whole guided UNet step of a 1024-pixel image
        {"name": "unet_step_1024px", "op": "unet", "B": 2, "H": 128, "W": 128},
        # decoding one 1024-pixel image
        {"name": "vae_decode_1024px", "op": "vae", "B": 1, "H": 128, "W": 128},
    ]


def _latent(rng, most=128 * 128):
    """Latent height and width, multiples of 4, of at most `most` pixels."""
    while True:
        h, w = (4 * round(math.exp(rng.uniform(math.log(8), math.log(48)))) for _ in range(2))
        if h * w <= most and max(h, w) <= 3 * min(h, w):
            return h, w


def _tokens(rng):
    """Tokens and channels of one transformer level."""
    h, w = _latent(rng)
    return (h * w // 4, 640) if rng.random() < 0.5 else (h * w // 16, 1280)


# resnet blocks by resolution level, with the channels of their input and skip
RESNETS = [("down_blocks.0.resnets.0", 0, 320, 0), ("down_blocks.1.resnets.0", 1, 320, 0),
           ("down_blocks.2.resnets.0", 2, 640, 0), ("mid_block.resnets.0", 2, 1280, 0),
           ("up_blocks.0.resnets.0", 2, 1280, 1280), ("up_blocks.0.resnets.2", 2, 1280, 640),
           ("up_blocks.1.resnets.0", 1, 1280, 640), ("up_blocks.1.resnets.2", 1, 640, 320),
           ("up_blocks.2.resnets.0", 0, 640, 320), ("up_blocks.2.resnets.2", 0, 320, 320)]


def draw(rng):
    op = rng.choice(["embeddings", "group_norm", "linear", "linear", "feed_forward", "self_attention",
                     "cross_attention", "attention_bhsd", "conv", "conv", "conv_nchw", "resnet", "unet", "vae"])
    B = rng.choice([1, 2, 2])
    if op == "embeddings":
        return {"op": op, "B": rng.randint(1, 8)}
    if op == "group_norm":
        h, w = _latent(rng)
        if rng.random() < 0.3:  # the decoder's fp32 stages
            return {"op": op, "B": 1, "H": 4 * h, "W": 4 * w, "Ca": rng.choice([128, 256, 512]), "Cb": 0, "f32": True}
        lv = rng.randrange(3)
        return {"op": op, "B": B, "H": h >> lv, "W": w >> lv, "Ca": 320 << lv,
                "Cb": rng.choice([0, 320, 640, 1280]), "f32": False}
    if op == "linear":
        S, C = _tokens(rng)
        N, K = rng.choice([(C, C), (3 * C, C), (C, 4 * C), (2 * C, C)])
        return {"op": op, "M": B * S, "N": N, "K": K, "residual": rng.random() < 0.5}
    if op in ("feed_forward", "self_attention", "cross_attention"):
        S, C = _tokens(rng)
        return {"op": op, "B": B, "S": S, "C": C}
    if op == "attention_bhsd":
        S = round(math.exp(rng.uniform(math.log(64), math.log(4096))))
        return {"op": op, "B": B, "heads": rng.choice([8, 10, 20]), "Sq": S,
                "Sk": CTX if rng.random() < 0.3 else S, "D": rng.choice([40, 64, 64, 64, 80])}
    if op in ("conv", "conv_nchw"):
        h, w = _latent(rng)
        lv = rng.randrange(3)
        h, w, ci = h >> lv, w >> lv, 320 << lv
        stride = rng.choice([1, 1, 2])
        if op == "conv_nchw":
            k = rng.choice([1, 3, 3])
            return {"op": op, "B": B, "H": h, "W": w, "Cin": 4 if lv == 0 and rng.random() < 0.3 else ci,
                    "Cout": rng.choice([4, 320, 640]), "k": k, "stride": stride}
        up = lv > 0 and stride == 1 and rng.random() < 0.3
        form = "plain" if up or stride == 2 else rng.choice(["tbias", "residual", "silu"])
        return {"op": op, "B": B, "H": h, "W": w, "Cin": ci, "Cout": ci if up or stride == 2 else
                rng.choice([320, 640, 1280]), "stride": stride, "up": up, "form": form}
    h, w = _latent(rng)
    if op == "resnet":
        block, lv, ca, cb = rng.choice(RESNETS)
        return {"op": op, "B": B, "H": h >> lv, "W": w >> lv, "block": block, "Ca": ca, "Cb": cb}
    if op == "vae":
        return {"op": op, "B": 1, "H": 8 * (h // 8) or 8, "W": 8 * (w // 8) or 8}
    return {"op": op, "B": B, "H": h, "W": w}


# ---------------------------------------------------------------------------
# Inputs: fp16 tensors from the seed alone, the same for run and exact.
# ---------------------------------------------------------------------------
def _inputs(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    op = case["op"]

    def rn(*shape, std=1.0, dtype=torch.float16):
        return (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)

    def weight(n, *k):  # unit gain
        return rn(n, *k, std=math.prod(k) ** -0.5)

    def norm(c):
        return 1.0 + rn(c, std=0.1), rn(c, std=0.1)

    t = {}
    if op == "embeddings":
        B = case["B"]
        t["timesteps"] = torch.full((B,), float(torch.randint(1, 1000, (1,), generator=g, device=DEV)), device=DEV)
        t["text"] = rn(B, 1280)
        t["ids"] = torch.tensor([1024, 1024, 0, 0, 1024, 1024], dtype=torch.float16, device=DEV)
        for name, n, k in (("t1", 1280, 320), ("t2", 1280, 1280), ("a1", 1280, 2816), ("a2", 1280, 1280)):
            t[name], t[name + "b"] = weight(n, k), rn(n, std=0.1)
    elif op == "group_norm":
        dt = torch.float32 if case["f32"] else torch.float16
        B, H, W, Ca, Cb = (case[k] for k in ("B", "H", "W", "Ca", "Cb"))
        t["x"] = rn(B, H, W, Ca, std=2.0, dtype=dt) + 0.5
        t["xb"] = rn(B, H, W, Cb) if Cb else None
        t["g"], t["b"] = norm(Ca + Cb)
    elif op == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        t["x"], t["w"], t["b"] = rn(M, K), weight(N, K), rn(N, std=0.1)
        t["res"] = rn(M, N) if case["residual"] else None
    elif op in ("feed_forward", "self_attention", "cross_attention"):
        B, S, C = case["B"], case["S"], case["C"]
        t["x"] = rn(B * S, C)
        t["g"], t["beta"] = norm(C)
        if op == "feed_forward":
            t["w1"], t["b1"] = weight(8 * C, C), rn(8 * C, std=0.1)
            t["w2"], t["b2"] = weight(C, 4 * C), rn(C, std=0.1)
        else:
            t["wo"], t["bo"] = weight(C, C), rn(C, std=0.1)
        if op == "self_attention":
            t["wqkv"] = weight(3 * C, C)
        if op == "cross_attention":
            t["wq"], t["wkv"] = weight(C, C), weight(2 * C, CROSS)
            t["ehs"] = rn(B * CTX, CROSS)
    elif op == "attention_bhsd":
        B, H, D = case["B"], case["heads"], case["D"]
        t["q"], t["k"], t["v"] = rn(B, H, case["Sq"], D), rn(B, H, case["Sk"], D), rn(B, H, case["Sk"], D)
    elif op in ("conv", "conv_nchw"):
        B, H, W, ci, co = (case[k] for k in ("B", "H", "W", "Cin", "Cout"))
        k = case.get("k", 3)
        t["x"] = rn(B, ci, H, W)
        t["w"], t["b"] = weight(co, ci, k, k), rn(co, std=0.1)
        if op == "conv":
            Ho, Wo = _conv_out(case)
            t["tbias"] = rn(B, co) if case["form"] == "tbias" else None
            t["res"] = rn(B, co, Ho, Wo) if case["form"] == "residual" else None
    elif op == "resnet":
        B, H, W = case["B"], case["H"], case["W"]
        t["x"], t["temb"] = rn(B, H, W, case["Ca"]), rn(B, 1280)
        t["xb"] = rn(B, H, W, case["Cb"]) if case["Cb"] else None
    elif op == "unet":
        B = case["B"]
        t["latent"] = rn(B, 4, case["H"], case["W"])
        t["timesteps"] = torch.full((B,), 1.0 + 50.0 * (seed % 20), device=DEV)
        t["ehs"], t["text"] = rn(B, CTX, CROSS), rn(B, 1280)
        px = [8.0 * case["H"], 8.0 * case["W"]]
        t["ids"] = torch.tensor(px + [0, 0] + px, dtype=torch.float16, device=DEV)
    elif op == "vae":
        t["latent"] = rn(case["B"], 4, case["H"], case["W"], std=7.0)  # 1 / scaling factor
    return t


def _conv_out(case):
    k, s = case.get("k", 3), case["stride"]
    f = 2 if case.get("up") else 1
    return tuple((f * case[d] + 2 * (k // 2) - k) // s + 1 for d in ("H", "W"))


# ---------------------------------------------------------------------------
# What a program holds, and one pass
# ---------------------------------------------------------------------------
def prepare(case, seed):
    t = _inputs(case, seed)
    op = case["op"]
    st = {"case": case, "t": t}
    if op == "feed_forward":
        M, C = t["x"].shape
        st["w1"], st["b1"] = ops.pack_geglu(t["w1"], t["b1"])
        st["n"], st["y"] = torch.empty_like(t["x"]), torch.empty_like(t["x"])
        st["h"] = torch.empty(M, 4 * C, dtype=torch.float16, device=DEV)
    elif op == "self_attention":
        st["qkv"] = ops.ln_fold(t["wqkv"], t["g"], t["beta"])
        st["o"], st["y"] = torch.empty_like(t["x"]), torch.empty_like(t["x"])
    elif op == "cross_attention":
        st["q"] = ops.ln_fold(t["wq"], t["g"], t["beta"])
        st["o"], st["y"] = torch.empty_like(t["x"]), torch.empty_like(t["x"])
    elif op == "attention_bhsd":
        st["o"] = torch.empty_like(t["q"])
    elif op == "conv":
        st["x"], st["w"] = ops.nchw_to_nhwc(t["x"]), ops.pack_conv_weight(t["w"])
        st["res"] = None if t["res"] is None else ops.nchw_to_nhwc(t["res"])
    elif op == "conv_nchw":
        st["y"] = torch.empty(case["B"], case["Cout"], *_conv_out(case), dtype=torch.float16, device=DEV)
    elif op == "resnet":
        st["net"] = U.UNet(RESNET_CFG)
        st["net"].set_weights(U.random_weights(RESNET_CFG, seed, device=DEV))
        st["net"].prepare()
    elif op == "unet":
        st["net"] = U.UNet(U.SDXL_CONFIG)
        st["net"].set_weights(U.random_weights(U.SDXL_CONFIG, seed, device=DEV))
        st["net"].prepare()
    elif op == "vae":
        st["vae"] = V.VAE(V.SDXL_VAE_CONFIG)
        st["vae"].set_weights(V.random_weights(V.SDXL_VAE_CONFIG, seed, device=DEV))
        st["vae"].prepare()
    return st


def run(st):
    case, t = st["case"], st["t"]
    op = case["op"]
    if op == "embeddings":
        te, ai = ops.sdxl_embed_inputs(t["timesteps"], t["text"], t["ids"])
        emb = ops.linear_small(ops.linear_small(te, t["t1"], t["t1b"], act=ops.ACT_SILU), t["t2"], t["t2b"])
        a = ops.linear_small(ai, t["a1"], t["a1b"], act=ops.ACT_SILU)
        return ops.linear_small(a, t["a2"], t["a2b"], out=emb, accumulate=True)
    if op == "group_norm":
        return ops.group_norm_nhwc(t["x"], t["g"], t["b"], 32, 1e-5, True, x_b=t["xb"])
    if op == "linear":
        return ops.linear(t["x"], t["w"], bias=t["b"], residual=t["res"])
    if op == "feed_forward":
        M, C = t["x"].shape
        ops.launch_layer_norm(t["x"], t["g"], t["beta"], st["n"], M, C, 1e-5)
        ops.linear(st["n"], st["w1"], bias=st["b1"], act=ops.ACT_GEGLU, out=st["h"])
        ops.linear(st["h"], t["w2"], bias=t["b2"], residual=t["x"], out=st["y"])
        return st["h"], st["y"]
    if op == "self_attention":
        B, S, C = case["B"], case["S"], case["C"]
        ld = (S + 7) & ~7
        qk, vt = ops.linear_vt_ln(t["x"], *st["qkv"], 1e-5, 2 * C, S, vt_ld=ld)
        ops.attention_vt(qk, qk[:, C:], vt, st["o"], B=B, H=C // 64, Sq=S, Sk=S, q_strides=(S * 2 * C, 2 * C, 64),
                         k_strides=(S * 2 * C, 2 * C, 64), vt_strides=(C * ld, 64 * ld), vt_ld=ld,
                         o_strides=(S * C, C, 64), scale=0.125)
        ops.linear(st["o"], t["wo"], bias=t["bo"], residual=t["x"], out=st["y"])
        return st["o"], st["y"]
    if op == "cross_attention":
        B, S, C = case["B"], case["S"], case["C"]
        ld = (CTX + 7) & ~7
        q = ops.linear_ln(t["x"], *st["q"], 1e-5)
        k, vt = ops.linear_vt(t["ehs"], t["wkv"], C, CTX, vt_ld=ld)
        ops.attention_vt(q, k, vt, st["o"], B=B, H=C // 64, Sq=S, Sk=CTX, q_strides=(S * C, C, 64),
                         k_strides=(CTX * C, C, 64), vt_strides=(C * ld, 64 * ld), vt_ld=ld,
                         o_strides=(S * C, C, 64), scale=0.125)
        ops.linear(st["o"], t["wo"], bias=t["bo"], residual=t["x"], out=st["y"])
        return st["o"], st["y"]
    if op == "attention_bhsd":
        ops.launch_attention(t["q"], t["k"], t["v"], st["o"], case["B"], case["heads"], case["Sq"], case["Sk"],
                             case["D"], case["D"] ** -0.5)
        return st["o"]
    if op == "conv":
        return ops.conv2d_nhwc(st["x"], st["w"], KH=3, KW=3, stride=case["stride"], pad=1, bias=t["b"],
                               tbias=t["tbias"], residual=st["res"], upsample=case["up"],
                               act=ops.ACT_SILU if case["form"] == "silu" else ops.ACT_NONE)
    if op == "conv_nchw":
        k, s = case["k"], case["stride"]
        ops.launch_conv2d(t["x"], t["w"], t["b"], st["y"], case["B"], case["Cin"], case["H"], case["W"],
                          case["Cout"], k, k, s, s, k // 2, k // 2)
        return st["y"]
    if op == "resnet":
        return st["net"].run_resnet(case["block"], t["x"], t["temb"], x_b=t["xb"])
    if op == "unet":
        return st["net"].forward(t["latent"], t["timesteps"], t["ehs"], t["text"], t["ids"])
    return st["vae"].decode(t["latent"])


# ---------------------------------------------------------------------------
# Work, tolerance
# ---------------------------------------------------------------------------
def _resnet_channels(block):
    return U.weight_specs(RESNET_CFG)[block + ".conv1.weight"][0]


def _vae_flops(B, h, w):
    """2 per multiply-add of the decoder's convs, projections and attention."""
    ch = V.SDXL_VAE_CONFIG.ch[::-1]
    S, C = h * w, ch[0]
    f = 2 * S * (4 * 4 + 9 * 4 * C) + 4 * 2 * S * 9 * C * C + 4 * 2 * S * C * C + 4 * S * S * C
    cin = C
    for b, co in enumerate(ch):
        px = S * 4 ** b
        for r in range(V.SDXL_VAE_CONFIG.layers):
            ci = cin if r == 0 else co
            f += 2 * px * (9 * ci * co + 9 * co * co + (ci * co if ci != co else 0))
        if b < 3:
            f += 2 * 4 * px * 9 * co * co
        cin = co
    return B * (f + 2 * 64 * S * 9 * cin * 3)


def work(case):
    op = case["op"]
    if op == "embeddings":
        B, w = case["B"], 1280 * (320 + 1280 + 2816 + 1280)
        return {"bytes": 2 * (w + 4 * 1280 + B * (1280 + 1280)) + 4 * B, "flops": 2 * B * w}
    if op == "group_norm":
        n = case["B"] * case["H"] * case["W"]
        return {"bytes": n * (case["Ca"] * (6 if case["f32"] else 4) + 4 * case["Cb"]),
                "flops": 8 * n * (case["Ca"] + case["Cb"])}
    if op == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 2 * (M * K + N * K + N + M * N * (2 if case["residual"] else 1)), "flops": 2 * M * N * K}
    if op in ("feed_forward", "self_attention", "cross_attention"):
        B, S, C = case["B"], case["S"], case["C"]
        M = B * S
        if op == "feed_forward":
            return {"bytes": 2 * (2 * M * C + 4 * M * C + 12 * C * C), "flops": 2 * M * 12 * C * C}
        if op == "self_attention":
            return {"bytes": 2 * (3 * M * C + 4 * C * C), "flops": 2 * M * 4 * C * C + 4 * B * S * S * C}
        return {"bytes": 2 * (3 * M * C + 2 * C * C + 2 * C * CROSS + B * CTX * CROSS),
                "flops": 2 * M * 2 * C * C + 2 * B * CTX * 2 * C * CROSS + 4 * B * S * CTX * C}
    if op == "attention_bhsd":
        n = case["B"] * case["heads"] * case["D"]
        return {"bytes": 2 * n * 2 * (case["Sq"] + case["Sk"]), "flops": 4 * n * case["Sq"] * case["Sk"]}
    if op in ("conv", "conv_nchw"):
        Ho, Wo = _conv_out(case)
        k, ci, co, B = case.get("k", 3), case["Cin"], case["Cout"], case["B"]
        outs = 2 if case.get("form") == "residual" else 1
        return {"bytes": 2 * (B * case["H"] * case["W"] * ci + co * ci * k * k + outs * B * Ho * Wo * co),
                "flops": 2 * B * Ho * Wo * co * ci * k * k}
    n = case["B"] * case["H"] * case["W"]
    if op == "resnet":
        ci, co = case["Ca"] + case["Cb"], _resnet_channels(case["block"])
        w = 9 * ci * co + 9 * co * co + (ci * co if ci != co else 0)
        return {"bytes": 2 * (n * (ci + co) + w + 1280 * co), "flops": 2 * n * w}
    if op == "unet":
        f = unet_step_flops(B=case["B"], H=case["H"], W=case["W"])
        return {"bytes": 2 * (2567463684 + 8 * n + case["B"] * CTX * CROSS), "flops": f["total"] + f["small"]}
    return {"bytes": 2 * (49490199 + n * (4 + 3 * 64)), "flops": _vae_flops(case["B"], case["H"], case["W"])}


def tolerance(case):
    # fp16 results of fp32 sums: one rounding is 2.1e-4 of the result, and a
    # layer of several roundings, a block and a whole model show more.  Stated
    # are four times the measured distances from the 64-bit results.
    return {"rel": {"unet": 6e-3, "vae": 4e-3, "resnet": 1.6e-3, "feed_forward": 1.5e-3, "self_attention": 1.5e-3,
                    "cross_attention": 2.2e-3, "attention_bhsd": 1.5e-3, "embeddings": 1.4e-3}.get(case["op"], 1e-3)}


# ---------------------------------------------------------------------------
# The same results by plain torch in 64 bits
# ---------------------------------------------------------------------------
def _d(t):
    return None if t is None else t.double()


def _linear(x, w, b=None):
    y = x @ w.double().t()
    return y if b is None else y + b.double()


def _layer_norm(x, g, b):
    return F.layer_norm(x, x.shape[-1:], g.double(), b.double(), 1e-5)


def _heads(x, B, D):  # [B * S, C] -> [B, heads, S, D]
    return x.reshape(B, -1, x.shape[-1] // D, D).transpose(1, 2).contiguous()


def _attention(q, k, v, scale):
    """softmax(q k^T scale) v over [B, H, S, D], one head at a time."""
    o = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            o[b, h] = torch.softmax((q[b, h] @ k[b, h].t()) * scale, -1) @ v[b, h]
    return o


def _merge(o):  # [B, heads, S, D] -> [B * S, C]
    return o.transpose(1, 2).reshape(o.shape[0] * o.shape[2], -1)


def _conv(x, w, b, stride=1, up=False):
    """Channels-last conv with padding k // 2, one product per tap."""
    if up:
        x = x.repeat_interleave(2, 1).repeat_interleave(2, 2)
    k = w.shape[-1]
    N, H, W, C = x.shape
    Ho, Wo = ((s + 2 * (k // 2) - k) // stride + 1 for s in (H, W))
    x = F.pad(x, (0, 0, k // 2, k // 2, k // 2, k // 2))
    y = b.double().expand(N, Ho, Wo, -1)
    for i in range(k):
        for j in range(k):
            s = x[:, i:i + stride * (Ho - 1) + 1:stride, j:j + stride * (Wo - 1) + 1:stride]
            y = y + (s.reshape(-1, C) @ w[:, :, i, j].double().t()).reshape(N, Ho, Wo, -1)
    return y


def _group_norm(x, g, b, eps, silu=True):
    """Channels-last GroupNorm over 32 groups."""
    y = F.group_norm(x.permute(0, 3, 1, 2), 32, g.double(), b.double(), eps).permute(0, 2, 3, 1)
    return F.silu(y) if silu else y


def _resnet(w, p, x, temb, eps):
    h = _conv(_group_norm(x, w[p + "norm1.weight"], w[p + "norm1.bias"], eps), w[p + "conv1.weight"],
              w[p + "conv1.bias"])
    if temb is not None:
        h = h + _linear(F.silu(temb), w[p + "time_emb_proj.weight"], w[p + "time_emb_proj.bias"])[:, None, None]
    h = _conv(_group_norm(h, w[p + "norm2.weight"], w[p + "norm2.bias"], eps), w[p + "conv2.weight"],
              w[p + "conv2.bias"])
    if p + "conv_shortcut.weight" in w:
        x = _conv(x, w[p + "conv_shortcut.weight"], w[p + "conv_shortcut.bias"])
    return x + h


def _sinusoid(t, dim):
    f = torch.exp(torch.arange(dim // 2, dtype=torch.float64, device=DEV) * (-math.log(10000.0) / (dim // 2)))
    a = t.double()[:, None] * f
    return torch.cat([a.cos(), a.sin()], 1)


def _size_inputs(text, ids):
    e = _sinusoid(ids.reshape(-1), 256).reshape(1, -1).expand(text.shape[0], -1)
    return torch.cat([text.double(), e], 1)


def _transformer(w, p, x, ehs, depth):
    B, H, W, C = x.shape
    h = _group_norm(x, w[p + "norm.weight"], w[p + "norm.bias"], 1e-6, silu=False).reshape(-1, C)
    h = _linear(h, w[p + "proj_in.weight"], w[p + "proj_in.bias"])
    for i in range(depth):
        k = f"{p}transformer_blocks.{i}."
        for a, norm in (("attn1.", "norm1"), ("attn2.", "norm2")):
            n = _layer_norm(h, w[k + norm + ".weight"], w[k + norm + ".bias"])
            src = n if a == "attn1." else ehs
            q, kk, v = (_heads(_linear(s, w[k + a + m + ".weight"]), B, 64)
                        for s, m in ((n, "to_q"), (src, "to_k"), (src, "to_v")))
            h = h + _linear(_merge(_attention(q, kk, v, 0.125)), w[k + a + "to_out.0.weight"],
                            w[k + a + "to_out.0.bias"])
        n = _layer_norm(h, w[k + "norm3.weight"], w[k + "norm3.bias"])
        v, g = _linear(n, w[k + "ff.net.0.proj.weight"], w[k + "ff.net.0.proj.bias"]).chunk(2, -1)
        h = h + _linear(v * F.gelu(g), w[k + "ff.net.2.weight"], w[k + "ff.net.2.bias"])
    return x + _linear(h, w[p + "proj_out.weight"], w[p + "proj_out.bias"]).reshape(B, H, W, C)


def _unet(w, t):
    def mlp(p, x):
        return _linear(F.silu(_linear(x, w[p + "linear_1.weight"], w[p + "linear_1.bias"])), w[p + "linear_2.weight"],
                       w[p + "linear_2.bias"])

    def conv(p, x, **kw):
        return _conv(x, w[p + ".weight"], w[p + ".bias"], **kw)

    depth = (0, U.SDXL_CONFIG.depth1, U.SDXL_CONFIG.depth2)
    temb = mlp("time_embedding.", _sinusoid(t["timesteps"], 320)) + mlp("add_embedding.",
                                                                        _size_inputs(t["text"], t["ids"]))
    ehs = t["ehs"].double().reshape(-1, CROSS)
    x = conv("conv_in", t["latent"].double().permute(0, 2, 3, 1))
    skips = [x]
    for lv in range(3):
        for r in range(2):
            x = _resnet(w, f"down_blocks.{lv}.resnets.{r}.", x, temb, 1e-5)
            if depth[lv]:
                x = _transformer(w, f"down_blocks.{lv}.attentions.{r}.", x, ehs, depth[lv])
            skips.append(x)
        if lv < 2:
            x = conv(f"down_blocks.{lv}.downsamplers.0.conv", x, stride=2)
            skips.append(x)
    x = _resnet(w, "mid_block.resnets.0.", x, temb, 1e-5)
    x = _transformer(w, "mid_block.attentions.0.", x, ehs, depth[2])
    x = _resnet(w, "mid_block.resnets.1.", x, temb, 1e-5)
    for u in range(3):
        for r in range(3):
            x = _resnet(w, f"up_blocks.{u}.resnets.{r}.", torch.cat([x, skips.pop()], -1), temb, 1e-5)
            if depth[2 - u]:
                x = _transformer(w, f"up_blocks.{u}.attentions.{r}.", x, ehs, depth[2 - u])
        if u < 2:
            x = conv(f"up_blocks.{u}.upsamplers.0.conv", x, up=True)
    x = conv("conv_out", _group_norm(x, w["conv_norm_out.weight"], w["conv_norm_out.bias"], 1e-5))
    return x.permute(0, 3, 1, 2)


def _vae(w, latent):
    w = {k.removeprefix("decoder."): v for k, v in w.items()}

    def conv(p, x, **kw):
        return _conv(x, w[p + ".weight"], w[p + ".bias"], **kw)

    x = conv("conv_in", conv("post_quant_conv", latent.double().permute(0, 2, 3, 1)))
    x = _resnet(w, "mid_block.resnets.0.", x, None, 1e-6)
    a, (B, H, W, C) = "mid_block.attentions.0.", x.shape
    h = _group_norm(x, w[a + "group_norm.weight"], w[a + "group_norm.bias"], 1e-6, silu=False).reshape(-1, C)
    q, k, v = (_heads(_linear(h, w[a + m + ".weight"], w[a + m + ".bias"]), B, C) for m in ("to_q", "to_k", "to_v"))
    o = _merge(_attention(q, k, v, C ** -0.5))
    x = x + _linear(o, w[a + "to_out.0.weight"], w[a + "to_out.0.bias"]).reshape(B, H, W, C)
    x = _resnet(w, "mid_block.resnets.1.", x, None, 1e-6)
    for b in range(4):
        for r in range(V.SDXL_VAE_CONFIG.layers):
            x = _resnet(w, f"up_blocks.{b}.resnets.{r}.", x, None, 1e-6)
        if b < 3:
            x = conv(f"up_blocks.{b}.upsamplers.0.conv", x, up=True)
    x = conv("conv_out", _group_norm(x, w["conv_norm_out.weight"], w["conv_norm_out.bias"], 1e-6))
    return x.permute(0, 3, 1, 2)


@torch.no_grad()
def exact(case, seed):
    t = _inputs(case, seed)
    op = case["op"]
    if op == "embeddings":
        e = _linear(F.silu(_linear(_sinusoid(t["timesteps"], 320), t["t1"], t["t1b"])), t["t2"], t["t2b"])
        a = F.silu(_linear(_size_inputs(t["text"], t["ids"]), t["a1"], t["a1b"]))
        return e + _linear(a, t["a2"], t["a2b"])
    if op == "group_norm":
        x = t["x"].double() if t["xb"] is None else torch.cat([t["x"].double(), t["xb"].double()], -1)
        return _group_norm(x, t["g"], t["b"], 1e-5)
    if op == "linear":
        y = _linear(_d(t["x"]), t["w"], t["b"])
        return y if t["res"] is None else y + t["res"].double()
    if op in ("feed_forward", "self_attention", "cross_attention"):
        B, C = case["B"], case["C"]
        x = t["x"].double()
        n = _layer_norm(x, t["g"], t["beta"])
        if op == "feed_forward":
            v, g = _linear(n, t["w1"], t["b1"]).chunk(2, -1)
            h = v * F.gelu(g)
            return h, x + _linear(h, t["w2"], t["b2"])
        if op == "self_attention":
            q, k, v = _linear(n, t["wqkv"]).chunk(3, -1)
        else:
            q, (k, v) = _linear(n, t["wq"]), _linear(_d(t["ehs"]), t["wkv"]).chunk(2, -1)
        o = _merge(_attention(_heads(q, B, 64), _heads(k, B, 64), _heads(v, B, 64), 0.125))
        return o, x + _linear(o, t["wo"], t["bo"])
    if op == "attention_bhsd":
        return _attention(_d(t["q"]), _d(t["k"]), _d(t["v"]), case["D"] ** -0.5)
    if op == "conv":
        y = _conv(_d(t["x"]).permute(0, 2, 3, 1), t["w"], t["b"], case["stride"], case["up"])
        if t["tbias"] is not None:
            y = y + t["tbias"].double()[:, None, None]
        if t["res"] is not None:
            y = y + t["res"].double().permute(0, 2, 3, 1)
        return F.silu(y) if case["form"] == "silu" else y
    if op == "conv_nchw":
        return _conv(_d(t["x"]).permute(0, 2, 3, 1), t["w"], t["b"], case["stride"]).permute(0, 3, 1, 2)
    if op == "resnet":
        w = U.random_weights(RESNET_CFG, seed, device=DEV)
        x = t["x"].double() if t["xb"] is None else torch.cat([t["x"].double(), t["xb"].double()], -1)
        return _resnet(w, case["block"] + ".", x, t["temb"].double(), 1e-5)
    if op == "unet":
        return _unet(U.random_weights(U.SDXL_CONFIG, seed, device=DEV), t)
    return _vae(V.random_weights(V.SDXL_VAE_CONFIG, seed, device=DEV), t["latent"])
