"""The calls whose speed is followed: encoder forwards, the attentive-pool head, the masked predictor and frame
preprocessing, through the library's public entry points (jepa_amd_encode_device, jepa_encode, jepa_amd_head_device,
jepa_predict_mod, jepa_amd_preprocess_frames_device).

A program loads a model once, keeps one context for it and sends it one input after another, each in a buffer of its
own; so the states here share a model and its context, and every state has its own input and output buffers.

Weights are synthetic (forge). Cases with fewer layers than the model has stand for its blocks: the same widths, heads,
token counts and weight types, with larger weights and random LayerNorm parameters, so that the attention depends on
its inputs. Cases with all layers use the benchmark's own models.
"""
import math
import os
import struct
import sys
from collections import OrderedDict
from dataclasses import replace

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "jepa.cpp_amd", "python"))

from jepa_amd import _lib, forge  # noqa: E402

# model -> forge configuration (family, widths, heads, patch and tubelet of the benchmark configurations)
MODELS = {"vits16": "vits16_f16", "vitb16": "vitb16_2_1_q8_0", "vitl16": "vitl16_q8_0", "levjepa": "levjepa_vitl16_q8_0",
          "vitg16": "vitg16_q8_0", "vith14": "vith14_ijepa_f16", "head": "vitl16_ssv2_q8_0", "pred": "vitl16_pred_q8_0"}
MEAN, STD = (0.485, 0.456, 0.406), (0.229, 0.224, 0.225)
MAX_FLOPS = 1.66e12     # a drawn case does no more than the whole ViT-L clip


def _enc(name, model, ftype, layers, batch, frames, height, width, via="device"):
    return {"name": name, "op": "encode", "model": model, "ftype": ftype, "layers": layers, "batch": batch, "frames": frames,
            "height": height, "width": width, "via": via}


def listed():
    return [
        # one image embedded at a time (LeJEPA ViT-S/16, all 12 layers, 197 tokens): latency, small kernels
        _enc("image_s16_f16", "vits16", "f16", 12, 1, 1, 224, 224),
        # one image through the reference's own call, host buffers in and out (V-JEPA 2.1 ViT-B/16 at 384: 576 tokens)
        _enc("image_b16_host_q8", "vitb16", "q8_0", 4, 1, 1, 384, 384, "host"),
        # a batch of images for a dataset's features (the 8-image benchmark shape)
        _enc("images_b16_q8", "vitb16", "q8_0", 4, 8, 1, 384, 384),
        # the headline: one 16-frame clip through all 24 layers of ViT-L/16 (2048 tokens)
        _enc("clip_l16_q8", "vitl16", "q8_0", 24, 1, 16, 256, 256),
        # the same clip with the smaller weight file
        _enc("clip_l16_q4k", "vitl16", "q4_k", 4, 1, 16, 256, 256),
        # several clips per call (a server's batch), 4-bit q4_0 weights
        _enc("clips_l16_q40", "vitl16", "q4_0", 2, 4, 16, 256, 256),
        # a long clip through the largest model's blocks (64 frames: 8192 tokens, width 1408, 22 heads)
        _enc("clip_g16_q8", "vitg16", "q8_0", 2, 1, 64, 256, 256),
        # block-causal video model, a ragged 3137 rows (16 slots of 196 patches and the CLS row)
        _enc("clip_levjepa_q8", "levjepa", "q8_0", 4, 1, 16, 224, 224),
        # heads of 80, f32 patch embedding of 14 x 14 patches, f16 weights (I-JEPA ViT-H/14)
        _enc("images_h14_f16", "vith14", "f16", 4, 4, 1, 224, 224),
        # video classification head on the encoder's rows: 3 pooler blocks, cross-attention, MLP, 174 classes
        {"name": "head_l16_q8", "op": "head", "model": "head", "ftype": "q8_0", "tokens": 2048},
        # masked prediction, half of the clip's tokens from the other half (12 blocks of 384), host buffers
        {"name": "predict_l16_q8", "op": "predict", "model": "pred", "ftype": "q8_0", "context": 1024, "target": 1024},
        # decoded 720p frames on the device to a normalised clip
        {"name": "frames_720p", "op": "frames", "frames": 16, "height": 720, "width": 1280, "short": 292, "crop": 256, "resample": 0},
    ]


def _between(rng, lo, hi):
    """A whole number spread evenly over the logarithm of lo..hi."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        c = _draw(rng)
        if work(c)["flops"] <= MAX_FLOPS:
            return c


def _draw(rng):
    op = rng.choice(["encode"] * 8 + ["head", "predict", "frames", "frames"])
    if op == "head":
        return {"op": op, "model": "head", "ftype": rng.choice(["q8_0", "f16", "q4_k"]), "tokens": _between(rng, 196, 4608)}
    if op == "predict":
        return {"op": op, "model": "pred", "ftype": rng.choice(["q8_0", "q8_0", "f16"]), "context": _between(rng, 64, 1024),
                "target": _between(rng, 32, 1024)}
    if op == "frames":
        h, w = rng.choice([(240, 320), (360, 640), (480, 854), (720, 1280), (1080, 1920), (rng.randint(200, 1100), rng.randint(200, 1900))])
        crop = rng.choice([224, 256, 384])
        return {"op": op, "frames": rng.choice([1, 8, 16, 32]), "height": h, "width": w, "short": rng.choice([crop, crop * 8 // 7]), "crop": crop,
                "resample": rng.choice([0, 0, 1])}
    model = rng.choice(["vits16", "vits16", "vitb16", "vitl16", "vitl16", "vitg16", "levjepa", "vith14"])
    ftype = rng.choice(["f16", "q8_0", "q8_0", "q4_0", "q4_k"])
    via = rng.choice(["device", "device", "device", "host"])
    side = lambda lo, hi, p: p * rng.randint(lo, hi)  # noqa: E731
    if model == "vits16":       # learned positions: square images of the model's own size
        s = side(6, 24, 16)
        return _enc_drawn(model, ftype, 12, _between(rng, 1, 16), 1, s, s, via)
    if model == "vith14":
        s = side(8, 24, 14)
        return _enc_drawn(model, rng.choice(["f16", "q8_0"]), 4, _between(rng, 1, 6), 1, s, s, via)
    if model == "vitb16":
        return _enc_drawn(model, ftype, 4, _between(rng, 1, 12), 1, side(12, 28, 16), side(12, 28, 16), via)
    if model == "vitg16":
        return _enc_drawn(model, rng.choice(["q8_0", "q4_k"]), 2, 1, 2 * rng.randint(4, 32), 256, 256, "device")
    if model == "levjepa":
        return _enc_drawn(model, rng.choice(["q8_0", "f16"]), 4, 1, rng.randint(2, 16), 224, 224, "device")
    return _enc_drawn(model, ftype, 4, _between(rng, 1, 4), 2 * rng.randint(1, 8), side(8, 18, 16), side(8, 18, 16), via)


def _enc_drawn(*a):
    c = _enc("", *a)
    del c["name"]
    return c


# ---- what a program has in hand -------------------------------------------------------------------------------

def _config(case):
    cfg = forge.CONFIGS[MODELS[case["model"]]]
    if case["op"] != "encode":      # the encoder's layers take no part
        return replace(cfg, n_layer=1, ftype=case["ftype"], ln_random=True, w_std=0.03)
    if case["layers"] != cfg.n_layer:
        cfg = replace(cfg, n_layer=case["layers"], ln_random=True, w_std=0.03)
    if cfg.family in ("hfvit", "ijepa"):
        cfg = replace(cfg, img_size=case["height"])
    return replace(cfg, ftype=case["ftype"])


_loaded = OrderedDict()      # model file -> context; the four that were used last


def _context(case):
    path = forge.cached_model(_config(case))
    if path not in _loaded:
        _loaded[path] = _lib.Context(_lib.Model(path, device=0))
        while len(_loaded) > 4:
            _loaded.popitem(last=False)
    _loaded.move_to_end(path)
    return _loaded[path], path


def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _pixels(seed, batch, frames, h, w):
    """Frames as cameras give them: uint8, smooth structure with finer noise on it, drifting from frame to frame."""
    g = _rng(seed)
    x = torch.zeros(batch, 3, frames, h, w, device="cuda")
    for cells, amp in ((4, 60.0), (16, 30.0), (64, 12.0)):
        for b in range(batch):
            coarse = torch.randn(1, 3, max(2, frames // 4), cells, cells, generator=g, device="cuda")
            x[b] += amp * torch.nn.functional.interpolate(coarse, size=(frames, h, w), mode="trilinear", align_corners=False)[0]
    x += 118.0 + 5.0 * torch.randn(x.shape, generator=g, device="cuda")
    return x.round_().clamp_(0, 255).to(torch.uint8)


def _clip(case, seed):
    u8 = _pixels(seed, case["batch"], case["frames"], case["height"], case["width"]).float()
    mean = torch.tensor(MEAN, device="cuda").view(1, 3, 1, 1, 1)
    std = torch.tensor(STD, device="cuda").view(1, 3, 1, 1, 1)
    return ((u8 / 255.0 - mean) / std).contiguous()


def _token_rows(case, seed, n, dim):
    """Encoder output rows: unit variance by the final LayerNorm, neighbouring tokens alike."""
    x = torch.randn(n, dim, generator=_rng(seed), device="cuda")
    x = x + 0.7 * torch.roll(x, 1, 0)
    return torch.nn.functional.layer_norm(x, (dim,)).contiguous()


def _ids(case, seed):
    perm = np.random.default_rng(int(seed)).permutation(2048).astype(np.int32)
    return np.sort(perm[:case["context"]]), np.sort(perm[case["context"]:case["context"] + case["target"]])


def _frames_params(case):
    p = _lib.lib().jepa_preprocess_default_params(None)
    p.resize_short, p.crop, p.resample = case["short"], case["crop"], case["resample"]
    return p


def prepare(case, seed):
    op = case["op"]
    if op == "frames":
        u8 = _pixels(seed, 1, case["frames"], case["height"], case["width"])[0].permute(1, 2, 3, 0).contiguous()
        out = torch.empty(3, case["frames"], case["crop"], case["crop"], device="cuda")
        state = {"op": op, "params": _frames_params(case), "in": u8, "out": out}
    else:
        ctx, _ = _context(case)
        m = ctx.model
        state = {"op": op, "ctx": ctx}
        if op == "head":
            state["in"] = _token_rows(case, seed, case["tokens"], m.dim)
            state["out"] = [torch.empty(m.dim, device="cuda"), torch.empty(m.n_classes, device="cuda")]
        elif op == "predict":
            state["in"] = _token_rows(case, seed, 2048, m.dim).cpu().numpy()
            state["ids"] = _ids(case, seed)
        else:
            x = _clip(case, seed)
            rows = m.token_grid(case["frames"], case["height"], case["width"])
            if case["via"] == "host":
                state["in"] = x.cpu().numpy()
            else:
                state["in"], state["out"] = x, torch.empty(case["batch"] * rows, m.dim, device="cuda")
    torch.cuda.synchronize()     # the library's streams do not wait for torch's
    return state


def run(state):
    op, x = state["op"], state["in"]
    if op == "frames":
        t, h, w, _ = x.shape
        L = _lib.lib()
        _lib.check(L.jepa_amd_preprocess_frames_device(0, state["params"], x.data_ptr(), t, h, w, state["out"].data_ptr(), state["out"].numel(),
                                                       None, None), "jepa_amd_preprocess_frames_device")
        return state["out"]
    ctx = state["ctx"]
    if op == "head":
        ctx.head_device(x.data_ptr(), x.shape[0], state["out"][0].data_ptr(), state["out"][1].data_ptr())
        return state["out"]
    if op == "predict":
        return ctx.predict(x, *state["ids"])
    if "out" not in state:
        return ctx.encode(x)
    ctx.encode_device(x.data_ptr(), tuple(x.shape), state["out"].data_ptr(), state["out"].numel())
    return state["out"]


# ---- what a pass cannot do without ----------------------------------------------------------------------------

_WBYTES = {"f16": 2.0, "q8_0": 34 / 32, "q4_0": 18 / 32, "q4_k": 144 / 256}


def _blocks(rows, seqs, d, f, n_layer, seen=1.0):
    """Multiply-adds (as 2 flops) of transformer blocks over rows tokens in seqs sequences, and the weights they read."""
    per = rows / seqs
    return n_layer * (2.0 * rows * (4 * d * d + 2 * d * f) + 4.0 * rows * per * d * seen), n_layer * (4.0 * d * d + 2.0 * d * f)


def work(case):
    op = case["op"]
    if op == "frames":
        src = case["frames"] * case["height"] * case["width"] * 3
        dst = case["frames"] * case["crop"] ** 2 * 3
        s = case["short"] / min(case["height"], case["width"])
        taps = (2 if case["resample"] == 0 else 4) * max(1.0, 1 / s)
        return {"bytes": src + 4.0 * dst, "flops": 2.0 * taps * dst * (1 + max(1.0, 1 / s))}
    cfg = _config(case)
    d, f, wb = cfg.embed_dim, cfg.ffn_dim, _WBYTES[case["ftype"]]
    if op == "head":
        n = case["tokens"]
        flops, weights = _blocks(n, 1, d, f, cfg.n_pool_layers)
        one_row = d * d + 2 * d * f + cfg.n_classes * d
        return {"bytes": wb * (weights + 2 * d * d + one_row) + 4.0 * (n * d + d + cfg.n_classes),
                "flops": flops + 4.0 * n * d * d + 2.0 * one_row + 4.0 * n * d}
    if op == "predict":
        n = case["context"] + case["target"]
        flops, weights = _blocks(n, 1, cfg.pred_dim, cfg.pred_ffn, cfg.pred_layers)
        return {"bytes": wb * (weights + 2 * d * cfg.pred_dim) + 4.0 * n * d, "flops": flops + 2.0 * n * d * cfg.pred_dim}
    rows_px = (case["height"] // cfg.patch) * (case["width"] // cfg.patch) * (case["frames"] // cfg.tubelet if case["frames"] > 1 else 1)
    prefix = (1 if cfg.cls_token else 0) + cfg.n_registers
    rows = case["batch"] * (rows_px + prefix)
    slots = case["frames"] if cfg.attn_mode == "block_causal" else 1
    flops, weights = _blocks(rows, case["batch"], d, f, cfg.n_layer, (slots + 1) / (2 * slots))
    kin = 3 * cfg.patch ** 2 * (cfg.tubelet if case["frames"] > 1 else 1)
    pixels = case["batch"] * 3 * case["frames"] * case["height"] * case["width"]
    return {"bytes": 4.0 * pixels + wb * weights + (4.0 if cfg.family in ("hfvit", "ijepa") else 2.0) * kin * d + 4.0 * rows * d,
            "flops": flops + 2.0 * case["batch"] * rows_px * kin * d}


def tolerance(case):
    if case["op"] == "frames":
        return "exact"          # integer resize, one division per value
    if case["ftype"] == "f16":
        return {"rel": 2e-3}    # 4e-4 to 6e-4 from the 64-bit result
    # A last-bit difference moves activation codes that sit on a rounding boundary, and each layer spreads it: two valid
    # orders of summation are 1e-2 apart after four layers and 1.6e-2 after 24, as either is from the 64-bit result.
    return {"rel": 0.03}


# ---- the same in 64 bits --------------------------------------------------------------------------------------

def _read_model(path):
    """name -> (ggml type, shape with the row length first, offset into the mapped file), and the file."""
    raw = np.memmap(path, dtype=np.uint8, mode="r")
    at = 0

    def take(fmt):
        nonlocal at
        v = struct.unpack_from("<" + fmt, raw, at)
        at += struct.calcsize("<" + fmt)
        return v[0] if len(v) == 1 else v

    def text():
        nonlocal at
        n = take("Q")
        at += n
        return bytes(raw[at - n:at]).decode()

    def value(kind):
        if kind == 8:
            return text()
        if kind == 9:
            inner, n = take("I"), take("Q")
            return [value(inner) for _ in range(n)]
        return take({0: "B", 1: "b", 2: "H", 3: "h", 4: "I", 5: "i", 6: "f", 7: "?", 10: "Q", 11: "q", 12: "d"}[kind])

    take("II")
    n_tensors, n_keys = take("Q"), take("Q")
    align = 32
    for _ in range(n_keys):
        key = text()
        v = value(take("I"))
        align = v if key == "general.alignment" else align
    infos = []
    for _ in range(n_tensors):
        name, nd = text(), take("I")
        shape = [take("Q") for _ in range(nd)]
        infos.append((name, take("I"), shape, take("Q")))
    base = (at + align - 1) // align * align
    return raw, {n: (t, s, base + o) for n, t, s, o in infos}


def _halves(b):
    return b.contiguous().view(torch.float16).double()


class _Weights:
    def __init__(self, path):
        self.raw, self.at = _read_model(path)

    def __contains__(self, name):
        return name in self.at

    def kind(self, name):
        return self.at[name][0]

    def __call__(self, name):
        """The tensor's values, float64 on the GPU, rows last dimension first of the file's shape."""
        kind, shape, off = self.at[name]
        n = int(np.prod(shape))
        block, size = {0: (1, 4), 1: (1, 2), 8: (32, 34), 2: (32, 18), 12: (256, 144)}[kind]
        b = torch.from_numpy(np.array(self.raw[off:off + n // block * size])).cuda()
        if kind == 0:
            v = b.view(torch.float32).double()
        elif kind == 1:
            v = _halves(b)
        else:
            b = b.view(-1, size)
            d = _halves(b[:, :2])
            if kind == 8:
                v = d * b[:, 2:].view(torch.int8).double()
            elif kind == 2:
                v = d * (torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8)
            else:
                sc, qs = b[:, 4:16].int(), b[:, 16:].view(-1, 4, 32)
                low, high = torch.arange(4), torch.arange(4, 8)
                s = torch.cat([sc[:, low] & 63, (sc[:, high + 4] & 15) | ((sc[:, low] >> 6) << 4)], 1).double()
                m = torch.cat([sc[:, high] & 63, (sc[:, high + 4] >> 4) | ((sc[:, high] >> 6) << 4)], 1).double()
                q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
                v = d[:, :, None] * s[:, :, None] * q - _halves(b[:, 2:4])[:, :, None] * m[:, :, None]
        return v.reshape(list(reversed(shape)))


def _input(x, kind):
    """What a weight of this type multiplies: the activations in its own format (blocks of 32 or 256, or f16)."""
    if kind == 0:
        return x
    if kind == 1:
        return x.half().double()
    if kind in (8, 2):
        v = x.reshape(-1, 32)
        top = v.abs().amax(1, keepdim=True)
        q = torch.where(top > 0, torch.round(v * (127.0 / top)), 0.0)
        return ((top / 127.0).half().double() * q).reshape(x.shape)
    v = x.reshape(-1, 256)
    top = v.gather(1, v.abs().argmax(1, keepdim=True))
    scale = -127.0 / top
    return torch.where(top != 0, torch.round(scale * v).clamp(max=127.0) / scale, 0.0).reshape(x.shape)


def _linear(w, name, x):
    y = _input(x, w.kind(name + ".weight")) @ w(name + ".weight").T
    return y + w(name + ".bias") if name + ".bias" in w else y


def _norm(w, name, x):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), w(name + ".weight"), w(name + ".bias"), 1e-6)


def _gelu(x):
    return torch.nn.functional.gelu(x)


def _rope(ids, grid, hd, interleaved, ref):
    """cos and sin [token, hd]: a third of the head (rounded to pairs) for each of t, h, w, the rest not turned."""
    gh, gw = grid
    d = 2 * ((hd // 3) // 2)
    half = d // 2
    pos = [ids // (gh * gw), ids % (gh * gw) // gw, ids % gw]
    pos = [p.double() for p in pos]
    if ref:
        pos[1] = pos[1] * ((ref - 1) / (gh - 1)) if gh > 1 else pos[1]
        pos[2] = pos[2] * ((ref - 1) / (gw - 1)) if gw > 1 else pos[2]
    j = torch.arange(d, device=ids.device)
    omega = 10000.0 ** -((j // 2 if interleaved else j % half).double() / half)
    ang = torch.cat([p[:, None] * omega for p in pos] + [torch.zeros(len(ids), hd - 3 * d, dtype=torch.float64, device=ids.device)], 1)
    return ang.cos(), ang.sin()


def _turn(x, cs):
    if cs is None:
        return x
    c, s = cs
    other = torch.stack([-x[..., 1::2], x[..., 0::2]], -1).flatten(-2)
    return x * c + other * s


def _block(w, p, x, heads, cs=None, mask=None):
    """One pre-LN block on x [sequences, tokens, width]; keys and values are kept in f16."""
    seqs, n, d = x.shape
    hd = d // heads
    qkv = _linear(w, p + "attn_qkv", _norm(w, p + "ln1", x)).view(seqs, n, 3, heads, hd)
    o = torch.empty(seqs, n, heads, hd, dtype=torch.float64, device=x.device)
    for b in range(seqs):
        for h in range(heads):
            q, k, v = (qkv[b, :, i, h].contiguous() for i in range(3))
            q, k, v = _turn(q, cs), _turn(k, cs).half().double(), v.half().double()
            s = q @ k.T.contiguous() / math.sqrt(hd)
            if mask is not None:
                s.masked_fill_(~mask, -math.inf)
            o[b, :, h] = s.softmax(-1) @ v
    x = x + _linear(w, p + "attn_out", o.view(seqs, n, d))
    return x + _linear(w, p + "ffn_down", _gelu(_linear(w, p + "ffn_up", _norm(w, p + "ln2", x))))


def _exact_encode(case, seed):
    cfg = _config(case)
    w = _Weights(_context(case)[1])
    x = _clip(case, seed).double()
    b, t, p = case["batch"], case["frames"], cfg.patch
    gh, gw = case["height"] // p, case["width"] // p
    image = cfg.family == "vjepa2_1" and t == 1
    tub = 1 if image or cfg.family in ("hfvit", "ijepa") else cfg.tubelet
    gt = t // tub
    x = x.view(b, 3, gt, tub, gh, p, gw, p).permute(0, 2, 4, 6, 1, 3, 5, 7).reshape(b, gt * gh * gw, -1)
    x = _linear(w, "enc.patch_embed_img" if image else "enc.patch_embed", x)
    if cfg.modality_embed:
        x = x + w("enc.mod_embed_img" if image else "enc.mod_embed_video")
    n_prefix = 1 if cfg.cls_token else 0
    if n_prefix:
        x = torch.cat([w("enc.cls_token").view(1, 1, -1).expand(b, 1, -1), x], 1)
    cs = mask = None
    if cfg.family in ("hfvit", "ijepa"):
        x = x + w("enc.pos_embed")
    else:
        ref = cfg.rope_ref_grid if cfg.rope_interpolate else 0
        cs = _rope(torch.arange(gt * gh * gw, device="cuda"), (gh, gw), cfg.embed_dim // cfg.n_head, cfg.rope_layout == "interleaved", ref)
        if n_prefix:
            cs = tuple(torch.cat([torch.full((1, v.shape[1]), one, dtype=torch.float64, device="cuda"), v]) for v, one in zip(cs, (1.0, 0.0)))
    if cfg.attn_mode == "block_causal":
        slot = torch.cat([torch.tensor([-1], device="cuda"), torch.arange(gt * gh * gw, device="cuda") // (gh * gw)])
        mask = (slot[:, None] < 0) | ((slot[None, :] >= 0) & (slot[None, :] <= slot[:, None]))
    for i in range(cfg.n_layer):
        x = _block(w, "enc.blk.%d." % i, x, cfg.n_head, cs, mask)
    return _norm(w, "enc.norm", x).view(-1, cfg.embed_dim)


def _exact_head(case, seed):
    cfg = _config(case)
    w = _Weights(_context(case)[1])
    d, heads = cfg.embed_dim, cfg.n_head
    x = _token_rows(case, seed, case["tokens"], d).double()[None]
    for i in range(cfg.n_pool_layers):
        x = _block(w, "head.blk.%d." % i, x, heads)
    kv = _norm(w, "head.xattn.ln_kv", x[0])
    k, v = (_linear(w, "head.xattn." + n, kv).view(-1, heads, d // heads) for n in "kv")
    q0 = w("head.query").view(1, d)
    q = _linear(w, "head.xattn.q", q0).view(heads, d // heads)
    a = ((k * q).sum(-1) / math.sqrt(d // heads)).softmax(0)
    y = (a[:, :, None] * v).sum(0).view(1, d) + q0
    y = y + _linear(w, "head.xattn.ffn_down", _gelu(_linear(w, "head.xattn.ffn_up", _norm(w, "head.xattn.ln2", y))))
    return [y[0], _linear(w, "head.cls", y)[0]]


def _exact_predict(case, seed):
    cfg = _config(case)
    w = _Weights(_context(case)[1])
    ctx, tgt = _ids(case, seed)
    rows = _token_rows(case, seed, 2048, cfg.embed_dim).double()
    ids = torch.from_numpy(np.concatenate([ctx, tgt])).cuda().long()
    x = _linear(w, "pred.embed", rows[ids[:len(ctx)]])
    x = torch.cat([x, w("pred.mask_tokens")[1].expand(len(tgt), -1)])[None]
    grid = cfg.img_size // cfg.patch
    cs = _rope(ids, (grid, grid), 32, False, 0)
    for i in range(cfg.pred_layers):
        x = _block(w, "pred.blk.%d." % i, x, cfg.pred_dim // 32, cs)
    return _linear(w, "pred.proj", _norm(w, "pred.norm", x[0, len(ctx):])).cpu().numpy()


def _exact_frames(case, seed):
    """torch's own uint8 antialiased resize on the CPU, centre crop, normalisation in 64 bits."""
    x = _pixels(seed, 1, case["frames"], case["height"], case["width"])[0].permute(1, 0, 2, 3).contiguous().cpu()
    h, w, short, crop = case["height"], case["width"], case["short"], case["crop"]
    rh, rw = (short * h // w, short) if w <= h else (short, short * w // h)
    x = torch.nn.functional.interpolate(x, size=(rh, rw), mode=("bilinear", "bicubic")[case["resample"]], antialias=True, align_corners=False)
    oy, ox = (rh - crop) // 2, (rw - crop) // 2
    x = x[:, :, oy:oy + crop, ox:ox + crop].double()
    mean, std = (torch.tensor(v, dtype=torch.float64).view(1, 3, 1, 1) for v in (MEAN, STD))
    return ((x / 255.0 - mean) / std).permute(1, 0, 2, 3).contiguous()


def exact(case, seed):
    out = {"encode": _exact_encode, "head": _exact_head, "predict": _exact_predict, "frames": _exact_frames}[case["op"]](case, seed)
    if case["op"] == "encode" and case["via"] == "host":
        out = out.cpu().numpy()
    return out
