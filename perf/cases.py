"""The work that the framework's speed is measured on: what a user's program
asks of it, through its public entry points, over the range of sizes, formats
and options in real use.

A case is a dict of plain values.  Its "kind" names the path:

  transcode   one .crn file to DXTn in device memory: begin, every level, end
              (an asset streamed in once)
  batch       one plan over many files' contexts (a scene's textures, or the
              copies of a frame loop), all levels in one run
  dxt1        plain DXT1 blocks of one image with the exact errors
  encode_set  plain encode of a set of textures with mip chains, mixed formats
  hc          dxt_hc: the clustered compressor behind .crn files
  qdxt        clustered DDS: qdxt1 for colour, qdxt5 for alpha
  mips        the mip chain of one image from a kept plan
  decode      DXTn blocks back to RGBA8
  learned     the learned DXT1 proposal with its fallback to the plain search
  train       one batch's loss and gradient of the proposal network

Everything but `train` gives whole numbers that have one right value.
"""
import ctypes as C
import math

import numpy as np
import torch

from crunch2_amd import crnd, dxt1, hc, learned, mips, qdxt, texture
from crunch2_amd._lib import (FMT_DXN_XY, FMT_DXT1, FMT_DXT5, FMT_DXT5A, EncodeItem, check, lib)
from crunch2_amd.train_learned import DEFAULT_OUT

FORMATS = {"dxt1": FMT_DXT1, "dxt5": FMT_DXT5, "dxt5a": FMT_DXT5A, "dxn": FMT_DXN_XY}
KINDS = {"dxt1": texture.RGB, "dxt5": texture.RGBA, "dxt5a": texture.RGBA, "dxn": texture.NORMAL}
FILTERS = {"box": mips.BOX, "tent": mips.TENT, "lanczos4": mips.LANCZOS4, "mitchell": mips.MITCHELL,
           "kaiser": mips.KAISER}
# colour distances that the uber search evaluates per block (the reference
# search, averaged over textures) and the integer operations of one
SEARCH_OPS_PER_BLOCK = 11200 * 9


def listed():
    return [
        # the smallest asset: launches, host work and latency are all there is
        {"name": "transcode_dxt1_256", "kind": "transcode", "format": "dxt1", "width": 256, "height": 256, "faces": 1},
        # an ordinary full-size texture with alpha, streamed in
        {"name": "transcode_dxt5_2048", "kind": "transcode", "format": "dxt5", "width": 2048, "height": 2048,
         "faces": 1},
        # a scene's textures in one plan: 8 files of mixed formats and sizes, 8 instances of each
        {"name": "transcode_batch_64", "kind": "batch", "files": 8, "copies": 8, "low": 64, "high": 1024},
        # one small texture encoded while an artist waits
        {"name": "dxt1_image_256", "kind": "dxt1", "width": 256, "height": 256, "quality": 4, "alpha_blocks": True},
        # a build farm's step: odd-sized textures with mips, DXT1 / DXT5 / DXN
        {"name": "encode_set_16", "kind": "encode_set", "files": 16, "low": 64, "high": 1024},
        # .crn of an opaque texture at quality 128
        {"name": "hc_dxt1_2048", "kind": "hc", "format": "dxt1", "width": 2048, "height": 2048, "perceptual": True},
        # .crn of a texture with alpha
        {"name": "hc_dxt5_1024", "kind": "hc", "format": "dxt5", "width": 1024, "height": 1024, "perceptual": True},
        # clustered DDS of a texture with alpha
        {"name": "qdxt_dxt5_1024", "kind": "qdxt", "width": 1024, "height": 1024, "quality": 128},
        # crunch's default mip chain of a large image that is no power of two
        {"name": "mips_3840x2160", "kind": "mips", "width": 3840, "height": 2160, "filter": "kaiser", "wrap": False,
         "normal": False},
        # a ragged level decoded for display or for an error metric
        {"name": "decode_dxt5_2047x1533", "kind": "decode", "format": "dxt5", "width": 2047, "height": 1533},
        # the fast encoder on a full-size texture
        {"name": "learned_2048", "kind": "learned", "width": 2048, "height": 2048, "percent": 8},
        # one batch of training the proposal network
        {"name": "train_32768", "kind": "train", "batch": 32768},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_size(rng, lo, hi):
    """A texture's sides: often square powers of two, else anything."""
    w = _log_int(rng, lo, hi)
    if rng.random() < 0.35:
        w = 1 << int(round(math.log2(w)))
        w = min(max(w, lo), hi)
        return w, w
    return w, min(max(int(w * math.exp(rng.uniform(-0.7, 0.7))), lo), hi)


def draw(rng):
    kind = rng.choice(["transcode", "transcode", "batch", "dxt1", "encode_set", "hc", "hc", "qdxt", "mips", "mips",
                       "decode", "learned", "train"])
    c = {"kind": kind}
    if kind == "transcode":
        w, h = _draw_size(rng, 64, 2048)
        faces = 6 if max(w, h) <= 512 and rng.random() < 0.2 else 1
        if faces == 6:
            h = w
        c.update(format=rng.choice(["dxt1", "dxt1", "dxt5", "dxn", "dxt5a"]), width=w, height=h, faces=faces)
    elif kind == "batch":
        c.update(files=rng.randint(2, 8), copies=rng.randint(1, 8), low=64, high=_log_int(rng, 128, 1024))
    elif kind == "dxt1":
        w, h = _draw_size(rng, 64, 2048)
        c.update(width=w, height=h, quality=rng.choice([4, 4, 3, 2, 1]), alpha_blocks=rng.random() < 0.6)
    elif kind == "encode_set":
        c.update(files=rng.randint(2, 16), low=32, high=_log_int(rng, 64, 1024))
    elif kind == "hc":
        fmt = rng.choice(["dxt1", "dxt1", "dxt5", "dxn"])
        w, h = _draw_size(rng, 128, 2048 if fmt == "dxt1" else 1024)
        c.update(format=fmt, width=w, height=h, perceptual=fmt != "dxn" and rng.random() < 0.8)
    elif kind == "qdxt":
        w, h = _draw_size(rng, 128, 1024)
        c.update(width=w, height=h, quality=rng.randint(40, 200))
    elif kind == "mips":
        w, h = _draw_size(rng, 100, 2880)
        normal = rng.random() < 0.25
        c.update(width=w, height=h, filter=rng.choice(["kaiser", "kaiser", "box", "tent", "lanczos4", "mitchell"]),
                 wrap=rng.random() < 0.3, normal=normal)
    elif kind == "decode":
        w, h = _draw_size(rng, 64, 2048)
        c.update(format=rng.choice(["dxt1", "dxt5", "dxn", "dxt5a"]), width=w, height=h)
    elif kind == "learned":
        w, h = _draw_size(rng, 64, 2048)
        c.update(width=w, height=h, percent=rng.choice([0, 4, 8, 16]))
    else:
        c.update(batch=_log_int(rng, 1000, 65536))
    return c


# ---------------------------------------------------------------- inputs
def _set_textures(case, seed, formats):
    """The set's (format, side, seed): sides log-uniform, shares as in the
    serving-style set (60 % colour, 25 % colour with alpha, 15 % normal maps).
    The first texture has the largest side.  The sides belong to the case, the
    images to the seed."""
    rng = np.random.default_rng([case["files"], case["low"], case["high"]])
    out = []
    for i in range(case["files"]):
        side = int(round(math.exp(rng.uniform(math.log(case["low"]), math.log(case["high"])))))
        u = rng.random()
        fmt = "dxt1" if u < 0.60 else ("dxt5" if u < 0.85 else "dxn")
        out.append((fmt if i >= len(formats) else formats[i], case["high"] if i == 0 else side, seed * 1000 + i))
    return out


def _chain(w, h, seed, fmt):
    return texture.mip_chain(texture.synth(w, h, seed, KINDS[fmt]))


def _crn(w, h, seed, fmt, faces=1):
    """A .crn of the clustered compressor at crnlib's quality-128 palette sizes."""
    levels = [_chain(w, h, seed + 7919 * f, fmt) for f in range(faces)]
    return texture.compress_hc(levels, FORMATS[fmt], texture.q128_palette_sizes(w, h, FORMATS[fmt]))


def _even_blocks(levels):
    """The pixel blocks of every level on its even-padded grid (edge texels
    repeated) and the (first, count, width, weight) of each level."""
    blocks, desc, first = [], [], 0
    for img in levels:
        h, w = img.shape[:2]
        ys = np.minimum(np.arange((h + 7) // 8 * 8), h - 1)
        xs = np.minimum(np.arange((w + 7) // 8 * 8), w - 1)
        b = dxt1.image_blocks(img[ys][:, xs])
        blocks.append(b)
        desc.append((first, len(b), len(xs) // 4, min(12.0, 1.3 ** len(desc))))
        first += len(b)
    return np.concatenate(blocks), desc


class _Batch:
    """A transcode plan over many contexts and the buffer it writes."""

    def __init__(self, files, copies):
        self.ctxs = [crnd.unpack_begin(d) for _ in range(copies) for d in files]
        sizes = [crnd.levels_size(c, 0, _levels(c)) for c in self.ctxs]
        ofs = np.concatenate([[0], np.cumsum([(s + 255) // 256 * 256 for s in sizes])])
        self.out = torch.zeros(int(ofs[-1]), dtype=torch.uint8, device="cuda")
        n = len(self.ctxs)
        self.plan = C.c_void_p()
        base = self.out.data_ptr()
        check(lib().crn2_batch_create((C.c_void_p * n)(*[c.handle for c in self.ctxs]), n,
                                      (C.c_void_p * n)(*[base + int(o) for o in ofs[:-1]]),
                                      (C.c_uint64 * n)(*sizes), C.byref(self.plan)), "crn2_batch_create")

    def run(self):
        check(lib().crn2_batch_run(self.plan, C.c_void_p(torch.cuda.current_stream().cuda_stream)), "crn2_batch_run")
        return self.out

    def __del__(self):
        torch.cuda.synchronize()
        lib().crn2_batch_destroy(self.plan)
        for c in self.ctxs:
            crnd.unpack_end(c)


class _EncodeSet:
    """The level images of a set of textures and the encoder over them."""

    def __init__(self, chains, fmts):
        self.src, items, ofs = [], [], 0
        for chain, fmt in zip(chains, fmts):
            for lv in chain:
                h, w = lv.shape[:2]
                self.src.append(torch.from_numpy(np.ascontiguousarray(lv).reshape(-1)).cuda())
                items.append((self.src[-1].data_ptr(), w, h, FORMATS[fmt], ofs))
                ofs += ((w + 3) // 4) * ((h + 3) // 4) * (8 if fmt in ("dxt1", "dxt5a") else 16)
        self.out = torch.zeros(ofs, dtype=torch.uint8, device="cuda")
        base = self.out.data_ptr()
        arr = (EncodeItem * len(items))(*[EncodeItem(p, w, h, f, base + o) for p, w, h, f, o in items])
        self.set = C.c_void_p()
        check(lib().crn2_encode_set_create(arr, len(items), dxt1.UBER, 1 | 2, C.byref(self.set)),
              "crn2_encode_set_create")

    def run(self):
        check(lib().crn2_encode_set_run(self.set, C.c_void_p(torch.cuda.current_stream().cuda_stream)),
              "crn2_encode_set_run")
        return self.out

    def __del__(self):
        torch.cuda.synchronize()
        lib().crn2_encode_set_destroy(self.set)


def _levels(ctx):
    return crnd.get_texture_info(ctx._keep)["levels"]


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "transcode":
        s["data"] = _crn(case["width"], case["height"], seed, case["format"], case["faces"])
        s["levels"] = crnd.get_texture_info(s["data"])["levels"]
    elif kind == "batch":
        s["batch"] = _Batch([_crn(side, side, sd, fmt)
                             for fmt, side, sd in _set_textures(case, seed, ["dxt5", "dxt1", "dxn"])], case["copies"])
    elif kind == "dxt1":
        s["img"] = torch.from_numpy(texture.synth(case["width"], case["height"], seed, texture.RGB)).cuda()
    elif kind == "encode_set":
        tex = _set_textures(case, seed, ["dxt1", "dxt5", "dxn"])
        s["set"] = _EncodeSet([_chain(side, side, sd, fmt) for fmt, side, sd in tex], [t[0] for t in tex])
    elif kind == "hc":
        blocks, s["desc"] = _even_blocks(_chain(case["width"], case["height"], seed, case["format"]))
        s["blocks"] = torch.from_numpy(blocks).cuda()
        s["sizes"] = tuple(max(8, v) for v in texture.q128_palette_sizes(case["width"], case["height"],
                                                                         FORMATS[case["format"]]))
        # palettes of the sizes asked for (the compressor may need fewer entries)
        s["palettes"] = [torch.zeros(n, dtype=torch.int64, device="cuda") for n in s["sizes"]]
    elif kind == "qdxt":
        blocks, s["desc"] = qdxt.level_blocks(_chain(case["width"], case["height"], seed, "dxt5"))
        s["blocks"] = torch.from_numpy(blocks).cuda()
    elif kind == "mips":
        img = texture.synth(case["width"], case["height"], seed, texture.NORMAL if case["normal"] else texture.RGBA)
        s["img"] = torch.from_numpy(img).cuda()
        flags = (mips.RENORMALIZE if case["normal"] else mips.SRGB | mips.ALPHA) | (mips.WRAP if case["wrap"] else 0)
        s["plan"] = mips.Plan(case["width"], case["height"], mips.params(FILTERS[case["filter"]], flags))
    elif kind == "decode":
        w, h, fmt = case["width"], case["height"], case["format"]
        img = torch.from_numpy(texture.synth(w, h, seed, KINDS[fmt])).cuda()
        bpb = 8 if fmt in ("dxt1", "dxt5a") else 16
        s["blocks"] = torch.zeros(((w + 3) // 4) * ((h + 3) // 4) * bpb, dtype=torch.uint8, device="cuda")
        check(lib().crn2_encode_image_device(img.data_ptr(), w, h, FORMATS[fmt], dxt1.FAST, 1 | 2,
                                             s["blocks"].data_ptr(),
                                             C.c_void_p(torch.cuda.current_stream().cuda_stream)),
              "crn2_encode_image_device")
        s["rgba"] = torch.zeros((h, w, 4), dtype=torch.uint8, device="cuda")
    elif kind == "learned":
        img = texture.synth(case["width"], case["height"], seed, texture.RGB)
        s["blocks"] = torch.from_numpy(dxt1.image_blocks(img)).cuda()
        s["theta"] = torch.from_numpy(np.load(DEFAULT_OUT)).cuda()
    else:
        n = case["batch"]
        side = int(math.ceil(math.sqrt(n))) * 4
        blocks = torch.from_numpy(dxt1.image_blocks(texture.synth(side, side, seed, texture.RGB))[:n]).cuda()
        s["X"] = learned.features(blocks)
        s["T"] = learned.plain_targets(blocks, dxt1.FAST)[0]
        s["trainer"] = learned.Trainer(seed=seed)
    return s


# ------------------------------------------------------------------- run
def run(s):
    case = s["case"]
    kind = case["kind"]
    st = torch.cuda.current_stream().cuda_stream
    if kind == "transcode":
        ctx = crnd.unpack_begin(s["data"])
        n = crnd.levels_size(ctx, 0, s["levels"])
        out = torch.empty(n, dtype=torch.uint8, device="cuda")
        crnd.unpack_levels_device(ctx, out.data_ptr(), n, 0, s["levels"], st)
        crnd.unpack_end(ctx)
        return out
    if kind == "batch":
        return s["batch"].run()
    if kind == "dxt1":
        n = ((case["width"] + 3) // 4) * ((case["height"] + 3) // 4)
        out = torch.empty(n, dtype=torch.int64, device="cuda")
        err = torch.empty(n, dtype=torch.int64, device="cuda")
        flags = dxt1.PERCEPTUAL | (dxt1.ALPHA_BLOCKS if case["alpha_blocks"] else 0)
        check(lib().crn2_encode_dxt1_image_device(s["img"].data_ptr(), case["width"], case["height"], case["quality"],
                                                  flags, out.data_ptr(), 1, err.data_ptr(), C.c_void_p(st)),
              "crn2_encode_dxt1_image_device")
        return out, err
    if kind == "encode_set":
        return s["set"].run()
    if kind == "hc":
        fmt = case["format"]
        got = hc.compress(s["blocks"], s["desc"], has_color=fmt != "dxn",
                          alpha_comp={"dxt1": (), "dxt5": (3,), "dxn": (0, 1)}[fmt], perceptual=case["perceptual"],
                          codebook_sizes=s["sizes"])
        for pal, p in zip(s["palettes"], got[2:]):
            if p is not None:
                pal[:p.shape[0]] = p
                pal[p.shape[0]:] = 0
        return got[0], got[1], s["palettes"]
    if kind == "qdxt":
        color = qdxt.Qdxt1(s["blocks"], s["desc"])
        c = color.pack(qdxt.params(case["quality"]), pow_mul=0.75)
        color.close()
        alpha = qdxt.Qdxt5(s["blocks"], s["desc"], 3)
        a = alpha.pack(qdxt.params5(case["quality"]))
        alpha.close()
        return c, a
    if kind == "mips":
        return s["plan"].run(s["img"])
    if kind == "decode":
        check(lib().crn2_decode_dxt_device(s["blocks"].data_ptr(), FORMATS[case["format"]], case["width"],
                                           case["height"], 0, s["rgba"].data_ptr(), 0, C.c_void_p(st)),
              "crn2_decode_dxt_device")
        return s["rgba"]
    if kind == "learned":
        return learned.encode(s["theta"], s["blocks"], fallback_frac=case["percent"] / 100.0)
    loss, grad = s["trainer"].gradients(s["X"], s["T"])
    return loss, grad


# ------------------------------------------------------ what a pass needs
def _texture_blocks(w, h, levels=None):
    n, l = 0, 0
    while True:
        n += ((max(1, w >> l) + 3) // 4) * ((max(1, h >> l) + 3) // 4)
        l += 1
        if l == levels or (not levels and max(w, h) >> l == 0):
            return n


def work(case):
    """Inputs read once, outputs written once; operations that no form of the
    path can leave out (the search's and the filters' arithmetic)."""
    kind = case["kind"]
    if kind in ("transcode", "batch", "encode_set"):
        if kind == "transcode":
            blocks = _texture_blocks(case["width"], case["height"]) * case["faces"]
            bpb = 8 if case["format"] in ("dxt1", "dxt5a") else 16
            # about 1.2 (one channel) and 2.4 bits per texel in the file
            return {"bytes": blocks * (bpb + 0.3 * bpb), "flops": 0}
        # the mean area of log-uniform sides, and the one largest texture
        lo, hi = case["low"], case["high"]
        mean = (hi * hi - lo * lo) / (2 * math.log(hi / lo)) if hi > lo else hi * hi
        blocks = (mean * (case["files"] - 1) + hi * hi) / 16 * 4 / 3
        if kind == "batch":
            return {"bytes": blocks * case["copies"] * 11.2 * 1.3, "flops": 0}
        return {"bytes": blocks * (64 + 11.2), "flops": blocks * SEARCH_OPS_PER_BLOCK}
    if kind == "dxt1":
        blocks = _texture_blocks(case["width"], case["height"], 1)
        share = {4: 1.0, 3: 0.55, 2: 0.3, 1: 0.2, 0: 0.15}[case["quality"]]
        return {"bytes": blocks * (64 + 16), "flops": blocks * SEARCH_OPS_PER_BLOCK * share}
    if kind == "hc":
        fmt = FORMATS[case["format"]]
        blocks = _texture_blocks(case["width"], case["height"])
        sizes = texture.q128_palette_sizes(case["width"], case["height"], fmt)
        ops = 0
        if case["format"] != "dxn":
            ops += 2 * blocks * sizes[1] * 64
        ops += 2 * blocks * sizes[3] * 128 * {"dxt1": 0, "dxt5": 1, "dxn": 2}[case["format"]]
        return {"bytes": blocks * (64 + 14), "flops": ops}
    if kind == "qdxt":
        blocks = _texture_blocks(case["width"], case["height"])
        # each tree level passes over the training vectors of 2, 6 and 16 floats
        return {"bytes": blocks * (64 + 16), "flops": 2 * blocks * 15 * (2 * 2 + 6 * 6 + 16 * 16)}
    if kind == "mips":
        w, h = case["width"], case["height"]
        levels = int(math.log2(max(w, h))) + 1
        taps = {"box": 1, "tent": 2, "mitchell": 4, "kaiser": 6, "lanczos4": 8}[case["filter"]] * 0.9
        comps = 3 if case["normal"] else 4
        return {"bytes": w * h * 4 + w * h * 4 / 3, "flops": 2 * comps * w * h * max(1, levels - 1) * max(1.0, taps)}
    if kind == "decode":
        blocks = _texture_blocks(case["width"], case["height"], 1)
        return {"bytes": blocks * (8 if case["format"] in ("dxt1", "dxt5a") else 16) + case["width"] * case["height"] * 4,
                "flops": 0}
    if kind == "learned":
        blocks = _texture_blocks(case["width"], case["height"], 1)
        net = 2 * (57 * 128 + 128 * 128 + 128 * 7)
        return {"bytes": blocks * (64 + 12),
                "flops": blocks * (net + SEARCH_OPS_PER_BLOCK * case["percent"] / 100.0 + 3 * 12 * 16 * 4 * 9)}
    n = case["batch"]
    net = 57 * 128 + 128 * 128 + 128 * 7
    return {"bytes": n * (57 + 6) * 4 + 2 * 4 * learned.N_PARAMS, "flops": n * (6 * net - 2 * 57 * 128)}


def tolerance(case):
    if case["kind"] == "train":
        # layer inputs are rounded to bfloat16: a sum in another order moves a
        # few of them by one step
        return {"rel": 1e-5, "max": 1e-4}
    return "exact"


def exact(case, seed):
    if case["kind"] != "train":
        return None
    s = prepare(case, seed)
    f8 = torch.float64

    def bf(t):
        return t.to(torch.float32).to(torch.bfloat16).to(f8)
    theta = s["trainer"].theta.cpu()
    p, o = {}, 0
    for name, shp in learned.SHAPES:
        k = int(np.prod(shp))
        p[name] = theta[o:o + k].reshape(shp).to(f8)
        o += k
    w1, w2, w3 = (bf(p[k]) for k in ("W1", "W2", "W3"))
    x, t = bf(s["X"].cpu()), s["T"].cpu().to(f8)
    n = x.shape[0]
    gc, ga = float(np.float32(0.7978845608028654)), float(np.float32(0.044715))

    def gelu(z):
        return 0.5 * z * (1.0 + torch.tanh(gc * (z + ga * z ** 3)))

    def gelu_grad(z):
        th = torch.tanh(gc * (z + ga * z ** 3))
        return 0.5 * (1.0 + th) + 0.5 * z * (1.0 - th * th) * gc * (1.0 + 3.0 * ga * z * z)
    z1 = x @ w1 + p["b1"]
    a1 = bf(gelu(z1))
    z2 = a1 @ w2 + p["b2"]
    a2 = bf(gelu(z2))
    y = a2 @ w3 + p["b3"]
    scale = torch.tensor([31.0, 63.0, 31.0, 31.0, 63.0, 31.0], dtype=f8)
    q = torch.minimum(torch.clamp(torch.round(y[:, :6] * scale), min=0.0), scale)
    lab = ((q - torch.round(t * scale)).abs() <= 1.0).all(1).to(f8)
    d, z = y[:, :6] - t, y[:, 6]
    loss = (d * d).sum() / n + 0.05 * (torch.nn.functional.softplus(z) - lab * z).sum() / n
    dy = torch.cat([2.0 / n * d, (0.05 / n * (torch.sigmoid(z) - lab))[:, None]], 1)
    dz2 = (dy @ w3.T) * gelu_grad(z2)
    dz1 = (dz2 @ w2.T) * gelu_grad(z1)
    grad = torch.cat([(x.T @ dz1).reshape(-1), dz1.sum(0), (a1.T @ dz2).reshape(-1), dz2.sum(0),
                      (a2.T @ dy).reshape(-1), dy.sum(0)])
    return loss.reshape(1), grad
