"""The work this framework is used for, as cases that can be timed and compared.

Every case goes through the public entry points of `cudacompress_amd` with the inputs of the
repository's configurations: turbulence-like fields (energy spectrum k^-5/3), fractional Brownian
heightfields, byte images, sparse Laplace symbol streams.  Volumes and coder calls that hand their
bitstream to the host do so here too; batches, plans, servers and the device coder keep it on the
device.  Coefficients are quantized, so a bitstream stays the same only while every transform keeps
its rounding: bitstreams, symbols, bytes and integers compare exactly.

A case is {"name", "kind", ...sizes and options of the kind}:
  volume    compressVolumeFloat and / or decompressVolumeFloat of one volume ("way")
  channels  decompressVolumeFloatMultiChannel of a vector field
  lossless  compressVolumeLossless + decompressVolumeLossless of int16 data, 2D (sz 1) or 3D
  short     compressVolumeFloatQuantFirst + decompressVolumeFloatQuantFirst
  dwt       multi-level dwtFloat3DForward, then dwtFloat3DInverse
  image     RGB bytes -> YCoCg -> 9/7 -> symbols per channel, and back to RGB bytes
  coder     encodeDevice + decodeDevice of symbol streams
  bricks    compressBricksFloat + decompressBricksFloat of bricks of mixed sizes
  plan      BricksPlan.run on bricks of mixed sizes
  serve     Server.run on decode requests over resident bricks
"""
import random

import numpy as np
import torch

import cudacompress_amd as cc

BRICK_AXES = (16, 32, 48, 64, 96, 128)


def listed():
    return [
        # one small brick through the plain calls: launches, synchronisations and host work
        {"name": "volume_32", "kind": "volume", "way": "both", "sx": 32, "sy": 32, "sz": 32, "levels": 2, "step": 0.01,
         "log2": 14, "block": 128, "lvl0": False},
        # the 128^3 configuration, written out to a host bitstream
        {"name": "volume_128", "kind": "volume", "way": "compress", "sx": 128, "sy": 128, "sz": 128, "levels": 2,
         "step": 0.01, "log2": 14, "block": 128, "lvl0": False},
        # loading a three-component vector field with sides that are no powers of two
        {"name": "channels_3", "kind": "channels", "channels": 3, "sx": 112, "sy": 96, "sz": 136, "levels": 3,
         "step": 0.01, "log2": 16, "block": 128, "lvl0": False},
        # the 4096^2 terrain configuration, lossless, there and back
        {"name": "lossless_4096", "kind": "lossless", "sx": 4096, "sy": 4096, "sz": 1, "levels": 3, "block": 128},
        # quantize first, integer wavelet, ragged sides
        {"name": "short_120", "kind": "short", "sx": 120, "sy": 88, "sz": 104, "levels": 3, "step": 0.01, "log2": 14,
         "block": 128},
        # one velocity component of the 256^3 configuration through the transforms alone
        {"name": "dwt_256", "kind": "dwt", "sx": 256, "sy": 256, "sz": 256, "levels": 3},
        # a full HD frame through the image path, there and back
        {"name": "image_1080", "kind": "image", "sx": 1920, "sy": 1080, "step": 2.0},
        # a caller's own symbols through the device-resident coder; an odd count, so no stream is aligned with the next
        {"name": "coder_3x", "kind": "coder", "streams": 3, "n": 700001, "rl": True, "log2": 14, "block": 128,
         "scale": 6.0, "density": 0.4},
        # a handful of bricks without a plan, as an importer codes them
        {"name": "bricks_64", "kind": "bricks", "count": 64, "axes_seed": 4, "levels": 2, "step": 0.005, "log2": 14,
         "block": 64},
        # the whole 2048-brick configuration as a captured plan
        {"name": "plan_2048", "kind": "plan", "count": 2048, "axes_seed": 4, "levels": 2, "step": 0.005, "log2": 14,
         "block": 64},
        # a viewer that waits for one brick
        {"name": "serve_1", "kind": "serve", "bricks": 64, "requests": 1, "most": 1, "trace_seed": 1, "block": 64},
        # a burst of requests of 1 to 64 bricks, half of them of the coarser level
        {"name": "serve_32", "kind": "serve", "bricks": 64, "requests": 32, "most": 64, "trace_seed": 2, "block": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _sides(rng, levels, lo, hi):
    f = 1 << levels
    return [max(f, f * round(_log_int(rng, lo, hi) / f)) for _ in range(3)]


def draw(rng):
    kind = rng.choice(("volume", "volume", "channels", "lossless", "short", "dwt", "image", "coder", "bricks", "plan",
                       "plan", "serve"))
    block = rng.choice((32, 64, 128, 256))
    c = {"kind": kind}
    if kind in ("volume", "channels", "short"):
        levels = rng.choice((1, 2, 3))
        sx, sy, sz = _sides(rng, levels, 16, 160)
        c.update(sx=sx, sy=sy, sz=sz, levels=levels, step=0.002 * 10 ** rng.random(), log2=rng.choice((14, 16)),
                 block=block)
        if kind == "volume":
            c.update(way=rng.choice(("compress", "decompress", "both")), lvl0=rng.random() < 0.25)
        if kind == "channels":
            c.update(channels=rng.choice((2, 3, 4)), lvl0=rng.random() < 0.25)
    elif kind == "lossless":
        levels = rng.choice((1, 2, 3))
        if rng.random() < 0.7:
            f = 1 << levels
            c.update(sx=f * _log_int(rng, 16, 4096 // f), sy=f * _log_int(rng, 16, 4096 // f), sz=1)
        else:
            sx, sy, sz = _sides(rng, levels, 16, 192)
            c.update(sx=sx, sy=sy, sz=sz)
        c.update(levels=levels, block=block)
    elif kind == "dwt":
        levels = rng.choice((1, 2, 3))
        sx, sy, sz = _sides(rng, levels, 16, 320)
        c.update(sx=sx, sy=sy, sz=sz, levels=levels)
    elif kind == "image":
        c.update(sx=4 * _log_int(rng, 16, 960), sy=4 * _log_int(rng, 16, 540), step=0.5 * 16 ** rng.random())
    elif kind == "coder":
        c.update(streams=rng.choice((1, 3, 7)), n=_log_int(rng, 1000, 1500000), rl=rng.random() < 0.7,
                 log2=rng.choice((14, 14, 16, 20)), block=block, scale=2.0 * 20 ** rng.random(),
                 density=0.1 * 9 ** rng.random())
    elif kind in ("bricks", "plan"):
        c.update(count=_log_int(rng, 1, 128) if kind == "bricks" else _log_int(rng, 16, 1024),
                 axes_seed=rng.randrange(1 << 20), levels=rng.choice((1, 2, 2, 3)), step=0.002 * 10 ** rng.random(),
                 log2=rng.choice((14, 16)), block=block)
    else:
        c.update(bricks=_log_int(rng, 4, 96), requests=_log_int(rng, 1, 40), most=_log_int(rng, 1, 64),
                 trace_seed=rng.randrange(1 << 20), block=rng.choice((64, 128)))
    return c


# ------------------------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _spectral(shape, exponent, seed):
    """Gaussian noise whose modes fall off as k^exponent, zero mean, unit deviation."""
    spec = torch.fft.rfftn(torch.randn(shape, generator=_generator(seed), device="cuda"))
    k2 = 0
    for a, n in enumerate(shape):
        f = (torch.fft.rfftfreq if a == len(shape) - 1 else torch.fft.fftfreq)(n, d=1.0 / n, device="cuda")
        view = [1] * len(shape)
        view[a] = -1
        k2 = k2 + f.view(view) ** 2
    spec *= torch.where(k2 > 0, k2.clamp_min(1e-30) ** (exponent / 2), torch.zeros_like(k2))
    f = torch.fft.irfftn(spec, s=shape)
    return (f - f.mean()) / f.std()


def _field(sz, sy, sx, seed):
    """A turbulence-like box: cut from a cube of energy spectrum k^-5/3."""
    n = 1 << (max(sx, sy, sz) - 1).bit_length()
    return _spectral((n, n, n), -11.0 / 6.0, seed)[:sz, :sy, :sx].contiguous()


def _shapes(case):
    """(z, y, x) of the bricks, the same for every seed."""
    rng = random.Random(case["axes_seed"])
    return [tuple(rng.choice(BRICK_AXES) for _ in range(3)) for _ in range(case["count"])]


def _packed(shapes):
    """One buffer and a view of it for every brick, each from a multiple of 64 elements on."""
    at, n = [], 0
    for s in shapes:
        at.append(n)
        n += -(-s[0] * s[1] * s[2] // 64) * 64
    buf = torch.zeros(n, device="cuda")
    return buf, [buf[o:o + s[0] * s[1] * s[2]].view(s) for o, s in zip(at, shapes)]


def _cut(field, shapes, views, seed):
    rng = random.Random(seed)
    n = field.shape[0]
    for s, v in zip(shapes, views):
        z, y, x = (rng.randint(0, n - d) for d in s)
        v.copy_(field[z:z + s[0], y:y + s[1], x:x + s[2]])


def _brick_inputs(case, seed):
    shapes = _shapes(case)
    src, srcs = _packed(shapes)
    _cut(_spectral((256, 256, 256), -11.0 / 6.0, seed), shapes, srcs, seed)
    stds = torch.stack([s.std() for s in srcs]).tolist()
    return shapes, src, srcs, [float(np.float32(case["step"] * s)) for s in stds]


def _serve_shapes(case):
    """Bricks of the full level (128^3), then as many of the level of detail (64^3)."""
    n = -(-case["bricks"] // 2)
    return [(128, 128, 128)] * n + [(64, 64, 64)] * n


def _trace(case):
    rng = random.Random(case["trace_seed"])
    n = -(-case["bricks"] // 2)
    return [[rng.randrange(n) + n * rng.randrange(2) for _ in range(rng.randint(1, case["most"]))]
            for _ in range(case["requests"])]


def _rgb(sy, sx, seed):
    """A byte image: three correlated smooth channels with a little noise."""
    n = 1 << (max(sx, sy) - 1).bit_length()
    grey = _spectral((n, n), -1.6, seed)[:sy, :sx]
    tint = _spectral((3, n, n), -1.8, seed + 1)[:, :sy, :sx]
    v = 128 + 45 * grey + 15 * tint + 2 * torch.randn((3, sy, sx), generator=_generator(seed + 2), device="cuda")
    return v.clamp(0, 255).to(torch.uint8).permute(1, 2, 0).contiguous()


def _file(elems):
    """Room for a bitstream on the host, as a caller's container or file buffer."""
    return np.zeros(elems + 65536, dtype=np.int32)


def _store(file, words):
    file[:words.size] = words.view(np.int32)
    return file


def _levels_of(case):
    """Divisor of the sides at every level."""
    return [1 << level for level in range(case["levels"])]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("volume", "channels", "short", "lossless", "dwt"):
        sx, sy, sz, levels = case["sx"], case["sy"], case["sz"], case["levels"]
        elems = sx * sy * sz
    if kind == "volume":
        src = _field(sz, sy, sx, seed)
        inst = cc.createInstance(0, 7, elems // 8, case["block"], case["log2"])
        words = None
        if case["way"] == "decompress":
            words = cc.compressVolumeFloat(inst, src, sx, sy, sz, levels, case["step"], case["lvl0"])
        return {"case": case, "inst": inst, "src": src, "rec": torch.empty_like(src), "words": words,
                "file": _file(elems)}
    if kind == "channels":
        inst = cc.createInstance(0, 7 * case["channels"], elems // 8, case["block"], case["log2"])
        channels = []
        for i in range(case["channels"]):
            src = _field(sz, sy, sx, seed * 8 + i)
            words = cc.compressVolumeFloat(inst, src, sx, sy, sz, levels, case["step"], case["lvl0"])
            channels.append((torch.empty_like(src), words, case["step"]))
        return {"case": case, "inst": inst, "channels": channels}
    if kind == "short":
        inst = cc.createInstance(0, 7, elems // 8, case["block"], case["log2"])
        src = _field(sz, sy, sx, seed)
        return {"case": case, "inst": inst, "src": src, "rec": torch.empty_like(src), "file": _file(elems)}
    if kind == "lossless":
        shape = (sy, sx) if sz == 1 else (sz, sy, sx)
        n = 1 << (max(shape) - 1).bit_length()
        h = _spectral((n,) * len(shape), -1.8 if sz == 1 else -11.0 / 6.0, seed)[tuple(slice(0, s) for s in shape)]
        lo, hi = h.amin(), h.amax()
        src = (torch.round((h - lo) / (hi - lo) * 65535.0) - 32768).to(torch.int16).contiguous()
        inst = cc.createInstance(0, 3 if sz == 1 else 7, elems // (4 if sz == 1 else 8), case["block"], 16)
        return {"case": case, "inst": inst, "src": src, "rec": torch.empty_like(src), "file": _file(elems)}
    if kind == "dwt":
        src = _field(sz, sy, sx, seed)
        return {"case": case, "src": src, "coef": torch.empty_like(src), "rec": torch.empty_like(src),
                "b1": torch.empty_like(src), "b2": torch.empty_like(src)}
    if kind == "image":
        sx, sy = case["sx"], case["sy"]
        rgb = _rgb(sy, sx, seed)
        planes = torch.empty((3, sy, sx), device="cuda")
        sym1 = torch.empty((3, 3, sy // 2, sx // 2), dtype=torch.int16, device="cuda")
        sym2 = torch.empty((3, 4, sy // 4, sx // 4), dtype=torch.int16, device="cuda")
        bands = torch.tensor([[[sym1[c, b].data_ptr() for b in range(3)], [sym2[c, 1 + b].data_ptr() for b in range(3)]]
                              for c in range(3)], dtype=torch.int64, device="cuda")
        return {"case": case, "rgb": rgb, "ycocg": torch.empty_like(rgb), "back": torch.empty_like(rgb),
                "out": torch.empty_like(rgb), "planes": planes, "work": torch.empty((sy, sx), device="cuda"),
                "low": torch.empty((sy // 2, sx // 2), device="cuda"), "sym1": sym1, "sym2": sym2, "bands": bands}
    if kind == "coder":
        n, dtype = case["n"], torch.int32 if case["log2"] > 16 else torch.int16
        g = _generator(seed)
        u = torch.rand((case["streams"], n), generator=g, device="cuda") - 0.5
        q = torch.round(-case["scale"] * u.sign() * torch.log1p(-2 * u.abs().clamp_max(0.4999995))).to(torch.int64)
        q[torch.rand(q.shape, generator=g, device="cuda") > case["density"]] = 0
        sym = torch.where(q >= 0, 2 * q, -2 * q - 1).clamp_max((1 << min(case["log2"], 14)) - 1).to(dtype)
        streams = [sym[i] for i in range(case["streams"])]
        outs = torch.empty_like(sym)
        inst = cc.createInstance(0, case["streams"], n, case["block"], case["log2"])
        words = torch.zeros(case["streams"] * (n + 65536), dtype=torch.int32, device="cuda")
        return {"case": case, "inst": inst, "streams": streams, "out": outs,
                "outs": [outs[i] for i in range(case["streams"])], "words": words}
    if kind in ("bricks", "plan"):
        shapes, src, srcs, steps = _brick_inputs(case, seed)
        rec, recs = _packed(shapes)
        words = torch.zeros(src.numel() // 2 + 2048 * len(shapes), dtype=torch.int32, device="cuda")
        inst = cc.createInstance(0, 7, 128 ** 3 // 8, case["block"], case["log2"])
        if kind == "bricks":
            return {"case": case, "inst": inst, "shapes": shapes, "srcs": srcs, "steps": steps, "rec": rec, "recs": recs,
                    "words": words}
        plan = cc.BricksPlan(inst, srcs, recs, shapes, steps, case["levels"], words)
        return {"plan": plan, "case": case, "rec": rec, "words": words, "inst": inst}
    if kind == "serve":
        shapes = _serve_shapes(case)
        n = len(shapes) // 2
        src, srcs = _packed(shapes)
        field = _spectral((256, 256, 256), -11.0 / 6.0, seed)
        _cut(field, shapes[:n], srcs[:n], seed)
        lod = field.view(128, 2, 128, 2, 128, 2).mean(dim=(1, 3, 5))
        _cut(lod, shapes[n:], srcs[n:], seed)
        steps = [0.005 * float(field.std())] * n + [0.005 * float(lod.std())] * n
        words = torch.empty(src.numel(), dtype=torch.int32, device="cuda")
        inst = cc.createInstance(0, 7, 128 ** 3 // 8, case["block"], 14)
        offsets, _ = cc.compressBricksFloat(inst, srcs, shapes, steps, 2, words)
        ranges = np.stack([offsets[:-1], offsets[1:]], axis=1)
        requests = _trace(case)
        rec, recs = _packed([shapes[b] for r in requests for b in r])
        outputs, k = [], 0
        for r in requests:
            outputs.append(recs[k:k + len(r)])
            k += len(r)
        server = cc.Server(inst, words, ranges, shapes, steps, 2, slots=8, workspaceBytes=8 << 30)
        return {"server": server, "case": case, "arrivals": [0.0] * len(requests), "requests": requests,
                "outputs": outputs, "rec": rec, "words": words, "inst": inst}
    raise ValueError(kind)


# ------------------------------------------------------------------------------------ one pass
def _run_image(s):
    c = s["case"]
    sx, sy, step, util = c["sx"], c["sy"], c["step"], cc.util
    hx, hy, qx, qy = sx // 2, sy // 2, sx // 4, sy // 4
    util.convertRGBtoYCoCg(s["ycocg"], s["rgb"], sx * sy, 3)
    for ch in range(3):
        plane = s["planes"][ch]
        util.dwtFloat2DForwardFromByte(plane, s["work"], s["ycocg"].data_ptr() + ch, sx, sy, 3, sx, 3 * sx)
        util.dwtFloat2DForward(plane, s["work"], plane, hx, hy, 1, sx, sx)
        base = plane.data_ptr()
        for b in range(1, 4):
            util.quantizeToSymbols(s["sym1"][ch, b - 1], base + 4 * (b % 2 * hx + b // 2 * hy * sx), hx, hy, 1, step, sx)
        for b in range(4):
            util.quantizeToSymbols(s["sym2"][ch, b], base + 4 * (b % 2 * qx + b // 2 * qy * sx), qx, qy, 1, step / 2, sx)
    for ch in range(3):
        low, band = s["low"], s["bands"][ch]
        util.unquantizeFromSymbols(low, s["sym2"][ch, 0], qx, qy, 1, step / 2, hx)
        util.dwtFloat2DInverseFromSymbols(low, s["work"], low, band[1], step / 2, hx, hy, 1, hx, hx)
        util.dwtFloat2DInverseFromSymbolsToByte(s["back"].data_ptr() + ch, s["work"], low, band[0], step, sx, sy, 3, 3 * sx,
                                                hx)
    util.convertYCoCgtoRGB(s["out"], s["back"], sx * sy, 3)
    return {"planes": s["planes"], "sym1": s["sym1"], "sym2": s["sym2"], "rgb": s["out"]}


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind in ("volume", "short", "lossless", "dwt"):
        sx, sy, sz, levels = c["sx"], c["sy"], c["sz"], c["levels"]
    if kind == "volume":
        out = {}
        words = s["words"]
        if c["way"] != "decompress":
            words = cc.compressVolumeFloat(s["inst"], s["src"], sx, sy, sz, levels, c["step"], c["lvl0"])
            out["words"] = _store(s["file"], words)
        if c["way"] != "compress":
            cc.decompressVolumeFloat(s["inst"], s["rec"], sx, sy, sz, levels, words, c["step"], c["lvl0"])
            out["rec"] = s["rec"]
        return out
    if kind == "channels":
        cc.decompressVolumeFloatMultiChannel(s["inst"], s["channels"], c["sx"], c["sy"], c["sz"], c["levels"], c["lvl0"])
        return [image for image, _, _ in s["channels"]]
    if kind == "short":
        words = cc.compressVolumeFloatQuantFirst(s["inst"], s["src"], sx, sy, sz, levels, c["step"])
        cc.decompressVolumeFloatQuantFirst(s["inst"], s["rec"], sx, sy, sz, levels, words, c["step"])
        return {"words": _store(s["file"], words), "rec": s["rec"]}
    if kind == "lossless":
        words = cc.compressVolumeLossless(s["inst"], s["src"], sx, sy, sz, levels)
        cc.decompressVolumeLossless(s["inst"], s["rec"], sx, sy, sz, levels, words)
        return {"words": _store(s["file"], words), "rec": s["rec"]}
    if kind == "dwt":
        coef, rec, row, plane = s["coef"], s["rec"], sx, sx * sy
        src = s["src"]
        for f in _levels_of(c):
            cc.util.dwtFloat3DForward(coef, s["b2"], s["b1"], src, sx // f, sy // f, sz // f, 1, row, plane, row, plane)
            src = coef
        rec.copy_(coef)
        for f in reversed(_levels_of(c)):
            cc.util.dwtFloat3DInverse(rec, s["b2"], s["b1"], rec, sx // f, sy // f, sz // f, 1, row, plane, row, plane)
        return {"coef": coef, "rec": rec}
    if kind == "image":
        return _run_image(s)
    if kind == "coder":
        n = cc.encodeDevice(s["inst"], c["rl"], s["streams"], c["n"], s["words"])
        cc.decodeDevice(s["inst"], c["rl"], s["words"], s["outs"], c["n"], n)
        return {"words": s["words"], "count": n, "symbols": s["out"]}
    if kind == "bricks":
        offsets, status = cc.compressBricksFloat(s["inst"], s["srcs"], s["shapes"], s["steps"], c["levels"], s["words"])
        cc.decompressBricksFloat(s["inst"], s["recs"], s["shapes"], s["steps"], c["levels"], s["words"], offsets)
        return {"offsets": offsets.view(np.int64), "status": status.view(np.int32),
                "words": s["words"], "rec": s["rec"]}
    if kind == "plan":
        offsets, status, _ = s["plan"].run()
        return {"offsets": offsets.view(np.int64), "status": status.view(np.int32),
                "words": s["words"], "rec": s["rec"]}
    if kind == "serve":
        latency, _ = s["server"].run(s["arrivals"], s["requests"], s["outputs"])
        return {"done": latency >= 0, "rec": s["rec"]}
    raise ValueError(kind)


# ------------------------------------------------------------------------------------ what a pass needs
RATIO = 4.0  # bytes of a field over bytes of its bitstream, about what these steps give


def work(case):
    """Inputs read once and outputs written once; the operations of the 9/7 filters (9 multiply-adds an output)."""
    kind = case["kind"]
    if kind == "volume":
        n = case["sx"] * case["sy"] * case["sz"]
        ways = 2 if case["way"] == "both" else 1
        return {"bytes": ways * n * 4 * (1 + 1 / RATIO), "flops": ways * 54 * n * 8 / 7}
    if kind == "channels":
        n = case["sx"] * case["sy"] * case["sz"] * case["channels"]
        return {"bytes": n * 4 * (1 + 1 / RATIO), "flops": 54 * n * 8 / 7}
    if kind == "short":
        n = case["sx"] * case["sy"] * case["sz"]
        return {"bytes": 2 * n * 4 * (1 + 1 / RATIO), "flops": 2 * 18 * n * 8 / 7}
    if kind == "lossless":
        n = case["sx"] * case["sy"] * case["sz"]
        return {"bytes": 2 * n * 2 * 1.5, "flops": 2 * 12 * n * 4 / 3}
    if kind == "dwt":
        n = case["sx"] * case["sy"] * case["sz"]
        g = sum(0.125 ** level for level in range(case["levels"]))
        return {"bytes": n * 4 * 3, "flops": 2 * 54 * n * g}
    if kind == "image":
        n = case["sx"] * case["sy"] * 3
        return {"bytes": n * (1 + 4 + 2 + 2 + 1), "flops": 2 * 36 * n * 5 / 4}
    if kind == "coder":
        n = case["streams"] * case["n"]
        return {"bytes": 2 * n * (4 if case["log2"] > 16 else 2) * 1.25, "flops": 0}
    if kind in ("bricks", "plan"):
        n = sum(z * y * x for z, y, x in _shapes(case))
        return {"bytes": 2 * n * 4 * (1 + 1 / RATIO), "flops": 2 * 54 * n * 8 / 7}
    if kind == "serve":
        shapes = _serve_shapes(case)
        n = sum(shapes[b][0] * shapes[b][1] * shapes[b][2] for r in _trace(case) for b in r)
        return {"bytes": n * 4 * (1 + 1 / RATIO), "flops": 54 * n * 8 / 7}
    raise ValueError(kind)


def tolerance(case):
    """Whole numbers (bitstreams, symbols, bytes, status) are the same; floats are 32-bit sums of nine products an
    axis: against 64 bits three levels there and back show 4e-7."""
    if case["kind"] in ("lossless", "coder"):
        return "exact"
    return {"rel": 1.6e-6, "max": 1.6e-5}


# ------------------------------------------------------------------------------------ 64 bits
_LO = (0.0267488, -0.0168641, -0.0782233, 0.2668641, 0.6029490, 0.2668641, -0.0782233, -0.0168641, 0.0267488)
_HI = (0.0456359, -0.0287718, -0.2956359, 0.5575435, -0.2956359, -0.0287718, 0.0456359)
_EVEN = (0.0337282, -0.0575435, -0.5337281, 1.1150871, -0.5337281, -0.0575435, 0.0337282)
_ODD = (0.0534975, -0.0912718, -0.1564465, 0.5912718, 1.2058980, 0.5912718, -0.1564465, -0.0912718, 0.0534975)
_MATRICES = {}


def _mirror(j, n):
    """Whole-sample symmetric extension of a line of n samples."""
    while not 0 <= j < n:
        j = -j if j < 0 else 2 * (n - 1) - j
    return j


def _matrices(n):
    """The analysis and synthesis of a line of n samples (n even) as matrices; the lowpass half comes first."""
    if n not in _MATRICES:
        m = n // 2
        fwd, inv = np.zeros((n, n)), np.zeros((n, n))
        for k in range(m):
            for i, t in enumerate(_LO):
                fwd[k, _mirror(2 * k + i - 4, n)] += t
            for i, t in enumerate(_HI):
                fwd[m + k, _mirror(2 * k + 1 + i - 3, n)] += t
        for j in range(n):
            taps = _ODD if j % 2 else _EVEN
            for i, t in enumerate(taps):
                p = _mirror(j + i - len(taps) // 2, n)  # of the interleaved line: low at even, high at odd places
                inv[j, p // 2 + (m if p % 2 else 0)] += t
        _MATRICES[n] = [torch.from_numpy(a).cuda() for a in (fwd, inv)]
    return _MATRICES[n]


def _along_all(v, which):
    """One analysis (0) or synthesis (1) of v, one axis after the other."""
    for a in range(v.dim()):
        w = v.movedim(a, 0)
        v = torch.matmul(_matrices(w.shape[0])[which], w.reshape(w.shape[0], -1)).view(w.shape).movedim(0, a)
    return v.contiguous()


def _corner(shape, f):
    return tuple(slice(0, n // f) for n in shape)


def _analysis(v, levels):
    v = v.clone()
    for level in range(levels):
        at = _corner(v.shape, 1 << level)
        v[at] = _along_all(v[at], 0)
    return v


def _synthesis(v, levels):
    v = v.clone()
    for level in reversed(range(levels)):
        at = _corner(v.shape, 1 << level)
        v[at] = _along_all(v[at], 1)
    return v


def _deadzone(v, step):
    q = torch.trunc(v / step)
    return (q + 0.5 * torch.sign(q)) * step


def _coded(v, levels, step):
    """v after analysis, quantization with step / 2^level and synthesis."""
    c = _analysis(v.double(), levels)
    low = _deadzone(c[_corner(v.shape, 1 << levels)], step / (1 << (levels - 1)))
    for level in reversed(range(levels)):
        at = _corner(v.shape, 1 << level)
        c[at] = _deadzone(c[at], step / (1 << level))
        c[_corner(v.shape, 2 << level)] = low
        low = c[at].clone()
    return _synthesis(c, levels)


def _coded_bricks(shapes, srcs, steps, levels):
    out, views = _packed(shapes)
    out = out.double()
    at = 0
    for s, src, step in zip(shapes, srcs, steps):
        n = s[0] * s[1] * s[2]
        out[at:at + n] = _coded(src, levels, step).reshape(-1)
        at += -(-n // 64) * 64
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("lossless", "coder"):
        return None
    if kind in ("volume", "channels", "short", "dwt"):
        shape = (case["sz"], case["sy"], case["sx"])
    step = float(np.float32(case["step"])) if "step" in case else None
    if kind == "volume":
        out = {} if case["way"] == "decompress" else {"words": None}
        if case["way"] != "compress":
            out["rec"] = _coded(_field(*shape, seed), case["levels"], step)
        return out if "rec" in out else None
    if kind == "channels":
        return [_coded(_field(*shape, seed * 8 + i), case["levels"], step) for i in range(case["channels"])]
    if kind == "short":
        v = _field(*shape, seed).double()
        return {"words": None, "rec": torch.trunc(v / step + 0.5 * torch.sign(v)) * step}
    if kind == "dwt":
        c = _analysis(_field(*shape, seed).double(), case["levels"])
        return {"coef": c, "rec": _synthesis(c, case["levels"])}
    if kind == "image":
        r, g, b = _rgb(case["sy"], case["sx"], seed).to(torch.int64).unbind(-1)
        half = lambda v, d: torch.div(v, d, rounding_mode="trunc")  # noqa: E731
        ycocg = (half(r + 2 * g + b + 2, 4), half(r - b + 1, 2) + 127, half(-r + 2 * g - b + 2, 4) + 127)
        return {"planes": torch.stack([_analysis((p - 128).double(), 2) for p in ycocg]), "sym1": None, "sym2": None,
                "rgb": None}
    if kind in ("bricks", "plan"):
        shapes, _, srcs, steps = _brick_inputs(case, seed)
        return {"offsets": None, "status": None, "words": None,
                "rec": _coded_bricks(shapes, srcs, steps, case["levels"])}
    if kind == "serve":
        shapes = _serve_shapes(case)
        n = len(shapes) // 2
        _, srcs = _packed(shapes)
        field = _spectral((256, 256, 256), -11.0 / 6.0, seed)
        _cut(field, shapes[:n], srcs[:n], seed)
        lod = field.view(128, 2, 128, 2, 128, 2).mean(dim=(1, 3, 5))
        _cut(lod, shapes[n:], srcs[n:], seed)
        steps = [float(np.float32(0.005 * float(field.std())))] * n + [float(np.float32(0.005 * float(lod.std())))] * n
        decoded = {}
        order = [b for r in _trace(case) for b in r]
        for b in set(order):
            decoded[b] = _coded(srcs[b], 2, steps[b]).reshape(-1)
        return {"done": None, "rec": torch.cat([decoded[b] for b in order])}
    raise ValueError(kind)
