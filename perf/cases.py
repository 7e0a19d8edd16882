"""The work that programs built on this package have it do, as cases that can be timed.

Every case goes through the public operators of ``mx_driving`` / ``drivingsdk_amd`` the way a model calls them: inference
passes under ``no_grad``, training passes through autograd with all the gradients that a training step asks for.

A case is a dict of plain values:

  op      msda (multi-scale deformable attention), fused (the same with the calling module's softmax and location
          arithmetic inside), dagg (deformable aggregation), gka (geometric kernel attention), grid (2-D grid sampler)
  train   False: forward only; True: forward and backward
  dtype   float32, float16 or bfloat16
  levels  the feature maps, finest first, as "HxW,HxW,..."
  bs, nq, nh, hd, np ...   sizes in the terms of the operator
  where   how the queries' sampling points lie (see ``_points``)
"""
import math

import torch

import drivingsdk_amd
import mx_driving

_DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
_SIZE = {"float32": 4, "float16": 2, "bfloat16": 2}

_DETR = "100x150,50x75,25x38,13x19"          # feature maps of a detection transformer, strides 8 to 64
_BEV = "116x200,58x100,29x50,15x25"          # feature maps of one camera of a surround-view model
_CAMERA = "64x176,32x88,16x44,8x22"          # the same for a 256 x 704 camera image


def listed():
    return [
        # a detection decoder at inference: 300 object queries of one image, the smallest call; latency is what counts
        dict(name="decoder_infer_f32", op="msda", train=False, dtype="float32", levels=_DETR, bs=1, nq=300, nh=8, hd=32, np=4,
             where="scattered"),
        # the decoder of a training step: 900 queries, two images
        dict(name="decoder_train_f32", op="msda", train=True, dtype="float32", levels=_DETR, bs=2, nq=900, nh=8, hd=32, np=4,
             where="scattered"),
        # the encoder at inference in half precision: every pixel of the pyramid is a query, in raster order
        dict(name="encoder_infer_f16", op="msda", train=False, dtype="float16", levels=_DETR, bs=1, nq=19947, nh=8, hd=32, np=4,
             where="raster"),
        # the encoder of a training step (the headline workload of bench.py): the same size with two images
        dict(name="encoder_train_f32", op="msda", train=True, dtype="float32", levels=_DETR, bs=2, nq=19947, nh=8, hd=32, np=4,
             where="raster"),
        # spatial cross attention of a bird's-eye-view model: six cameras, eight points around each query's anchor
        dict(name="cross_attn_train_f16", op="msda", train=True, dtype="float16", levels=_BEV, bs=6, nq=9675, nh=8, hd=32, np=8,
             where="anchors"),
        # wide heads in bfloat16
        dict(name="wide_heads_train_bf16", op="msda", train=True, dtype="bfloat16", levels=_DETR, bs=1, nq=19947, nh=8, hd=128,
             np=4, where="scattered"),
        # a head size that no vector width divides, an odd number of levels and points, four heads
        dict(name="odd_heads_train_f32", op="msda", train=True, dtype="float32", levels="60x40,60x40,60x40,60x40,60x40", bs=6,
             nq=9680, nh=4, hd=37, np=3, where="scattered"),
        # the attention module as a whole, from logits and offsets, as a training step in mixed precision calls it
        dict(name="module_train_bf16", op="fused", train=True, dtype="bfloat16", levels=_DETR, bs=2, nq=19947, nh=8, hd=32, np=4,
             where="raster"),
        # deformable aggregation, 900 anchors of 13 points in six cameras: one frame at inference, and a training step
        dict(name="aggregate_infer_f16", op="dagg", train=False, dtype="float16", levels=_CAMERA, bs=1, cams=6, nq=900, np=13,
             nh=8, hd=32, where="cameras"),
        dict(name="aggregate_train_f32", op="dagg", train=True, dtype="float32", levels=_CAMERA, bs=6, cams=6, nq=900, np=13,
             nh=8, hd=32, where="cameras"),
        # geometric kernel attention of a map model: pixel indices that reach a little beyond the map
        dict(name="geometric_train_f32", op="gka", train=True, dtype="float32", levels="15x25", bs=24, nq=7156, nh=4, hd=64,
             np=15, where="indices"),
        # a feature map warped by a displacement field, in torch's default memory format
        dict(name="warp_train_f32", op="grid", train=True, dtype="float32", levels="64x176", bs=24, nh=1, hd=128, out="24x176",
             np=1, where="warp"),
    ]


def draw(rng):
    """One more case: the same kinds of call over the range of sizes, head widths, data types and directions."""
    limits = {}
    for c in listed():
        cost = _cost(c)
        limits[c["op"]] = max(limits.get(c["op"], 0), cost)
    while True:
        c = _draw_one(rng)
        if _cost(c) <= limits[c["op"]]:
            return c


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_one(rng):
    op = rng.choices(["msda", "fused", "dagg", "gka", "grid"], [10, 4, 3, 2, 3])[0]
    c = dict(op=op, train=rng.random() < 0.6, dtype=rng.choice(["float32", "float16", "bfloat16"]))
    if op in ("msda", "fused"):
        h, w = _log_uniform(rng, 20, 130), _log_uniform(rng, 20, 200)
        nl = rng.randint(1, 5)
        c.update(levels=_pyramid(h, w, nl), bs=rng.choice([1, 1, 2, 2, 3, 6]), nh=rng.choice([4, 8, 8, 8, 16]),
                 hd=rng.choice([16, 24, 32, 32, 32, 37, 48, 64, 128]), np=rng.choice([1, 2, 3, 4, 4, 4, 6, 8]))
        c["where"] = rng.choice(["raster", "scattered", "anchors"])
        c["nq"] = _keys(c) if c["where"] == "raster" else _log_uniform(rng, 100, 20000)
    elif op == "dagg":
        h, w = _log_uniform(rng, 16, 64), _log_uniform(rng, 22, 176)
        c.update(levels=_pyramid(h, w, rng.randint(1, 4)), bs=rng.choice([1, 1, 2, 4, 6]), cams=rng.randint(1, 6),
                 nq=_log_uniform(rng, 50, 1200), np=rng.randint(5, 31), nh=rng.choice([4, 8, 16]), hd=rng.choice([4, 8, 16, 32]),
                 where="cameras")
    elif op == "gka":
        c.update(levels="%dx%d" % (_log_uniform(rng, 8, 64), _log_uniform(rng, 12, 100)), bs=rng.randint(1, 24),
                 nq=_log_uniform(rng, 200, 8000), nh=rng.choice([2, 4, 8]), hd=rng.choice([16, 32, 64]), np=rng.randint(4, 20),
                 where="indices")
    else:
        c.update(levels="%dx%d" % (_log_uniform(rng, 16, 100), _log_uniform(rng, 20, 180)), bs=rng.randint(1, 24), nh=1,
                 hd=rng.choice([3, 16, 32, 64, 80, 128]), np=1, where="warp",
                 out="%dx%d" % (_log_uniform(rng, 12, 100), _log_uniform(rng, 20, 180)))
    return c


def _pyramid(h, w, nl):
    maps = []
    for _ in range(nl):
        maps.append("%dx%d" % (h, w))
        h, w = max(1, (h + 1) // 2), max(1, (w + 1) // 2)
    return ",".join(maps)


def _maps(c):
    return [tuple(int(v) for v in m.split("x")) for m in c["levels"].split(",")]


def _keys(c):
    return sum(h * w for h, w in _maps(c))


def _queries(c):
    if c["op"] == "grid":
        h, w = c["out"].split("x")
        return int(h) * int(w)
    return c["nq"]


def _samples(c):
    """Sampling points of one pass (each reads up to four rows of ``hd`` channels)."""
    return c["bs"] * _queries(c) * c["nh"] * len(_maps(c)) * c["np"] * c.get("cams", 1)


def _cost(c):
    return max(work(c)["bytes"] / 4e12, work(c)["flops"] / 4e12)


def _level_tensors(c, dtype, device):
    shapes = torch.tensor(_maps(c), dtype=dtype)
    starts = torch.cat((shapes.new_zeros(1), shapes.prod(1).cumsum(0)[:-1])).to(dtype)
    return shapes.to(device), starts.to(device)


def _points(c, g, dev):
    """Reference points in [0, 1], [bs, nq, 1, 1, 1, 2], and the spread of the samples around them per level, [nl, 1, 2]:

    raster     self attention over the pyramid: query i sits on the centre of pixel i, samples a few pixels away
    scattered  object queries: anywhere in the image, samples a few pixels away on the coarse maps and wide of it on the fine
    anchors    projected anchors: anywhere in the image, samples in a box of a tenth of it
    """
    bs, nq = c["bs"], c["nq"]
    maps = torch.tensor(_maps(c), dtype=torch.float32, device=dev)                     # (h, w)
    if c["where"] == "raster":
        centres = []
        for h, w in _maps(c):
            y, x = torch.meshgrid(torch.arange(h, device=dev), torch.arange(w, device=dev), indexing="ij")
            centres.append(torch.stack(((x.flatten() + 0.5) / w, (y.flatten() + 0.5) / h), -1))
        ref = torch.cat(centres).expand(bs, nq, 2)
        spread = 2.0 / maps.flip(1)
    else:
        ref = torch.rand(bs, nq, 2, generator=g, device=dev)
        spread = torch.full_like(maps, 0.05 if c["where"] == "anchors" else 0.02)
    return ref.reshape(bs, nq, 1, 1, 1, 2), spread.reshape(-1, 1, 2)


def prepare(case, seed):
    c, dev, dt = case, torch.device("cuda"), _DTYPES[case["dtype"]]
    g = torch.Generator(device=dev).manual_seed(int(seed))

    def randn(*shape):
        return torch.randn(*shape, generator=g, device=dev, dtype=torch.float32)

    def rand(*shape):
        return torch.rand(*shape, generator=g, device=dev, dtype=torch.float32)

    bs, nq, nh, hd, npts, nl, nk = c["bs"], _queries(c), c["nh"], c["hd"], c["np"], len(_maps(c)), _keys(c)
    if c["op"] in ("msda", "fused"):
        ref, spread = _points(c, g, dev)
        shift = randn(bs, nq, nh, nl, npts, 2) if c["where"] != "anchors" else 2 * rand(bs, nq, nh, nl, npts, 2) - 1
        logits = randn(bs, nq, nh, nl * npts)
        value, (shapes, starts) = randn(bs, nk, nh, hd), _level_tensors(c, torch.int64, dev)
        if c["op"] == "msda":
            attn = torch.softmax(logits, -1).reshape(bs, nq, nh, nl, npts)
            tensors = [value, ref + shift * spread, attn]
        else:
            pixels = shift * spread * shapes.flip(1).reshape(nl, 1, 2)                 # offsets are in pixels of their level
            tensors = [value, ref.reshape(bs, nq, 1, 2).expand(bs, nq, nl, 2).contiguous(), pixels, logits]
    elif c["op"] == "dagg":
        cams = c["cams"]
        shapes, starts = _level_tensors(c, torch.int32, dev)
        starts = (starts + torch.arange(cams, dtype=torch.int32, device=dev)[:, None] * nk).contiguous()
        shapes = shapes.expand(cams, nl, 2).contiguous()
        # an anchor's points lie around its centre, which projects into some of the cameras and misses the others
        centre = rand(bs, nq, 1, cams, 2) * 1.6 - 0.3
        loc = centre + 0.05 * randn(bs, nq, npts, cams, 2)
        weights = torch.softmax(randn(bs, nq, npts * cams * nl, nh), 2).reshape(bs, nq, npts, cams, nl, nh)
        tensors = [randn(bs, cams * nk, nh * hd), loc, weights]
    elif c["op"] == "gka":
        shapes, starts = _level_tensors(c, torch.int32, dev)
        h, w = _maps(c)[0]
        loc = rand(bs, nq, nh, nl, npts, 2) * torch.tensor([w + 6.0, h + 6.0], device=dev) - 3
        tensors = [randn(bs, nk, nh, hd), rand(bs, nq, nh, nl, npts)]
    else:
        shapes = starts = None
        (h, w), (ho, wo) = _maps(c)[0], (int(v) for v in c["out"].split("x"))
        y, x = torch.meshgrid(torch.linspace(-1, 1, ho, device=dev), torch.linspace(-1, 1, wo, device=dev), indexing="ij")
        tensors = [randn(bs, hd, h, w), torch.stack((x, y), -1) + 0.1 * randn(bs, ho, wo, 2)]
    s = dict(op=c["op"], train=bool(c["train"]), shapes=shapes, starts=starts,
             inputs=[t.to(dt).requires_grad_(bool(c["train"])) for t in tensors])
    if c["op"] == "gka":
        s["indices"] = loc.trunc()                                                     # whole numbers, float32 in every case
    if c["train"]:
        out = (bs, hd, ho, wo) if c["op"] == "grid" else (bs, nq, nh * hd)
        s["grad"] = randn(*out).to(dt)
    return s


def _forward(s):
    x = s["inputs"]
    if s["op"] == "msda":
        return mx_driving.multi_scale_deformable_attn(x[0], s["shapes"], s["starts"], x[1], x[2])
    if s["op"] == "fused":
        return drivingsdk_amd.multi_scale_deformable_attn_fused(x[0], s["shapes"], s["starts"], x[1], x[2], x[3])
    if s["op"] == "dagg":
        return mx_driving.deformable_aggregation(x[0], s["shapes"], s["starts"], x[1], x[2])
    if s["op"] == "gka":
        return mx_driving.geometric_kernel_attention(x[0], s["shapes"], s["starts"], s["indices"], x[1])
    return mx_driving.grid_sampler2d_v2(x[0], x[1], "bilinear", "zeros", False)


def run(state):
    if not state["train"]:
        with torch.no_grad():
            return _forward(state)
    out = _forward(state)
    return (out.detach(),) + torch.autograd.grad(out, state["inputs"], state["grad"])


def work(case):
    """Bytes: every input read once and every output written once (rows of the feature maps that no sample reaches are not
    read: where the samples' four rows are fewer than the maps have, those).  Operations: four rows per sample (one for geometric
    kernel attention), a multiply-add per channel in the forward, two more (dots, scatter) in the backward."""
    c = case
    es, bs, nq, nh, hd, nl = _SIZE[c["dtype"]], c["bs"], _queries(c), c["nh"], c["hd"], len(_maps(c))
    samples, rows = _samples(c), 1 if c["op"] == "gka" else 4
    value = bs * _keys(c) * c.get("cams", 1) * nh * hd
    read = min(value, samples * rows * hd) * es
    out = bs * nq * nh * hd * es
    if c["op"] == "dagg":
        loc, weights = bs * nq * c["np"] * c["cams"] * 2 * es, samples * es
    elif c["op"] == "gka":
        loc, weights = samples * 2 * 4, samples * es
    elif c["op"] == "grid":
        loc, weights = samples * 2 * es, 0
    else:
        loc, weights = samples * 2 * es, samples * es
    refs = bs * nq * nl * 2 * es if c["op"] == "fused" else 0
    ins = read + loc + weights + refs
    flops = 2.0 * samples * rows * hd
    if not c["train"]:
        return {"bytes": ins + out, "flops": flops}
    grads = value * es + (0 if c["op"] == "gka" else loc) + weights + refs
    return {"bytes": 2 * (ins + out) + grads, "flops": 3.0 * flops}


def tolerance(case):
    """float32: sums of a few dozen to a few thousand products in another order.  16-bit types: one rounding at the store of each
    result (float16 keeps 11 significant bits, bfloat16 8), so a result may fall on the neighbouring value."""
    return {"float32": {"rel": 1e-5, "max": 1e-3}, "float16": {"rel": 1e-3, "max": 4e-3}, "bfloat16": {"rel": 6e-3, "max": 3e-2}}[
        case["dtype"]]
