"""What a user has this framework do, as measurable cases.

Each case is one pass through public entry points (insta_amd.capi): a frame
render, a new pose with its set-up, a batch of served requests, a training
step, a density-grid update, the network alone (inference and the trainable
plugin) and the geometry queries.  Two workload shapes occur throughout, the
repository's own configurations: "small" (small_config: a 2,048-triangle
sphere, L=8, T=2^14, 64^3 grid, step 1/256) and "head" (full_config: a
9,976-triangle head, L=16, T=2^19, 128^3 grid, step sqrt(3)/1024).

Two states of the network occur in use: "initial" parameters (Xavier MLPs,
tables U(-1e-4, 1e-4): a thin translucent volume, the benchmark's render
workload) and a "surface" (tables of trained scale whose density rises from
empty to opaque across the avatar's skin, as a trained avatar's does).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from insta_amd import synth
from insta_amd.capi import (PRECISION_BF16, PRECISION_FP16, PRECISION_FP32, Context, Server, default_frame_config,
                            default_server_config, default_train_config, full_config, make_camera, small_config)

PRECISIONS = {"fp32": PRECISION_FP32, "fp16": PRECISION_FP16, "bf16": PRECISION_BF16}
# per shape: levels, log2 table size, growth, camera radius, mesh occupancy threshold, triangles, vertices,
# depth under the skin at which the density logit has risen from 0 to 8 (opaque within a step or two)
SHAPES = {
    "small": dict(levels=8, log2_t=14, growth=1.5, radius=1.0, threshold=0.05, tris=2048, verts=1026, ramp=0.02),
    "head": dict(levels=16, log2_t=19, growth=math.exp(math.log(2048.0 / 16.0) / 15.0), radius=0.7, threshold=0.015,
                 tris=9976, verts=5023, ramp=0.006),
}
FRAMES = 4            # posed frames of a render, query or density-grid context
TRAIN_FRAMES = 16     # posed frames (and images) of a training set
TRAIN_RES = 512       # training image side
# composited samples per pixel of a frame (30 degree field of view, the mesh's occupancy shell), measured
SAMPLES_PER_PIXEL = {("small", "initial"): 85.0, ("head", "initial"): 17.2,
                     ("small", "surface"): 30.0, ("head", "surface"): 8.7}


# ----------------------------------------------------------------------------
# cases
# ----------------------------------------------------------------------------

def listed():
    return [
        # the smallest frame a user renders (a thumbnail of the small avatar): launches and latency
        dict(name="render_small_64", kind="render", shape="small", precision="fp32", scene="initial", extra=0,
             width=64, height=64),
        # the benchmark's frame: a full-size head at 512^2 in FP32, every marched sample composited
        dict(name="render_head_512", kind="render", shape="head", precision="fp32", scene="initial", extra=0,
             width=512, height=512),
        # the largest frame served: a trained head at 1024^2 through the render buffer (shade, tonemap) in FP16
        # with the 16 expression dims of the reference's network
        dict(name="frame_head_fp16_1024", kind="frame", shape="head", precision="fp16", scene="surface", extra=16,
             width=1024, height=1024),
        # an animated avatar: every frame a new expression (mesh blend, BVH, occupancy, lists), then the image;
        # an odd viewport
        dict(name="pose_head_301x257", kind="pose", shape="head", precision="fp32", scene="surface", extra=0,
             width=301, height=257),
        # the serving loop under load: eight queued requests of mixed sizes on four workers
        dict(name="serve_small_8", kind="serve", shape="small", precision="fp16", scene="surface", extra=0,
             requests=8, most=512),
        # a training step late in training at the small shapes, FP32 grid gradients
        dict(name="train_small", kind="train", shape="small", scene="surface", extra=0, rays=8000, grid_fp16=False,
             supervised=False),
        # the same at full size with segmentation and depth supervision, expression dims and FP16 grid gradients
        dict(name="train_head_fp16grid", kind="train", shape="head", scene="surface", extra=16, rays=24000,
             grid_fp16=True, supervised=True),
        # the density-grid update of the training loop after its first 256 steps (G^3/4 + G^3/4 samples)
        dict(name="density_grid_head", kind="density", shape="head", scene="surface", extra=0,
             uniform=128 ** 3 // 4, nonuniform=128 ** 3 // 4),
        # the network alone on a large ragged batch of coordinates
        dict(name="infer_head_bf16_1m", kind="infer", shape="head", precision="bf16", scene="surface", n=1000003),
        # the network as a trainable plugin, forward and backward with input gradients: a large batch and a small one
        dict(name="plugin_head_100k", kind="plugin", shape="head", scene="surface", extra=16, n=100003),
        dict(name="plugin_small_1k", kind="plugin", shape="small", scene="surface", extra=0, n=1027),
        # geometry alone: nearest triangles of free points and the posed-to-canonical warp of coordinates
        dict(name="query_head_200k", kind="query", shape="head", extra=0, n=200003),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["render", "render", "frame", "pose", "serve", "train", "train", "density", "infer", "plugin",
                       "plugin", "query"])
    shape = rng.choice(["small", "head"])
    scene = rng.choice(["initial", "surface", "surface"])
    precision = rng.choice(["fp32", "fp16", "bf16"])
    extra = rng.choice([0, 0, 16])
    if kind in ("render", "frame"):
        # a small-shape frame marches five times the samples of a head's
        side = 1024 if shape == "head" else 480
        return dict(kind=kind, shape=shape, precision=precision, scene=scene, extra=extra, width=_log(rng, 40, side),
                    height=_log(rng, 40, side))
    if kind == "pose":
        return dict(kind=kind, shape=shape, precision=precision, scene="surface", extra=extra,
                    width=_log(rng, 64, 512), height=_log(rng, 64, 512))
    if kind == "serve":
        return dict(kind=kind, shape="small", precision="fp16", scene="surface", extra=0, requests=rng.randint(1, 8),
                    most=_log(rng, 128, 512))
    if kind == "train":
        return dict(kind=kind, shape=shape, scene="surface", extra=extra,
                    rays=_log(rng, 1000, 8000 if shape == "small" else 24000), grid_fp16=rng.random() < 0.5,
                    supervised=rng.random() < 0.5)
    if kind == "density":
        g3 = (64 if shape == "small" else 128) ** 3
        return dict(kind=kind, shape=shape, scene="surface", extra=extra, uniform=_log(rng, g3 // 16, g3 // 4),
                    nonuniform=_log(rng, g3 // 16, g3 // 4))
    if kind == "infer":
        return dict(kind=kind, shape=shape, precision=precision, scene="surface", n=_log(rng, 300, 1000000))
    if kind == "plugin":
        return dict(kind=kind, shape=shape, scene="surface", extra=extra, n=_log(rng, 300, 120000))
    return dict(kind="query", shape=shape, extra=extra, n=_log(rng, 300, 250000))


# ----------------------------------------------------------------------------
# inputs
# ----------------------------------------------------------------------------

def _levels(shape):
    """(offset, entries, resolution, scale, dense) of each hash-grid level."""
    s = SHAPES[shape]
    out, off = [], 0
    for l in range(s["levels"]):
        scale = np.float32(2.0 ** (l * math.log2(float(np.float32(s["growth"])))) * 16 - 1.0)
        res = int(math.ceil(float(scale))) + 1
        dense = res ** 3 <= 1 << s["log2_t"]
        size = (res ** 3 + 7) // 8 * 8 if dense else 1 << s["log2_t"]
        out.append((off, size, res, float(scale), dense))
        off += size
    return out


def _mlp_shapes(shape, extra):
    din = 2 * SHAPES[shape]["levels"] + extra
    return [(64, din), (16, 64), (64, 32), (64, 64), (3, 64)]


def _skin_depth(shape, x):
    """Signed depth of points [n, 3] under the avatar's mean canonical surface (positive inside)."""
    c = x - 0.5
    if shape == "small":
        return 0.3 - np.sqrt((c ** 2).sum(-1))
    axes = np.array([0.09, 0.12, 0.11])
    return 0.105 * (1.0 - np.sqrt(((c / axes) ** 2).sum(-1)))


def _params(shape, extra, scene, seed):
    """Flat FP32 parameters, MLPs then tables; the surface adds two density neurons that carry feature 0 of the
    finest dense level (both signs) to the density logit, and writes the skin's ramp there."""
    rng = np.random.default_rng(seed)
    mats = []
    for o, i in _mlp_shapes(shape, extra):
        a = math.sqrt(6.0 / (o + i))
        mats.append(rng.uniform(-a, a, (o, i)).astype(np.float32))
    levels = _levels(shape)
    n = 2 * (levels[-1][0] + levels[-1][1])
    tables = (rng.random(n, dtype=np.float32) - 0.5) * np.float32(2e-4 if scene == "initial" else 0.2)
    if scene == "surface":
        l = max(i for i, lv in enumerate(levels) if lv[4])
        off, _, res, scale, _ = levels[l]
        ax = (np.arange(res) - 0.5) / scale
        z, y, x = np.meshgrid(ax, ax, ax, indexing="ij")
        f = _skin_depth(shape, np.stack([x, y, z], -1).reshape(-1, 3)) / SHAPES[shape]["ramp"]
        tables[2 * off:2 * (off + res ** 3):2] = np.clip(f, -2.0, 2.0)
        w0, w1 = mats[0], mats[1]
        w0[0], w0[1] = 0.0, 0.0
        w0[0, 2 * l], w0[1, 2 * l] = 1.0, -1.0
        w1[0] *= 0.1
        w1[0, 0], w1[0, 1] = 8.0, -8.0
    return np.concatenate([m.ravel() for m in mats] + [tables])


def _avatar(shape, seed, frames, bases=0):
    if shape == "small":
        return synth.small_sphere_avatar(seed=seed, n_frames=frames, n_bases=bases)
    return synth.head_avatar(seed=seed, n_frames=frames, n_bases=bases or 50)


def _context(case, seed, av, max_frames, **kw):
    make = small_config if case["shape"] == "small" else full_config
    cfg = make(max_frames=max_frames, precision=PRECISIONS[case.get("precision", "fp32")],
               n_extra_dims=case.get("extra", 0), **kw)
    ctx = Context(cfg)
    ctx.set_canonical_mesh(av.canonical, av.faces, av.masks)
    if av.frames:
        ctx.set_frames(0, torch.from_numpy(np.stack(av.frames)).cuda())
    if "scene" in case:
        ctx.set_params(torch.from_numpy(_params(case["shape"], case.get("extra", 0), case["scene"], seed)).cuda())
    if cfg.n_extra_dims and av.frames:
        v = np.random.default_rng(seed + 1).standard_normal((len(av.frames), cfg.n_extra_dims)).astype(np.float32)
        ctx.set_frame_extra_dims(0, torch.from_numpy(v).cuda())
    return ctx


def _camera(shape, rng, height, front=True):
    return make_camera(synth.random_camera(rng, SHAPES[shape]["radius"], front_bias=front),
                       synth.focal_from_fov(height, 30.0))


def _images(rng, n, res):
    """Smooth RGB fields in [0, 1], alpha 1, [n, res, res, 4] on the device."""
    u = (torch.arange(res, dtype=torch.float64, device="cuda") + 0.5) / res
    p = torch.from_numpy(rng.uniform(0.0, 1.0, (5, n, 3, 4))).cuda()
    wave = torch.sin(2 * math.pi * ((1 + 3 * p[0])[..., None] * u + p[1][..., None]))
    rise = torch.cos(2 * math.pi * ((1 + 3 * p[2])[..., None] * u + p[3][..., None]))
    out = torch.ones((n, res, res, 4), dtype=torch.float32, device="cuda")
    for c in range(3):
        s = sum(p[4, :, c, k, None, None] * rise[:, c, k, :, None] * wave[:, c, k, None, :] for k in range(4))
        out[..., c] = (0.5 + 0.5 * s / p[4, :, c].sum(-1)[:, None, None]).float()
    return out


def _coords(case, seed):
    """NerfCoordinate rows around the canonical surface, directions uniform, extra dims N(0, 1)."""
    rng = np.random.default_rng(seed + 2)
    n, X = case["n"], case.get("extra", 0)
    d = rng.standard_normal((n, 3))
    u = d / np.linalg.norm(d, axis=1, keepdims=True)
    axes = np.array([0.3, 0.3, 0.3]) if case["shape"] == "small" else np.array([0.09, 0.12, 0.11])
    t = SHAPES[case["shape"]]["threshold"]
    pos = 0.5 + u * axes + rng.uniform(-t, t, (n, 1)) * u
    v = rng.standard_normal((n, 3))
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    c = np.zeros((n, 11 + X), np.float32)
    c[:, 0:3] = pos
    c[:, 8:11] = (v + 1.0) * 0.5
    if X:
        c[:, 11:] = rng.standard_normal((n, X))
    return c


def _upstream(case, seed):
    """dL/d(network output) of a loss averaged over the batch."""
    rng = np.random.default_rng(seed + 3)
    return (rng.standard_normal((case["n"], 4)) / case["n"]).astype(np.float32)


def _query_inputs(case, seed):
    """Coordinates around the posed skins (each row names its frame) and free points for nearest-triangle queries of
    frame 0: half near the skin, half anywhere in the unit cube."""
    av = _avatar(case["shape"], seed, FRAMES)
    rng = np.random.default_rng(seed + 2)
    n, t = case["n"], SHAPES[case["shape"]]["threshold"]

    def near(verts, k):
        tri = verts[av.faces[rng.integers(0, len(av.faces), k)]].astype(np.float64)
        bary = rng.dirichlet([1.0, 1.0, 1.0], k)
        off = rng.standard_normal((k, 3))
        off *= rng.uniform(0.0, t, (k, 1)) / np.linalg.norm(off, axis=1, keepdims=True)
        return (bary[:, :, None] * tri).sum(1) + off

    c = np.zeros((n, 11 + case["extra"]), np.float32)
    edges = np.linspace(0, n, FRAMES + 1).astype(int)
    for f in range(FRAMES):
        c[edges[f]:edges[f + 1], 0:3] = near(av.frames[f], edges[f + 1] - edges[f])
        c[edges[f]:edges[f + 1], 4] = f
    v = rng.standard_normal((n, 3))
    c[:, 8:11] = (v / np.linalg.norm(v, axis=1, keepdims=True) + 1.0) * 0.5
    pts = rng.uniform(0.0, 1.0, (n, 3))
    pts[: n // 2] = near(av.frames[0], n // 2)
    return av, c, pts.astype(np.float32)


class _Serving:
    """A server with its avatars; closed before the avatars go."""

    def __init__(self, case, seed):
        rng = np.random.default_rng(seed)
        self.avatars, self.bases = [], []
        self.server = Server(default_server_config(n_slots=4, hbm_budget_bytes=6 << 30,
                                                   occupancy_threshold=SHAPES[case["shape"]]["threshold"]))
        for a in range(4):
            av = _avatar(case["shape"], seed + a, 0, 50)
            ctx = _context(case, seed + 10 * a, av, 4, cell_split=2)
            self.avatars.append(ctx)
            self.bases.append(torch.from_numpy(av.bases).cuda())
            self.server.add_avatar(ctx, self.bases[a])
        self.requests = []
        for k in range(case["requests"]):
            res = int(min(case["most"], (128, 256, 512, case["most"])[k % 4]))
            self.requests.append((k % 4, rng.normal(0.0, 1.0, 50).astype(np.float32),
                                  _camera(case["shape"], rng, res, front=False), res,
                                  torch.empty((res * res, 4), dtype=torch.float32, device="cuda")))
        torch.cuda.synchronize()  # the workers' streams read what was uploaded here

    def __del__(self):
        self.server.close()


def prepare(case, seed):
    kind, shape = case["kind"], case["shape"]
    rng = np.random.default_rng(seed)
    t = SHAPES[shape]["threshold"]
    if kind in ("render", "frame"):
        av = _avatar(shape, seed, 1)
        ctx = _context(case, seed, av, FRAMES)
        ctx.build_occupancy(0, t)
        w, h = case["width"], case["height"]
        out = [torch.empty((h * w, 4), dtype=torch.float32, device="cuda"),
               torch.empty(h * w, dtype=torch.float32, device="cuda")]
        if kind == "render":
            out.append(torch.empty(h * w, dtype=torch.int32, device="cuda"))
        else:
            out.append(torch.zeros((h * w, 4), dtype=torch.float32, device="cuda"))
        ctx.reserve(render_pixels=w * h)
        return dict(case=case, ctx=ctx, cam=_camera(shape, rng, h), out=out, fc=default_frame_config())
    if kind == "pose":
        av = _avatar(shape, seed, 0, 50)
        ctx = _context(case, seed, av, FRAMES)
        w, h = case["width"], case["height"]
        ctx.reserve(render_pixels=w * h)
        return dict(case=case, ctx=ctx, cam=_camera(shape, rng, h), bases=torch.from_numpy(av.bases).cuda(),
                    coeffs=torch.from_numpy(rng.standard_normal(50).astype(np.float32)).cuda(),
                    out=(torch.empty((h * w, 4), dtype=torch.float32, device="cuda"),
                         torch.empty(h * w, dtype=torch.float32, device="cuda"),
                         torch.empty(h * w, dtype=torch.int32, device="cuda")))
    if kind == "serve":
        return dict(case=case, serving=_Serving(case, seed))
    if kind == "train":
        av = _avatar(shape, seed, TRAIN_FRAMES)
        ctx = _context(case, seed, av, TRAIN_FRAMES)
        for f in range(TRAIN_FRAMES):
            ctx.build_occupancy(f, t)
        cams = [_camera(shape, rng, TRAIN_RES, front=False) for _ in range(TRAIN_FRAMES)]
        ctx.set_training_set(_images(rng, TRAIN_FRAMES, TRAIN_RES), cams, list(range(TRAIN_FRAMES)))
        if case["supervised"]:
            size = (TRAIN_FRAMES, TRAIN_RES // 8, TRAIN_RES // 8)
            grow = torch.nn.Upsample(scale_factor=8)
            ids = np.array([30, 100, 120, 130, 140, 200, 255], np.float32)
            seg = grow(torch.from_numpy(ids[rng.integers(0, len(ids), size)])[None].cuda())[0].to(torch.uint8)
            depth = rng.uniform(0.9, 1.1, size) * SHAPES[shape]["radius"] * (rng.random(size) > 0.2)
            ctx.set_training_supervision(seg, grow(torch.from_numpy(depth.astype(np.float32))[None].cuda())[0])
        # the learning rate of a late step; ray counts whose batch stays below its 2^18-sample target
        tc = default_train_config(seed=seed & 0xFFFF, n_rays=case["rays"], learning_rate=1e-4,
                                  grid_grad_fp16=int(case["grid_fp16"]),
                                  loss_scale=128.0 if case["grid_fp16"] else 1.0)
        ctx.reserve(train_rays=case["rays"], train_samples=tc.max_samples, train_batch=tc.target_samples)
        return dict(case=case, ctx=ctx, tc=tc)
    if kind == "density":
        av = _avatar(shape, seed, FRAMES)
        ctx = _context(case, seed, av, FRAMES)
        for f in range(FRAMES):
            ctx.build_occupancy(f, t)
        g3 = ctx.cfg.grid_size ** 3
        ctx.update_density_grid(-1, FRAMES, n_uniform=g3, seed=seed & 0xFFFF)   # the loop's first updates
        return dict(case=case, ctx=ctx, seed=seed & 0xFFFF)
    if kind == "infer":
        ctx = _context(case, seed, _avatar(shape, seed, 0), 1)
        return dict(case=case, ctx=ctx, coords=torch.from_numpy(_coords(case, seed)).cuda())
    if kind == "plugin":
        ctx = _context(case, seed, _avatar(shape, seed, 0), 1)
        c = torch.from_numpy(_coords(case, seed)).cuda()
        ctx.reserve(train_samples=case["n"], train_batch=case["n"])
        return dict(case=case, ctx=ctx, coords=c, dout=torch.from_numpy(_upstream(case, seed)).cuda(),
                    din=torch.zeros_like(c))
    av, c, pts = _query_inputs(case, seed)
    ctx = _context(case, seed, av, FRAMES)
    for f in range(FRAMES):
        ctx.build_occupancy(f, t)
    return dict(case=case, ctx=ctx, coords=torch.from_numpy(c).cuda(), pts=torch.from_numpy(pts).cuda())


# ----------------------------------------------------------------------------
# one pass
# ----------------------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "serve":
        s = state["serving"]
        for a, coeffs, cam, res, out in s.requests:
            s.server.submit(a, coeffs, cam, res, res, out)
        done = []
        while len(done) < len(s.requests):
            done += s.server.poll(wait=True)
        return [out for *_, out in s.requests], sum(r.status for r in done)
    ctx = state["ctx"]
    if kind == "render":
        return ctx.render(state["cam"], case["width"], case["height"], 0, 0, 0, tuple(state["out"]))
    if kind == "frame":
        image, depth, accum = state["out"]
        ctx.render_frame(state["cam"], case["width"], case["height"], 0, 0, 0, state["fc"], accum, image, depth)
        return image, depth, accum
    if kind == "pose":
        ctx.set_frame_expression(0, state["bases"], state["coeffs"])
        bits = ctx.build_occupancy(0, SHAPES[case["shape"]]["threshold"])
        return ctx.render(state["cam"], case["width"], case["height"], 0, 0, 0, state["out"]), bits
    if kind == "train":
        st = ctx.train_step(state["tc"])
        return dict(gradients=ctx.gradients(), params=ctx.params(), loss=st.loss)
    if kind == "density":
        grid, mean = ctx.update_density_grid(-1, FRAMES, n_uniform=case["uniform"], n_nonuniform=case["nonuniform"],
                                             seed=state["seed"], want_grid=True)
        return grid, mean, ctx.get_occupancy(-1)
    if kind == "infer":
        return ctx.network_inference(state["coords"])
    if kind == "plugin":
        out = ctx.network_forward(state["coords"])
        grads = ctx.network_backward(state["coords"], state["dout"], dL_dinput_dev=state["din"])
        return dict(out=out, grads=grads, din=state["din"])
    ids, dist = ctx.closest(0, state["pts"])
    coords = state["coords"].clone()
    ctx.deform_samples(coords)
    return dict(ids=ids, dist=dist, coords=coords)


# ----------------------------------------------------------------------------
# the least work of a pass
# ----------------------------------------------------------------------------

def work(case):
    kind, shape = case["kind"], case["shape"]
    s = SHAPES[shape]
    mats = _mlp_shapes(shape, case.get("extra", 0))
    mlp = 2 * sum(o * i for o, i in mats)            # FLOP per sample
    corners = s["levels"] * 8 * 2 * 2                # interpolation FLOP per sample
    lv = _levels(shape)
    table = 8.0 * (lv[-1][0] + lv[-1][1])            # FP32 bytes
    touched = lambda n: min(table, s["levels"] * 64.0 * n)   # noqa: E731  entries n samples can touch
    mesh = s["tris"] * 48.0
    if kind in ("render", "frame", "pose", "serve"):
        if kind == "serve":
            px = sum(min(case["most"], (128, 256, 512, case["most"])[k % 4]) ** 2 for k in range(case["requests"]))
        else:
            px = case["width"] * case["height"]
        n = px * SAMPLES_PER_PIXEL[shape, case["scene"]]
        images = {"render": 24, "frame": 36, "pose": 24, "serve": 16}[kind] * px
        b = images + touched(n) + mesh
        if kind == "pose":
            b += 51 * 12.0 * s["verts"] + (64 if shape == "small" else 128) ** 3 / 8
        if kind == "serve":
            b += case["requests"] * 51 * 12.0 * s["verts"]
        return dict(bytes=b, flops=n * (mlp + corners))
    if kind == "train":
        # composited samples a ray, times forward (inference and batch), both products of the backward; parameters,
        # moments and gradients of the update
        n = case["rays"] * SAMPLES_PER_PIXEL[shape, "surface"]
        return dict(bytes=28.0 * (table / 4 + mlp / 2) + touched(n), flops=n * 4 * (mlp + corners))
    if kind == "density":
        n = case["uniform"] + case["nonuniform"]
        g3 = (64 if shape == "small" else 128) ** 3
        # the density MLP's hidden layer and its first output
        return dict(bytes=8.0 * g3 + g3 / 8 + touched(n), flops=n * (2 * (mats[0][0] * mats[0][1] + 64) + corners))
    n = case["n"]
    if kind == "infer":
        return dict(bytes=n * (44 + 16) + touched(n), flops=n * (mlp + corners))
    if kind == "plugin":
        row = 44 + 4 * case["extra"]
        return dict(bytes=n * (2 * row + 16 + 16) + 2 * touched(n) + table, flops=n * 3 * (mlp + corners))
    # two queries a row against the triangles next to it (about 8 exact distances of 100 FLOP each)
    return dict(bytes=n * (12 + 8 + 2 * (44 + 4 * case["extra"])) + FRAMES * mesh, flops=n * 2 * 8 * 100)


# ----------------------------------------------------------------------------
# the values in 64 bits
# ----------------------------------------------------------------------------

def _encode64(tables, shape, x):
    feats = []
    for off, size, res, scale, dense in _levels(shape):
        p = x * scale + 0.5
        g = torch.floor(p.detach()).to(torch.int64)
        f = p - g
        acc = 0.0
        for c in range(8):
            w, q = 1.0, []
            for k in range(3):
                up = (c >> k) & 1
                w = w * (f[:, k] if up else 1.0 - f[:, k])
                q.append(g[:, k] + up)
            if dense:
                i = (q[0] + q[1] * res + q[2] * res * res) % size
            else:
                i = (q[0] ^ (q[1] * 2654435761) ^ (q[2] * 805459861)) & (size - 1)
            acc = acc + w[:, None] * tables[off + i]
        feats.append(acc)
    return torch.cat(feats, 1)


def _sh64(d):
    """Real spherical harmonics of degrees 0..3, m = -l..l, with the Condon-Shortley phase."""
    x, y, z = d[:, 0], d[:, 1], d[:, 2]
    r = math.sqrt
    pi = math.pi
    c = [r(1 / (4 * pi)), r(3 / (4 * pi)), r(15 / (4 * pi)), r(5 / (16 * pi)), r(15 / (16 * pi)), r(35 / (32 * pi)),
         r(105 / (4 * pi)), r(21 / (32 * pi)), r(7 / (16 * pi)), r(105 / (16 * pi))]
    return torch.stack([
        c[0] + 0 * x, -c[1] * y, c[1] * z, -c[1] * x,
        c[2] * x * y, -c[2] * y * z, c[3] * (3 * z * z - 1), -c[2] * x * z, c[4] * (x * x - y * y),
        c[5] * y * (y * y - 3 * x * x), c[6] * x * y * z, c[7] * y * (1 - 5 * z * z), c[8] * z * (5 * z * z - 3),
        c[7] * x * (1 - 5 * z * z), c[9] * z * (x * x - y * y), c[5] * x * (3 * y * y - x * x)], 1)


def _network64(params, case, c):
    shapes = _mlp_shapes(case["shape"], case.get("extra", 0))
    mats, at = [], 0
    for o, i in shapes:
        mats.append(params[at:at + o * i].view(o, i))
        at += o * i
    x = _encode64(params[at:].view(-1, 2), case["shape"], c[:, 0:3])
    if case.get("extra", 0):
        x = torch.cat([x, c[:, 11:]], 1)
    d = torch.relu(x @ mats[0].t().contiguous()) @ mats[1].t().contiguous()
    h = torch.cat([d, _sh64(c[:, 8:11] * 2 - 1)], 1)
    for m in mats[2:4]:
        h = torch.relu(h @ m.t().contiguous())
    return torch.cat([h @ mats[4].t().contiguous(), d[:, :1]], 1)


def _tri_dist64(v, p):
    """Distances of points [n, 3] to triangles [m, 3, 3]: smallest over the triangles."""
    a, b, c = v[:, 0], v[:, 1], v[:, 2]
    nor = torch.linalg.cross(b - a, a - c)
    best = torch.full((len(p),), math.inf, dtype=torch.float64, device=p.device)
    for q, e in ((a, b - a), (b, c - b), (c, a - c)):
        d = p[:, None] - q[None]
        t = ((d * e).sum(-1) / (e * e).sum(-1)).clamp(0.0, 1.0)
        best = torch.minimum(best, ((t[..., None] * e - d) ** 2).sum(-1).min(1).values)
    inside = 0
    for q, e in ((a, b - a), (b, c - b), (c, a - c)):
        inside = inside + torch.sign((torch.linalg.cross(e, nor)[None] * (p[:, None] - q[None])).sum(-1))
    d = ((p[:, None] - a[None]) * nor).sum(-1) ** 2 / (nor * nor).sum(-1)
    d = torch.where(inside < 2, torch.full_like(d, math.inf), d)
    return torch.sqrt(torch.minimum(best, d.min(1).values))


def exact(case, seed):
    """Network outputs and gradients, and nearest distances.  A rendered image, a training step and the density grid
    have no value of their own here: each sample's frame is that of its nearest triangle, which changes at once where
    two are nearly as near, so another arithmetic's samples go elsewhere; the same holds for warped coordinates."""
    kind = case["kind"]
    if kind in ("infer", "plugin"):
        params = torch.from_numpy(_params(case["shape"], case.get("extra", 0), case["scene"], seed)).cuda().double()
        c = torch.from_numpy(_coords(case, seed)).cuda().double()
        if kind == "infer":
            return torch.cat([_network64(params, case, part) for part in c.split(1 << 17)])
        params.requires_grad_(True)
        c.requires_grad_(True)
        out = _network64(params, case, c)
        up = torch.from_numpy(_upstream(case, seed)).cuda().double()
        grads, din = torch.autograd.grad(out, (params, c), up)
        din = din.clone()
        din[:, 11:] = 0.0      # the entry point writes the position and direction columns
        return dict(out=out.detach(), grads=grads, din=din)
    if kind == "query" and case["n"] <= 300000:
        av, _, pts = _query_inputs(case, seed)
        v = torch.from_numpy(av.frames[0][av.faces]).cuda().double()
        p = torch.from_numpy(pts).cuda().double()
        return dict(ids=None, dist=torch.cat([_tri_dist64(v, part) for part in p.split(2048)]), coords=None)
    return None
