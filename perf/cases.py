"""The work that users of this framework have it do, as cases that can be timed
and compared: whole frames (plain, learned, voxel view), the upsampler's
forward pass and its training, through the C ABI and its Python handle.

  listed()             the cases, plain dicts
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  what a program holds before the call
  run(state)           one pass; returns its outputs
  work(case)           bytes and floating-point operations of a pass
  exact(case, seed)    the outputs in 64 bits (the upsampler's forward pass)

Frames.  A frame is what a headless program does per frame: queue the models
and lights, render, read the image back into a pinned host buffer it keeps
(voxelize, mip, G-buffer and trace all run again every frame, as in the
reference's render loop).  Scenes are the two generators of the framework, the
Cornell box and the triangle soup, in the sizes of the benchmark workloads and
around them; the camera, the soup and its materials come from the seed.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from voxel_cone_tracing_amd import _lib as L
from voxel_cone_tracing_amd.context import Context
from voxel_cone_tracing_amd.scene import C_add_material_records, look_at, perspective, soup_materials_fast

DTYPES = {"rgba8": L.RGBA8, "fp16": L.FP16, "bf16": L.BF16, "fp32": L.FP32}
CONES = {"ref9": (L.CONES_REF9, 9), "wide5": (L.CONES_5_WIDE, 5), "ring16": (L.CONES_16, 16)}
TEXEL = {"rgba8": 4, "fp16": 8, "bf16": 8, "fp32": 16}


def _frame(kind="plain", scene="soup", ntri=0, mu=-4.0, models=1, mats=0, res=128, dtype="rgba8", mean="reference",
           width=1280, height=720, cones="ref9", direct=False, shadow=False, lights=1):
    """mu: log of the soup's mean edge; mats: material palette (0: one material per triangle)."""
    return dict(kind=kind, scene=scene, ntri=ntri, mu=mu, models=models, mats=mats, res=res, dtype=dtype, mean=mean,
                width=width, height=height, cones=cones, direct=direct, shadow=shadow, lights=lights)


def listed():
    return [
        # the smallest frame anyone renders: the demo program's Cornell box (34
        # triangles, every phase on), where launches and waits count
        dict(_frame(scene="cornell", ntri=34, res=64, width=512, height=512, cones="wide5", direct=True, shadow=True),
             name="frame_cornell64"),
        # the drop-in's defaults (128^3, RGBA8, the reference's running average,
        # every phase) on an ordinary scene: a few models, a palette of materials
        dict(_frame(ntri=20_000, mu=-3.0, models=6, mats=32, direct=True, shadow=True), name="frame_default128"),
        # the 200k-triangle workload in the reference's storage and averaging
        dict(_frame(ntri=200_000, width=1920, height=1080), name="frame_soup128_rgba8"),
        # the benchmark frame, plain form
        dict(_frame(ntri=1_000_000, res=256, dtype="fp16", mean="exact", width=2560, height=1440),
             name="frame_soup256_fp16"),
        # the same frame in the reference's storage and averaging
        dict(_frame(ntri=1_000_000, res=256, width=2560, height=1440), name="frame_soup256_rgba8"),
        # a window of no round size, BF16 storage, direct light with shadows of
        # three lights
        dict(_frame(ntri=300_000, mu=-3.7, models=3, mats=500, res=256, dtype="bf16", mean="exact", width=1363,
                    height=767, direct=True, shadow=True, lights=3), name="frame_ragged_bf16"),
        # full-precision storage at an odd window, a scene of few and large
        # triangles (architecture rather than scans)
        dict(_frame(ntri=4_000, mu=-1.8, models=2, mats=40, res=128, dtype="fp32", mean="exact", width=1001,
                    height=563, cones="wide5", direct=True), name="frame_odd_fp32"),
        # the largest workload: 5M triangles, 512^3, 3840x2160, 16 cones
        dict(_frame(ntri=5_000_000, mats=4096, res=512, dtype="fp16", mean="exact", width=3840, height=2160,
                    cones="ring16"), name="frame_soup512_fp16"),
        # the benchmark frame, learned form (committed network, 40 dB fallback)
        dict(_frame(kind="learned", ntri=1_000_000, res=256, dtype="fp16", mean="exact", width=2560, height=1440),
             name="learned_soup256_fp16"),
        # the voxel view of an ordinary scene (the reference's inspection mode)
        dict(_frame(kind="view", ntri=20_000, mu=-3.0, models=6, mats=32), name="view_default128"),
        # the network on a serving program's own device buffers, at no round
        # number of rows
        dict(kind="forward", rows=200_003, name="mlp_forward"),
        # training: 32 Adam steps on minibatches of a resident sample set
        dict(kind="train", rows=65_536, batch=8192, steps=32, name="mlp_train"),
    ]


def _between(rng, lo, hi):
    """Spread over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    k = rng.random()
    if k < 0.12:
        return dict(kind="forward", rows=_between(rng, 64, L.MLP_NOALLOC_MAX_ROWS))
    if k < 0.22:
        batch = 64 * _between(rng, 1, 256)
        return dict(kind="train", rows=batch + _between(rng, 64, 65_536), batch=batch, steps=rng.randint(8, 40))
    kind = "learned" if k < 0.34 else ("view" if k < 0.42 else "plain")
    dtype = rng.choice(["rgba8", "rgba8", "fp16", "fp16", "bf16", "fp32"])
    mean = "reference" if dtype == "rgba8" and rng.random() < 0.7 else "exact"
    width = _between(rng, 64, 2560)
    height = max(16, int(width * rng.uniform(0.45, 0.8)))
    if kind == "learned":
        width, height = max(64, width // 4 * 4), max(32, height // 4 * 4)
    if kind != "view" and rng.random() < 0.1:
        return _frame(kind, "cornell", 34, res=rng.choice([32, 64, 128]), dtype=dtype, mean=mean, width=width,
                      height=height, cones=rng.choice(list(CONES)), direct=True, shadow=True)
    res = rng.choice([64, 128, 128, 256]) if kind == "view" else rng.choice([32, 64, 128, 128, 256, 256])
    ntri = _between(rng, 500, 40_000 if kind == "view" else 1_000_000)
    # denser soups have smaller triangles
    mu = min(-1.2, rng.uniform(-0.4, 0.4) - 0.5 * math.log(max(ntri, 2000) / 340.0))
    direct = rng.random() < 0.5 and kind == "plain"
    return _frame(kind, "soup", ntri, round(mu, 3), rng.choice([1, 1, 2, 5, 12]), rng.choice([0, 1, 37, 1000]), res,
                  dtype, mean, width, height, rng.choice(["ref9", "ref9", "wide5", "ring16"]), direct,
                  direct and rng.random() < 0.7, rng.choice([1, 1, 2, 4]) if direct else 1)


# ---- frames -------------------------------------------------------------------
class _FrameState:
    pass


def _prepare_frame(case, seed):
    rng = np.random.default_rng(seed)
    W, H = case["width"], case["height"]
    ctx = Context(W, H)
    average = L.AVG_REFERENCE if case["mean"] == "reference" else L.AVG_EXACT
    ctx.set_grid(case["res"], min(7, case["res"].bit_length()), DTYPES[case["dtype"]], average)
    ctx.set_cone_set(CONES[case["cones"]][0])
    ctx.set_phases(case["direct"], True, True, case["shadow"])
    ctx.set_voxel_view(int(rng.integers(0, 6)) if case["kind"] == "view" else 7, 0.5)
    ctx.set_pass_timing(0)
    s = _FrameState()
    turn = rng.uniform(-0.35, 0.35)
    if case["scene"] == "cornell":
        ctx.set_grid_size(0.55)
        pos, nrm, tm, mats = L.cornell(int(seed))
        base = ctx.add_materials(mats)
        s.models = [ctx.model_create(pos, nrm, tm + base)]
        turn *= 0.3
        eye, target, fovy = (1.55 * math.sin(turn), rng.uniform(-0.1, 0.1), 1.55 * math.cos(turn)), (0, 0, 0), 45.0
        s.lights = [((rng.uniform(-0.2, 0.2), 0.45, rng.uniform(-0.2, 0.2)), (1, 1, 1), 1.0, L.LIGHT_POINT)]
    else:
        ctx.set_grid_size(1.1)
        n, palette = case["ntri"], case["mats"]
        pos, nrm, ar = L.soup(int(seed), n, 1.0, case["mu"])
        first = C_add_material_records(ctx, soup_materials_fast(ar[:palette] if palette else ar))
        if palette:
            tm = rng.integers(0, min(palette, n), n).astype(np.uint32) + np.uint32(first)
        else:
            tm = np.arange(n, dtype=np.uint32) + np.uint32(first)
        cuts = np.linspace(0, n, case["models"] + 1).astype(int)
        s.models = [ctx.model_create(pos[a:b], nrm[a:b], tm[a:b]) for a, b in zip(cuts, cuts[1:]) if b > a]
        for i, m in enumerate(s.models):  # models of a scene stand at transforms of their own
            if i:
                c, d = math.cos(0.3 * i), math.sin(0.3 * i)
                ctx.set_model_transform(m, np.array([[c, 0, -d, 0], [0, 1, 0, 0], [d, 0, c, 0], [0, 0, 0, 1]],
                                                    np.float32))
        eye, target, fovy = (3.2 * math.sin(turn), 0.3, 3.2 * math.cos(turn)), (0, 0, 0), 50.0
        s.lights = [((0.4, 1.0, 0.6), (1.0, 1.0, 1.0), 1.0, L.LIGHT_DIRECTIONAL)]
    for _ in range(case["lights"] - 1):
        s.lights.append((tuple(rng.uniform(-0.8, 0.8, 3)), tuple(rng.uniform(0.3, 1.0, 3)), 1.0, L.LIGHT_POINT))
    ctx.set_camera(look_at(eye, target, (0, 1, 0)), perspective(math.radians(fovy), W / H, 0.1, 100.0))
    if case["kind"] == "learned":
        ctx.mlp_set_params(_network())
    s.ctx, s.learned, s.pixels = ctx, case["kind"] == "learned", W * H
    s.image = torch.empty((H, W, 4), dtype=torch.float32, pin_memory=torch.cuda.is_available())
    s.ptr = C.cast(s.image.data_ptr(), C.POINTER(C.c_float))
    ctx.sync()
    return s


def _run_frame(s):
    ctx = s.ctx
    for m in s.models:
        ctx.queue_model(m)
    for p, c, i, k in s.lights:
        ctx.queue_light(p, c, i, k)
    if s.learned:
        ctx.render_learned()
    else:
        ctx.render()
    L.check(ctx.lib.vct_image_download(ctx.h, s.ptr, s.pixels))
    return s.image


# ---- the upsampler's network ----------------------------------------------------
def _network():
    return np.load(L.LIB_PATH.parent / "weights" / "upsampler_soup256.npy")


def _features(n, seed, device):
    """Rows as the upsampler builds them: 9 taps of indirect light times their
    weights, a unit normal, the relative depth, the albedo."""
    g = torch.Generator(device=device).manual_seed(int(seed))
    x = torch.rand((n, 34), generator=g, device=device)
    x[:, :27] *= torch.rand((n, 1), generator=g, device=device) * 0.3
    v = torch.randn((n, 3), generator=g, device=device)
    x[:, 27:30] = v / v.norm(dim=1, keepdim=True)
    x[:, 30] = (x[:, 30] - 0.5) * 0.1
    return x


_stream = []  # the no-allocation entry point's calls share one staging array per GPU, so one stream orders them


def _prepare_forward(case, seed):
    s = _FrameState()
    s.ctx = Context(16, 16)
    s.ctx.mlp_set_params(_network())
    s.ctx.sync()
    s.rows = case["rows"]
    s.x = _features(s.rows, seed, "cuda")
    s.y = torch.empty((s.rows, 3), dtype=torch.float32, device="cuda")
    if not _stream:
        _stream.append(torch.cuda.Stream())
    torch.cuda.synchronize()
    return s


def _run_forward(s):
    L.check(s.ctx.lib.vct_mlp_forward_noalloc(s.ctx.h, s.x.data_ptr(), s.rows, s.y.data_ptr(),
                                              _stream[0].cuda_stream))
    return s.y


def _prepare_train(case, seed):
    s = _FrameState()
    s.ctx = Context(16, 16)
    s.ctx.mlp_set_params(_network())
    x = _features(case["rows"], seed, "cpu").numpy()
    rng = np.random.default_rng(seed)
    target = (0.2 * x[:, 12:15] - 0.05 * x[:, 0:3] + 0.02 * rng.standard_normal((case["rows"], 3))).astype(np.float32)
    s.ctx.upsample_set_samples(x, x[:, 31:34], target)
    s.steps, s.batch, s.seed = case["steps"], case["batch"], int(seed)
    s.ctx.sync()
    return s


def _run_train(s):
    loss = s.ctx.upsample_train(s.steps, s.batch, 1e-4, s.seed)
    return {"loss": loss, "params": s.ctx.mlp_params()}


# ---- the interface ----------------------------------------------------------------
def prepare(case, seed):
    if case["kind"] == "forward":
        return "forward", _prepare_forward(case, seed)
    if case["kind"] == "train":
        return "train", _prepare_train(case, seed)
    return "frame", _prepare_frame(case, seed)


def run(state):
    kind, s = state
    if kind == "forward":
        return _run_forward(s)
    if kind == "train":
        return _run_train(s)
    return _run_frame(s)


def exact(case, seed):
    if case["kind"] != "forward":
        return None  # whole frames and training runs: many passes of rasterisation and marching, or rounding steps
    p = torch.from_numpy(_network().astype(np.float64)).cuda()
    x = _features(case["rows"], seed, "cuda").double()
    o = 0
    for rows, cols, relu in ((64, 34, True), (64, 64, True), (3, 64, False)):
        w = p[o:o + rows * cols].reshape(rows, cols)
        b = p[o + rows * cols:o + rows * cols + rows]
        o += rows * cols + rows
        x = x @ w.t() + b
        x = x.clamp(min=0) if relu else x
    return x


def work(case):
    if case["kind"] == "forward":
        return {"bytes": case["rows"] * 37 * 4, "flops": case["rows"] * 12_928}
    if case["kind"] == "train":
        n = case["steps"] * case["batch"]
        return {"bytes": n * (34 * 2 + 24), "flops": n * 34_432}
    # geometry read by voxelize and by the G-buffer, level 0 and the mip chain
    # written and read once, the image written on the GPU and to the host
    bpe, res, pixels = TEXEL[case["dtype"]], case["res"], case["width"] * case["height"]
    volume = res ** 3 * bpe + sum(6 * (res >> k) ** 3 * bpe for k in range(1, min(7, res.bit_length())))
    traced = pixels / 16 if case["kind"] == "learned" else pixels
    cones = CONES[case["cones"]][1] + 1 + (case["lights"] if case["shadow"] else 0)
    # half the pixels covered, about 6 steps a cone, two levels of three
    # trilinear samples of four channels a step
    steps = 0 if case["kind"] == "view" else 0.5 * traced * cones * 6
    flops = steps * 2 * 3 * 8 * 4 * 2 + (12_928 * pixels if case["kind"] == "learned" else 0)
    return {"bytes": 2 * 76 * case["ntri"] + 2 * volume + 2 * 16 * pixels, "flops": flops + 200.0 * case["ntri"]}
