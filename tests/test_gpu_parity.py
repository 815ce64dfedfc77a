"""GPU parity of the three passes against the CPU oracle (through the C ABI).

Bit-exact: voxel occupancy, coordinates and stored level-0 values (both
averaging modes), every mip level of every direction map, G-buffer coverage,
positions, normals and material ids.  Tolerance: the cone-traced image
(FP32 on both sides; max-abs stated per test) and its PSNR against the FP64
ideal oracle.
"""
from __future__ import annotations

import sys

import numpy as np
import pytest

from voxel_cone_tracing_amd import _lib as L
from voxel_cone_tracing_amd.context import Context

from helpers import SceneSpec, bits, decode_level, encode_level

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


# ---- mip (kernel b) ---------------------------------------------------------------
def _random_level0(rng, res, dtype):
    n = res ** 3
    if dtype == L.RGBA8:
        v = rng.integers(0, 2 ** 32, size=n, dtype=np.uint64).astype(np.uint32)
        # a share of empty and of opaque voxels, as voxelisation produces
        v[rng.random(n) < 0.3] = 0
        op = rng.random(n) < 0.3
        v[op] = (v[op] & 0x00FFFFFF) | 0xFF000000
        return v.reshape(res, res, res)
    f = rng.random((n, 4)).astype(np.float32)
    f[rng.random(n) < 0.3] = 0
    f[rng.random(n) < 0.3, 3] = 1.0
    return encode_level(f.reshape(res, res, res, 4), dtype)


@pytest.mark.parametrize("dtype", [L.RGBA8, L.FP16, L.BF16, L.FP32])
@pytest.mark.parametrize("res,levels", [(32, 6), (64, 7), (256, 7)])
def test_mip_bit_exact(gpu_available, orc, dtype, res, levels):
    say(f"mip parity dtype={dtype} res={res} levels={levels}")
    rng = np.random.default_rng(res * 10 + dtype)
    l0 = _random_level0(rng, res, dtype)
    with Context(16, 16) as ctx:
        ctx.set_grid(res, levels, dtype)
        ctx.upload_level(0, 0, l0)
        ctx.mip()
        ctx.sync()
        ref = orc.mip_f32(res, levels, dtype, decode_level(l0, dtype))
        for l in range(1, levels):
            for d in range(6):
                got = ctx.download_level(l, d)
                want = encode_level(ref[(l, d)], dtype)
                assert np.array_equal(bits(got), bits(want)), f"level {l} dir {d} differs"


# ---- voxelize (kernel a) ----------------------------------------------------------
@pytest.mark.parametrize("kind,res,ntri", [("cornell", 64, 34), ("soup", 64, 3000), ("soup", 128, 20000)])
def test_voxelize_reference_average_bit_exact(gpu_available, orc, kind, res, ntri):
    say(f"voxelize reference average kind={kind} res={res}")
    sc = SceneSpec(kind, res=res, ntri=ntri)
    with Context(32, 32) as ctx:
        sc.build(ctx, L.RGBA8, L.AVG_REFERENCE)
        ctx.voxelize()
        got = ctx.download_level(0)
        nfrag, ncand = ctx.voxelize_stats()
    want = orc.voxelize(res, sc.cube_size, sc.M, sc.pos, sc.nrm, sc.tri_mat, sc.mat_records, sc.lights,
                        want=("ref", "count"))
    assert nfrag == want["fragments"]
    occ_g, occ_w = got != 0, want["ref"] != 0
    assert np.array_equal(occ_g, occ_w), f"occupancy differs at {np.argwhere(occ_g != occ_w)[:5]}"
    assert np.array_equal(got, want["ref"]), f"{np.count_nonzero(got != want['ref'])} voxels differ"


def test_voxelize_reference_average_many_models(gpu_available, orc):
    """37 queued models: the texels equal the oracle's for the same triangles
    as one list, since the canonical order runs over the queue."""
    say("voxelize reference average over 37 models")
    sc = SceneSpec("soup", res=64, ntri=3000)
    cuts = np.linspace(0, 3000, 38).astype(int)
    with Context(32, 32) as ctx:
        sc.build(ctx, L.RGBA8, L.AVG_REFERENCE)
        ctx.clear_queues()
        for a, b in zip(cuts[:-1], cuts[1:]):
            ctx.queue_model(ctx.model_create(sc.pos[a:b], sc.nrm[a:b], sc.tri_mat[a:b]))
        for (p, c, i, k) in sc.lights:
            ctx.queue_light(p, c, i, k)
        for _ in range(2):  # the second frame checks that the per-voxel counts start again from zero
            ctx.voxelize()
            got = ctx.download_level(0)
        nfrag, _ = ctx.voxelize_stats()
    want = orc.voxelize(sc.res, sc.cube_size, sc.M, sc.pos, sc.nrm, sc.tri_mat, sc.mat_records, sc.lights,
                        want=("ref", "count"))
    assert nfrag == want["fragments"]
    assert np.array_equal(got, want["ref"]), f"{np.count_nonzero(got != want['ref'])} voxels differ"


@pytest.mark.parametrize("dtype", [L.FP32, L.FP16, L.BF16, L.RGBA8])
@pytest.mark.parametrize("kind,res,ntri", [("cornell", 64, 34), ("soup", 128, 20000), ("cornell", 8, 34),
                                           ("soup", 256, 60000)])
def test_voxelize_exact_mean_bit_exact(gpu_available, orc, dtype, kind, res, ntri):
    say(f"voxelize exact mean dtype={dtype} kind={kind} res={res}")
    sc = SceneSpec(kind, res=res, ntri=ntri)
    with Context(32, 32) as ctx:
        sc.build(ctx, dtype, L.AVG_EXACT)
        for _ in range(2):  # the second frame checks that the sums were re-zeroed
            ctx.voxelize()
            got = ctx.download_level(0)
    want = orc.voxelize(res, sc.cube_size, sc.M, sc.pos, sc.nrm, sc.tri_mat, sc.mat_records, sc.lights,
                        want=("q32", "f64", "count"))
    w = encode_level(want["q32"], dtype)
    assert np.array_equal(bits(got), bits(w)), "level 0 differs"
    # error of the stored radiance against the FP64 exact mean
    err = np.abs(decode_level(got, dtype).astype(np.float64) - want["f64"]).max()
    bound = {L.FP32: 2e-5, L.FP16: 1e-3, L.BF16: 4.0e-3, L.RGBA8: 2.0e-3}[dtype]
    say(f"  max-abs vs FP64 = {err:.3e}")
    assert err <= bound


def test_voxelize_lists_past_their_capacity_bit_exact(gpu_available, orc):
    """Brick lists sized from an earlier frame's (triangle, brick) count: a
    frame whose geometry outgrew them (the same triangles, grown tenfold by
    the model matrix) has its overflowing bricks walk every triangle's brick
    box and stays bit-exact, and so does the frame after it (sized from the
    grown count)."""
    say("voxelize lists past their capacity")
    res = 256
    sc = SceneSpec("cornell", res=res)
    ntri = sc.pos.reshape(-1, 9).shape[0]
    small = np.diag([0.1, 0.1, 0.1, 1.0]).astype(np.float32)
    with Context(32, 32) as ctx:
        sc.build(ctx, L.FP16, L.AVG_EXACT)
        ctx.set_model_transform(sc.model, small)
        ctx.voxelize()  # the first frame waits for its count: the lists are sized from it
        _, small_pairs = ctx.voxelize_stats()
        ctx.set_model_transform(sc.model, sc.M)
        got = []
        for _ in range(2):
            ctx.voxelize()
            got.append(ctx.download_level(0))
        _, pairs = ctx.voxelize_stats()
    cap = max(small_pairs + small_pairs // 4, 2 * ntri + 1024)
    say(f"  pairs: shrunk box {small_pairs}, full box {pairs}, capacity of the second frame {cap}")
    assert pairs > cap
    want = orc.voxelize(res, sc.cube_size, sc.M, sc.pos, sc.nrm, sc.tri_mat, sc.mat_records, sc.lights,
                        want=("q32",))
    w = encode_level(want["q32"], L.FP16)
    for k, g in enumerate(got):
        assert np.array_equal(bits(g), bits(w)), f"frame {k + 2}: level 0 differs"


@pytest.mark.parametrize("dtype,average", [(L.FP16, L.AVG_EXACT), (L.RGBA8, L.AVG_REFERENCE)])
def test_voxelize_follows_material_changes_bit_exact(gpu_available, orc, dtype, average):
    """The set-up keeps the queued models' per-triangle material terms from
    frame to frame; a material upload (upload_material_data), a model's
    material assignment (set_model_material) and another model in the queue
    with the same triangle count each rebuild them, so every frame matches
    the oracle for the materials then in force."""
    import ctypes as C

    say(f"voxelize after material changes dtype={dtype} average={average}")
    sc = SceneSpec("cornell", res=64)
    recs = sc.mat_records.copy()
    with Context(32, 32) as ctx:
        sc.build(ctx, dtype, average)

        def check(tri_mat, tag):
            ctx.voxelize()
            got = ctx.download_level(0)
            want = orc.voxelize(sc.res, sc.cube_size, sc.M, sc.pos, sc.nrm, tri_mat, recs, sc.lights,
                                want=("ref", "q32"))
            w = want["ref"] if average == L.AVG_REFERENCE else encode_level(want["q32"], dtype)
            assert np.array_equal(bits(got), bits(w)), f"{tag}: level 0 differs"

        check(sc.tri_mat, "first frame")
        check(sc.tri_mat, "second frame")
        # a wall (material 2) turns green, emissive and transmissive
        r = recs[2].copy()
        r[4:7] = (0.1, 0.7, 0.3)
        r[12:15] = (0.5, 0.6, 0.7)
        r[16:19] = (0.2, 0.0, 0.05)
        r[21] = 0.4
        r[22] = np.array([4], np.int32).view(np.float32)[0]
        recs[2] = r
        m = L.Material.from_buffer_copy(np.ascontiguousarray(r).tobytes())
        L.check(ctx.lib.vct_upload_material_data(ctx.h, C.byref(m), 2))
        check(sc.tri_mat, "after the upload")
        check(sc.tri_mat, "the frame after the upload")
        ctx.set_model_material(2, sc.model)
        every2 = np.full_like(sc.tri_mat, 2)
        check(every2, "after set_model_material")
        # another model with the same triangles and count, in the original materials
        other = ctx.model_create(sc.pos, sc.nrm, sc.tri_mat)
        ctx.set_model_transform(other, sc.M)
        ctx.clear_queues()
        ctx.queue_model(other)
        for (p, c, i, k) in sc.lights:
            ctx.queue_light(p, c, i, k)
        check(sc.tri_mat, "another model queued")
        ctx.clear_queues()
        ctx.queue_model(sc.model)
        for (p, c, i, k) in sc.lights:
            ctx.queue_light(p, c, i, k)
        check(every2, "the first model queued again")


@pytest.mark.parametrize("dtype,average", [(L.FP16, L.AVG_EXACT), (L.RGBA8, L.AVG_REFERENCE)])
@pytest.mark.parametrize("change", ["grid", "transform", "cube"])
def test_voxelize_keeps_terms_of_undrawn_triangles(gpu_available, orc, dtype, average, change):
    """The per-triangle material terms kept from the first frame hold for
    every queued triangle, drawn then or not: triangles that the first frame
    dropped (between the pixel centres of a coarse grid, off the grid by the
    model matrix, or too small in a larger cube) and the second frame draws
    have their own materials there."""
    say(f"voxelize: undrawn, then drawn; dtype={dtype} average={average} change={change}")
    res = 128
    sc = SceneSpec("soup", res=res, ntri=6000, mu=-4.0, model="rot_scale")
    with Context(32, 32) as ctx:
        sc.build(ctx, dtype, average)
        if change == "grid":
            ctx.set_grid(8, 4, dtype, average)
        elif change == "transform":
            away = sc.M.copy().reshape(-1)
            away[12:15] += 50.0
            ctx.set_model_transform(sc.model, away.reshape(4, 4))
        else:
            ctx.set_grid_size(60.0)
        ctx.voxelize()
        if change == "grid":
            ctx.set_grid(res, 7, dtype, average)
        elif change == "transform":
            ctx.set_model_transform(sc.model, sc.M)
        else:
            ctx.set_grid_size(sc.cube_size)
        ctx.voxelize()
        got = ctx.download_level(0)
    want = orc.voxelize(res, sc.cube_size, sc.M, sc.pos, sc.nrm, sc.tri_mat, sc.mat_records, sc.lights,
                        want=("ref", "q32", "count"))
    assert want["count"].sum() > 6000
    w = want["ref"] if average == L.AVG_REFERENCE else encode_level(want["q32"], dtype)
    assert np.array_equal(bits(got), bits(w)), f"{np.count_nonzero(bits(got) != bits(w))} values differ"


# ---- voxelize under a model matrix (voxelize.vert:24-30) ----------------------------
@pytest.mark.parametrize("dtype,average", [(L.RGBA8, L.AVG_REFERENCE), (L.FP16, L.AVG_EXACT), (L.FP32, L.AVG_EXACT)])
def test_voxelize_with_model_matrix_bit_exact(gpu_available, orc, dtype, average):
    """Rotation, translation and non-uniform scale: world positions through
    the model matrix, normals through its inverse transpose."""
    say(f"voxelize with a model matrix dtype={dtype} average={average}")
    sc = SceneSpec("soup", res=128, ntri=20000, model="rot_scale")
    with Context(32, 32) as ctx:
        sc.build(ctx, dtype, average)
        ctx.voxelize()
        got = ctx.download_level(0)
    want = orc.voxelize(sc.res, sc.cube_size, sc.M, sc.pos, sc.nrm, sc.tri_mat, sc.mat_records, sc.lights,
                        want=("ref", "q32"))
    w = want["ref"] if average == L.AVG_REFERENCE else encode_level(want["q32"], dtype)
    assert np.array_equal(bits(got), bits(w)), "level 0 differs"


@pytest.mark.parametrize("dtype,average", [(L.RGBA8, L.AVG_REFERENCE), (L.FP16, L.AVG_EXACT)])
def test_voxelize_many_models_bit_exact(gpu_available, orc, dtype, average):
    """Any number of queued models (renderer.cpp:242-256): 37 draws, two of
    them with a model matrix, in one frame; two frames in a row."""
    say(f"voxelize over 37 models dtype={dtype} average={average}")
    from helpers import model_matrix

    sc = SceneSpec("soup", res=128, ntri=20000)
    cuts = np.linspace(0, 20000, 38).astype(int)
    draws = []
    with Context(32, 32) as ctx:
        sc.build(ctx, dtype, average)
        ctx.clear_queues()
        for k, (a, b) in enumerate(zip(cuts[:-1], cuts[1:])):
            m = ctx.model_create(sc.pos[a:b], sc.nrm[a:b], sc.tri_mat[a:b])
            M = model_matrix("rot_scale") if k in (3, 30) else sc.M
            ctx.set_model_transform(m, M)
            ctx.queue_model(m)
            draws.append((M, sc.pos[a:b], sc.nrm[a:b], sc.tri_mat[a:b]))
        for (p, c, i, k) in sc.lights:
            ctx.queue_light(p, c, i, k)
        for _ in range(2):  # the second frame reuses the draw table
            ctx.voxelize()
        got = ctx.download_level(0)
    want = orc.voxelize_draws(sc.res, sc.cube_size, draws, sc.mat_records, sc.lights, want=("ref", "q32"))
    w = want["ref"] if average == L.AVG_REFERENCE else encode_level(want["q32"], dtype)
    assert np.array_equal(bits(got), bits(w)), "level 0 differs"


# ---- G-buffer -----------------------------------------------------------------------
INSIDE = dict(eye=(0.12, 0.05, 0.2), target=(-0.25, -0.1, -0.5), fovy_deg=75.0)


@pytest.mark.parametrize("kind,ntri,W,H,extra", [
    ("cornell", 34, 96, 64, {}), ("soup", 5000, 160, 90, {}), ("cornell", 34, 512, 512, {}),
    ("soup", 40000, 640, 360, {}), ("soup", 3000, 100, 70, {}),
    # the camera inside the box: walls crossing the near plane are clipped and drawn as fans
    ("cornell", 34, 128, 96, INSIDE), ("cornell", 34, 640, 480, INSIDE),
    # a camera among the soup's triangles: many cross the near plane
    ("soup", 20000, 320, 180, dict(eye=(0.05, 0.02, 0.1), target=(0.4, -0.1, -1.0), fovy_deg=90.0)),
    # a model matrix (voxel_cone_tracing.vert:22-28)
    ("soup", 20000, 160, 90, dict(model="rot_scale"))],
    ids=["cornell", "soup", "cornell512", "soup640", "ragged", "inside", "inside640", "in_soup", "model"])
def test_gbuffer_bit_exact(gpu_available, orc, kind, ntri, W, H, extra):
    say(f"gbuffer parity kind={kind} {W}x{H} {extra}")
    sc = SceneSpec(kind, ntri=ntri, W=W, H=H, **extra)
    with Context(W, H) as ctx:
        sc.build(ctx, L.FP16)
        for _ in range(2):  # the second frame reuses the tile lists and counters
            ctx.gbuffer()
        gp, gn = ctx.download_gbuffer()
    p32, n32, _, _, keys = orc.gbuffer(W, H, sc.view, sc.proj, [(sc.M, sc.pos, sc.nrm, sc.tri_mat)])
    cov_g, cov_w = gp[..., 3] != 0, p32[..., 3] != 0
    assert cov_w.any()
    fans = int(((keys & np.uint64(7)) != 0).sum())
    say(f"  covered {int(cov_w.sum())} pixels, {fans} of them by fan triangles beyond the first")
    assert np.array_equal(cov_g, cov_w)
    assert np.array_equal(bits(gp), bits(p32))
    assert np.array_equal(bits(gn), bits(n32))


@pytest.mark.parametrize("ntri,W,H,extra", [
    (20000, 16, 16, {}), (129, 33, 31, {}), (128, 64, 64, {}), (60000, 83, 61, {}), (5000, 2048, 1024, {}),
    (20000, 70, 45, {"eye": (0.0, 0.1, 0.6), "target": (0.3, 0.0, -1.0)})])
def test_gbuffer_shared_tiles_bit_exact(gpu_available, orc, ntri, W, H, extra):
    """Viewports whose tiles several workgroups share: one tile, lists of one
    chunk and of one chunk and a triangle, more chunks than sharers, the last
    tile count with two sharers, clipped triangles from an eye inside; every
    frame twice, the second on the keys the first left."""
    say(f"gbuffer shared tiles {ntri} triangles {W}x{H}")
    sc = SceneSpec("soup", ntri=ntri, W=W, H=H, mu=-2.0, **extra)
    with Context(W, H) as ctx:
        sc.build(ctx, L.FP16)
        for _ in range(2):
            ctx.gbuffer()
            gp, gn = ctx.download_gbuffer()
            p32, n32, _, _, _ = orc.gbuffer(W, H, sc.view, sc.proj, [(sc.M, sc.pos, sc.nrm, sc.tri_mat)])
            assert (p32[..., 3] != 0).any()
            assert np.array_equal(bits(gp), bits(p32))
            assert np.array_equal(bits(gn), bits(n32))


@pytest.mark.parametrize("dtype,average", [(L.RGBA8, L.AVG_REFERENCE), (L.FP16, L.AVG_EXACT)])
@pytest.mark.parametrize("res,ntri", [(4, 300), (8, 2000), (16, 5000), (32, 40000), (64, 3000)])
def test_voxelize_small_grids_bit_exact(gpu_available, orc, res, ntri, dtype, average):
    """Grids on both sides of the brick edge's rule (4^3 bricks up to 32^3),
    down to the one that is a single brick."""
    say(f"voxelize small grid {res}^3 {ntri} triangles dtype={dtype}")
    sc = SceneSpec("soup", ntri=ntri, res=res, mu=-2.5)
    with Context(sc.W, sc.H) as ctx:
        sc.build(ctx, dtype, average)
        ctx.voxelize()
        lvl = ctx.download_level(0)
    key = "ref" if average == L.AVG_REFERENCE else "q32"
    want = orc.voxelize(res, sc.cube_size, sc.M, sc.pos, sc.nrm, sc.tri_mat, sc.mat_records, sc.lights, want=(key,))[key]
    assert np.array_equal(bits(lvl), bits(want if key == "ref" else encode_level(want, dtype)))


@pytest.mark.parametrize("W,H", [(4096, 4096), (4128, 4096)])
def test_gbuffer_tile_count_past_one_scan_workgroup(gpu_available, orc, W, H):
    """16,384 tiles, the most whose counts one workgroup scans, and 16,512,
    which take the three-launch scan."""
    say(f"gbuffer parity at {W}x{H}")
    sc = SceneSpec("soup", ntri=1500, W=W, H=H)
    with Context(W, H) as ctx:
        sc.build(ctx, L.RGBA8)
        ctx.gbuffer()
        gp, gn = ctx.download_gbuffer()
    p32, n32, _, _, _ = orc.gbuffer(W, H, sc.view, sc.proj, [(sc.M, sc.pos, sc.nrm, sc.tri_mat)])
    assert (p32[..., 3] != 0).any()
    assert np.array_equal(bits(gp), bits(p32))
    assert np.array_equal(bits(gn), bits(n32))


def test_gbuffer_many_models(gpu_available, orc):
    """Any number of queued models (renderer.cpp:242-256): 37 draws, two of
    them with a model matrix, camera inside the soup (clipped triangles)."""
    say("gbuffer parity over 37 models")
    from helpers import model_matrix

    sc = SceneSpec("soup", ntri=6000, W=200, H=120, eye=(0.05, 0.02, 0.6), target=(0.0, 0.0, -1.0), fovy_deg=80.0)
    cuts = np.linspace(0, 6000, 38).astype(int)
    draws = []
    with Context(sc.W, sc.H) as ctx:
        sc.build(ctx, L.FP16)
        ctx.clear_queues()
        for k, (a, b) in enumerate(zip(cuts[:-1], cuts[1:])):
            m = ctx.model_create(sc.pos[a:b], sc.nrm[a:b], sc.tri_mat[a:b])
            M = model_matrix("rot_scale") if k in (3, 30) else sc.M
            ctx.set_model_transform(m, M)
            ctx.queue_model(m)
            draws.append((M, sc.pos[a:b], sc.nrm[a:b], sc.tri_mat[a:b]))
        for _ in range(2):  # the second frame reuses the draw table and the lists
            ctx.gbuffer()
        gp, gn = ctx.download_gbuffer()
    p32, n32, _, _, _ = orc.gbuffer(sc.W, sc.H, sc.view, sc.proj, draws)
    assert (p32[..., 3] != 0).any()
    assert np.array_equal(bits(gp), bits(p32))
    assert np.array_equal(bits(gn), bits(n32))


def test_equal_draw_tables_on_both_streams(gpu_available):
    """An unchanged draw table is copied once, for the frame's second stream or
    the context's: passes called one by one and whole frames in turn, with the
    table unchanged, changed and changed back, give the buffers of a context
    that only runs that call."""
    say("draw tables, frames and single passes in turn")
    W, H = 320, 200
    sc = SceneSpec("soup", res=64, ntri=4000, W=W, H=H, mu=-3.0)
    moved = sc.M.copy().reshape(-1)
    moved[12:15] += 0.2

    def passes(ctx, whole, M):
        ctx.set_model_transform(sc.model, M)
        ctx.clear_queues()
        ctx.queue_model(sc.model)
        for (p, c, i, k) in sc.lights:
            ctx.queue_light(p, c, i, k)
        if whole:
            ctx.render()
        else:
            ctx.gbuffer()
            ctx.voxelize()
        return [bits(a) for a in (*ctx.download_gbuffer(), ctx.download_level(0))]

    want = {}
    for key, M in (("home", sc.M), ("moved", moved.reshape(4, 4))):
        with Context(W, H) as ctx:
            sc.build(ctx, L.FP16)
            want[key] = passes(ctx, False, M)
    assert not np.array_equal(want["home"][0], want["moved"][0])
    with Context(W, H) as ctx:
        sc.build(ctx, L.FP16)
        for whole, key in [(True, "home"), (False, "home"), (True, "home"), (True, "moved"), (False, "moved"),
                           (False, "home"), (True, "home"), (False, "home")]:
            got = passes(ctx, whole, sc.M if key == "home" else moved.reshape(4, 4))
            for g, w in zip(got, want[key]):
                assert np.array_equal(g, w), (whole, key)


def large_triangles(n, seed):
    """Triangles of 0.01 to 3 world units around and across the grid, every
    fourth a sliver, every fifth flat in a coordinate plane."""
    rng = np.random.default_rng(seed)
    size = np.exp(rng.uniform(np.log(0.01), np.log(3.0), (n, 1, 1)))
    p = rng.uniform(-1.3, 1.3, (n, 1, 3)) + size * rng.standard_normal((n, 3, 3)) * 0.5
    k = np.arange(n)
    sl = k % 4 == 0
    p[sl, 2] = p[sl, 0] + (p[sl, 1] - p[sl, 0]) * rng.uniform(0, 1, (sl.sum(), 1)) + \
        1e-3 * rng.standard_normal((sl.sum(), 3))
    for a in range(3):
        f = (k % 5 == 0) & (k % 3 == a)
        p[f, :, a] = p[f, :1, a]
    nrm = np.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0])
    nrm /= np.maximum(np.linalg.norm(nrm, axis=1, keepdims=True), 1e-12)
    return (np.ascontiguousarray(p.reshape(n, 9).astype(np.float32)),
            np.ascontiguousarray(np.repeat(nrm[:, None], 3, 1).reshape(n, 9).astype(np.float32)))


@pytest.mark.parametrize("n,res,W,H", [(1, 64, 40, 40), (65, 128, 700, 500), (4096, 64, 333, 190), (4097, 32, 64, 64),
                                       (20000, 128, 200, 120)])
def test_large_triangles_bit_exact(gpu_available, orc, n, res, W, H):
    """The set-up and list kernels take 64, 32 (4097 triangles) or 8 lanes per
    triangle here; boxes of more than 8 bricks or tiles go to the whole wave,
    which drops bricks and tiles the triangle cannot reach.  Level 0 in both
    averaging modes and the G-buffer must not notice."""
    say(f"large triangles n={n} res={res} {W}x{H}")
    sc = SceneSpec("soup", ntri=n, res=res, W=W, H=H)
    sc.pos, sc.nrm = large_triangles(n, n)
    want = orc.voxelize(res, sc.cube_size, sc.M, sc.pos, sc.nrm, sc.tri_mat, sc.mat_records, sc.lights,
                        want=("q32", "ref"))
    p32, n32, _, _, _ = orc.gbuffer(W, H, sc.view, sc.proj, [(sc.M, sc.pos, sc.nrm, sc.tri_mat)])
    with Context(W, H) as ctx:
        sc.build(ctx, L.FP16, L.AVG_EXACT)
        for _ in range(2):  # the second frame sizes its lists from the first one's count
            ctx.voxelize()
            got = ctx.download_level(0)
            assert np.array_equal(bits(got), bits(encode_level(want["q32"], L.FP16)))
        ctx.gbuffer()
        gp, gn = ctx.download_gbuffer()
        ctx.set_grid(res, 6, L.RGBA8, L.AVG_REFERENCE)
        ctx.voxelize()
        ref = ctx.download_level(0)
    assert np.array_equal(ref, want["ref"])
    assert np.array_equal(bits(gp), bits(p32))
    assert np.array_equal(bits(gn), bits(n32))


@pytest.mark.parametrize("res,n,size", [(4, 3, 1.0), (8, 1, 2.0), (8, 64, 1.0), (8, 129, 0.02), (8, 1024, 0.3),
                                        (8, 1025, 0.3), (16, 9000, 0.1), (64, 3000, 1.0)])
def test_reference_average_rounds_bit_exact(gpu_available, orc, res, n, size):
    """The reference average takes a brick's triangles sorted by original
    index (in LDS up to 1024 of them, by radix passes past that) in rounds of
    up to 128 whose fragments fit in LDS, halving a round that does not.
    Grids of one brick or few (8^3 voxels) with 1 to 9000 triangles each,
    from tiny ones (whole rounds) to ones that fill the brick's footprint
    (three a round), the triangles' order shuffled by the upload's own sort."""
    say(f"reference average rounds res={res} n={n} size={size}")
    rng = np.random.default_rng(n + res)
    p = rng.uniform(-1.0, 1.0, (n, 1, 3)) + size * rng.standard_normal((n, 3, 3))
    nrm = np.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0])
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    sc = SceneSpec("soup", ntri=n, res=res, W=16, H=16)
    sc.pos = np.ascontiguousarray(p.reshape(n, 9).astype(np.float32))
    sc.nrm = np.ascontiguousarray(np.repeat(nrm[:, None], 3, 1).reshape(n, 9).astype(np.float32))
    want = orc.voxelize(res, sc.cube_size, sc.M, sc.pos, sc.nrm, sc.tri_mat, sc.mat_records, sc.lights,
                        want=("ref", "count"))
    with Context(16, 16) as ctx:
        sc.build(ctx, L.RGBA8, L.AVG_REFERENCE)
        for _ in range(2):
            ctx.voxelize()
            got = ctx.download_level(0)
            assert np.array_equal(got, want["ref"])
        nfrag, _ = ctx.voxelize_stats()
    say(f"  {nfrag} fragments, up to {int(want['count'].max())} in a voxel")
    assert nfrag == int(want["count"].sum())


@pytest.mark.parametrize("res,n,size", [(64, 2000, 1.0), (64, 1200, 0.3)])
def test_reference_average_of_large_triangles_in_proportion(gpu_available, orc, res, n, size):
    """Bricks of triangles that fill their footprint, a few of which fit in a
    round, and of mixed sizes: the texels are the oracle's, and the average
    takes at most 12 times as long as the exact mean, which tests the same
    pixels once (a round that always starts from 128 triangles tests them 30
    to 60 times: 28.6 times as long at 2,000 triangles, 5.3 when rounds follow
    the fragments of the one before)."""
    say(f"reference average, large triangles, res={res} n={n} size={size}")
    rng = np.random.default_rng(n + res)
    p = rng.uniform(-1.0, 1.0, (n, 1, 3)) + size * rng.standard_normal((n, 3, 3))
    nrm = np.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0])
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    sc = SceneSpec("soup", ntri=n, res=res, W=16, H=16)
    sc.pos = np.ascontiguousarray(p.reshape(n, 9).astype(np.float32))
    sc.nrm = np.ascontiguousarray(np.repeat(nrm[:, None], 3, 1).reshape(n, 9).astype(np.float32))
    want = orc.voxelize(res, sc.cube_size, sc.M, sc.pos, sc.nrm, sc.tri_mat, sc.mat_records, sc.lights,
                        want=("ref", "count"))
    ms = {}
    for average in (L.AVG_REFERENCE, L.AVG_EXACT):
        with Context(16, 16) as ctx:
            sc.build(ctx, L.RGBA8, average)
            t = []
            for _ in range(6):
                ctx.voxelize()
                ctx.sync()
                t.append(float(ctx.pass_times()[0]))
            ms[average] = min(t)
            if average == L.AVG_REFERENCE:
                assert np.array_equal(ctx.download_level(0), want["ref"])
                assert ctx.voxelize_stats()[0] == int(want["count"].sum())
    say(f"  reference {ms[L.AVG_REFERENCE]:.3f} ms, exact mean {ms[L.AVG_EXACT]:.3f} ms")
    assert ms[L.AVG_REFERENCE] <= 12.0 * ms[L.AVG_EXACT]


@pytest.mark.parametrize("n", [2, 64, 65, 128, 129, 256, 257, 1024, 1025])
def test_reference_average_one_brick_bit_exact(gpu_available, orc, n):
    """n triangles inside one 8^3 brick of a 64^3 grid: the list sorted by rank
    (1, 2 or 4 lanes a triangle), by a bitonic sort past 256 triangles and by
    radix passes past 1024, and voxels with many fragments each."""
    say(f"reference average, {n} triangles in one brick")
    res = 64
    rng = np.random.default_rng(n)
    sc = SceneSpec("soup", ntri=n, res=res, W=16, H=16)
    centre = 0.125 * sc.cube_size  # the middle of the brick after the grid's
    p = centre * (1.0 + rng.uniform(-0.6, 0.6, (n, 1, 3))) + 0.02 * sc.cube_size * rng.uniform(-1.0, 1.0, (n, 3, 3))
    nrm = np.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0])
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    sc.pos = np.ascontiguousarray(p.reshape(n, 9).astype(np.float32))
    sc.nrm = np.ascontiguousarray(np.repeat(nrm[:, None], 3, 1).reshape(n, 9).astype(np.float32))
    want = orc.voxelize(res, sc.cube_size, sc.M, sc.pos, sc.nrm, sc.tri_mat, sc.mat_records, sc.lights,
                        want=("ref", "count"))
    z, y, x = np.nonzero(want["count"])
    assert (np.stack([z, y, x]) // 8 == 4).all()
    with Context(16, 16) as ctx:
        sc.build(ctx, L.RGBA8, L.AVG_REFERENCE)
        for _ in range(2):
            ctx.voxelize()
            assert np.array_equal(ctx.download_level(0), want["ref"])
        nfrag, _ = ctx.voxelize_stats()
    say(f"  {nfrag} fragments, up to {int(want['count'].max())} in a voxel")
    assert nfrag == int(want["count"].sum())


# ---- trace (kernel c) ----------------------------------------------------------------
@pytest.mark.parametrize("kind,dtype,res,ntri", [("cornell", L.RGBA8, 64, 34), ("cornell", L.FP16, 64, 34),
                                                 ("soup", L.FP16, 64, 4000), ("soup", L.BF16, 64, 4000),
                                                 ("soup", L.FP32, 64, 4000)])
def test_trace_matches_oracle(gpu_available, orc, kind, dtype, res, ntri):
    say(f"trace parity kind={kind} dtype={dtype}")
    W, H = 96, 64
    sc = SceneSpec(kind, res=res, ntri=ntri, W=W, H=H)
    levels = 7
    with Context(W, H) as ctx:
        sc.build(ctx, dtype)
        ctx.voxelize()
        ctx.mip()
        ctx.gbuffer()
        ctx.trace()
        img = ctx.download_image()
        gp, gn = ctx.download_gbuffer()
        l0 = decode_level(ctx.download_level(0), dtype)
        mips = {(l, d): decode_level(ctx.download_level(l, d), dtype) for l in range(1, levels) for d in range(6)}
    rng = np.random.default_rng(7)
    pix = np.sort(rng.choice(W * H, size=min(W * H, 1500), replace=False)).astype(np.int64)
    want, _ = orc.trace(np.float32, res, levels, l0, mips, gp, gn, sc.mat_records, sc.lights, sc.cam, sc.cube_size,
                        cone_set=sc.cone_set, pixels=pix)
    got = img.reshape(-1, 4)[pix]
    err = np.abs(got[:, :3] - want[:, :3]).max()
    say(f"  max-abs vs FP32 oracle = {err:.3e}")
    assert err <= 2e-3


@pytest.mark.parametrize("case", ["cones16", "lights3"])
def test_trace_full_block_shape_matches_oracle(gpu_available, orc, case):
    """Configurations beyond the 128-pixel block shape (more than 9 diffuse
    cones, or shadow cones of more than 2 lights) run the 64-pixel shape with
    every LDS slot; same oracle bar as the other trace tests."""
    say(f"trace parity, full block shape: {case}")
    W, H, res = 96, 64, 64
    if case == "cones16":
        sc = SceneSpec("soup", res=res, ntri=4000, W=W, H=H)
        sc.cone_set = L.CONES_16
    else:
        sc = SceneSpec("cornell", res=res, W=W, H=H, glass=True, phases=(True, True, True, True))
        sc.lights = sc.lights + [((0.3, 0.2, 0.35), (0.9, 0.6, 0.4), 0.7, L.LIGHT_POINT),
                                 ((-0.6, 1.0, 0.8), (0.5, 0.6, 1.0), 0.8, L.LIGHT_DIRECTIONAL)]
    with Context(W, H) as ctx:
        sc.build(ctx, L.FP16)
        ctx.render()
        img = ctx.download_image()
        gp, gn = ctx.download_gbuffer()
        l0 = decode_level(ctx.download_level(0), L.FP16)
        mips = {(l, d): decode_level(ctx.download_level(l, d), L.FP16) for l in range(1, 7) for d in range(6)}
    cov = gp[..., 3].reshape(-1) != 0
    pix = np.flatnonzero(cov).astype(np.int64)
    assert pix.size > 0
    want, _ = orc.trace(np.float32, res, 7, l0, mips, gp, gn, sc.mat_records, sc.lights, sc.cam, sc.cube_size,
                        cone_set=sc.cone_set, phases=sc.phases, pixels=pix)
    err = np.abs(img.reshape(-1, 4)[pix, :3] - want[:, :3]).max()
    say(f"  max-abs vs FP32 oracle = {err:.3e}")
    assert err <= 2e-3


@pytest.mark.parametrize("dtype", [L.RGBA8, L.FP16])
def test_full_compose_matches_oracle(gpu_available, orc, dtype):
    """All phases on (direct light + shadow cones, diffuse, specular and
    refraction cones, emission, the transmissive override), on the GPU's own
    volume and G-buffer."""
    say(f"full compose parity dtype={dtype}")
    W, H, res = 128, 96, 64
    sc = SceneSpec("cornell", res=res, W=W, H=H, glass=True, phases=(True, True, True, True))
    with Context(W, H) as ctx:
        sc.build(ctx, dtype)
        ctx.render()
        img = ctx.download_image()
        gp, gn = ctx.download_gbuffer()
        l0 = decode_level(ctx.download_level(0), dtype)
        mips = {(l, d): decode_level(ctx.download_level(l, d), dtype) for l in range(1, 7) for d in range(6)}
    cov = gp[..., 3].reshape(-1) != 0
    pix = np.flatnonzero(cov).astype(np.int64)
    want, _ = orc.trace(np.float32, res, 7, l0, mips, gp, gn, sc.mat_records, sc.lights, sc.cam, sc.cube_size,
                        cone_set=sc.cone_set, phases=sc.phases, pixels=pix)
    err = np.abs(img.reshape(-1, 4)[pix, :3] - want[:, :3]).max()
    say(f"  max-abs vs FP32 oracle = {err:.3e}")
    assert err <= 2e-3


def test_pass_timing_mask(gpu_available):
    """vct_set_pass_timing: with timing off the frame is the same bit for bit
    and every pass reads 0 ms; a pass left out of the mask reads 0 while the
    others are timed; a mask past pass 5 is an error."""
    say("pass timing mask")
    W, H, res = 96, 64, 64
    sc = SceneSpec("cornell", res=res, W=W, H=H)

    def frame(ctx):
        ctx.clear_queues()
        ctx.queue_model(sc.model)
        for (p, c, i, k) in sc.lights:
            ctx.queue_light(p, c, i, k)
        ctx.render()
        return ctx.download_image(), ctx.pass_times()

    with Context(W, H) as ctx:
        sc.build(ctx, L.FP16)
        img_on, t_on = frame(ctx)
        ctx.set_pass_timing(0)
        img_off, t_off = frame(ctx)
        ctx.set_pass_timing(0x3F & ~(1 << 3))  # all but the trace
        _, t_some = frame(ctx)
        with pytest.raises(L.VctError):
            ctx.set_pass_timing(0x40)
    say(f"  on {np.round(t_on[:4], 4)}, off {t_off[:4]}, no trace {np.round(t_some[:4], 4)}")
    assert np.array_equal(img_on, img_off)
    assert (t_on[:4] > 0).all() and (t_off == 0).all()
    assert t_some[3] == 0 and (t_some[[0, 1, 2]] > 0).all()


def test_trace_ragged_viewport_matches_oracle(gpu_available, orc):
    """A viewport whose block grid is ragged: 88x100 is 6 x 13 blocks of
    16x8 pixels, partial on the right and bottom edges, 8 block rows in the
    XCD-interleaved order and 5 left in dispatch order.  The Cornell scene
    covers every pixel, so a block traced twice or not at all shows up."""
    say("trace parity, ragged 88x100 viewport")
    W, H, res = 88, 100, 64
    sc = SceneSpec("cornell", res=res, W=W, H=H, glass=True, phases=(True, True, True, True))
    with Context(W, H) as ctx:
        sc.build(ctx, L.FP16)
        ctx.render()
        img = ctx.download_image()
        gp, gn = ctx.download_gbuffer()
        l0 = decode_level(ctx.download_level(0), L.FP16)
        mips = {(l, d): decode_level(ctx.download_level(l, d), L.FP16) for l in range(1, 7) for d in range(6)}
    cov = gp[..., 3].reshape(-1) != 0
    assert cov.all()
    pix = np.arange(W * H, dtype=np.int64)
    want, _ = orc.trace(np.float32, res, 7, l0, mips, gp, gn, sc.mat_records, sc.lights, sc.cam, sc.cube_size,
                        cone_set=sc.cone_set, phases=sc.phases, pixels=pix)
    err = np.abs(img.reshape(-1, 4)[:, :3] - want[:, :3]).max()
    say(f"  max-abs vs FP32 oracle = {err:.3e}")
    assert err <= 2e-3


@pytest.mark.parametrize("dtype", [L.RGBA8, L.FP16, L.BF16, L.FP32])
def test_trace_wide_blocks_ragged_viewport_matches_oracle(gpu_available, orc, dtype):
    """A viewport past the small block shape (over 2^18 pixels) that no block
    width divides (521 = 21 x 24 + 17 = 32 x 16 + 9; 509 = 63 x 8 + 5): the
    wide shape of each storage type, its partial blocks on both edges and the
    block rows past a multiple of 8.  A block's pixels are queued in sorted
    order, so a pixel dropped or taken twice by the sort shows up as well."""
    say(f"trace parity, ragged 521x509 viewport, dtype={dtype}")
    W, H, res = 521, 509, 64
    sc = SceneSpec("cornell", res=res, W=W, H=H, glass=True, phases=(True, True, True, True))
    with Context(W, H) as ctx:
        sc.build(ctx, dtype)
        ctx.render()
        img = ctx.download_image()
        gp, gn = ctx.download_gbuffer()
        l0 = decode_level(ctx.download_level(0), dtype)
        mips = {(l, d): decode_level(ctx.download_level(l, d), dtype) for l in range(1, 7) for d in range(6)}
    edge = np.zeros((H, W), bool)
    edge[-6:, :] = True
    edge[:, -18:] = True
    edge[248:256, 240:288] = True  # two whole 24-pixel blocks, three 16-pixel ones
    edge.reshape(-1)[np.random.default_rng(3).choice(W * H, 2000, replace=False)] = True
    cov = gp[..., 3] != 0
    pix = np.flatnonzero(edge & cov).astype(np.int64)
    assert pix.size > 10000
    want, _ = orc.trace(np.float32, res, 7, l0, mips, gp, gn, sc.mat_records, sc.lights, sc.cam, sc.cube_size,
                        cone_set=sc.cone_set, phases=sc.phases, pixels=pix)
    err = np.abs(img.reshape(-1, 4)[pix, :3] - want[:, :3]).max()
    say(f"  {pix.size} pixels, max-abs vs FP32 oracle = {err:.3e}")
    assert err <= 2e-3


@pytest.mark.parametrize("dtype", [L.RGBA8, L.FP16, L.BF16, L.FP32])
@pytest.mark.parametrize("W,H", [(811, 653), (1013, 781)])
def test_trace_block_shapes_ragged_viewport_matches_oracle(gpu_available, orc, dtype, W, H):
    """The shapes of viewports past 2^19 pixels (811 = 50 x 16 + 11, 653 = 81 x 8
    + 5: 128-pixel blocks) and past 3 * 2^18 (1013 = 42 x 24 + 5 = 63 x 16 + 5,
    781 = 97 x 8 + 5: 192-pixel blocks in the 16-bit types): partial blocks on
    both edges, block rows past a multiple of 8, whole blocks inside."""
    say(f"trace parity, ragged {W}x{H} viewport, dtype={dtype}")
    assert (1 << 19) < W * H and (W * H <= 3 << 18) == (W == 811)
    res = 64
    sc = SceneSpec("cornell", res=res, W=W, H=H, glass=True, phases=(True, True, True, True),
                   fovy_deg=40.0)  # the box fills the window, edges included
    with Context(W, H) as ctx:
        sc.build(ctx, dtype)
        ctx.render()
        img = ctx.download_image()
        gp, gn = ctx.download_gbuffer()
        l0 = decode_level(ctx.download_level(0), dtype)
        mips = {(l, d): decode_level(ctx.download_level(l, d), dtype) for l in range(1, 7) for d in range(6)}
    pick = np.zeros((H, W), bool)
    pick[-6:, :] = True
    pick[:, -6:] = True
    pick[392:400, 480:528] = True  # two whole 24-pixel blocks, three 16-pixel ones
    pick.reshape(-1)[np.random.default_rng(W).choice(W * H, 2000, replace=False)] = True
    pix = np.flatnonzero(pick & (gp[..., 3] != 0)).astype(np.int64)
    assert pix.size > 8000
    want, _ = orc.trace(np.float32, res, 7, l0, mips, gp, gn, sc.mat_records, sc.lights, sc.cam, sc.cube_size,
                        cone_set=sc.cone_set, phases=sc.phases, pixels=pix)
    err = np.abs(img.reshape(-1, 4)[pix, :3] - want[:, :3]).max()
    say(f"  {pix.size} pixels, max-abs vs FP32 oracle = {err:.3e}")
    assert err <= 2e-3


@pytest.mark.parametrize("view_dir,lod,extra,dtype", [
    (0, 0.0, {}, L.RGBA8), (3, 1.5, {}, L.RGBA8), (5, 4.0, {}, L.FP16),
    # the camera inside the box: clipped walls drawn as fans, in draw order
    (1, 0.5, dict(eye=(0.12, 0.05, 0.2), target=(-0.25, -0.1, -0.5), fovy_deg=75.0), L.RGBA8)])
def test_voxel_view_matches_oracle(gpu_available, orc, view_dir, lod, extra, dtype):
    """The voxel-view debug path (voxel_cone_tracing.frag:253-257) with GL's
    in-order SRC_ALPHA blending of every fragment that passes the depth test
    (renderer.cpp:384-388), against the oracle's sequential draw."""
    say(f"voxel view dir={view_dir} lod={lod} {extra} dtype={dtype}")
    W, H, res = 96, 64, 64
    sc = SceneSpec("cornell", res=res, W=W, H=H, **extra)
    with Context(W, H) as ctx:
        sc.build(ctx, dtype)
        ctx.set_voxel_view(view_dir, lod)
        ctx.render()
        # a second frame reuses the sort buffers
        ctx.queue_model(sc.model)
        for (p, c, i, k) in sc.lights:
            ctx.queue_light(p, c, i, k)
        ctx.render()
        img = ctx.download_image()
        l0 = decode_level(ctx.download_level(0), dtype)
        mips = {(l, d): decode_level(ctx.download_level(l, d), dtype) for l in range(1, 7) for d in range(6)}
    want = orc.voxel_view(W, H, sc.view, sc.proj, [(sc.M, sc.pos)], res, 7, l0, mips, sc.cube_size, view_dir, lod)
    err = np.abs(img - want).max()
    say(f"  max-abs vs FP32 oracle = {err:.3e}")
    assert err == 0.0  # the same float operations in the same order (measured bit-exact)


@pytest.mark.parametrize("n,W,H,extra", [(64, 70, 45, {}), (65, 33, 64, {}), (400, 96, 64, {}),
                                         (150, 61, 47, dict(eye=(0.05, 0.02, 0.1), target=(0.4, -0.1, -1.0),
                                                            fovy_deg=90.0))])
def test_voxel_view_chunks_match_oracle(gpu_available, orc, n, W, H, extra):
    """Tiles with more entries than the composite stages at a time (64), at
    viewports that cut its 8x8 blocks, with overlapping triangles of all sizes
    in draw order, the last case clipped around the eye."""
    say(f"voxel view chunks n={n} {W}x{H} {extra}")
    res = 32
    sc = SceneSpec("soup", ntri=n, res=res, W=W, H=H, **extra)
    sc.pos, sc.nrm = large_triangles(n, n + 1)
    with Context(W, H) as ctx:
        sc.build(ctx, L.FP16)
        ctx.set_voxel_view(3, 0.6)
        ctx.render()
        img = ctx.download_image()
        l0 = decode_level(ctx.download_level(0), L.FP16)
        mips = {(l, d): decode_level(ctx.download_level(l, d), L.FP16) for l in range(1, 6) for d in range(6)}
    want = orc.voxel_view(W, H, sc.view, sc.proj, [(sc.M, sc.pos)], res, 6, l0, mips, sc.cube_size, 3, 0.6)
    err = np.abs(img - want).max()
    say(f"  max-abs vs FP32 oracle = {err:.3e}")
    assert err == 0.0


def test_voxel_view_over_many_models(gpu_available, orc):
    """Draw order runs over the queued models (renderer.cpp:242-256): the
    Cornell box split into 5 models queued in reverse, two of them moved."""
    say("voxel view over 5 models")
    from helpers import model_matrix

    W, H, res = 96, 64, 64
    sc = SceneSpec("cornell", res=res, W=W, H=H)
    cuts = np.linspace(0, sc.pos.shape[0], 6).astype(int)
    draws = []
    with Context(W, H) as ctx:
        sc.build(ctx, L.RGBA8)
        ctx.clear_queues()
        models = []
        for k, (a, b) in enumerate(zip(cuts[:-1], cuts[1:])):
            m = ctx.model_create(sc.pos[a:b], sc.nrm[a:b], sc.tri_mat[a:b])
            M = model_matrix("rot_scale") if k in (1, 3) else sc.M
            ctx.set_model_transform(m, M)
            models.append((m, M, sc.pos[a:b]))
        for m, M, pos in reversed(models):
            ctx.queue_model(m)
            draws.append((M, pos))
        for (p, c, i, k) in sc.lights:
            ctx.queue_light(p, c, i, k)
        ctx.set_voxel_view(2, 0.7)
        ctx.render()
        img = ctx.download_image()
        l0 = decode_level(ctx.download_level(0), L.RGBA8)
        mips = {(l, d): decode_level(ctx.download_level(l, d), L.RGBA8) for l in range(1, 7) for d in range(6)}
    want = orc.voxel_view(W, H, sc.view, sc.proj, draws, res, 7, l0, mips, sc.cube_size, 2, 0.7)
    err = np.abs(img - want).max()
    say(f"  max-abs vs FP32 oracle = {err:.3e}")
    assert err == 0.0  # the same float operations in the same order (measured bit-exact)


@pytest.mark.parametrize("dtype", [L.RGBA8, L.FP16, L.BF16, L.FP32])
@pytest.mark.parametrize("view_dir,lod", [(1, 0.0), (2, 0.6), (4, 2.3)])
def test_sampler_at_the_volume_faces(gpu_available, orc, dtype, view_dir, lod):
    """The marcher's sampler (x-paired texels for 8- and 16-bit storage) on a
    random volume at points spread over the whole cube and up to half a texel
    past its faces, where the zero border and the first / last columns meet
    (the voxel view samples exactly one textureLod per pixel)."""
    say(f"sampler at faces dtype={dtype} dir={view_dir} lod={lod}")
    W, H, res, levels = 64, 32, 8, 4
    sc = SceneSpec("cornell", res=res, W=W, H=H)
    rng = np.random.default_rng(100 + dtype)
    with Context(W, H) as ctx:
        sc.build(ctx, dtype, levels=levels)
        want_levels = {}
        for lvl in range(levels):
            s = res >> lvl
            for d in range(1 if lvl == 0 else 6):
                f = rng.random((s, s, s, 4)).astype(np.float32)
                enc = encode_level(f, dtype)
                ctx.upload_level(lvl, d, enc)
                want_levels[(lvl, d)] = decode_level(enc, dtype)
        # biased coordinates in [-0.06, 0.999]: columns -1 and s-1 of every level are hit
        b = rng.uniform(-0.06, 0.999, (H, W, 3)).astype(np.float32)
        b[0, :, 0] = -0.5 / res + 1e-3  # the first texel's left border, level 0
        b[1, :, 0] = 1.0 - 0.5 / res + 1e-3  # past the last texel centre, level 0
        world = (b - 0.5) * 2.0 * sc.cube_size
        gp = np.concatenate([world, np.ones((H, W, 1), np.float32)], -1).astype(np.float32)
        gn = np.zeros((H, W, 4), np.float32)
        gn[..., 1] = 1.0
        gn[..., 3] = np.uint32(1).view(np.float32)
        ctx.upload_gbuffer(gp, gn)
        ctx.set_voxel_view(view_dir, lod)
        ctx.trace()
        img = ctx.download_image()
    l0 = want_levels[(0, 0)]
    mips = {(lv, d): want_levels[(lv, d)] for lv in range(1, levels) for d in range(6)}
    want, _ = orc.trace(np.float32, res, levels, l0, mips, gp, gn, sc.mat_records, sc.lights, sc.cam, sc.cube_size,
                        cone_set=sc.cone_set, phases=sc.phases, view_dir=view_dir, view_lod=lod)
    err = np.abs(img.reshape(-1, 4) - want).max()
    say(f"  max-abs vs FP32 oracle = {err:.3e}")
    # 16-bit pairs blend with weights rounded to the storage type (2^-11 / 2^-8)
    assert err <= {L.RGBA8: 1e-5, L.FP16: 2e-3, L.BF16: 1.6e-2, L.FP32: 1e-5}[dtype]


@pytest.mark.parametrize("dtype", [L.RGBA8, L.FP16, L.BF16, L.FP32])
@pytest.mark.parametrize("res,levels,lod", [(8, 4, 3.0), (8, 4, 2.5), (4, 3, 1.3), (4, 1, 0.0), (4, 2, 7.0),
                                            (32, 6, 0.5), (128, 2, 0.4)])
def test_sampler_far_past_the_faces(gpu_available, orc, dtype, res, levels, lod):
    """One sample per pixel at points from 1.5 texels of the coarsest level
    before the cube to as far behind it, in levels down to a single texel: the
    two texels an axis reads are clamped into the level, so the weights alone
    have to make the border zero, on both sides and in the level of one texel
    (where the second texel has no place at all)."""
    say(f"sampler past faces dtype={dtype} res={res} levels={levels} lod={lod}")
    W, H = 64, 48
    sc = SceneSpec("cornell", res=res, W=W, H=H)
    rng = np.random.default_rng(7 + dtype)
    far = 1.5 * 2.0 ** (levels - 1) / res
    with Context(W, H) as ctx:
        sc.build(ctx, dtype, levels=levels)
        maps = {}
        for lvl in range(levels):
            s = res >> lvl
            for d in range(1 if lvl == 0 else 6):
                enc = encode_level(rng.random((s, s, s, 4)).astype(np.float32), dtype)
                ctx.upload_level(lvl, d, enc)
                maps[(lvl, d)] = decode_level(enc, dtype)
        b = rng.uniform(-far, 1.0 + far, (H, W, 3)).astype(np.float32)
        b[: H // 2] = np.clip(b[: H // 2], 0.01, 0.99)  # half of them inside
        b[0, :, 1] = 1.0 + 0.25 * far
        b[1, :, 2] = -0.25 * far
        world = (b - 0.5) * 2.0 * sc.cube_size
        gp = np.concatenate([world, np.ones((H, W, 1), np.float32)], -1).astype(np.float32)
        gn = np.zeros((H, W, 4), np.float32)
        gn[..., 1] = 1.0
        gn[..., 3] = np.uint32(1).view(np.float32)
        ctx.upload_gbuffer(gp, gn)
        ctx.set_voxel_view(3, lod)
        ctx.trace()
        img = ctx.download_image()
    mips = {k: v for k, v in maps.items() if k[0] > 0}
    want, _ = orc.trace(np.float32, res, levels, maps[(0, 0)], mips, gp, gn, sc.mat_records, sc.lights, sc.cam,
                        sc.cube_size, cone_set=sc.cone_set, phases=sc.phases, view_dir=3, view_lod=lod)
    err = np.abs(img.reshape(-1, 4) - want).max()
    say(f"  max-abs vs FP32 oracle = {err:.3e}")
    # 16-bit pairs blend with weights rounded to the storage type (2^-11 / 2^-8)
    assert err <= {L.RGBA8: 1e-5, L.FP16: 2e-3, L.BF16: 1.6e-2, L.FP32: 1e-5}[dtype]


@pytest.mark.parametrize("dtype,res,levels", [(L.RGBA8, 32, 1), (L.FP32, 32, 2), (L.FP16, 64, 4), (L.RGBA8, 16, 5)])
def test_cones_end_past_the_volume(gpu_available, orc, dtype, res, levels):
    """Cones that leave the volume through every face, with mip chains cut
    short (the coarsest texel sets how far out a cone still reads): the exit
    distance changes no pixel, and the steps taken are those of the oracle's
    loop that tests the position at every step."""
    say(f"cone exits dtype={dtype} res={res} levels={levels}")
    W, H = 96, 64
    sc = SceneSpec("soup", res=res, ntri=20000, W=W, H=H)
    with Context(W, H) as ctx:
        sc.build(ctx, dtype, levels=levels)
        ctx.render()
        img = ctx.download_image()
        steps = ctx.trace_steps()
        gp, gn = ctx.download_gbuffer()
        l0 = decode_level(ctx.download_level(0), dtype)
        mips = {(l, d): decode_level(ctx.download_level(l, d), dtype) for l in range(1, levels) for d in range(6)}
    want, (_, live) = orc.trace(np.float32, res, levels, l0, mips, gp, gn, sc.mat_records, sc.lights, sc.cam,
                                sc.cube_size, cone_set=sc.cone_set, early_exit_steps=True)
    cov = (gp[..., 3] != 0).reshape(-1)
    assert cov.sum() > 500
    err = np.abs(img.reshape(-1, 4)[cov, :3] - want[cov, :3]).max()
    rel = abs(int(steps) - int(live)) / live
    say(f"  {int(cov.sum())} pixels, max-abs vs FP32 oracle = {err:.3e}; steps GPU {steps}, oracle {live}")
    assert err <= 2e-3
    assert rel <= 1e-3
