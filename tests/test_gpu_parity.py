"""GPU parity: libvpt.so (through the C ABI) against the CPU oracle.

Bar: bit-exact distance field, hit cells, faces, block ids and shadow masks;
hit distance within 1e-5 relative (the kernels reproduce the oracle's IEEE
operation sequence, so in practice t is bit-exact too); GI radiance and SVGF
planes compared exactly where the operation sequences coincide and at most
1e-3 relative mean radiance after the full SVGF chain.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import oracle
from tests.helpers import (OracleSVGF, camera, f16, gi_planes_from_oracle, random_world, rel_l1, svgf_camera_path,
                           terrain, u8n)
from voxelpathtracer_amd import World, decode_texels, gi_params, viewproj
from voxelpathtracer_amd._lib import Hit, Ray
from voxelpathtracer_amd.world import DeviceGBuffer

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    return torch


def _world(ctx, grid):
    nz, ny, nx = grid.shape
    w = World(ctx, nx, ny, nz)
    w.m_WorldData[...] = grid
    w.Buffer()
    w.GenerateDistanceField()
    return w


# ---------------------------------------------------------------- DF build

@pytest.mark.parametrize("shape,density,seed", [
    ((32, 16, 32), 0.0, 1),        # empty world: 254 everywhere
    ((32, 16, 32), 1.0, 2),        # full world: 0 everywhere
    ((32, 16, 32), 0.002, 3),
    ((48, 8, 16), 0.05, 4),
    ((64, 32, 64), 0.3, 5),
    ((16, 8, 8), 0.1, 6),          # smallest allowed dims
    # rows of one to four 256-cell chunks of the slab X pass, partial last
    # chunks, and more rows than one batch of a wavefront (with columns
    # longer than the register-held Y segments)
    ((80, 16, 16), 0.02, 7),
    ((400, 24, 16), 0.01, 8),
    ((640, 32, 16), 0.01, 11),
    ((1008, 16, 8), 0.005, 9),
    ((1024, 8, 16), 0.3, 10),
    ((128, 512, 8), 0.01, 12),
    ((64, 16, 256), 0.02, 13),     # 16-layer Z segments
])
def test_df_random_worlds(ctx, shape, density, seed):
    rng = np.random.default_rng(seed)
    nx, ny, nz = shape
    g = random_world(rng, nx, ny, nz, density)
    print(f"df parity {shape} density {density}", flush=True)
    w = _world(ctx, g)
    np.testing.assert_array_equal(w.download_grid(), g)
    np.testing.assert_array_equal(w.download_df(), oracle.df_build(g))
    w.close()


def test_df_single_voxel(ctx):
    g = np.zeros((64, 64, 64), np.uint8)
    g[17, 40, 5] = 9
    w = _world(ctx, g)
    df = w.download_df()
    z, y, x = np.meshgrid(np.arange(64), np.arange(64), np.arange(64), indexing="ij")
    expect = np.minimum(254, np.abs(x - 5) + np.abs(y - 40) + np.abs(z - 17)).astype(np.uint8)
    np.testing.assert_array_equal(df, expect)
    w.close()


@pytest.mark.parametrize("dims", [(384, 128, 384), (512, 256, 512)])
def test_df_terrain_full_size(ctx, dims):
    nx, ny, nz = dims
    print(f"df parity terrain {dims}", flush=True)
    g = terrain(nx, ny, nz)
    w = _world(ctx, g)
    np.testing.assert_array_equal(w.download_df(), oracle.df_build(g))
    w.close()


def test_df_after_edits(ctx):
    """Block edits then a rebuild (World.cpp:367-375 + GenerateDistanceField)."""
    g = terrain(128, 64, 128, h_min=10, h_max=40)
    w = _world(ctx, g)
    rng = np.random.default_rng(11)
    for _ in range(50):
        x, y, z = int(rng.integers(0, 128)), int(rng.integers(0, 64)), int(rng.integers(0, 128))
        b = int(rng.integers(0, 5))
        w.SetBlock(x, y, z, b)
        g[z, y, x] = b
    w.GenerateDistanceField()
    np.testing.assert_array_equal(w.download_grid(), g)
    np.testing.assert_array_equal(w.download_df(), oracle.df_build(g))
    w.close()


# ---------------------------------------------------------------- rays

def _check_gbuffer(gb, ref):
    np.testing.assert_array_equal(gb["face"], ref["face"])
    np.testing.assert_array_equal(gb["block"], ref["block"])
    np.testing.assert_array_equal(gb["voxel"], ref["voxel"])
    hit = ref["face"] != 255
    t, rt = gb["t"], ref["t"]
    rel = np.abs(t[hit] - rt[hit]) / np.maximum(np.abs(rt[hit]), 1e-30)
    assert rel.size == 0 or rel.max() <= 1e-5, rel.max()
    np.testing.assert_array_equal(t[~hit], rt[~hit])
    return float((t == rt).mean())


@pytest.fixture(scope="module")
def terrain_world(ctx):
    g = terrain()
    w = _world(ctx, g)
    df = oracle.df_build(g)
    yield g, df, w
    w.close()


@pytest.mark.parametrize("W,H", [(640, 360), (1920, 1080), (333, 97)])
def test_primary_parity(terrain_world, W, H):
    g, df, w = terrain_world
    torch = _torch()
    print(f"primary parity {W}x{H}", flush=True)
    cam, view, proj, iv, ip = camera(W, H)
    gb = DeviceGBuffer(W, H)
    w.trace_primary(cam, gb, 350)
    torch.cuda.synchronize()
    ref = oracle.trace_primary(g, df, iv, ip, W, H, 350)
    exact = _check_gbuffer(gb.numpy(), ref)
    assert exact == 1.0, f"t bit-exact fraction {exact}"


@pytest.fixture(scope="module")
def gbuffer_1080(terrain_world):
    g, df, w = terrain_world
    torch = _torch()
    W, H = 1920, 1080
    cam, view, proj, iv, ip = camera(W, H)
    gb = DeviceGBuffer(W, H)
    w.trace_primary(cam, gb, 350)
    torch.cuda.synchronize()
    return cam, iv, ip, gb


def test_shadow_parity(terrain_world, gbuffer_1080):
    g, df, w = terrain_world
    torch = _torch()
    cam, iv, ip, gb = gbuffer_1080
    prm = gi_params()
    mask = torch.empty((cam.height, cam.width), dtype=torch.uint8, device="cuda")
    w.trace_shadow(cam, gb, list(prm.sun_dir), mask, 350)
    torch.cuda.synchronize()
    host = gb.numpy()
    ref = oracle.trace_shadow(g, df, iv, ip, host["t"], host["face"], np.array(prm.sun_dir, np.float32), 350)
    np.testing.assert_array_equal(mask.cpu().numpy(), ref["mask"])
    assert 0.05 < ref["mask"].mean() < 0.95


def test_gi_parity(terrain_world, gbuffer_1080):
    g, df, w = terrain_world
    torch = _torch()
    cam, iv, ip, gb = gbuffer_1080
    prm = gi_params(frame=3)
    rgb = torch.empty((cam.height, cam.width, 3), dtype=torch.float32, device="cuda")
    tex = torch.empty((cam.height, cam.width, 8), dtype=torch.int16, device="cuda")
    w.trace_gi(cam, gb, prm, rgb, tex)
    torch.cuda.synchronize()
    host = gb.numpy()
    ref = oracle.trace_gi(g, df, iv, ip, host["t"], host["face"], oracle.gi_params_from(prm))
    np.testing.assert_array_equal(rgb.cpu().numpy(), ref["rgb"])
    d = decode_texels(tex.cpu().numpy().view(np.uint16))
    planes = gi_planes_from_oracle(ref)
    np.testing.assert_array_equal(d["sh"], planes["sh"])
    np.testing.assert_array_equal(d["cocg"], planes["cocg"])
    np.testing.assert_array_equal(d["x"], planes["luma"])
    np.testing.assert_array_equal(d["ao"], planes["ao"])


@pytest.mark.parametrize("W,H,gi_iter", [
    (17, 9, 48),        # one 16x16 tile row, fewer tiles than XCDs
    (40, 40, 48),       # 9 tiles: one per XCD plus a leftover
    (129, 3, 48),       # ragged last tile, 1-pixel-high rows
    (333, 97, 48),
    (640, 360, 0),      # no bounce step at all
    (640, 360, 1),
    (640, 360, 24),     # exactly the bounce kernel's step budget: no continuation
    (640, 360, 25),     # continued rays take one more step
    (640, 360, 200),
])
def test_gi_parity_sizes_and_caps(terrain_world, W, H, gi_iter):
    """The GI pass (bounce kernel, continuations after 24 steps, shadow
    jobs; per-XCD queues sized from the tile layout) equals the oracle at
    sizes with fewer tiles than XCDs, ragged tiles and iteration caps on
    both sides of the bounce kernel's 24 steps, and counts the oracle's DF
    samples and rays."""
    g, df, w = terrain_world
    torch = _torch()
    print(f"gi parity {W}x{H} gi_iter {gi_iter}", flush=True)
    cam, view, proj, iv, ip = camera(W, H)
    gb = DeviceGBuffer(W, H)
    w.trace_primary(cam, gb, 350)
    prm = gi_params(frame=5)
    prm.gi_iter = gi_iter
    rgb = torch.empty((H, W, 3), dtype=torch.float32, device="cuda")
    tex = torch.empty((H, W, 8), dtype=torch.int16, device="cuda")
    counter = torch.zeros(2, dtype=torch.int64, device="cuda")
    w.set_sample_counter(counter)
    w.trace_gi(cam, gb, prm, rgb, tex)
    w.set_sample_counter(None)
    torch.cuda.synchronize()
    host = gb.numpy()
    ref = oracle.trace_gi(g, df, iv, ip, host["t"], host["face"], oracle.gi_params_from(prm))
    np.testing.assert_array_equal(rgb.cpu().numpy(), ref["rgb"])
    d = decode_texels(tex.cpu().numpy().view(np.uint16))
    planes = gi_planes_from_oracle(ref)
    np.testing.assert_array_equal(d["sh"], planes["sh"])
    np.testing.assert_array_equal(d["ao"], planes["ao"])
    c = counter.cpu().numpy()
    assert int(c[0]) == int(ref["samples"].sum()) and int(c[1]) == int(ref["rays"].sum()), (c, ref["samples"].sum(),
                                                                                         ref["rays"].sum())


def test_trace_frame_parity(terrain_world):
    """vpt_trace_frame (shadow pass beside GI on the context's side stream)
    equals the oracle's three passes, frame after frame, with the DF samples
    and rays of all three counted."""
    g, df, w = terrain_world
    torch = _torch()
    W, H = 640, 360
    cam, view, proj, iv, ip = camera(W, H)
    gb = DeviceGBuffer(W, H)
    mask = torch.full((H, W), 7, dtype=torch.uint8, device="cuda")
    rgb = torch.empty((H, W, 3), dtype=torch.float32, device="cuda")
    tex = torch.empty((H, W, 8), dtype=torch.int16, device="cuda")
    counter = torch.zeros(2, dtype=torch.int64, device="cuda")
    for frame in range(3):
        prm = gi_params(frame=frame)
        print(f"trace_frame {W}x{H} frame {frame}", flush=True)
        counter.zero_()
        w.set_sample_counter(counter)
        w.trace_frame(cam, gb, prm, mask, rgb, tex)
        w.set_sample_counter(None)
        torch.cuda.synchronize()
        host = gb.numpy()
        p = oracle.trace_primary(g, df, iv, ip, W, H, 350)
        _check_gbuffer(host, p)
        sd = np.array(prm.sun_dir, np.float32)
        sh = oracle.trace_shadow(g, df, iv, ip, host["t"], host["face"], sd, 350)
        np.testing.assert_array_equal(mask.cpu().numpy(), sh["mask"])
        gi = oracle.trace_gi(g, df, iv, ip, host["t"], host["face"], oracle.gi_params_from(prm))
        np.testing.assert_array_equal(rgb.cpu().numpy(), gi["rgb"])
        # the same work as the three passes called one after another
        c = counter.cpu().numpy().copy()
        counter.zero_()
        w.set_sample_counter(counter)
        w.trace_primary(cam, gb, 350)
        w.trace_shadow(cam, gb, list(prm.sun_dir), mask, 350)
        w.trace_gi(cam, gb, prm, rgb, tex)
        w.set_sample_counter(None)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(c, counter.cpu().numpy())
        assert c[1] > W * H
    # with the transversal: the shadow pass is vpt_trace_shadow2's
    tv = torch.empty((H, W), dtype=torch.int16, device="cuda")
    w.trace_frame(cam, gb, prm, mask, rgb, tex, transversal=tv)
    torch.cuda.synchronize()
    host = gb.numpy()
    sh2 = oracle.trace_shadow2(g, df, iv, ip, host["t"], host["face"], np.array(prm.sun_dir, np.float32), 350)
    np.testing.assert_array_equal(mask.cpu().numpy(), sh2["mask"])
    np.testing.assert_array_equal(tv.cpu().numpy().view(np.uint16), sh2["transversal"])
    from voxelpathtracer_amd._lib import VptError
    with pytest.raises(VptError):
        w.trace_frame(cam, gb, prm, None, rgb, tex)
    with pytest.raises(VptError):
        w.trace_frame(cam, gb, prm, mask, rgb, tex, primary_iter=-1)


def test_ray_queries_parity(terrain_world):
    g, df, w = terrain_world
    torch = _torch()
    rng = np.random.default_rng(7)
    n = 200_000
    org = np.stack([rng.uniform(-20, 404, n), rng.uniform(-10, 140, n), rng.uniform(-20, 404, n)], 1)
    d = rng.normal(size=(n, 3))
    # axis-aligned and zero-component directions (the DDA tie/zero rules)
    d[:2000] = 0.0
    d[np.arange(2000), rng.integers(0, 3, 2000)] = rng.choice([-1.0, 1.0], 2000)
    d[2000:4000, rng.integers(0, 3)] = 0.0
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rays = np.concatenate([org, d], 1).astype(np.float32)
    rays[4000:4100, 0:3] = np.floor(rays[4000:4100, 0:3])   # origins on cell corners
    dev_rays = torch.from_numpy(rays.view(np.uint8).copy()).cuda()
    hits = torch.empty(n * C.sizeof(Hit), dtype=torch.uint8, device="cuda")
    w.trace_rays(dev_rays, hits, n, 350)
    torch.cuda.synchronize()
    dt = np.dtype([("t", "<f4"), ("voxel", "<u4"), ("face", "u1"), ("block", "u1"), ("samples", "<u2")])
    got = hits.cpu().numpy().view(dt)
    ref = oracle.trace_rays(g, df, rays, 350)
    np.testing.assert_array_equal(got["face"], ref["face"])
    np.testing.assert_array_equal(got["block"], ref["block"])
    np.testing.assert_array_equal(got["t"], ref["t"])
    np.testing.assert_array_equal(got["samples"], ref["samples"])
    cell = ref["cell"]
    vox = np.where(cell[:, 0] < 0, np.uint32(0xFFFFFFFF),
                   (cell[:, 0] | (cell[:, 1] << 10) | (cell[:, 2] << 20)).astype(np.uint32))
    np.testing.assert_array_equal(got["voxel"], vox)


def test_sample_counter(terrain_world):
    g, df, w = terrain_world
    torch = _torch()
    W, H = 640, 360
    cam, view, proj, iv, ip = camera(W, H)
    gb = DeviceGBuffer(W, H)
    counter = torch.zeros(2, dtype=torch.int64, device="cuda")
    w.set_sample_counter(counter)
    w.trace_primary(cam, gb, 350)
    w.set_sample_counter(None)
    torch.cuda.synchronize()
    ref = oracle.trace_primary(g, df, iv, ip, W, H, 350)
    got = counter.cpu().numpy()
    assert int(got[0]) == int(ref["samples"].sum())
    assert int(got[1]) == W * H


# ---------------------------------------------------------------- SVGF

def _run_svgf(ctx, w, g, df, W, H, frames, tol_final=1e-3):
    """Runs the SVGF camera path for `frames` frames through the kernels and
    the oracle on the same GPU-rendered inputs; compares every plane of
    every frame.  Returns per-frame match fractions and the oracle's
    temporal utility of the last frame (for branch-coverage checks)."""
    torch = _torch()
    from voxelpathtracer_amd import SVGF
    sv = SVGF(ctx, W, H)
    orc = OracleSVGF(W, H)
    gbs = [DeviceGBuffer(W, H), DeviceGBuffer(W, H)]
    rgb = torch.empty((H, W, 3), dtype=torch.float32, device="cuda")
    tex = torch.empty((H, W, 8), dtype=torch.int16, device="cuda")
    out = torch.empty((H, W, 3), dtype=torch.float32, device="cuda")
    plane = torch.empty((H, W, 8), dtype=torch.int16, device="cuda")
    util = torch.empty((H, W, 4), dtype=torch.int16, device="cuda")
    prev_view = prev_proj = None
    prev_host = None
    results = []
    spp_hist = []
    for f in range(frames):
        pos, yaw, pitch = svgf_camera_path(f)
        cam, view, proj, iv, ip = camera(W, H, pos, yaw, pitch)
        cur = gbs[f % 2]
        prev = gbs[(f + 1) % 2] if f > 0 else cur
        if prev_view is None:
            prev_view, prev_proj = view, proj
        vp = viewproj(prev_view, prev_proj)
        w.trace_primary(cam, cur, 350)
        prm = gi_params(frame=f)
        w.trace_gi(cam, cur, prm, rgb, tex)
        sv.frame(cam, vp, cur, prev, tex, out, time=f / 60.0)
        torch.cuda.synchronize()
        host = cur.numpy()
        prev_h = host if prev_host is None else prev_host
        raw = decode_texels(tex.cpu().numpy().view(np.uint16))
        raw = dict(sh=raw["sh"], cocg=raw["cocg"], luma=raw["x"], ao=raw["ao"])
        # history length entering this frame's temporal pass (oracle state)
        spp_in = orc.hist["util"][..., 0].copy()
        ref = orc.frame(iv, ip, vp, host, prev_h, raw, f / 60.0)
        # per-plane comparison of this frame
        sv.read_plane(0, plane)
        pre = decode_texels(plane.cpu().numpy().view(np.uint16))
        sv.read_plane(1, plane)
        tmp = decode_texels(plane.cpu().numpy().view(np.uint16))
        sv.read_utility(util)
        ut = util.cpu().numpy().view(np.float16).astype(np.float32)[..., :3]
        sv.read_plane(2, plane)
        var = decode_texels(plane.cpu().numpy().view(np.uint16))
        sv.read_plane(3, plane)
        fin = decode_texels(plane.cpu().numpy().view(np.uint16))
        torch.cuda.synchronize()
        stats = dict(
            pre=float((pre["sh"] == ref["pre"]["sh"]).mean()),
            temporal=float((tmp["sh"] == ref["temporal"]["sh"]).mean()),
            util=float((ut == ref["temporal"]["util"]).mean()),
            var=float((var["x"] == ref["variance"]["var"]).mean()),
            var_sh=float((var["sh"] == ref["variance"]["sh"]).mean()),
            final=float((fin["sh"] == ref["final"]["sh"]).mean() * (fin["cocg"] == ref["final"]["cocg"]).mean()),
            final_var=float((fin["x"] == ref["final"]["var"]).mean()),
            rgb_rel_l1=rel_l1(out.cpu().numpy(), ref["rgb"]),
        )
        print(f"svgf frame {f} {W}x{H}: {stats}", flush=True)
        results.append(stats)
        spp_hist.append(spp_in)
        assert stats["rgb_rel_l1"] <= tol_final, stats
        prev_view, prev_proj = view, proj
        prev_host = host
    sv.close()
    return results, spp_hist, ref["temporal"]["util"]


def _assert_exact(res):
    for f, r in enumerate(res):
        bad = {k: v for k, v in r.items() if k != "rgb_rel_l1" and v != 1.0}
        assert not bad, f"frame {f}: planes not bit-exact {bad}"


def test_svgf_parity_small(ctx, terrain_world):
    g, df, w = terrain_world
    res, _, _ = _run_svgf(ctx, w, g, df, 320, 180, 6)
    # the kernels follow the oracle's operation sequence: planes agree exactly
    _assert_exact(res)


@pytest.mark.parametrize("W,H", [(2, 2), (5, 3), (33, 9), (70, 41), (260, 241)])
def test_svgf_parity_ragged(ctx, terrain_world, W, H):
    """Images smaller than a tile and its 9x9 apron, and ones a tile does not
    divide: taps off the image in every pass; and one of more than 256 tiles
    whose last column is narrow; bit-exact."""
    g, df, w = terrain_world
    res, _, _ = _run_svgf(ctx, w, g, df, W, H, 3)
    _assert_exact(res)


def test_svgf_parity_steady_state(ctx, terrain_world):
    """24 frames of the SVGF camera path at 640x360, every plane bit-exact on
    every frame, with the oracle's state shown to reach the long-history
    branches: VarianceEstimate.glsl:172-176 (history >= 12, and 32x8 pixel
    blocks whose every pixel has it, which skip the 9x9 staging),
    SpatialFilter.glsl:219,293 at steps <= 8 with history > 8 (non-strong
    weights), and the TemporalFilter.glsl:322-323 blend floor 0.05 (history
    >= 20 entering the temporal pass)."""
    g, df, w = terrain_world
    W, H = 640, 360
    res, spp_in, util = _run_svgf(ctx, w, g, df, W, H, 24)
    _assert_exact(res)
    spp = util[..., 0]
    assert (spp >= 12).mean() > 0.3, "variance long-history branch not reached"
    assert (spp > 8).mean() > 0.3, "non-strong a-trous branch not reached"
    assert (spp_in[-1] >= 20).mean() > 0.3, "temporal 0.05 blend floor not reached"
    assert (spp < 12).mean() > 0.05, "short-history branch not exercised"
    blk = (spp >= 12).reshape(H // 8, 8, W // 32, 32).all(axis=(1, 3))
    assert blk.mean() > 0.1 and (~blk).mean() > 0.1, "variance block skip not exercised both ways"


@pytest.mark.timeout(600)
def test_svgf_parity_1080p(ctx, terrain_world):
    """13 frames at 1920x1080 (the workload's resolution): every plane
    bit-exact; the last frames run with history >= 12."""
    g, df, w = terrain_world
    res, spp_in, util = _run_svgf(ctx, w, g, df, 1920, 1080, 13)
    for r in res:
        assert r["rgb_rel_l1"] <= 1e-3
    _assert_exact(res)
    assert (util[..., 0] >= 12).mean() > 0.3


@pytest.mark.parametrize("max_iter", [0, 1, 2, 65535])
def test_ray_queries_iteration_caps(terrain_world, max_iter):
    """The loop cap at its edges: 0 (no sample), 1, 2 and the largest cap."""
    g, df, w = terrain_world
    torch = _torch()
    rng = np.random.default_rng(31 + max_iter)
    n = 20_000
    org = np.stack([rng.uniform(0, 384, n), rng.uniform(0, 128, n), rng.uniform(0, 384, n)], 1)
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rays = np.concatenate([org, d], 1).astype(np.float32)
    dev_rays = torch.from_numpy(rays.view(np.uint8).copy()).cuda()
    hits = torch.empty(n * C.sizeof(Hit), dtype=torch.uint8, device="cuda")
    w.trace_rays(dev_rays, hits, n, max_iter)
    torch.cuda.synchronize()
    dt = np.dtype([("t", "<f4"), ("voxel", "<u4"), ("face", "u1"), ("block", "u1"), ("samples", "<u2")])
    got = hits.cpu().numpy().view(dt)
    ref = oracle.trace_rays(g, df, rays, max_iter)
    for k in ("t", "face", "block", "samples"):
        np.testing.assert_array_equal(got[k], ref[k], err_msg=k)
    assert got["samples"].max() <= max_iter


@pytest.mark.parametrize("n", [20_000, 300_000])
@pytest.mark.parametrize("max_iter", [23, 24, 25, 48, 350])
def test_ray_queries_long_rays(terrain_world, n, max_iter):
    """Launches below and above 262,144 rays, where the traversal takes its
    eager form at once or after 24 steps, with caps around that step: random
    rays, grazing ones that walk far, axis-aligned directions, -0 and
    on-boundary origins, and direction components near zero."""
    g, df, w = terrain_world
    torch = _torch()
    rng = np.random.default_rng(57 + max_iter)
    org = np.stack([rng.uniform(0, 384, n), rng.uniform(0, 128, n), rng.uniform(0, 384, n)], 1)
    d = rng.normal(size=(n, 3))
    kind = rng.integers(0, 8, n)
    low = kind < 3
    d[low, 1] *= 0.02
    org[low, 1] = rng.uniform(60, 95, int(low.sum()))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    axis = np.flatnonzero(kind == 3)
    d[axis] = 0.0
    d[axis, rng.integers(0, 3, axis.size)] = rng.choice([-1.0, 1.0], axis.size)
    flat = np.flatnonzero(kind == 4)
    d[flat, rng.integers(0, 3, flat.size)] = 0.0
    tiny = np.flatnonzero(kind == 5)
    d[tiny, rng.integers(0, 3, tiny.size)] = rng.choice([1e-38, -1e-20, 1e-7], tiny.size)
    edge = np.flatnonzero(kind == 6)
    org[edge] = np.round(org[edge])
    rays = np.concatenate([org, d], 1).astype(np.float32)
    zero = np.flatnonzero(kind == 7)[::2]
    rays[zero, rng.integers(0, 3, zero.size)] = -0.0
    dev_rays = torch.from_numpy(rays.view(np.uint8).copy()).cuda()
    hits = torch.empty(n * C.sizeof(Hit), dtype=torch.uint8, device="cuda")
    w.trace_rays(dev_rays, hits, n, max_iter)
    torch.cuda.synchronize()
    dt = np.dtype([("t", "<f4"), ("voxel", "<u4"), ("face", "u1"), ("block", "u1"), ("samples", "<u2")])
    got = hits.cpu().numpy().view(dt)
    ref = oracle.trace_rays(g, df, rays, max_iter)
    for k in ("t", "face", "block", "samples"):
        np.testing.assert_array_equal(got[k], ref[k], err_msg=k)
    assert got["samples"].max() == max_iter if max_iter < 100 else got["samples"].max() > 60


@pytest.mark.parametrize("dims", [(16, 8, 8), (1024, 16, 8), (16, 1024, 16), (16, 8, 1024)])
def test_extreme_world_shapes(ctx, dims):
    """Smallest world and worlds at the 1024 limit along each axis: DF and
    ray queries against the oracle."""
    torch = _torch()
    nx, ny, nz = dims
    rng = np.random.default_rng(nx + 3 * ny + 7 * nz)
    g = random_world(rng, nx, ny, nz, 0.05)
    w = World(ctx, nx, ny, nz)
    w.m_WorldData[...] = g
    w.Buffer()
    w.GenerateDistanceField()
    df = oracle.df_build(g)
    np.testing.assert_array_equal(w.download_df(), df)
    n = 5000
    org = np.stack([rng.uniform(-2, nx + 2, n), rng.uniform(-2, ny + 2, n), rng.uniform(-2, nz + 2, n)], 1)
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rays = np.concatenate([org, d], 1).astype(np.float32)
    dev_rays = torch.from_numpy(rays.view(np.uint8).copy()).cuda()
    hits = torch.empty(n * C.sizeof(Hit), dtype=torch.uint8, device="cuda")
    w.trace_rays(dev_rays, hits, n, 350)
    torch.cuda.synchronize()
    dt = np.dtype([("t", "<f4"), ("voxel", "<u4"), ("face", "u1"), ("block", "u1"), ("samples", "<u2")])
    got = hits.cpu().numpy().view(dt)
    ref = oracle.trace_rays(g, df, rays, 350)
    for k in ("t", "face", "block", "samples"):
        np.testing.assert_array_equal(got[k], ref[k], err_msg=k)
    w.close()
