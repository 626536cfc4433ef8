"""Closest hits for the forms of rays and scenes at which the box tests' number formats could go
wrong, bit-exact against the oracle's brute force on every tree: geometry far from the origin, tiny
and huge, negative; rays along the axes and with zero components, directions of any length, intervals
that start below zero, end at zero or are empty; odd ray counts from a single ray up; no triangles."""
import numpy as np
import pytest

from merian_amd import abi, scenes
from merian_amd.runtime import pt_params
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TREES = [(4, 4, 0), (4, 1, 0), (8, 2, 0), (8, 2, 1)]


def _scene(ctx, pos, idx, tree):
    ds = ctx.triangles(pos, idx)
    t = ds.tuning()
    t.bvh_width, t.bvh_max_leaf, t.bvh8_order = tree
    ds.set_tuning(t)
    return ds


def _same(a, b):
    assert np.array_equal(a["triangle"], b["triangle"]), int((a["triangle"] != b["triangle"]).sum())
    hit = b["triangle"] != 0xFFFFFFFF
    for k in ("t", "u", "v"):
        assert np.array_equal(a[k][hit].view(np.uint32), b[k][hit].view(np.uint32)), k
    return hit


def _rays(n, seed, scale, shift):
    r = scenes.incoherent_rays(n, seed=seed)
    r["origin"] = (r["origin"] * np.float32(scale) + np.float32(shift)).astype(np.float32)
    d = r["direction"]
    k = np.arange(n)
    d[k % 7 == 0] = np.eye(3, dtype=np.float32)[k[k % 7 == 0] % 3] * np.where(k[k % 7 == 0] % 2, 1, -1)[:, None]
    d[k % 7 == 1, 0] = 0.0
    d[k % 7 == 2, 1] = -0.0
    d[k % 7 == 3] *= np.float32(1e-4)
    d[k % 7 == 4] *= np.float32(1e3)
    r["tmax"][k % 11 == 0] = np.float32(0.3 * scale)
    r["tmin"][k % 11 == 1] = np.float32(-0.5 * scale)
    r["tmax"][k % 11 == 2] = -0.0
    r["tmin"][k % 11 == 3], r["tmax"][k % 11 == 3] = np.float32(scale), np.float32(0.5 * scale)
    r["tmin"][k % 11 == 4], r["tmax"][k % 11 == 4] = np.float32(-scale), np.float32(-0.01 * scale)
    return r


@pytest.mark.parametrize("tree", TREES)
@pytest.mark.parametrize("scale,shift", [(1.0, 0.0), (1.0, -0.5), (1e-3, -0.25), (1e-2, 40.0), (1e5, -3e4), (1e8, 0.0)])
def test_forms_vs_bruteforce(ctx, tree, scale, shift):
    pos, idx = scenes.ray_query(seed=9, n_tri=1500)
    pos = (pos * np.float32(scale) + np.float32(shift)).astype(np.float32)
    rays = _rays(6001, 4, scale, shift)
    ref = O.OracleScene(triangles=(pos, idx), use_bvh=False).trace(rays)
    ds = _scene(ctx, pos, idx, tree)
    got = ctx.trace(ds, rays)
    ds.destroy()
    assert _same(got, ref).mean() > 0.1


@pytest.mark.parametrize("tree", TREES)
@pytest.mark.parametrize("ahead", [True, False])
def test_interval_of_one_point(ctx, tree, ahead):
    """tmin = tmax = the hit's own distance, ahead of the origin and behind it: the limits of the box
    tests are rounded outward on both sides, so the hit stays."""
    pos, idx = scenes.ray_query(seed=11, n_tri=4000)
    rays = scenes.incoherent_rays(20_001, seed=6)
    osc = O.OracleScene(triangles=(pos, idx), use_bvh=False)
    if not ahead:
        rays["direction"] *= -1
        rays["tmin"], rays["tmax"] = -np.inf, 0.0
    first = osc.trace(rays)
    t = np.where(first["triangle"] != 0xFFFFFFFF, first["t"], np.float32(-1.0 if not ahead else 1.0))
    rays["tmin"] = rays["tmax"] = t
    ref = osc.trace(rays)
    ds = _scene(ctx, pos, idx, tree)
    got = ctx.trace(ds, rays)
    ds.destroy()
    hit = _same(got, ref)
    assert hit.mean() > 0.3 and (got["t"][hit] == t[hit]).all()  # 39.6 % of these rays hit (brute force)


@pytest.mark.parametrize("tree", TREES)
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1000, 16385, 400_003])
def test_ray_counts(ctx, tree, n):
    pos, idx = scenes.ray_query(seed=3, n_tri=3000)
    rays = scenes.incoherent_rays(n, seed=5)
    ref = O.OracleScene(triangles=(pos, idx), use_bvh=True).trace(rays)
    ds = _scene(ctx, pos, idx, tree)
    for _ in range(2):
        _same(ctx.trace(ds, rays), ref)
    ds.destroy()


@pytest.mark.parametrize("tree", TREES)
def test_no_triangles_and_one(ctx, tree):
    rays = _rays(500, 1, 1.0, 0.0)
    tri = np.array([[0.1, 0.1, 0.5], [0.9, 0.1, 0.5], [0.5, 0.9, 0.5]], np.float32)
    for idx in (np.zeros(0, np.uint32), np.arange(3, dtype=np.uint32)):
        ds = _scene(ctx, tri, idx, tree)
        got = ctx.trace(ds, rays)
        ds.destroy()
        if len(idx):
            _same(got, O.OracleScene(triangles=(tri, idx), use_bvh=False).trace(rays))
        else:
            assert (got["triangle"] == 0xFFFFFFFF).all()


@pytest.fixture(scope="module")
def soup():
    pos, idx = scenes.ray_query(seed=21, n_tri=20_000)
    rays = scenes.incoherent_rays((3 << 20) + 65, seed=22)
    return pos, idx, rays, O.OracleScene(triangles=(pos, idx), use_bvh=True).trace(rays)


@pytest.mark.parametrize("tree", [(4, 2, 0), (8, 2, 0), (8, 4, 1)])
@pytest.mark.parametrize("refill,grid", [(1, 100), (16, 3), (64, 100), (64, 1), (63, 1)])
def test_shared_rays_and_refill(ctx, soup, tree, refill, grid):
    """Launches whose lanes share rays (up to 3 << 20 of them), with every kind of refill and few or many
    rays per wave, and one just above that limit."""
    pos, idx, rays, ref = soup
    ds = _scene(ctx, pos, idx, tree)
    t = ds.tuning()
    t.refill_lanes, t.grid_percent, t.leaf_lanes = refill, grid, 64 if refill == 63 else 8
    ds.set_tuning(t)
    for n in (17, 4097, 130_001, *([3 << 20, len(rays)] if grid == 100 else [])):
        _same(ctx.trace(ds, rays[:n]), ref[:n])
    ds.destroy()


@pytest.mark.parametrize("tree", [(4, 2, 0), (8, 2, 0), (8, 4, 1)])
@pytest.mark.parametrize("grid", [100, 3, 1])
def test_ray_counts_around_the_cursors(ctx, soup, tree, grid):
    """Arrays on both sides of the limits of the several cursors, 2^20 and 2^23 rays, with grids that make
    many, few and no whole rounds of them. The first 3.1 M rays against the oracle; longer arrays repeat
    them and repeat their hits."""
    import torch
    pos, idx, rays, ref = soup
    ds = _scene(ctx, pos, idx, tree)
    t = ds.tuning()
    t.grid_percent = grid
    ds.set_tuning(t)
    for n in (54_785, (1 << 20) - 1, 1 << 20, (1 << 20) + 1, 1_310_721, 2_097_153, 3 << 20, (3 << 20) + 64):
        _same(ctx.trace(ds, rays[:n]), ref[:n])
    if grid == 100:
        one = torch.from_numpy(rays.view(np.float32).reshape(-1, 8)).cuda()
        d_rays = torch.cat([one, one, one])[:(1 << 23) + 1].contiguous()
        want = torch.from_numpy(ctx.trace(ds, rays).view(np.int32).reshape(-1, 4)).cuda()
        want = torch.cat([want, want, want])[:len(d_rays)]
        for n in ((1 << 23) - 1023, 1 << 23, (1 << 23) + 1):
            got = torch.full((len(d_rays), 4), -2, dtype=torch.int32, device="cuda")
            torch.cuda.synchronize()
            ctx.trace_dev(ds, d_rays.data_ptr(), n, got.data_ptr(), stream=torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            assert torch.equal(got[:n], want[:n]) and bool((got[n:] == -2).all())
    ds.destroy()


@pytest.fixture(scope="module")
def room():
    return scenes.full_scene(seed=4, instances=12, env_size=(64, 32), name="room")


@pytest.mark.parametrize("tree", [(4, 4, 0), (8, 2, 0), (8, 2, 1)])
@pytest.mark.parametrize("w,h", [(2053, 2051), (2047, 2049), (701, 503)])
def test_gbuffer_matches_ray_queries(ctx, room, tree, w, h):
    """GBuffer passes above and below the 2^22 rays up to which lanes share rays, every pixel against the
    closest hit of its camera ray (another kernel): the packed record bit for bit."""
    import torch
    ds = ctx.scene(room)
    t = ds.tuning()
    t.bvh_width, t.bvh_max_leaf, t.bvh8_order = tree
    ds.set_tuning(t)
    cam = ctx.camera(room.camera, 3)
    rays, hits = (torch.zeros(w * h, k, device="cuda") for k in (8, 4))
    gb = torch.full((w * h, 4), -2, dtype=torch.int32, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    ctx.camera_rays_dev(cam, w, h, rays.data_ptr(), stream=stream)
    ctx.trace_dev(ds, rays.data_ptr(), w * h, hits.data_ptr(), stream=stream)
    ctx.gbuffer_dev(ds, cam, w, h, gb.data_ptr(), stream=stream)
    torch.cuda.synchronize()
    ds.destroy()
    got, hits = gb.cpu().numpy().view(np.uint32), hits.cpu().numpy()
    tri = hits[:, 0].copy().view(np.uint32)
    hit = tri != 0xFFFFFFFF
    first = np.concatenate([[0], np.cumsum(room.geometries["primitive_count"].astype(np.int64))])
    geom = np.searchsorted(first, tri.astype(np.int64), side="right") - 1
    uv = hits[:, 2:4].astype(np.float16).view(np.uint16).astype(np.uint32)
    want = np.empty_like(got)
    want[:, :3], want[:, 3] = 0xFFFFFFFF, 0
    want[hit, 0], want[hit, 1], want[hit, 2] = 0, (tri - first[np.where(hit, geom, 0)])[hit], geom[hit]
    want[hit, 3] = (uv[:, 0] | uv[:, 1] << 16)[hit]
    assert 0.2 < hit.mean() <= 1.0 and np.array_equal(got, want)


@pytest.mark.parametrize("mode", [abi.MODE_BSDF, abi.MODE_NEE])
@pytest.mark.parametrize("tree", [(4, 4, 0), (8, 2, 0), (8, 2, 1)])
def test_frame_of_large_passes_matches_small(ctx, room, tree, mode):
    """Passes above the 2^22 paths up to which lanes share rays (path and shadow queues): the frame in one
    pass of 8.4 M paths equals the same frame in passes of 2.1 M bit for bit."""
    ds = ctx.scene(room)
    W = H = 1024
    cam = ctx.camera(room.camera, 7)
    frames = []
    for spp in (8, 2):
        t = ds.tuning()
        t.bvh_width, t.bvh_max_leaf, t.bvh8_order = tree
        t.max_paths = spp * W * H
        ds.set_tuning(t)
        img, sig, _, st = ctx.render(ds, pt_params(spp=8, max_path_length=4, mode=mode), cam, 7, W, H)
        frames.append((img.tobytes(), sig.tobytes(), int(st.continuation_segments)))
    ds.destroy()
    assert frames[0][2] > 1 << 22 and frames[0] == frames[1]
