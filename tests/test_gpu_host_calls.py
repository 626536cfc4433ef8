"""Host-buffer entry points keep their device block between calls: calls of growing and shrinking sizes
return what a fresh context returns, blocks beyond the kept size are given back, and a kept block makes
way for an allocation that the budget could hold without it."""
import ctypes as C

import numpy as np
import pytest

from merian_amd import scenes
from merian_amd.runtime import Context, pt_params
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def test_ray_calls_of_changing_size(ctx):
    pos, idx = scenes.ray_query(seed=2, n_tri=2000)
    rays = scenes.incoherent_rays(1_500_000, seed=3)
    ref = O.OracleScene(triangles=(pos, idx), use_bvh=True).trace(rays)
    ds = ctx.triangles(pos, idx)
    for n in (3, 20_000, 7, 1_500_000, 21_846, 1):  # 21,846 rays: just above the pinned staging
        got = ctx.trace(ds, rays[:n])
        assert np.array_equal(got["triangle"], ref["triangle"][:n])
        hit = got["triangle"] != 0xFFFFFFFF
        assert np.array_equal(got["t"][hit], ref["t"][:n][hit])
    ds.destroy()


def test_frame_calls_of_changing_size_and_statistics(ctx):
    sc = scenes.plain_small(seed=0)
    ds = ctx.scene(sc)
    first = {}
    for rep in range(2):
        for w, h, spp, length in ((16, 9, 1, 3), (200, 120, 2, 5), (1, 1, 1, 1), (33, 65, 3, 4), (1, 1, 1, 1)):
            cam = ctx.camera(sc.camera, 4)
            img, sig, gb, st = ctx.render(ds, pt_params(spp=spp, max_path_length=length), cam, 4, w, h)
            key = (w, h, spp, length)
            if key in first:
                assert all(a.tobytes() == b.tobytes() for a, b in zip(first[key], (img, sig, gb)))
            first[key] = (img, sig, gb)
            assert st.trace_launches == length - 1 and st.primary_segments == w * h
            assert st.ms_gbuffer > 0 and st.ms_total >= st.ms_trace + st.ms_shade - 1e-3 and st.ms_shade > 0
            assert (st.ms_trace > 0) == (length > 1)
            plain, _, _, _ = ctx.render(ds, pt_params(spp=spp, max_path_length=length), cam, 4, w, h, signature=False,
                                        gbuffer=False)
            assert plain.tobytes() == img.tobytes()
    ds.destroy()


def test_kept_block_makes_way():
    with Context(0, hbm_budget=1 << 30) as ctx:
        pos, idx = scenes.ray_query(seed=2, n_tri=500)
        ds = ctx.triangles(pos, idx)
        ctx.trace(ds, scenes.incoherent_rays(10, seed=1))
        base = ctx.memory_in_use
        ctx.trace(ds, scenes.incoherent_rays(1_300_000, seed=1))  # 62.4 MB: kept
        kept = ctx.memory_in_use
        assert kept > base
        ctx.trace(ds, scenes.incoherent_rays(3_000_000, seed=1))  # 144 MB: not kept
        assert ctx.memory_in_use == kept
        p = C.c_void_p()
        ctx._check(ctx.lib.mrt_alloc_dev(ctx.h, (1 << 30) - base - 4096, C.byref(p)))  # needs the kept block's room
        ctx._check(ctx.lib.mrt_free_dev(ctx.h, p))
        assert len(ctx.trace(ds, scenes.incoherent_rays(100, seed=1))) == 100
        ds.destroy()
