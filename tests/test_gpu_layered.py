"""Shading kernels with and without the coat / sheen levels of the material tree: a scene takes the
full tree when any of its materials has such a lobe. An unused coated material must not change a
bit of any mode's image (the two routes compute the same values), and materials that use the lobes
must match the oracle."""
import numpy as np
import pytest

from merian_amd import abi, scenes
from merian_amd.runtime import Guide, Mcpg, guide_config, mcpg_config, pt_params
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _coated(coat=0.6, sheen=0.3):
    m = scenes.pbrt_diffuse((0.6, 0.4, 0.3))
    m["features"] = abi.PBR_CLEARCOAT | abi.PBR_SHEEN
    m["coat_weight"], m["coat_alpha"], m["sheen_weight"], m["sheen_alpha"] = coat, 0.05, sheen, 0.2
    m["sheen_color"] = (0.8, 0.7, 0.9)
    return m


def _mixed(**kw):
    m = scenes.pbrt_conductor((0.7, 0.6, 0.4), 0.09)
    for k, v in kw.items():
        m[k] = v
    return m


def _scene(extra=None, used=False):
    """Spheres of every lobe mix on a ground under a small sky; `extra` is one more material, worn
    by a sphere if `used`."""
    b = scenes.SceneBuilder("layered")
    glass = _mixed(features=abi.PBR_TRANSMISSION, metalness=0.0, transmission_weight=0.5, transmission_color=(1, 1, 1))
    mats = [scenes.diffuse_material((0.5, 0.6, 0.7)), scenes.pbrt_diffuse((0.3, 0.6, 0.2)), _mixed(),
            scenes.pbrt_dielectric(1.5, 0.01), _mixed(metalness=0.5), glass, _mixed(metalness=0.0, specular_weight=1.0)]
    ids = [b.add_material(m) for m in mats]
    if extra is not None:
        e = b.add_material(extra)
        if used:
            ids.append(e)
    P, T = scenes.icosphere(2)
    N = scenes.vertex_normals(P, T)
    for k, mid in enumerate(ids):
        tr = mid < len(mats) and bool(mats[mid]["features"][0] & abi.PBR_TRANSMISSION)
        b.add_mesh(P * 0.45 + np.array([(k % 3 - 1) * 1.1, 0.45, (k // 3 - 1) * 1.1]), N, T, mid,
                   abi.GEOM_TWO_SIDED if tr else 0)
    P, N, T = scenes.quad((-3, 0, -3), (-3, 0, 3), (3, 0, 3), (3, 0, -3))
    b.add_mesh(P, N, T, ids[1])
    cam = scenes.CameraSpec((0.0, 3.0, 4.5), (0.0, 0.3, 0.0), (0.0, 1.0, 0.0), 0.8, 96, 64)
    return b.build(camera=cam, **scenes.sky_env(64, 32, dynamic_range=100.0))


def _frame(ctx, sc, mode, spp=3, demodulate=False):
    W, H = (1, 1) if mode == "mcpg" else (75, 53)
    ds = ctx.scene(sc)
    cam = ctx.camera(sc.camera, 5)
    gbp, out = ctx_alloc(ctx, W * H * 16), ctx_alloc(ctx, W * H * 16)
    try:
        if mode in ("bsdf", "nee"):
            p = pt_params(spp=spp, max_path_length=6, mode=abi.MODE_BSDF if mode == "bsdf" else abi.MODE_NEE,
                          demodulate_albedo=demodulate)
            return ctx.render(ds, p, cam, 5, W, H)[0]
        ctx.gbuffer_dev(ds, cam, W, H, gbp)
        if mode == "guided":
            g = Guide(ctx, ds, guide_config(seed=3))
            g.render_dev(ds, pt_params(spp=spp, max_path_length=6, mode=abi.MODE_GUIDED, record_signature=False), cam, 5,
                         W, H, gbp, out, train=False)
        else:
            g = Mcpg(ctx, mcpg_config(mc_buffer_size=4093, lc_buffer_size=1021))
            for f in range(8):  # chains to guide by; one path in flight is deterministic
                g.render_dev(ds, pt_params(spp=8, max_path_length=6, record_signature=False), cam, f, W, H, gbp, out)
        img = np.zeros(W * H * 4, np.float32)
        ctx._check(ctx.lib.mrt_download(ctx.h, img.ctypes.data, out, img.nbytes))
        g.close()
        return img
    finally:
        for p in (gbp, out):
            ctx._check(ctx.lib.mrt_free_dev(ctx.h, p))
        ds.destroy()


def ctx_alloc(ctx, n):
    import ctypes as C
    p = C.c_void_p()
    ctx._check(ctx.lib.mrt_alloc_dev(ctx.h, n, C.byref(p)))
    return p.value


@pytest.mark.parametrize("mode", ["bsdf", "nee", "guided", "mcpg"])
def test_unused_layered_material_changes_nothing(ctx, mode):
    a = _frame(ctx, _scene(), mode)
    b = _frame(ctx, _scene(extra=_coated()), mode)
    assert a.any() and a.tobytes() == b.tobytes()


def test_unused_layered_material_demodulated(ctx):
    a = _frame(ctx, _scene(), "bsdf", demodulate=True)
    b = _frame(ctx, _scene(extra=_coated()), "bsdf", demodulate=True)
    assert a.tobytes() == b.tobytes()


@pytest.mark.parametrize("extra", [None, _coated(), _coated(coat=0.0, sheen=1.0), _coated(coat=1.0, sheen=0.0)])
def test_layered_scene_matches_oracle(ctx, extra):
    sc = _scene(extra=extra, used=extra is not None)
    ds, osc = ctx.scene(sc), O.OracleScene(sc)
    cam = ctx.camera(sc.camera, 2)
    img, sig, gb, _ = ctx.render(ds, pt_params(spp=4, max_path_length=6), cam, 2, 96, 64)
    ds.destroy()
    ref, ref_sig, _ = osc.render(O.pt_params(4, 6), cam, 2, 96, 64, gb)
    m = sig == ref_sig
    assert m.mean() >= 0.999
    assert (img[m].view(np.uint32) == ref[m].view(np.uint32)).all()
