"""Shading of every kind of geometry (the flags and the material entry that a hit triangle's shading
record carries) against the oracle, bit for bit: flat and flipped, two-sided, with tangents and with
texture coordinates, geometries that show the environment, more materials than eight bits hold."""
import numpy as np
import pytest

from merian_amd import abi, scenes
from merian_amd.runtime import pt_params
from oracle import oracle as O

pytestmark = pytest.mark.gpu

FLAGS = [0, abi.GEOM_FLAT_SHADING, abi.GEOM_TWO_SIDED, abi.GEOM_FLIP_FACING | abi.GEOM_TWO_SIDED, abi.GEOM_HAS_TANGENTS,
         abi.GEOM_HAS_TANGENTS | abi.GEOM_FLAT_SHADING | abi.GEOM_TWO_SIDED, abi.GEOM_USE_ENV_MAP,
         abi.GEOM_FLIP_FACING | abi.GEOM_FLAT_SHADING | abi.GEOM_TWO_SIDED | abi.GEOM_HAS_TANGENTS]


def _scene(env):
    rng = np.random.default_rng(4)
    b = scenes.SceneBuilder("shade_forms")
    for _ in range(300):  # ids above 255 are the ones used
        b.add_material(scenes.diffuse_material(rng.uniform(0.1, 0.9, 3)))
    mats = [b.add_material(scenes.pbrt_conductor((0.8, 0.7, 0.5), a)) for a in (0.02, 0.2)]
    mats += [b.add_material(scenes.pbrt_diffuse((0.3, 0.5, 0.7))), b.add_material(scenes.pbrt_dielectric(1.5, 0.02))]
    P, T = scenes.icosphere(2)
    N = scenes.vertex_normals(P, T)
    for k, flags in enumerate(FLAGS):
        b.add_mesh(P * 0.4 + np.array([(k % 4 - 1.5) * 1.0, 0.45, (k // 4 - 0.5) * 1.2]), N, T, mats[k % len(mats)], flags)
    P, N, T = scenes.quad((-3, 0, -3), (-3, 0, 3), (3, 0, 3), (3, 0, -3))
    b.add_mesh(P, N, T, 299)
    cam = scenes.CameraSpec((0.0, 2.6, 4.0), (0.0, 0.3, 0.0), (0.0, 1.0, 0.0), 0.8, 101, 67)
    sc = b.build(camera=cam, **env)
    # texture coordinates and tangents that vary over the meshes
    n = len(sc.vertices)
    sc.vertices["uv"] = scenes.f16_bits(rng.uniform(0, 1, (n, 2)))
    t = rng.normal(size=(n, 3))
    sc.vertices["encoded_tangent"] = scenes.encode_normals((t / np.linalg.norm(t, axis=1, keepdims=True)).astype(np.float32))
    return sc


@pytest.mark.parametrize("env", [scenes.sky_env(64, 32, dynamic_range=50.0), scenes.constant_env((0.7, 0.8, 0.9))],
                         ids=["latlong", "equal_area"])
@pytest.mark.parametrize("demodulate", [False, True])
def test_geometry_forms_match_oracle(ctx, env, demodulate):
    sc = _scene(env)
    ds, osc = ctx.scene(sc), O.OracleScene(sc)
    cam = ctx.camera(sc.camera, 1)
    p = pt_params(spp=3, max_path_length=6, demodulate_albedo=demodulate)
    img, sig, gb, _ = ctx.render(ds, p, cam, 1, 101, 67)
    ds.destroy()
    ref, ref_sig, _ = osc.render(O.pt_params(3, 6, demodulate_albedo=demodulate), cam, 1, 101, 67, gb)
    m = sig == ref_sig
    assert m.mean() >= 0.999
    assert (img[m].view(np.uint32) == ref[m].view(np.uint32)).all()
