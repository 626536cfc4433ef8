"""Guide inference at the edges of its split: a query's outputs do not depend on how many queries share
the call (partial tiles, one to four tiles per wave iteration, uneven last iterations), with dense and
hashed levels, positions outside the scene and on its faces, and agree with the oracle at both ends."""
import numpy as np
import pytest

from merian_amd import scenes
from merian_amd.runtime import Guide, guide_config
from oracle import oracle as O
from test_gpu_guide import _random_params, _records, _spec

pytestmark = pytest.mark.gpu

WAVES = 512 * 8  # resident waves: beyond 16 queries each, an iteration takes more than one tile
SIZES = (1, 15, 16, 17, 63, 64, 65, 129, 16 * WAVES + 17, 16 * WAVES * 4 + 1, 16 * WAVES * 5 - 3)


@pytest.mark.parametrize("config", [dict(log2_table=12, base_resolution=2, max_resolution=64), dict(log2_table=10, base_resolution=2, max_resolution=512)])
def test_outputs_do_not_depend_on_the_call(ctx, config):
    sc = scenes.plain_small(seed=3, subdiv=1, grid=2)
    ds = ctx.scene(sc)
    g = Guide(ctx, ds, guide_config(seed=1, **config))
    try:
        W, G = _random_params(g, 5, scale=1.5)
        g.set_params(W, G)
        lo, hi = np.asarray(sc.bounds())
        R = _records(max(SIZES), lo - 0.1 * (hi - lo), hi + 0.1 * (hi - lo), 6)
        R[1::101, 0:3], R[2::101, 0:3] = lo, hi
        pos, wo = np.ascontiguousarray(R[:, 0:3]), np.ascontiguousarray(R[:, 4:7])
        whole = g.forward(pos, wo)
        for n in SIZES:
            assert g.forward(pos[:n], wo[:n]).tobytes() == whole[:n].tobytes(), n
        for part in (slice(0, 2000), slice(len(pos) - 2000, len(pos))):
            cpu = O.guide_forward(_spec(g), W, G, pos[part], wo[part])
            err, scale = np.abs(whole[part] - cpu), np.abs(cpu).max()
            # fp16 rounding points of the mirror, the bounds of the oracle comparison of 3,000 queries
            assert err.max() <= 2e-2 * scale and err.mean() <= 1e-3 * scale
    finally:
        g.close()
        ds.destroy()
