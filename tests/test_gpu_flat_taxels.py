"""The flat sensor of a plain call at the edges of its work split -- one taxel,
taxel counts on both sides of the four-wave / one-wave line, fans of fewer and
of many more rays than the split's line between small and large fans, and
lists of several chunks per wave -- against the oracle's sampling of the
oracle's polygons."""
import numpy as np
import pytest

import oracle as O
from mujoco_contact_surfaces_amd import scenes as S
from test_gpu_parity import add_scene, oracle_soft_rigid, pair_of

pytestmark = pytest.mark.gpu

# as for the sensors of the batched step
RTOL = 1e-10

FINE, COARSE, TINY = dict(L=4, K=4, m=48), dict(L=2, K=2, m=4), dict(L=1, K=1, m=1)


@pytest.mark.parametrize("shape,taxels,rays,window,sigma", [
    (FINE, 1, 24, 0, 0.0),  # one taxel holds every polygon
    (FINE, 3, 7, 1, 0.3),
    (FINE, 16, 20, 0, 0.0),
    (FINE, 45, 5, 3, 0.0),  # 2025 taxels: four waves each
    (FINE, 46, 5, 3, 0.0),  # 2116: one wave
    (COARSE, 2, 24, 2, 0.5),  # a fan holds a whole taxel's rays
    (COARSE, 16, 8, 0, 0.0),  # a range of 8 x 8 rays: the largest small fan
    (COARSE, 16, 9, 0, 0.0),
    (TINY, 5, 24, 1, 0.3),
    (TINY, 60, 3, 0, 0.0),  # few polygons over many taxels: the lists outgrow their first buffer
    (COARSE, 91, 2, 0, 0.0),  # 8281 taxels: more than the kernel writes to host memory itself
    (TINY, 1025, 1, 0, 0.0),  # more than a million: copied straight to the caller
])
def test_flat_sensor_work_split(engine, shape, taxels, rays, window, sigma):
    print("[case] flat", shape, taxels, rays, window, flush=True)
    sc = S.tactile_pad(5, **shape)
    ha, hb = add_scene(engine, sc)
    engine.contact_step([pair_of(sc, ha, hb)], keep_polygons=True)
    _check(engine, sc, hb, taxels, rays, window, sigma)


@pytest.mark.parametrize("pairs", [256, 257])
def test_flat_sensor_sees_its_pairs_only(engine, pairs):
    """The pairs a sensor sees travel with the launch up to 256 of them: the
    last pair's pad under its sensor, the others in contact with another."""
    print("[case] pairs", pairs, flush=True)
    sc, other = S.tactile_pad(5, **FINE), S.tactile_pad(6, **COARSE)
    ha, hb = add_scene(engine, sc)
    hc, hd = add_scene(engine, other)
    engine.contact_step([pair_of(other, hc, hd)] * (pairs - 1) + [pair_of(sc, ha, hb)], keep_polygons=True)
    _check(engine, sc, hb, 9, 12, 0, 0.0)


def _check(engine, sc, hb, taxels, rays, window, sigma):
    ref = oracle_soft_rigid(sc)
    zs = sc["grid"]["half_size"][2]
    half = (0.0303, 0.0303, zs)  # rays off the polygons' edges
    res = 2 * half[0] / taxels * (1 + 1e-9)
    got = engine.taxels([dict(geom=hb, X_W_sensor=sc["X_WB"], half_size=half, resolution=res,
                              sampling_resolution=rays, window=window, sigma=sigma)])[0]
    want = O.taxels(ref["polys"], sc["X_WB"], half, res, rays, window, sigma)
    assert got.shape == want.shape == (taxels, taxels) and np.abs(want).max() > 0
    np.testing.assert_allclose(got, want, rtol=RTOL, atol=RTOL * np.abs(want).max())
