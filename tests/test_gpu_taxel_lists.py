"""Flat sensors whose polygon lists may pass 2^32 entries, which is what their
32-bit offsets number: counted in 64 bits, and refused when they do."""
import numpy as np
import pytest

from mujoco_contact_surfaces_amd import scenes as S
from mujoco_contact_surfaces_amd.engine import HcsError
from test_gpu_parity import add_scene, pair_of

pytestmark = pytest.mark.gpu

HCS_ERR_CAPACITY = -4
RTOL = 1e-10  # as for the sensors of the batched step


def _grid(sc, geom, half, taxels, rays, at=(0.0, 0.0)):
    X = sc["X_WB"].copy()
    X[9:11] += at
    return dict(geom=geom, X_W_sensor=X, half_size=(half, half, sc["grid"]["half_size"][2]),
                resolution=2 * half / taxels * (1 + 1e-9), sampling_resolution=rays)


def test_lists_beyond_32_bits_are_refused(engine):
    """4400 pads over one sensor of 1000 x 1000 taxels within 0.2 mm, which a
    polygon of every pad covers: 4.4e9 entries, 1.1e8 in 32 bits."""
    sc = S.tactile_pad(3, L=1, K=1, m=2)
    ha, hb = add_scene(engine, sc)
    _, cnt = engine.contact_step([pair_of(sc, ha, hb)] * 4400, keep_polygons=True)
    np.testing.assert_array_equal(cnt, np.tile(cnt[:1], (4400, 1)))
    with pytest.raises(HcsError) as e:
        engine.taxels([_grid(sc, hb, 1e-4, 1000, 1, (0.0013, 0.0007))])
    assert e.value.code == HCS_ERR_CAPACITY
    many = engine.taxels([_grid(sc, hb, 0.03, 16, 8)])[0]
    engine.contact_step([pair_of(sc, ha, hb)], keep_polygons=True)
    one = engine.taxels([_grid(sc, hb, 0.03, 16, 8)])[0]
    assert np.abs(one).max() > 0
    np.testing.assert_array_equal(many, one)  # every hit ties with its copies


def test_many_polygons_under_a_million_taxels(engine):
    """More polygons x taxels than 2^32, far fewer entries: plain call and
    batched step, against sixteen rays per taxel of a coarser grid."""
    sc = S.tactile_pad(5, L=4, K=4, m=48)
    ha, hb = add_scene(engine, sc)
    pair = pair_of(sc, ha, hb)
    _, cnt = engine.contact_step([pair], keep_polygons=True)
    assert cnt[0, 1] * 1024 ** 2 > 2 ** 32
    half = 0.0303  # rays off the polygons' edges
    fine = engine.taxels([_grid(sc, hb, half, 1024, 1)])[0]
    want = engine.taxels([_grid(sc, hb, half, 256, 4)])[0]
    got = fine.reshape(256, 4, 256, 4).mean((1, 3))
    assert np.abs(want).max() > 0
    np.testing.assert_allclose(got, want, rtol=RTOL, atol=RTOL * np.abs(want).max())
    b = engine.batch([pair[:2]])
    b.set_sensors([0], [_grid(sc, hb, half, 1024, 1)])
    b.set_state(np.concatenate(pair[2:])[None, :])
    b.step()
    np.testing.assert_array_equal(b.taxels()[0], fine)
    b.close()
