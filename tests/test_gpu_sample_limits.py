"""Taxel sensors that ask for more samples than 32-bit offsets number are
refused before a buffer is sized by the count; the next call is served."""
import numpy as np
import pytest

import oracle as O
from mujoco_contact_surfaces_amd import Engine
from mujoco_contact_surfaces_amd import scenes as S
from mujoco_contact_surfaces_amd.engine import HcsError
from test_gpu_parity import add_scene, oracle_soft_rigid, pair_of

pytestmark = pytest.mark.gpu

HCS_ERR_LIMIT = -6
TAXELS = np.array([[x, 0.0, 0.002] for x in np.linspace(-0.02, 0.02, 5)])


def _step(engine, npairs):
    sc = S.tactile_pad(3, L=1, K=1, m=2)
    ha, hb = add_scene(engine, sc)
    _, cnt = engine.contact_step([pair_of(sc, ha, hb)] * npairs, keep_polygons=True)
    assert (cnt[:, 1] > 0).all()
    return hb, sc["X_WB"]


# one surface of 1 / resolution samples, and 1100 surfaces of 4e6 each: no
# surface's count passes 32 bits there, the sum 4.4e9 does (and would wrap to
# 1e8)
@pytest.mark.parametrize("npairs,resolution", [(1, 1e-10), (1, 1e-17), (1100, 2.5e-7)])
def test_area_importance_samples_beyond_32_bits(engine, npairs, resolution):
    print("[case] area importance", npairs, resolution, flush=True)
    geom, X = _step(engine, npairs)
    with pytest.raises(HcsError) as e:
        engine.taxel_sensor(geom, X, TAXELS, 0.004, resolution, "squared", "area_importance")
    assert e.value.code == HCS_ERR_LIMIT
    _, m = engine.taxel_sensor(geom, X, TAXELS, 0.004, 0.002, "squared", "area_importance")
    assert 499 * npairs <= m <= 502 * npairs


# one triangle's samples pass 32 bits; its steps pass an int; and 1100 pairs
# of 1.8e7 samples each, whose sum does (2e10)
@pytest.mark.parametrize("npairs,resolution", [(1, 2e-7), (1, 1e-12), (1100, 1.5e-5)])
def test_default_samples_beyond_32_bits(engine, npairs, resolution):
    print("[case] default", npairs, resolution, flush=True)
    geom, X = _step(engine, npairs)
    _, one = engine.taxel_sensor(geom, X, TAXELS, 0.004, 0.002)
    with pytest.raises(HcsError) as e:
        engine.taxel_sensor(geom, X, TAXELS, 0.004, resolution)
    assert e.value.code == HCS_ERR_LIMIT
    _, m = engine.taxel_sensor(geom, X, TAXELS, 0.004, 0.002)
    assert m == one > 0


def _passes(st):
    n, a = 0, 0.0
    while a <= 1:
        n, a = n + 1, a + 1.0 / st
    return n


def test_a_large_share_of_one_triangle_is_counted():
    """One of 111 triangles has more than its share of 2^32 samples while their
    sum, 7e8, does not pass it: counted again in 64 bits and served."""
    sc = S.tactile_pad(3, L=1, K=1, m=2)
    P = oracle_soft_rigid(sc)["polys"]
    T = O.fan_triangles(P, np.zeros(len(P), int))[0][:, :9].reshape(-1, 3, 3)
    res = 2.4e-6
    steps = [(int(np.linalg.norm(t[1] - t[0]) / res) + 1, int(np.linalg.norm(t[2] - t[0]) / res) + 1) for t in T]
    each = [_passes(max(st)) * _passes(st[1]) for st in steps]
    assert max(each) > 0xffffffff // len(T) and sum(each) < 0xffffffff
    e = Engine(0)
    try:
        geom, X = _step(e, 1)
        _, m = e.taxel_sensor(geom, X, TAXELS, 0.004, res)
        assert m == sum(each)
    finally:
        e.close()
