"""Sensor polygons whose keys (pair, element of A, element of B) need 64 bits
or more together are sorted in two stages."""
import numpy as np
import pytest

from mujoco_contact_surfaces_amd import Engine
from mujoco_contact_surfaces_amd import scenes as S
from test_gpu_parity import add_scene, pair_of

pytestmark = pytest.mark.gpu


def test_polygons_in_order_of_keys_beyond_64_bits():
    """Two pads among 65546 pairs, one of them of a 2.3M tet body and a 16.8M
    triangle grid (17 + 22 + 25 bits): the samples, whose sequence depends on the
    order of the polygons, are those of a call of the two pairs."""
    e = Engine(0)
    try:
        a, b = S.tactile_pad(5, L=4, K=4, m=60), S.tactile_pad(6, L=4, K=4, m=60)
        ha = add_scene(e, a)
        two = [pair_of(a, *ha), pair_of(b, add_scene(e, b)[0], ha[1])]
        tax = np.array([[x, y, 0.002] for y in np.linspace(-0.03, 0.03, 9) for x in np.linspace(-0.03, 0.03, 7)])

        def sensors():
            return [e.taxel_sensor(ha[1], a["X_WB"], tax, 0.004, res, method, sampling, True)
                    for method, sampling, res in (("closest", "area_importance", 0.002), ("closest", "default", 0.001),
                                                  ("squared", "area_importance", 0.002))]

        _, cnt = e.contact_step(two, keep_polygons=True)
        want = sensors()
        V, T, p = S.soft_mesh(7, 3, 1, 0.04, 0.03, 0.02, 5e4)
        VR, FR = S.rigid_mesh(1, 2900, 0.4)
        hs = e.add_soft_mesh(V, T, p, dict(S.SOFT_PROPS, hydroelastic_modulus=5e4), 900)
        hr = e.add_rigid_mesh(VR, FR, S.RIGID_PROPS, 901)
        ball, z = S.sphere_box(1), np.zeros(6)
        pairs = [pair_of(dict(ball, X_WA=ball["X_WA"] + np.r_[np.zeros(11), 5.0]), *add_scene(e, ball))] * 65546
        pairs[7] = (hs, hr, S.pose(np.eye(3), [0, 0, 5.0]), S.pose(np.eye(3), [0, 0, 0]), z, z)
        pairs[100], pairs[65000] = two
        assert len(pairs).bit_length() + len(T).bit_length() + len(FR).bit_length() >= 64
        _, c = e.contact_step(pairs, keep_polygons=True)
        np.testing.assert_array_equal(c[[100, 65000]], cnt)
        np.testing.assert_array_equal(c.sum(0), cnt.sum(0))
        for (v, m), (w, k) in zip(sensors(), want):
            assert m == k > 0 and np.abs(w).max() > 0
            np.testing.assert_array_equal(v, w)
    finally:
        e.close()
