"""The sensor kernels at the edges of their tiles: sample counts around a
wave, and few to many fan triangles, against the oracle's sensors on the
oracle's polygons."""
import numpy as np
import pytest

import oracle as O
from mujoco_contact_surfaces_amd import scenes as S
from test_gpu_parity import add_scene, oracle_soft_rigid, pair_of

pytestmark = pytest.mark.gpu

# the kernels run the oracle's arithmetic; only sums of n terms are added in
# another order, n eps of relative rounding (all terms have one sign): at most
# 1e5 samples reach a taxel here
RTOL = 1e5 * 2.3e-16

SMALL = dict(L=1, K=1, m=2)  # a handful of fan triangles, under one tile of 64
LARGE = dict(L=3, K=3, m=24)


def _pad(engine, shape, depth=0.003):
    sc = S.tactile_pad(3, depth=depth, **shape)
    ha, hb = add_scene(engine, sc)
    engine.contact_step([pair_of(sc, ha, hb)], keep_polygons=True)
    ref = oracle_soft_rigid(sc)
    tris, surf = O.fan_triangles(ref["polys"], np.zeros(len(ref["polys"]), int))
    return sc, hb, tris, surf


@pytest.mark.parametrize("shape", [SMALL, LARGE], ids=["few", "many"])
@pytest.mark.parametrize("m", [1, 63, 64, 65, 1000])
def test_curved_sensor_sample_and_slice_edges(engine, shape, m):
    print("[case] curved", shape, m, flush=True)
    sc, hb, tris, _ = _pad(engine, shape)
    rng = np.random.default_rng(m)
    # samples over the contact patch (where the fans are), the last one outside
    c = tris[:, :9].reshape(-1, 3, 3).mean(1)
    P = c[rng.integers(0, len(c), m)] + rng.uniform(-2e-4, 2e-4, (m, 3))
    P[:, 2] += 0.0007
    if m > 1:
        P[-1, :2] += 1.0
    N = np.tile([0.0, 0.0, 1.0], (m, 1))
    ptr = np.arange(m + 1, dtype=np.int32)
    vals = engine.curved_sensor(hb, sc["X_WB"], P, N, ptr, np.arange(m, dtype=np.int32), np.ones(m), 0.002)
    ref, hits = O.curved_sensor(tris, sc["X_WB"], P, N, ptr, np.arange(m, dtype=np.int32), np.ones(m), 0.002)
    assert hits > 0
    np.testing.assert_allclose(vals, ref, rtol=1e-12, atol=1e-12 * np.abs(ref).max())


@pytest.mark.parametrize("shape,npad", [(dict(L=1, K=1, m=2), 1), (dict(L=4, K=4, m=60), 1), (dict(L=4, K=4, m=70), 3)],
                         ids=["one-block", "rank", "radix"])
def test_sensor_polygons_are_read_in_key_order(engine, shape, npad):
    """The area-importance sequence and the first of equally near samples
    depend on the order of the polygons: a few of them, some thousand (rank
    sort) and more than the rank sort takes (packed radix sort), with the
    polygons of another pair left out."""
    print("[case] order", shape, npad, flush=True)
    other = S.sphere_box(2)
    hc, hd = add_scene(engine, other)
    scs = [S.tactile_pad(10 + k, **shape) for k in range(npad)]
    ha, hb = add_scene(engine, scs[0])
    pairs = [pair_of(other, hc, hd)]
    for sc in scs:  # the same pad handle under several bodies: one sensor, several surfaces
        a = ha if sc is scs[0] else add_scene(engine, sc)[0]
        pairs.append(pair_of(sc, a, hb))
    _, cnt = engine.contact_step(pairs, keep_polygons=True)
    if npad > 1:
        assert cnt[:, 1].sum() > 16384
    polys = [oracle_soft_rigid(sc)["polys"] for sc in scs]
    tris, surf = O.fan_triangles(np.concatenate(polys), np.repeat(np.arange(npad), [len(p) for p in polys]).astype(int))
    taxels = np.array([[x, y, 0.002] for y in np.linspace(-0.03, 0.03, 9) for x in np.linspace(-0.03, 0.03, 7)])
    X = scs[0]["X_WB"]
    for method, sampling, res in (("closest", "area_importance", 0.002), ("closest", "default", 0.001)):
        vals, m = engine.taxel_sensor(hb, X, taxels, 0.004, res, method, sampling, True)
        ref, rm = O.taxel_sensor(tris, surf, X, taxels, 0.004, res, method, sampling, True)
        assert m == rm and m > 0
        np.testing.assert_array_equal(vals, ref)
