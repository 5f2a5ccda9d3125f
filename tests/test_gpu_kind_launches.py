"""Launches whose pairs share one kind run kernels built for it, mixed ones
the general kernel: item counts around a wave, against the oracle."""
import numpy as np
import pytest

import oracle as O
from mujoco_contact_surfaces_amd import scenes as S
from test_gpu_parity import add_scene, assert_wrench_close, oracle_soft_rigid, pair_of

pytestmark = pytest.mark.gpu


def _plane_scene(engine, k, L, K):
    """A soft ellipsoid of 20 * 4^L (1 + 3 (K - 1)) tets on a tilted plane."""
    sc = S.soft_plane_env(5, k)
    V, T, p = S.soft_mesh(L, K, 1, 0.05, 0.04, 0.03, 1e5)
    props = dict(sc["soft"]["props"], hydroelastic_modulus=1e5)
    n, c = sc["X_WB"][:9].reshape(3, 3)[:, 2], sc["X_WB"][9:]
    R = sc["X_WA"][:9].reshape(3, 3)
    low = float((V @ R.T @ n).min())
    X = np.concatenate([R.reshape(9), c - (low + 0.006) * n])
    ha = engine.add_soft_mesh(V, T, p, props, 2 * k)
    hb = engine.add_rigid_plane(sc["plane"]["props"], 2 * k + 1)
    ref = O.soft_plane(V, T, p, X, sc["X_WB"], sc["V_WA"], sc["V_WB"], 1e5, props["dissipation"],
                       props["dynamic_friction"], sc["plane"]["props"]["dynamic_friction"])
    return (ha, hb, X, sc["X_WB"], sc["V_WA"], sc["V_WB"]), ref


# 20, 80 and 320 tets in one layer (less than an item, one item and a part,
# five items), and several hundred items
@pytest.mark.parametrize("sizes", [[(0, 1)], [(1, 1)], [(2, 1)], [(0, 1), (1, 1), (2, 2), (3, 4)]],
                         ids=["20", "80", "320", "mixed sizes"])
@pytest.mark.parametrize("queues", [1, 8])
def test_half_space_launch(engine, sizes, queues):
    print("[case] half-space", sizes, queues, flush=True)
    got = [_plane_scene(engine, k, L, K) for k, (L, K) in enumerate(sizes)]
    pairs, refs = [g[0] for g in got], [g[1] for g in got]
    W, cnt = engine.contact_step(pairs)
    b = engine.batch([p[:2] for p in pairs])
    b.set_state(np.array([np.concatenate(p[2:]) for p in pairs]))
    b.set_config(4, 1, 64, 2048, queues, 0)
    b.step()
    Wb, cb = b.get()
    st = b.item_stats()
    b.close()
    for i, r in enumerate(refs):
        np.testing.assert_array_equal(cnt[i], r["counts"])
        np.testing.assert_array_equal(cb[i], r["counts"])
        assert r["counts"][1] > 0
        assert_wrench_close(W[i], r["wrench"])
        assert_wrench_close(Wb[i], r["wrench"])
        assert st[st[:, 0] == i, 5].sum() == r["counts"][0]


# few survivors (less than a wave), some hundred, some thousand a pair
@pytest.mark.parametrize("size", [(0, 1), (1, 1), (3, 2)], ids=["20", "80", "5120"])
@pytest.mark.parametrize("representation", [0, 1])
@pytest.mark.parametrize("friction", [True, False])
def test_mixed_launch_clips_like_the_launches_of_one_kind(engine, size, representation, friction):
    """A half-space, a triangle and a soft pair in one call against calls of
    one pair: the same faces, record for record; the wrenches' sums differ in
    order only."""
    print("[case] mixed clip", size, representation, friction, flush=True)
    plane, _ = _plane_scene(engine, 1, *size)
    pad = S.tactile_pad(3, L=size[0], K=size[1], m=20, depth=0.006)
    soft = S.soft_soft_env(3, 0, nt_range=(3e3, 6e3))
    pairs = [plane]
    for sc in (pad, soft):
        pairs.append(pair_of(sc, *add_scene(engine, sc)))
    opts = dict(representation=representation, apply_forces=friction, face_capacity=1 << 18)

    def ordered(rec, key):
        o = np.lexsort(key.T[::-1])
        return rec[o], key[o]

    W, cnt, (rec, key) = engine.contact_step(pairs, **opts)
    rec, key = ordered(rec, key)
    assert (cnt[:, 2] > 0).all() and len(rec) == cnt[:, 2].sum()
    for k, p in enumerate(pairs):
        W1, c1, (r1, k1) = engine.contact_step([p], **opts)
        np.testing.assert_array_equal(cnt[k], c1[0])
        if friction:
            assert_wrench_close(W[k], W1[0], rtol=1e-12)
        r1, k1 = ordered(r1, k1)
        mine = key[:, 0] == k
        np.testing.assert_array_equal(key[mine][:, 1:], k1[:, 1:])
        np.testing.assert_array_equal(rec[mine], r1)
