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
