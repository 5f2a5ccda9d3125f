"""When a batch is planned: a configuration set before the first state is
honoured once there is one, and a batch that was never configured stays one
whose items are cut in every step, also after a mesh is replaced."""
import numpy as np
import pytest

from mujoco_contact_surfaces_amd import scenes as S
from test_gpu_parity import add_scene, pair_of

pytestmark = pytest.mark.gpu


def _pairs(engine):
    """A pad (triangle queries), a ball on a box (tet queries where allowed)
    and a soft pair, twice."""
    out = []
    for sc in (S.tactile_pad(2, L=4, K=3, m=40, depth=0.006), S.sphere_box(1), S.soft_soft_env(3, 0, nt_range=(3e3, 6e3))):
        out.append(pair_of(sc, *add_scene(engine, sc)))
    return out + out


def _state(pairs):
    return np.array([np.concatenate(p[2:]) for p in pairs])


# tet queries on and off, one and eight queues, whole items and split ones
@pytest.mark.parametrize("cfg", [(4, 1, 64, 64, 1, 1), (12, 1, 0, 64, 8, 0), (8, 1, 64, 0, 1, 1)])
def test_configuration_before_the_state(engine, cfg):
    print("[case] config first", cfg, flush=True)
    pairs = _pairs(engine)
    after, before = engine.batch([p[:2] for p in pairs]), engine.batch([p[:2] for p in pairs])
    after.set_state(_state(pairs))
    after.set_config(*cfg)
    before.set_config(*cfg)
    before.set_state(_state(pairs))
    for b in (after, before):
        b.step()
    Wa, ca = after.get()
    Wb, cb = before.get()
    np.testing.assert_array_equal(ca, cb)
    np.testing.assert_array_equal(Wa, Wb)
    sa, sb = after.item_stats(), before.item_stats()
    # pair, kind, queries, candidates and survivors of every item
    np.testing.assert_array_equal(sa[:, [0, 1, 2, 5, 6]], sb[:, [0, 1, 2, 5, 6]])
    assert before.config() == after.config()
    after.close(), before.close()


def test_unconfigured_batch_after_a_mesh_is_replaced(engine):
    pairs = _pairs(engine)
    V, T, p = S.soft_mesh(3, 4, 1, 0.04, 0.03, 0.02, 5e4)
    b = engine.batch([q[:2] for q in pairs])
    b.set_state(_state(pairs))
    b.step()
    b.get()
    engine.replace_soft_mesh(pairs[0][0], V, T, p)
    fresh = engine.batch([q[:2] for q in pairs])
    fresh.set_state(_state(pairs))
    got = []
    for x in (b, fresh):
        x.step()
        got.append(x.get() + (x.item_stats(),))
    np.testing.assert_array_equal(got[0][0], got[1][0])
    np.testing.assert_array_equal(got[0][1], got[1][1])
    assert len(got[0][2]) == len(got[1][2]) and got[0][1][0, 1] > 0
    b.close(), fresh.close()


def test_item_profile_runs_the_step(engine):
    """The profile of a batch that is not planned steps the batch, as that of a
    planned one does."""
    pairs = _pairs(engine)
    moved = _state(pairs)
    moved[:, 23] -= 0.0005
    b, ref = engine.batch([p[:2] for p in pairs]), engine.batch([p[:2] for p in pairs])
    b.set_state(_state(pairs))
    b.step()
    b.get()
    ref.set_state(moved)
    ref.step()
    b.set_state(moved)
    st = b.item_stats()
    W, cnt = b.get()
    Wr, cr = ref.get()
    np.testing.assert_array_equal(cnt, cr)
    np.testing.assert_array_equal(W, Wr)
    for k in range(len(pairs)):
        assert st[st[:, 0] == k, 5].sum() == cnt[k, 0]
    b.close(), ref.close()
