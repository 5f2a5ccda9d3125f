"""Steps of very many work items: a per-call step whose two culls both take
more blocks than add up their counts themselves, and unconfigured batches on
both sides of the lines between items cut evenly, cut by their expected
candidates, and left whole.  Results are those of calls of one pair."""
import numpy as np
import pytest

from mujoco_contact_surfaces_amd import Engine
from mujoco_contact_surfaces_amd import scenes as S
from test_gpu_parity import assert_wrench_close

pytestmark = pytest.mark.gpu


def _pairs(e, m, n):
    """A soft body on a plane grid of 2 m^2 triangles (m^2 / 32 chunks), in
    three poses, the first away from the grid; n pairs of them in turn."""
    V, T, p = S.soft_mesh(2, 2, 1, 0.04, 0.03, 0.02, 5e4)
    VR, FR = S.rigid_mesh(1, m, 0.4)
    ha = e.add_soft_mesh(V, T, p, dict(S.SOFT_PROPS, hydroelastic_modulus=5e4), 0)
    hb = e.add_rigid_mesh(VR, FR, S.RIGID_PROPS, 1)
    XB, z = S.pose(np.eye(3), [0, 0, 0]), np.zeros(6)
    base = [(ha, hb, S.pose(np.eye(3), at), XB, z, z) for at in ([0, 0, 5.0], [0.013, 0.007, 0.019], [-0.11, 0.09, 0.0185])]
    one = [e.contact_step([q]) for q in base]
    assert one[0][1][0, 1] == 0 and one[1][1][0, 1] > 0 and one[2][1][0, 1] > 0
    return [base[k % 3] for k in range(n)], one


def _check(W, cnt, one):
    for k in range(len(W)):
        w, c = one[k % 3]
        np.testing.assert_array_equal(cnt[k], c[0])
        assert_wrench_close(W[k], w[0], rtol=1e-12)


def test_step_of_a_million_items():
    """140 pairs of 8192 chunks: 4480 blocks in the first cull, and as many
    places for live items as make 4480 in the second."""
    e = Engine(0)
    try:
        pairs, one = _pairs(e, 512, 140)
        W, cnt = e.contact_step(pairs)
        _check(W, cnt, one)
    finally:
        e.close()


# 512 chunks a pair: 4096 and 4608 items, 262144 and 262656, 2097152 and
# 2097664
@pytest.mark.parametrize("n", [8, 9, 512, 513, 4096, 4097])
def test_unconfigured_batch_of_many_items(n):
    print("[case] batch items", 512 * n, flush=True)
    e = Engine(0)
    try:
        pairs, one = _pairs(e, 128, n)
        b = e.batch([p[:2] for p in pairs])
        b.set_state(np.array([np.concatenate(p[2:]) for p in pairs]))
        for _ in range(2):
            b.step()
            W, cnt = b.get()
            _check(W, cnt, one)
        b.close()
    finally:
        e.close()
