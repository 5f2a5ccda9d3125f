"""The clip of launches that mix pair kinds (hcs_clip.h) built for the CPU:
against the clip of the launches of one kind, value for value, and its
divisions against the division."""
import ctypes as C

import numpy as np
import pytest

from mujoco_contact_surfaces_amd import scenes as S
from test_emu_kernels import KPLANE, KSOFT, KTET, KTRI, _D, _I32, _dp, _scene, emu, run_pair  # noqa: F401


@pytest.fixture(scope="module")
def clip(emu):  # noqa: F811
    emu.emu_clip_differences.restype = C.c_int64
    emu.emu_div3.argtypes = [_D, C.c_int64, _D]
    emu.emu_div_by.argtypes = [_D, _D, C.c_int64, _D]
    emu.emu_clip_planes.argtypes = [_D, _I32, _D, C.c_int64, C.c_int]
    for f in (emu.emu_div3, emu.emu_div_by, emu.emu_clip_planes):
        f.restype = None
    return emu


# survivors of every kind, fewer and more than a wave's, both representations
@pytest.mark.parametrize("kind", [KTRI, KTET, KSOFT, KPLANE])
@pytest.mark.parametrize("representation", [0, 1])
def test_contributions_of_every_survivor(clip, kind, representation):
    _, counts, _ = run_pair(clip, _scene(kind), kind, representation=representation)
    assert counts[1] > (64 if kind != KPLANE else 0)
    assert clip.emu_clip_differences() == 0


@pytest.mark.parametrize("kind", [KTRI, KTET])
def test_contributions_of_meshes_far_from_their_origin(clip, kind):
    sc = dict(S.tactile_pad(3, L=1, K=1, m=2) if kind == KTET else S.tactile_pad(3, L=2, K=2, m=12))
    s, r = dict(sc["soft"]), dict(sc["rigid"])
    XA, XB = sc["X_WA"].copy(), sc["X_WB"].copy()
    for m, X, o in ((s, XA, np.array([3e3, -2e3, 1e3])), (r, XB, np.array([-1e3, 3e3, 2e3]))):
        m["V"] = m["V"] + o
        X[9:] -= X[:9].reshape(3, 3) @ o
    sc.update(soft=s, rigid=r, X_WA=XA, X_WB=XB)
    _, counts, _ = run_pair(clip, sc, kind)
    assert counts[1] > 0
    assert clip.emu_clip_differences() == 0


def _values(rng, n, lo, hi):
    return rng.choice([-1.0, 1.0], n) * (1 + rng.random(n)) * 2.0 ** rng.integers(lo, hi, n)


def test_division_by_three(clip):
    rng, n = np.random.default_rng(3), 2000000
    k = rng.integers(1, 2 ** 51, n).astype(float)
    x = np.concatenate([_values(rng, n, -900, 1000), 3 * k, 3 * k + 1, 3 * k + 2, np.nextafter(3 * k, 0),
                        [0.0, np.inf, -np.inf, np.finfo(float).max, 1.0, 2.0]])
    q = np.zeros_like(x)
    clip.emu_div3(_dp(x), len(x), _dp(q))
    np.testing.assert_array_equal(q, x / 3.0)
    nan = np.array([np.nan])
    clip.emu_div3(_dp(nan), 1, _dp(nan))
    assert np.isnan(nan[0])


def test_division_by_a_slip_speed(clip):
    """Divisors as the caller allows them: 1e-6 (the regularised slip speed at
    rest) to 1e100, and 1e-4; dividends a component of the slip, or the speed."""
    rng, n = np.random.default_rng(4), 3000000
    b = np.exp(rng.uniform(np.log(1e-6), np.log(1e100), n))
    x = np.concatenate([b * rng.uniform(-1, 1, n), b * _values(rng, n, -60, 0), _values(rng, n, -200, 300), b,
                        np.nextafter(b, 0), np.zeros(n)])
    b = np.concatenate([b, b, b, np.full(n, 1e-4), b, b])
    q = np.zeros_like(x)
    clip.emu_div_by(_dp(x), _dp(b), len(x), _dp(q))
    np.testing.assert_array_equal(q, x / b)


@pytest.mark.parametrize("n", [3, 4, 5, 6, 7])
def test_clipping_plane(clip, n):
    """Convex polygons against planes through them, past them, along their own
    plane within rounding (more than two crossings), through vertices, and
    without a value."""
    rng, m = np.random.default_rng(n), 60000
    a = np.sort(rng.uniform(0, 2 * np.pi, (m, n)), 1)
    e = np.linalg.qr(rng.normal(size=(m, 3, 3)))[0]
    size = 10 ** rng.uniform(-6, 0, m)
    at = rng.uniform(-1, 1, (m, 3)) * rng.choice([0, 1e-2, 1, 1e3], m)[:, None]
    V = (np.cos(a)[..., None] * e[:, None, 0] + np.sin(a)[..., None] * e[:, None, 1]) * size[:, None, None] + at[:, None]
    nh = np.linalg.qr(rng.normal(size=(m, 3, 3)))[0][:, 0]
    kind = rng.integers(0, 5, m)
    nh = np.where((kind == 1)[:, None], e[:, 2], nh)  # the polygon's own plane
    P = at + np.where(kind == 2, 3.0, rng.uniform(-1, 1, m))[:, None] * size[:, None] * e[:, 0]
    P = np.where((kind == 1)[:, None], at, P)
    P = np.where((kind == 3)[:, None], V[np.arange(m), rng.integers(0, n, m)], P)  # through a vertex
    off = -(nh * P).sum(1)
    off[:3] = np.nan, np.inf, -np.inf
    planes = np.ascontiguousarray(np.concatenate([nh, off[:, None]], 1))
    pad = np.zeros((m, 8, 3))
    pad[:, :n] = V
    out = []
    for wave in (0, 1):
        v, k = pad.copy(), np.full(m, n, np.int32)
        clip.emu_clip_planes(_dp(v), k.ctypes.data_as(_I32), _dp(planes), m, wave)
        out.append((v, k))
    np.testing.assert_array_equal(out[0][1], out[1][1])
    np.testing.assert_array_equal(out[0][0], out[1][0])
    assert {0, n, n + 1} <= set(out[0][1])
