"""The work items of per-call steps and unconfigured batches (hcs_items.h) built
for the CPU: every cut of a tree holds each leaf once, the pieces fit their
room, and a pair stepped over items enumerated, culled and cut that way has the
oracle's counts and wrench."""
import ctypes as C

import numpy as np
import pytest

from mujoco_contact_surfaces_amd import scenes as S
from test_emu_kernels import (KPLANE, KSOFT, KTET, KTRI, _D, _I32, _dp, _scene, assert_wrench_close, emu,  # noqa: F401
                              oracle, run_pair)

_U32 = C.POINTER(C.c_uint32)


@pytest.fixture(scope="module")
def items(emu):  # noqa: F811
    emu.emu_cover_errors.argtypes = [_D, C.c_int, _I32, C.c_int, _D]
    emu.emu_pieces.restype = C.c_int64
    emu.emu_pieces.argtypes = [_U32, C.c_uint32, C.c_uint32, C.c_uint32, _U32]
    emu.emu_set_items.argtypes = [C.c_int, C.c_int, C.c_uint32]
    emu.emu_set_items.restype = None
    return emu


def _one_tet():
    return (np.array([[0.0, 0, 0], [0.1, 0, 0], [0, 0.1, 0], [0, 0, 0.1]]), np.array([[0, 1, 2, 3]], np.int32),
            np.array([0.0, 0, 0, 1e4]))


# one tet, two, fewer than a frontier holds, some thousand
@pytest.mark.parametrize("body", ["1", "2", "20", "80", "1280", "5120"])
def test_cuts_hold_every_leaf_once(items, body):
    V, T, p = _one_tet() if body in "12" else S.soft_mesh(*{"20": (0, 1), "80": (1, 1), "1280": (2, 2), "5120": (3, 2)}[body],
                                                          1, 0.04, 0.03, 0.02, 5e4)
    if body == "2":
        V, T, p = np.vstack([V, [[0.1, 0.1, 0.1]]]), np.vstack([T, [[1, 2, 3, 4]]]).astype(np.int32), np.append(p, 0.0)
    V, T, p = np.ascontiguousarray(V), np.ascontiguousarray(T, np.int32), np.ascontiguousarray(p)
    assert items.emu_cover_errors(_dp(V), len(V), T.ctypes.data_as(_I32), len(T), _dp(p)) == 0


@pytest.mark.parametrize("n,room", [(1, 2), (5, 5), (5, 6), (1000, 1500), (65536, 65536 + 262144), (200000, 200000 + 262144)])
@pytest.mark.parametrize("largest", [1, 700, 200000, (1 << 27) - 1])
def test_pieces_fit_their_room(items, n, room, largest):
    rng = np.random.default_rng(n + largest)
    est = np.minimum(np.exp(rng.uniform(0, np.log(largest + 1), n)), largest).astype(np.uint32)
    word = est | rng.integers(0, 16, n).astype(np.uint32) << np.uint32(28)
    target = np.zeros(1, np.uint32)
    all_ = items.emu_pieces(word.ctypes.data_as(_U32), n, 256 * 32, room, target.ctypes.data_as(_U32))
    assert n <= all_ <= room and target[0] >= 512


@pytest.mark.parametrize("kind", [KTRI, KTET, KSOFT, KPLANE])
@pytest.mark.parametrize("mode,depth,room", [(1, 0, 1), (1, 2, 128), (1, 4, 256), (2, 0, 64), (2, 3, 128)])
def test_steps_over_enumerated_items(items, kind, mode, depth, room):
    sc = _scene(kind)
    items.emu_set_items(mode, depth, room)
    try:
        W, counts, stats = run_pair(items, sc, kind)
    finally:
        items.emu_set_items(0, 0, 0)
    ref = oracle(sc, kind)
    np.testing.assert_array_equal(counts, ref["counts"])
    assert_wrench_close(W[0], ref["wrench"])
    assert ref["counts"][1] > 0 and stats[4] == 0
