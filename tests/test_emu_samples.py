"""hcs_samples.h built for the CPU.  Sample counts of the taxel sensor: offsets
of samples are 32-bit, so a count beyond 2^32 - 1 has to be refused before
anything is sized by it.  The curved sensor's ray cull: it may skip no triangle
that the hit test accepts."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_D = C.POINTER(C.c_double)


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("emusmp") / "libemu_samples.so")
    cmd = ["g++", "-O2", "-std=c++20", "-ffp-contract=off", "-fPIC", "-shared", "-Wno-unknown-pragmas",
           "-I", os.path.join(ROOT, "tests", "emu", "include"),
           "-I", os.path.join(ROOT, "mujoco_contact_surfaces_amd", "csrc"),
           os.path.join(ROOT, "tests", "emu", "emu_samples.cpp"), "-o", out, "-lpthread"]
    subprocess.run(cmd, check=True, timeout=600)
    lib = C.CDLL(out)
    lib.emu_area_chain.restype = C.c_int64
    lib.emu_area_chain.argtypes = [C.c_double, C.c_double, _D, C.c_int64]
    lib.emu_grid_samples.restype = C.c_int64
    lib.emu_grid_samples.argtypes = [_D, C.c_double]
    lib.emu_lines_miss.restype = None
    lib.emu_lines_miss.argtypes = [_D, _D, _D, C.c_int64, C.POINTER(C.c_ubyte)]
    return lib


@pytest.mark.parametrize("top,step", [(0.0, 0.0), (1.0, 1.0), (1.0, 0.3), (3.7e-3, 1.1e-6), (np.inf, np.inf),
                                      (2.0, np.nan)])
def test_area_chain_counts_the_sums_below_the_top(emu, top, step):
    ref, a = [], 0.0
    while a < top:
        ref.append(a)
        a = a + step
    acc = np.zeros(max(1, len(ref)))
    assert emu.emu_area_chain(top, step, acc.ctypes.data_as(_D), len(acc)) == len(ref)
    np.testing.assert_array_equal(acc[:len(ref)], ref)


# steps that 32 bits cannot count, that never leave a rounding interval of
# the top, and none at all
@pytest.mark.parametrize("res", [2.2e-10, 1e-13, 1e-18, 0.0])
@pytest.mark.parametrize("top", [1e-4, 1.0, 3e5])
def test_area_chain_refuses_more_than_32_bits_count(emu, top, res):
    assert emu.emu_area_chain(top, res * top, None, 0) == -1


def _triangle(l01, l02):
    return np.array([0.1, 0.2, 0.3, 0.1 + l01, 0.2, 0.3, 0.1, 0.2 + l02, 0.3])


def _passes(st):
    n, a = 0, 0.0
    while a <= 1:
        n, a = n + 1, a + 1.0 / st
    return n


@pytest.mark.parametrize("l01,l02,res", [(1e-3, 2e-3, 5e-3), (3e-3, 1e-3, 1e-3), (0.02, 0.013, 3.7e-4), (0.3, 1e-4, 1e-3),
                                         (0.0, 0.0, 1e-3), (0.1, 1e-6, 1e-6)])
def test_grid_samples_are_the_passes_of_the_loops(emu, l01, l02, res):
    t = _triangle(l01, l02)
    n0, n1 = np.linalg.norm(t[3:6] - t[:3]) / res, np.linalg.norm(t[6:9] - t[:3]) / res
    st2 = int(n1) + 1
    st = max(int(n0) + 1, st2)
    assert emu.emu_grid_samples(t.ctypes.data_as(_D), res) == _passes(st) * _passes(st2)


# 1e5 x 1e5 passes (a product that wraps 32 bits), steps beyond an int, and
# edges without an end
@pytest.mark.parametrize("l01,l02,res", [(0.05, 0.05, 5e-7), (0.05, 0.05, 2e-11), (0.05, 1e-9, 1e-18),
                                         (1e-9, 0.05, 1e-300), (np.inf, 0.05, 1e-3)])
def test_grid_samples_refuse_more_than_32_bits_count(emu, l01, l02, res):
    assert emu.emu_grid_samples(_triangle(l01, l02).ctypes.data_as(_D), res) == -1


def _dot(a, b):
    return (a[:, 0] * b[:, 0] + a[:, 1] * b[:, 1]) + a[:, 2] * b[:, 2]


def _cross(a, b):
    return np.stack([a[:, 1] * b[:, 2] - a[:, 2] * b[:, 1], a[:, 2] * b[:, 0] - a[:, 0] * b[:, 2],
                     a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0]], 1)


def _accepted(T, O, D):
    """The hit test of the curved sensor's rays."""
    e1, e2, s = T[:, 3:6] - T[:, :3], T[:, 6:] - T[:, :3], O - T[:, :3]
    h = _cross(D, e2)
    det = _dot(e1, h)
    f = 1.0 / det
    u, q = f * _dot(s, h), _cross(s, e1)
    v, t = f * _dot(D, q), f * _dot(e2, q)
    return (np.abs(det) >= 1e-10) & (u >= 0) & (u <= 1) & (v >= 0) & (u + v <= 1) & (t > 0)


@pytest.mark.parametrize("size", [0.05, 0.01, 0.003])
@pytest.mark.parametrize("length", [1e-2, 1.0, 1.99, 2.01, 10.0, 1e3, 1e5, 1e7])
def test_no_accepted_hit_is_skipped(emu, size, length):
    """Rays that graze a triangle's plane just beyond its outermost vertex,
    with a determinant just over the hit test's limit: rounding accepts some
    whose line passes outside the bounding sphere, the farther the longer
    their direction."""
    rng, n = np.random.default_rng(1), 200000
    at = rng.uniform(-0.1, 0.1, (n, 3))
    V = at[:, None] + rng.normal(size=(n, 3, 3)) * size
    C0 = V.mean(1)
    F = V[np.arange(n), np.argmax(((V - C0[:, None]) ** 2).sum(2), 1)]
    nr = _cross(V[:, 1] - V[:, 0], V[:, 2] - V[:, 0])
    area = np.linalg.norm(nr, axis=1)
    nr /= area[:, None]
    out = (F - C0) / np.linalg.norm(F - C0, axis=1)[:, None]
    tilt = 1e-10 / (area * length) * 10 ** rng.uniform(0, 1, n) * rng.choice([-1, 1], n)
    Dh = _cross(nr, out) + np.clip(tilt, -1, 1)[:, None] * nr
    Dh /= np.linalg.norm(Dh, axis=1)[:, None]
    O = F + out * 10 ** rng.uniform(-9, -3, n)[:, None] - Dh * rng.uniform(1e-3, 5e-2, n)[:, None]
    T, O, D = (np.ascontiguousarray(x) for x in (V.reshape(n, 9), O, Dh * length))
    skip = np.zeros(n, np.uint8)
    emu.emu_lines_miss(*(x.ctypes.data_as(_D) for x in (T, O, D)), n, skip.ctypes.data_as(C.POINTER(C.c_ubyte)))
    hit = _accepted(T, O, D)
    assert hit.sum() > 0 or length < 1e5
    assert skip.sum() > n // 100 or length > 10  # (beyond, the widening covers all of these rays)
    assert not (hit & (skip != 0)).any()
