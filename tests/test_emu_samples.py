"""Sample counts of the taxel sensor (hcs_samples.h) built for the CPU:
offsets of samples are 32-bit, so a count beyond 2^32 - 1 has to be refused
before anything is sized by it."""
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
