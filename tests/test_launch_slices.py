"""Launches of any number of workgroups (noa_amd/csrc/launch_slices.hh, compiled here for the host): every workgroup
once and in order, each launch below HIP's 2^32 work items along x, one launch wherever one is enough."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def slices(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("slices") / "libslices.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC",
                    os.path.join(HERE, "native", "launch_slices_host.cc"), "-o", so], check=True)
    f = ctypes.CDLL(so).slices
    f.argtypes = [ctypes.c_int64, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_int]

    def call(workgroups, lanes, fail_at=-1):
        first, count = np.zeros(600, dtype=np.int64), np.zeros(600, dtype=np.uint32)
        n = f(workgroups, lanes, first.ctypes.data, count.ctypes.data, 600, fail_at)
        return n, first[:max(n, 0)], count[:max(n, 0)].astype(np.int64)
    return call


@pytest.mark.parametrize("lanes", [64, 256, 512, 1024])
def test_ranges(slices, lanes):
    most = (2 ** 32 - 1) // lanes
    for workgroups in (1, 2, most - 1, most, most + 1, 2 * most, 2 * most + 1, 2 ** 31 - 1, 2 ** 31, 5 * most + 3):
        n, first, count = slices(workgroups, lanes)
        assert n == -(-workgroups // most) and first[0] == 0 and count.sum() == workgroups
        assert np.array_equal(first[1:], (first + count)[:-1])
        assert count.min() >= 1 and (count * lanes).max() < 2 ** 32
    assert slices(0, lanes)[0] == 0


def test_stops_at_an_error(slices):
    assert slices(2 ** 31, 256, fail_at=3)[0] == -7
    assert slices(2 ** 20, 256, fail_at=1)[0] == 1
