"""Index arithmetic of the PUMAS table search (noa_amd/csrc/pumas_search.hh, compiled here for the host)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("search") / "libsearch.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC",
                    os.path.join(HERE, "native", "pumas_search_host.cc"), "-o", so], check=True)
    handle = ctypes.CDLL(so)
    handle.pumas_tree_levels.restype = ctypes.c_uint32
    handle.pumas_cell.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_float, ctypes.c_int]
    return handle


@pytest.mark.parametrize("n", [2, 3, 5, 35, 36, 64, 65, 145, 192])
def test_cell(lib, n):
    """The bracketing cell for every point between the nodes, and a cell of
    the table in every other lane: for points beyond the nodes, for NaN, and
    for the all-zero nodes of the first element."""
    t = np.sort(np.random.default_rng(n).uniform(-14, 0, n)).astype(np.float32)
    for i in range(n - 1):
        for x in (t[i], np.float32(0.5 * (float(t[i]) + float(t[i + 1]))), np.nextafter(t[i + 1], np.float32(-99))):
            assert lib.pumas_cell(t.ctypes.data, n, x, 1) == np.searchsorted(t, x, side="right") - 1
    zeros = np.zeros(n, dtype=np.float32)
    for nodes in (t, zeros):
        assert lib.pumas_cell(nodes.ctypes.data, n, np.nan, 1) == 0
        for x in (nodes[0], nodes[-1], 0.0, -1.0, 1.0, np.inf, -np.inf, np.nan):
            assert lib.pumas_cell(nodes.ctypes.data, n, x, 0) == 0


def test_tree_levels(lib):
    """The masks of 0 to 5 levels of a 31-node tree, and the whole tree for a level beyond its last."""
    assert [lib.pumas_tree_levels(n) for n in range(7)] == [0, 1, 7, 127, 0x7fff, 0x7fffffff, 0x7fffffff]
