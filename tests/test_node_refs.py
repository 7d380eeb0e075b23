"""How far the indices of a traversal reach, compiled for the host: records stand
for the nodes of a scene only where a reference can number every item and an
offset of 32 bits finds every record, and the place of a node in its pool is
computed in 64 bits."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "barnacle_amd", "csrc")
SRC = """
#include "node_ref.hpp"
extern "C" int reach(size_t t, size_t b, size_t i, size_t n) { return bnd::records_reach(t, b, i, n); }
extern "C" size_t at(int i, int half) { return bnd::node_at(i, half); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("node_ref")
    (d / "t.cpp").write_text(SRC)
    subprocess.run(["g++", "-O2", "-shared", "-fPIC", "-I", CSRC, str(d / "t.cpp"), "-o", str(d / "t.so")], check=True)
    lib = ctypes.CDLL(str(d / "t.so"))
    lib.reach.argtypes = [ctypes.c_size_t] * 4
    lib.at.restype = ctypes.c_size_t
    return lib


def test_records_reach(lib):
    items, nodes = 2**24 - 1, 2**26
    ok = [2, 1, 1, 1]
    assert lib.reach(*ok)
    for k, most in enumerate((items - 1, nodes, items - 1, nodes)):
        args = list(ok)
        args[k] = most
        assert lib.reach(*args)
        args[k] = most + 1
        assert not lib.reach(*args)
    # the last record of the largest pool starts below 4 GiB
    assert (nodes - 1) * 64 < 2**32 <= nodes * 64


@pytest.mark.parametrize("i", [0, 1, 2**30 - 1, 2**30, 2**30 + 5, 2**31 - 1])
def test_place_of_a_node(lib, i):
    assert [lib.at(i, 0), lib.at(i, 1)] == [2 * i, 2 * i + 1]
