"""Scalar pieces of the shared search space (csrc/multik_math.hpp), compiled for the host."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "optimode.jl_amd", "csrc")
CXX = shutil.which("g++") or shutil.which("c++")
pytestmark = pytest.mark.skipif(CXX is None, reason="no host C++ compiler")

SOURCE = """
#include "multik_math.hpp"
extern "C" int position(const double* d, int n, int a) { return omx::mk_position(d, n, a); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("multik_math")
    src, out = d / "m.cpp", d / "m.so"
    src.write_text(SOURCE)
    subprocess.run([CXX, "-O1", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(src), "-o", str(out)], check=True)
    return ctypes.CDLL(str(out))


NAN, INF = float("nan"), float("inf")


@pytest.mark.parametrize("d", [[3.0, 1.0, 2.0], [1.0, 1.0, 0.0, 1.0], [NAN] * 5, [2.0, NAN, 1.0, NAN], [INF, -INF, NAN, INF],
                               [0.0, -0.0, 0.0], list(np.linspace(1, 0, 54)), [7.0]])
def test_positions_are_a_permutation(lib, d):
    """Each Ritz pair is looked up by its position: every position has exactly one owner, also
    when the small matrix holds values that are not numbers."""
    a = np.array(d)
    pos = [lib.position(a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), len(a), i) for i in range(len(a))]
    assert sorted(pos) == list(range(len(a)))
    order = np.empty(len(a), dtype=int)
    order[pos] = np.arange(len(a))
    assert list(order) == list(np.argsort(a, kind="stable"))  # numpy sorts NaN last too
