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
extern "C" void interpolation(const double* k, int n, double at, double* nodes, double* w, double* dw) {
  double lo, hi;
  omx::mk_extent(k, n, lo, hi);
  const omx::MkRange r = omx::mk_range(lo, hi);
  double x[omx::MK_NODES];
  for (int t = 0; t < omx::MK_NODES; ++t) {
    x[t] = omx::mk_node(r, t);
    nodes[t] = exp(x[t]);
  }
  for (int t = 0; t < omx::MK_NODES; ++t) omx::mk_weight(x, t, at, w[t], dw[t]);
}
extern "C" double bytes(long N, long ld, long P, long ninst, long M) { return double(omx::group_bytes(N, 2 * N, ld, P, ninst, M)); }
extern "C" int nodes() { return omx::MK_NODES; }
extern "C" int position(const double* d, int n, int a) { return omx::mk_position(d, n, a); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("multik_math")
    src, out = d / "m.cpp", d / "m.so"
    src.write_text(SOURCE)
    subprocess.run([CXX, "-O1", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(src), "-o", str(out)], check=True)
    L = ctypes.CDLL(str(out))
    L.bytes.restype, L.bytes.argtypes = ctypes.c_double, [ctypes.c_long] * 5
    return L


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


def _interpolation(lib, ks, at):
    n = lib.nodes()
    out = [np.zeros(n) for _ in range(3)]
    p = ctypes.POINTER(ctypes.c_double)
    k = np.array(ks)
    lib.interpolation(k.ctypes.data_as(p), len(k), ctypes.c_double(at), *(a.ctypes.data_as(p) for a in out))
    return out


def test_norm_weights_by_the_width_of_the_k_range(lib):
    """1 / (rho^2 + k^2) and its k-derivative from the nodes, against the stated worst relative
    errors (half a digit of slack for their rounding and the sampling here).  A derivative of the
    interpolant loses up to the square of its degree over the half-width of the range."""
    for ratio, bound in ((1.01, 1e-14), (1.2, 2e-12), (1.5, 1e-9), (2.0, 9e-8), (3.0, 5e-6), (5.0, 1.3e-4)):
        for base in (0.02, 0.4, 1.3):
            lo, hi = base, base * ratio
            err = der = 0.0
            for at in np.geomspace(lo, hi, 33):
                nodes, w, dw = _interpolation(lib, [hi, lo, 0.5 * (lo + hi)], at)
                for rho in np.r_[0.0, lo * np.geomspace(0.03, 100, 25)]:
                    f = 1 / (rho ** 2 + nodes ** 2)
                    exact, slope = 1 / (rho ** 2 + at ** 2), -2 * at / (rho ** 2 + at ** 2) ** 2
                    err = max(err, abs(w @ f / exact - 1))
                    der = max(der, abs(dw @ f - slope) / (exact / at))
            assert err < 1.5 * bound
            assert der < 1.5 * bound * 49 / max(np.log(ratio) / 2, 0.01) + 1e-11


def test_norm_weights_at_a_node_and_for_negative_k(lib):
    nodes, _, _ = _interpolation(lib, [0.9, 1.2], 1.0)
    for t, at in enumerate(nodes):
        _, w, _ = _interpolation(lib, [0.9, 1.2], at)
        assert np.allclose(w, np.arange(len(nodes)) == t, atol=1e-12)
    _, w, dw = _interpolation(lib, [0.9, 1.2], 1.1)
    _, wn, dwn = _interpolation(lib, [-0.9, -1.2], -1.1)
    assert np.allclose(w, wn) and np.allclose(dw, -dwn)


@pytest.mark.parametrize("P,nev", [(1, 1), (40, 1), (40, 2), (12, 4), (5, 16)])
def test_launch_group_bytes_cover_both_forms(lib, P, nev):
    """What a launch group holds at once, counted buffer by buffer: the shared search space's
    columns (X and P twice, W; seven single-precision planes each, for nev + 2 columns a
    problem) and transform buffer, the blocks it hands over (X, M X, three components, and
    their single-precision copy and residuals), the refinement's seven vectors and the
    correction solves' eight with three components; or the per-band form's eleven blocks."""
    N = 128 * 96
    ld, ninst, m = 2 * N, P * nev, nev + 2
    shared = P * m * (5 * 7 + 3) * 8 * N + ninst * m * (2 * 16 * ld + 16 * 3 * N + 2 * 8 * ld)
    vectors = ninst * (5 * 16 * ld + 3 * 8 * ld + 8 * 8 * ld + 8 * 3 * N) + P * 6 * N * 2 * (4 + 8)
    per_band = 24 * ninst * nev * (11 * ld + 3 * N)
    got = lib.bytes(N, ld, P, ninst, nev)
    assert got >= vectors + shared
    assert got >= vectors + per_band
    assert got < 3 * (vectors + max(shared, per_band))


def test_launch_group_bytes_of_refused_mode_counts(lib):
    for nev in (-3, 0, 17, 2 ** 31 - 1):
        assert 0 < lib.bytes(256, 512, 1, 1, nev) < 1e9
