"""CPU check of the sorted nearest-codeword search (qs_e8_search.h, the code
the encode kernels run, compiled here with g++): wherever it calls its answer
certain, the row and shift bit are the oracle's, on Gaussian vectors over a
range of scales, near-ties, lattice points, midpoints and large inputs; and on
Gaussian vectors it is certain nearly always (the rest is evaluated candidate
by candidate)."""
import ctypes
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

from oracle import cref

CSRC = Path(__file__).resolve().parents[1] / "quipsharp_amd" / "csrc"

SRC = r"""
#include <stdint.h>
#include "qs_e8_search.h"
static constexpr qs::E8Luts luts = qs::make_e8_luts();
extern "C" void search(const float* x, int64_t n, int one, int32_t* row, int32_t* sb, int32_t* certain) {
  for (int64_t v = 0; v < n; ++v) {
    float y[8];
    for (int i = 0; i < 8; ++i) y[i] = x[8 * v + i];
    bool ok;
    int s = 0;
    qs::E8Best b = one ? qs::e81_search(y, ok) : qs::e8p_search2(y, s, ok);
    row[v] = one ? (int)(b.sel < 256 ? b.sel : luts.pair[b.sel - 256]) : (int)(luts.sel[b.sel] & 255);
    sb[v] = s;
    certain[v] = ok;
  }
}
"""


@pytest.fixture(scope="module")
def search(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("search")
    (d / "s.cpp").write_text(SRC)
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-I", str(CSRC),
                        str(d / "s.cpp"), "-o", str(d / "s.so")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    lib = ctypes.CDLL(str(d / "s.so"))

    def run(x, one=False):
        x = np.ascontiguousarray(x, dtype=np.float32)
        out = [np.zeros(len(x), np.int32) for _ in range(3)]
        lib.search(x.ctypes.data_as(ctypes.c_void_p), ctypes.c_int64(len(x)), int(one),
                   *[o.ctypes.data_as(ctypes.c_void_p) for o in out])
        return out
    return run


def inputs(kind, rng, n):
    x = rng.standard_normal((n, 8))
    if kind.startswith("gauss"):
        return x * float(kind[5:])
    if kind == "codewords":  # codewords and points just beside them
        c = cref.e8p_decode(rng.integers(0, 65536, n)).reshape(n, 8)
        return c + x * rng.choice([0.0, 1e-6, 1e-4, 1e-2], (n, 1))
    if kind == "midpoints":  # half-way between two codewords: ties and near-ties
        c = cref.e8p_decode(rng.integers(0, 65536, 2 * n)).reshape(2, n, 8)
        return (c[0] + c[1]) / 2 + x * rng.choice([0.0, 1e-6, 1e-4], (n, 1))
    if kind == "grid":  # equal magnitudes in many coordinates
        return rng.integers(-6, 7, (n, 8)) * 0.25 + x * rng.choice([0.0, 1e-7, 1e-5], (n, 1))
    if kind == "sparse":
        return x * (rng.random((n, 8)) < 0.4)
    return x * 10.0 ** rng.uniform(-8, 15, (n, 1))  # "wide"


KINDS = ["gauss0.3", "gauss1.0", "gauss1.6", "gauss6", "codewords", "midpoints", "grid", "sparse", "wide"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("one", [False, True])
def test_certain_answers_are_the_oracles(search, kind, one):
    rng = np.random.default_rng(KINDS.index(kind) + 17 * one)
    x = inputs(kind, rng, 60000).astype(np.float32)
    row, sb, certain = search(x, one)
    if one:
        _, want = cref.e81_encode(x)
        wrow, wsb = want, 0 * want
    else:
        _, want = cref.e8p_encode(x)
        wrow, wsb = (want >> 8) & 255, want & 1
    ok = certain.astype(bool)
    assert np.array_equal(row[ok], wrow[ok]) and np.array_equal(sb[ok], wsb[ok])
    if kind.startswith("gauss"):
        assert ok.mean() > 0.99


def test_non_finite_and_zero_inputs_are_never_certain_by_mistake(search):
    x = np.zeros((6, 8), np.float32)
    x[1, 3], x[2, 0], x[3, 7] = np.inf, np.nan, -np.inf
    x[4] = 3e38
    x[5, :4] = np.nan
    for one in (False, True):
        row, sb, certain = search(x, one)
        assert not certain[1:].any()
    row, sb, certain = search(x[:1])
    assert not certain[0]  # zero: the two shifts tie
