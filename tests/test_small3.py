"""The index arithmetic of the windowed 3D small scatter (csrc/k_small3.h),
compiled for the host.  CPU only."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "k_small3.h"
using namespace s2g;
// Every deposit that a wave can make for a box at window offset 8 (the last
// one), whatever its weights are: the number of cells that are not the box's,
// are past the plane, or are not met exactly once; x-table reads past the end
extern "C" int bad_cells(int iw, int jw, int kw)
{
    static int hit[2 * kSW3 * kSW3x];
    for (int &h : hit)
        h = 0;
    const int R = small3_planes(jw * kw), o = kST3 - 1;
    int bad = 0;
    for (int ln = 0; ln < 64; ++ln) {
        const Small3Lane l = small3_lane(ln, iw, jw, kw);
        for (int st = 0; st * R < iw; ++st) {
            if ((l.left > 0 ? l.ri : 0) + st * R >= 2 * kSmallSide3D)
                ++bad;
            if (!(st * R < l.left))
                continue;
            const int c = (o + l.ri + st * R) * kSW3x + (o + l.dj) * kSW3y + o + l.dk;
            if (c < 0 || c >= kSW3 * kSW3x)
                ++bad;
            else
                ++hit[c];
        }
    }
    for (int i = 0; i < iw; ++i)
        for (int j = 0; j < jw; ++j)
            for (int k = 0; k < kw; ++k)
                hit[(o + i) * kSW3x + (o + j) * kSW3y + o + k] -= 1;
    for (int h : hit)
        bad += h != 0;
    return bad;
}
extern "C" int side() { return kSmallSide3D; }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("small3")
    (d / "t.cpp").write_text(SRC)
    so = str(d / "t.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", so, str(d / "t.cpp"),
                    "-I", os.path.join(ROOT, "sphtogrid.jl_amd", "csrc")], check=True)
    return C.CDLL(so)


def test_lanes_cover_the_box_and_nothing_else(lib):
    """A lane deposits by its index alone, so a scale that is not finite (0
    times it is NaN, not 0) reaches the particle's own box only."""
    n = lib.side()
    assert n == 8
    for iw in range(1, n + 1):
        for jw in range(1, n + 1):
            for kw in range(1, n + 1):
                assert lib.bad_cells(iw, jw, kw) == 0, (iw, jw, kw)
