"""The index arithmetic of the windowed 3D small scatter and the rule between it
and the flat one (csrc/k_small3.h), compiled for the host.  CPU only."""
import ctypes as C
import os
import subprocess

import numpy as np
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
extern "C" int blocks() { return kSmall3Blocks; }
extern "C" int tiles() { return kSmall3Tiles; }
extern "C" int block(int i, int stride, int64_t n) { return small3_block(i, stride, n); }
extern "C" double share(const int *s, int64_t n) { return small3_share((const Small3Sample *)s, n); }
extern "C" int windowed(int64_t ns, int64_t npix, const int *s, int64_t n, int light)
{
    return small3_windowed(ns, npix, (const Small3Sample *)s, n, light != 0);
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("small3")
    (d / "t.cpp").write_text(SRC)
    so = str(d / "t.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", so, str(d / "t.cpp"),
                    "-I", os.path.join(ROOT, "sphtogrid.jl_amd", "csrc")], check=True)
    L = C.CDLL(so)
    L.share.restype = C.c_double
    L.share.argtypes = [C.c_void_p, C.c_int64]
    L.block.argtypes = [C.c_int, C.c_int, C.c_int64]
    L.windowed.argtypes = [C.c_int64, C.c_int64, C.c_void_p, C.c_int64, C.c_int]
    return L


def test_lanes_cover_the_box_and_nothing_else(lib):
    """A lane deposits by its index alone, so a scale that is not finite (0
    times it is NaN, not 0) reaches the particle's own box only."""
    n = lib.side()
    assert n == 8
    for iw in range(1, n + 1):
        for jw in range(1, n + 1):
            for kw in range(1, n + 1):
                assert lib.bad_cells(iw, jw, kw) == 0, (iw, jw, kw)


def _sample(lib, tile, vox):
    """What the set-up samples of particles in this order (blocks of 256, the
    first particle of every run of 16)."""
    nblk = -(-len(tile) // 256)
    stride = -(-nblk // lib.blocks())
    out = []
    for i in range(-(-nblk // stride)):
        b = lib.block(i, stride, nblk)
        assert i * stride <= b < min((i + 1) * stride, nblk)
        t, v = tile[256 * b: 256 * (b + 1)], vox[256 * b: 256 * (b + 1)]
        first = np.full(lib.tiles(), -1)
        first[: -(-len(t) // 16)] = t[::16]
        out.append([v.sum(), len(t), *first])
    return np.ascontiguousarray(out, dtype=np.int32)


@pytest.mark.parametrize("npix,n,box,clump,want", [
    (48, 1000000, 29, 1.0, 0),    # flat 450 us, windowed 720
    (33, 400000, 25, 1.0, 0),     # 262, 450
    (96, 1000000, 150, 1.0, 1),   # 1820, 960
    (48, 1000000, 35, 0.3, 1),    # many in few cells
    (18, 3000, 300, 1.0, 1),
    (24, 2000000, 6, 1.0, 1),     # 633, 518
    (40, 262144, 50, 1.0, 0),     # 297, 360
])
def test_rule_does_not_depend_on_the_order(lib, npix, n, box, clump, want):
    """The same set with its crowded part first, shuffled, and tile by tile."""
    r = np.random.default_rng(n + npix)
    x = r.random((n, 3))
    x[: n // 2] = 0.5 + clump * (x[: n // 2] - 0.5)
    c = (x * npix).astype(np.int64) // 9
    nt = -(-npix // 9)
    tile = (c[:, 0] * nt + c[:, 1]) * nt + c[:, 2]
    vox = np.full(n, box)
    true = ((np.bincount(tile) / n) ** 2).sum()
    for order in (np.arange(n), r.permutation(n), np.argsort(tile, kind="stable")):
        s = _sample(lib, tile[order], vox)
        # systematic samples of 192 to 1024 particles: the chance within a half
        assert 0.5 * true < max(lib.share(s.ctypes.data, len(s)), 1 / nt ** 3) < 1.5 * true
        assert lib.windowed(n, npix, s.ctypes.data, len(s), n <= 1 << 18) == want


def test_share_of_a_lattice(lib):
    """A lattice in its natural order, a plane of it as long as a sampled group
    of blocks."""
    npix, side = 24, 64
    i = np.arange(side ** 3)
    c = np.stack([i // side ** 2, i // side % side, i % side], 1) * npix // side // 9
    tile = (c[:, 0] * 3 + c[:, 1]) * 3 + c[:, 2]
    true = ((np.bincount(tile) / side ** 3) ** 2).sum()
    s = _sample(lib, tile, np.full(side ** 3, 23))
    assert abs(lib.share(s.ctypes.data, len(s)) / true - 1) < 0.5
    assert lib.windowed(side ** 3, npix, s.ctypes.data, len(s), 1) == 0


def _boxes(x, h, npix):
    """Voxels and first tile of the footprint boxes of particles at x (box
    units around 0), as the set-up clips them."""
    g = x * npix + 0.5 * npix
    lo = np.clip(np.floor(g - h[:, None] * npix), 0, npix - 1).astype(np.int64)
    hi = np.clip(np.floor(g + h[:, None] * npix), 0, npix - 1).astype(np.int64)
    c, nt = lo // 9, -(-npix // 9)
    return (hi - lo + 1).prod(1), (c[:, 0] * nt + c[:, 1]) * nt + c[:, 2]


@pytest.mark.parametrize("npix,n,hpix,clump,want", [
    (18, 3000, 0.4, 1.0, 0),
    (18, 3000, 3.4, 1.0, 1),
    (27, 300000, 0.4, 1.0, 0),
    (27, 300000, 2.0, 1.0, 1),
    (48, 300000, 0.5, 0.05, 1),
])
def test_which_scatter_the_gpu_tests_take(lib, npix, n, hpix, clump, want):
    """The sets of test_gpu_cic3d.py's test_small_scatter_rule: both scatters,
    the windowed one on the lists of small passes and on sorted ones."""
    r = np.random.default_rng(n + npix)
    x = clump * r.uniform(-0.5, 0.5, (n, 3))
    h = hpix / npix * r.uniform(0.9, 1.0, n)
    vox, tile = _boxes(x, h, npix)
    s = _sample(lib, tile, vox)
    assert lib.windowed(n, npix, s.ctypes.data, len(s), n <= 1 << 18) == want


def test_the_special_value_sets_are_windowed(lib):
    """The sets of test_gpu_small3.py."""
    import test_gpu_small3 as t
    for seed, lo, hi in ((11, 0.0, t.NPIX), (12, 0.0, t.NPIX), (13, 0.0, 8.0)):
        p = t._set(3000, seed, lo, hi)
        if seed == 12:
            p[1][::5] = 0.4 / t.NPIX
        vox, tile = _boxes(p[0], p[1], t.NPIX)
        s = _sample(lib, tile, vox)
        assert lib.windowed(3000, t.NPIX, s.ctypes.data, len(s), 1) == 1
