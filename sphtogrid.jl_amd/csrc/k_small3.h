// k_small3.h -- index arithmetic of the windowed 3D small scatter and the rule
// between it and the flat one, in plain C++ so that it can be checked on the
// host.
#pragma once

#include <algorithm>
#include <cstdint>

namespace s2g {

// 3D: footprint box side <= 8 voxels goes to the scatter path.
constexpr int kSmallSide3D = 8;
// side of the windowed 3D scatter's tiles
constexpr int kST3 = 9;
// its LDS window, the tile and the largest box; strides with one voxel of
// padding against bank conflicts
constexpr int kSW3 = kST3 + kSmallSide3D - 1;
constexpr int kSW3y = kSW3 + 1, kSW3x = kSW3 * kSW3y;

// Of a box of iw x jw x kw voxels, iw, jw, kw <= kSmallSide3D: a wave's 64
// lanes take R = small3_planes(jw kw) x planes of jw x kw voxels per step.
constexpr int small3_planes(int jk)
{
    const int r = (int)(64.5f * (1.0f / (float)jk));
    return r < kSmallSide3D ? r : kSmallSide3D;
}

// Lane ln's voxel of step 0: (ri, dj, dk) of the box; at step st it has (ri +
// st R, dj, dk), which is a voxel of the box while st R < left.  A lane past
// the R planes (left 0) or past the box's last plane has none, and deposits
// nothing whatever the particle's scale: its weight is 0, but 0 times an
// infinite scale is not.
struct Small3Lane {
    int ri, dj, dk, left;
};
constexpr Small3Lane small3_lane(int ln, int iw, int jw, int kw)
{
    const int jk = jw * kw;
    const int ri = (int)(((float)ln + 0.5f) * (1.0f / (float)jk)), rem = ln - ri * jk;
    const int dj = (int)(((float)rem + 0.5f) * (1.0f / (float)kw));
    return Small3Lane{ri, dj, rem - dj * kw, ri < small3_planes(jk) ? iw - ri : 0};
}

// A sampled set-up block's small particles: voxels of their boxes, particles,
// and the kST3^3 tile in which the first one of each run of 16 starts (-1: a
// run without any).
constexpr int kSmall3Blocks = 64, kSmall3Tiles = 16;
struct Small3Sample {
    int voxels, n, tile[kSmall3Tiles];
};

// The block sampled of group i, blocks [i stride, (i + 1) stride) of nblk: not
// the same one of each group, since a lattice's rows may be as long as a group.
constexpr int small3_block(int i, int stride, int64_t nblk)
{
    const int64_t left = nblk - (int64_t)i * stride;
    const uint32_t size = (uint32_t)(left < stride ? left : stride);
    return i * stride + (int)(((uint32_t)i * 2654435769u >> 8) % size);
}

// The chance that two small particles start in the same tile: over the pairs
// of sampled particles of different blocks, each standing for its share of its
// block.  (Particles near each other in the caller's order are left out: in a
// spatially ordered set they share a tile however sparse the set is.)
inline double small3_share(const Small3Sample *sample, int64_t nsample)
{
    // the tiles' weights, of all blocks and of the block in hand
    constexpr uint32_t kSlots = 2 * kSmall3Blocks * kSmall3Tiles;
    static_assert((kSlots & (kSlots - 1)) == 0, "a power of two");
    struct Slot {
        int tile = -1;
        double all = 0.0, block = 0.0;
    };
    Slot slots[kSlots];
    double all = 0.0, same = 0.0, pairs = 0.0;
    for (int64_t b = 0; b < nsample && b < kSmall3Blocks; ++b) {
        const Small3Sample &s = sample[b];
        int held = 0;
        for (int t : s.tile)
            held += t >= 0;
        if (held == 0)
            continue;
        const double w = (double)s.n / held;
        Slot *of[kSmall3Tiles];
        int m = 0;
        for (int t : s.tile) {
            if (t < 0)
                continue;
            uint32_t k = (uint32_t)t * 2654435761u >> 20 & (kSlots - 1);
            while (slots[k].tile >= 0 && slots[k].tile != t)
                k = (k + 1) & (kSlots - 1);
            slots[k].tile = t;
            // pairs with the blocks before, then into this block's weight
            same += 2.0 * w * slots[k].all;
            slots[k].block += w;
            of[m++] = &slots[k];
        }
        pairs += 2.0 * (double)s.n * all;
        all += (double)s.n;
        for (int i = 0; i < m; ++i) {
            of[i]->all += of[i]->block;
            of[i]->block = 0.0;
        }
    }
    return pairs > 0.0 ? same / pairs : 0.0;
}

// The rule between the windowed and the flat scatter.  At least 32 particles
// per tile, so that adding a window to the image costs less than their own
// atomics (10^5 of the cluster set on 200^3, 7 per tile: 887 / 737 us), and
// then the difference of the two, fitted to whole calls: a window saves 7.2 ps
// of global atomics per voxel, 0.54 us for every voxel of a mean box (a wave's
// chain), and what the flat scatter waits where many particles share few
// voxels; it costs the sort (139 us, 83 us for the lists that need none,
// `light`) and 0.23 ns per particle (boxes of at most 2^3, which it takes eight
// to a wave: it saves 0.13).  The crowding is the chance of a shared tile over
// that of a uniform set: beyond 1 it costs the flat scatter 0.28 us for every
// deposit on a mean voxel and 18 ps per particle (up to 20 times).
// Whole calls, windowed / flat, us: uniform sets, 10^6 particles of 29 voxels on
// 48^3 762 / 488, in Morton order 721 / 497, 4 10^5 of 14 on 24^3 435 / 183,
// 10^6 of 150 on 96^3 963 / 1846, 2.5 10^5 of 85 on 48^3 330 / 370; the cluster
// set, 2 10^6 on 48^3 1169 / 2015, on 128^3 3198 / 4036, 3 10^4 on 24^3 145 /
// 107.  Over 392 sets (uniform, lattices, clusters; shuffled and in Morton
// order) the choice loses 1.3 % on average and 1.5 times at most (2 10^6 in 20
// clumps on 48^3, Morton order, 657 / 999).
inline bool small3_dense(int64_t ns, int64_t nstiles)
{
    return ns > 0 && nstiles < ((int64_t)1 << 30) && ns >= 32 * nstiles;
}
inline bool small3_windowed(int64_t ns, int64_t npix, const Small3Sample *sample,
                            int64_t nsample, bool light)
{
    const int64_t nt = (npix + kST3 - 1) / kST3;
    if (!small3_dense(ns, nt * nt * nt))
        return false;
    double voxels = 0.0, boxes = 0.0;
    for (int64_t k = 0; k < nsample; ++k) {
        voxels += sample[k].voxels;
        boxes += sample[k].n;
    }
    const double n = (double)ns, box = boxes > 0.0 ? voxels / boxes : 1.0, vox = box * n;
    const double gain = 7.2e-12 * vox + 0.54e-6 * box - (light ? 83e-6 : 139e-6) +
                        (box <= 8.0 ? 0.135e-9 : -0.228e-9) * n;
    if (gain > 0.0)
        return true;
    // the chance of a uniform set, whose last tile of an axis may be cut
    const double w = (double)npix, last = w - (double)(kST3 * (nt - 1));
    const double axis = ((double)(nt - 1) * kST3 * kST3 + last * last) / (w * w);
    const double ex = std::max(small3_share(sample, nsample) / (axis * axis * axis) - 1.0, 0.0);
    return gain + 0.283e-6 * ex * vox / (w * w * w) + 18e-12 * n * std::min(ex, 20.0) > 0.0;
}

}  // namespace s2g
