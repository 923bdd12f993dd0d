// k_cic3d.h -- launchers of the 3D deposit kernels (k_cic3d.hip).
#pragma once

#include "k_cic2d.h"

namespace s2g {

using Map3DArgs = Map2DArgs;  // same fields; binq is scalar (nq == 1)

struct Gather3Args {
    int dtype, kernel, np, plane0, nq, nb;
    int64_t ntiles, nitems, npix;  // nitems: the count, or its upper bound with d_nitems
    const int64_t *d_nitems = nullptr;
    const int4 *items;
    const int32_t *pairs;  // particle index per (tile, particle) pair
    const Rec3 *rec;
    const void *binq;
    double *partial;
    const int64_t *tile_items;
    double *image;
    int add = 0;  // finalize adds its sums to the image instead of storing them
};

struct Small3Args {
    int dtype, kernel;
    int64_t ns, npix;
    const int32_t *list;
    const Rec3 *rec;
    const void *binq;
    double *image;
};

// counts: the partition's per-block class counts
// box: null, or a sample of one of every stride blocks of partition_blocks(a.n)
void launch_3d_setup(const Map3DArgs &a, Rec3 *rec, int32_t *cls, int64_t *counts,
                     Small3Sample *box, int stride, hipStream_t s);
// explicit normalisation sums (flags: S2G_FLAG_EXACT_NORM turns off the
// border-cut closed form)
void launch_3d_norm(int kernel, const int32_t *list, int64_t ne, int64_t npix, uint32_t flags,
                    Rec3 *rec, hipStream_t s);
void launch_3d_gather(const Gather3Args &g, hipStream_t s);
void launch_3d_finalize(const Gather3Args &g, hipStream_t s);
void launch_3d_small(const Small3Args &a, hipStream_t s);
// windowed small scatter: particles sorted by the kST3^3 tile (nt per side)
// of their box's first voxel, one block per work item (at most max_items)
void launch_3d_small_keys(const int32_t *list, int64_t ns, const Rec3 *rec, int nt,
                          uint32_t *keys, int32_t *vals, hipStream_t s);
void launch_3d_small_window(const Small3Args &a, const int4 *items, const int64_t *nitems,
                            int64_t max_items, const int32_t *plist, int nt, hipStream_t s);
void launch_3d_reduce(const double *image, int64_t npix, int reduce, double *out, hipStream_t s);

}  // namespace s2g
