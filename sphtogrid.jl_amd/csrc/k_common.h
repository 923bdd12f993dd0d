// k_common.h -- dimension-independent stages shared by the 2D and 3D
// deposits (class partition, tile pair lists, work items).
#pragma once

#include "s2g_internal.h"

namespace s2g {

constexpr int kPartBlock = 256;
// largest usual count of large-list entries per counting-sort chunk (one LDS
// histogram per chunk, one wave per chunk in the fill); the host sizes each
// map's chunks from 256 up to this, larger only to bound the counters
constexpr int kPairChunk = 4096;
// per-workgroup LDS bound of the tile histograms (ints): tiles of one map
constexpr int kMaxTiles = 16384;

int64_t partition_blocks(int64_t n);
// counts: class_count_elems(n) int64, of which the first 3*partition_blocks(n)+1
// are the per-block class counts as the setup kernels write them
// (block_class_counts); afterwards counts[c*nb] is
// the first index of class c in the concatenation and counts[3*nb] the grand
// total
void launch_partition(const int32_t *cls, int64_t n, int64_t *counts, int64_t *scan_tmp,
                      int32_t *l0, int32_t *l1, int32_t *l2, hipStream_t s);
// The partition and the class bounds of a small pass (at most kPartLight
// blocks) in one launch instead of four: every block adds up the counts of
// the blocks before it.  out as launch_class_bounds writes it, and after it, in
// out[2 nmaps + 6], the (tile, particle) pairs of the large particles; counts
// is left as it is.
constexpr int64_t kPartLight = 1024;
void launch_partition_light(const int32_t *cls, int64_t n, const int64_t *counts,
                            const int64_t *pbase, int nmaps, int32_t *l0, int32_t *l1,
                            int32_t *l2, int64_t *out, hipStream_t s);

// class membership of the three lists: small, large (closed form or explicit
// normalisation), large with explicit normalisation
__device__ __forceinline__ void part_flags(int cls, int &f0, int &f1, int &f2)
{
    f0 = cls == kClsSmall;
    f1 = cls == kClsLargeAn || cls == kClsLargeEx;
    f2 = cls == kClsLargeEx;
}

__device__ __forceinline__ void tile_rect(const Rec2 &r, int &a0, int &a1, int &b0, int &b1,
                                          int &c0, int &c1)
{
    a0 = r.i0 / kGT;
    a1 = r.i1 / kGT;
    b0 = r.j0 / kGT;
    b1 = r.j1 / kGT;
    c0 = c1 = 0;
}

__device__ __forceinline__ void tile_rect(const Rec3 &r, int &a0, int &a1, int &b0, int &b1,
                                          int &c0, int &c1)
{
    a0 = r.i0 / kBT;
    a1 = r.i1 / kBT;
    b0 = r.j0 / kBT;
    b1 = r.j1 / kBT;
    c0 = r.k0 / kBT;
    c1 = r.k1 / kBT;
}

// tiles (bricks) that a footprint meets, and a block's large particles together:
// from kPairsMost on just that
constexpr int64_t kPairsMost = ((int64_t)1 << 24) - 1;
template <typename R>
__device__ __forceinline__ int tile_count(const R &r)
{
    int a0, a1, b0, b1, c0, c1;
    tile_rect(r, a0, a1, b0, b1, c0, c1);
    const int64_t t = (int64_t)(a1 - a0 + 1) * (b1 - b0 + 1) * (c1 - c0 + 1);
    return (int)(t < kPairsMost ? t : kPairsMost);
}

// int64 elements of `counts` for n particles: the class counts, their sentinel,
// and for a small pass each block's pairs
inline int64_t class_count_elems(int64_t n)
{
    const int64_t nb = (n + kPartBlock - 1) / kPartBlock;
    return 3 * nb + 1 + (nb <= kPartLight ? nb : 0);
}

// Per-block class counts of the partition, from the setup kernel's blocks of
// kPartBlock threads (cls: this thread's particle's class, kClsSkip past the
// end; every thread of the block calls it).  tiles: the tile_count of a large
// particle; a small pass sizes its pair lists and partial sums by their sum.
__device__ __forceinline__ void block_class_counts(int cls, int tiles,
                                                   int64_t *__restrict__ counts)
{
    __shared__ int s[3][kPartBlock / kWave];
    __shared__ int s_tiles[kPartBlock / kWave];
    int f0, f1, f2;
    part_flags(cls, f0, f1, f2);
    const int wv = threadIdx.x / kWave, ln = threadIdx.x % kWave;
    const uint64_t b0 = __ballot(f0), b1 = __ballot(f1), b2 = __ballot(f2);
    const bool light = gridDim.x <= kPartLight;  // uniform
    if (light) {
        tiles = f1 ? tiles : 0;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1)
            tiles += __shfl_xor(tiles, o, kWave);  // below 2^30
    }
    if (ln == 0) {
        s[0][wv] = __popcll(b0);
        s[1][wv] = __popcll(b1);
        s[2][wv] = __popcll(b2);
        s_tiles[wv] = tiles;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        int t = 0;
        for (int k = 0; k < kPartBlock / kWave; ++k)
            t += s[threadIdx.x][k];
        counts[(int64_t)threadIdx.x * gridDim.x + blockIdx.x] = t;
    }
    if (light && threadIdx.x == 4) {
        int64_t t = 0;
        for (int k = 0; k < kPartBlock / kWave; ++k)
            t += s_tiles[k];
        counts[3 * (int64_t)gridDim.x + 1 + blockIdx.x] = t < kPairsMost ? t : kPairsMost;
    }
    if (blockIdx.x == 0 && threadIdx.x == 3)
        counts[3 * (int64_t)gridDim.x] = 0;  // becomes the grand total after the scan
}
// After launch_partition over the particles of several maps: out[0..3] =
// class offsets counts[0], counts[nb], counts[2nb], counts[3nb]; out[4 + m] =
// first entry of map m in the large list (particles of map m are
// [pbase[m], pbase[m+1]), and the partition is stable), out[4 + nmaps] = size
// of the large list; out[5 + nmaps + m]: the same for the small list, and
// out[5 + 2 nmaps] its size (out: 2 nmaps + 6 entries).
void launch_class_bounds(const int64_t *counts, int64_t nb, const int32_t *small,
                         const int32_t *large, const int64_t *pbase, int nmaps, int64_t *out,
                         hipStream_t s);

// Tile grid of one map in the (tile, particle) counting sort.  Local tile id
// t = (a * nt + b) * ntc + c; global tile id tbase + t.  The map's count block
// is cnt[cbase + t * nch + k] for its chunks k < nch.
struct TileMap {
    int64_t cbase;
    int32_t tbase, ntiles;
    int32_t nt, ntc;
    int32_t nch;
    int32_t csz;  // entries per chunk when the chunk ranges are taken on the device
};
// chunk k of map `map`: list entries lbase[map] + k csz .. (clipped to the
// map's list), with lbase the per-map list starts on the device
struct PairChunk {
    int32_t map, k;
};

// fill == false: count + scan into cnt (ncnt int64, the last is the total)
// fill == true : fill pairs (particle indices) from the scanned cnt
// lbase: per-map large-list starts on the device (nmaps + 1 entries); a map's
// segment is taken in the order f_j = e_{(j r) mod L} (L its length, r the
// integer nearest to L / phi made coprime to L), so every tile list follows
// that order; cap: entries of pairs (slots past it are not written)
template <typename R>
void launch_pairs(const int32_t *large, const R *rec, const PairChunk *chunks, int nchunks,
                  const TileMap *tmaps, int max_tiles, int64_t *cnt, int64_t ncnt,
                  int64_t *scan_tmp, int32_t *pairs_or_null, bool fill, hipStream_t s,
                  const int64_t *lbase, int64_t cap = INT64_MAX, bool scan = true);
// small-footprint buckets as per-tile lists (fill == false: counts per
// (tile, chunk) + scan into cnt; fill == true: out = the particles, tile t of
// map m at cnt[cbase + t nch] ..), chunk ranges from lbase as for the pairs
template <typename R>
void launch_anchor_lists(const int32_t *list, const R *rec, const PairChunk *chunks,
                         int nchunks, const TileMap *tmaps, int max_tiles, int64_t *cnt,
                         int64_t ncnt, int64_t *scan_tmp, int32_t *out, bool fill,
                         const int64_t *lbase, hipStream_t s, bool scan = true);
// The scan of the counts of launch_pairs / launch_anchor_lists (called with
// scan == false) and both steps of launch_items in one block, for counts of a
// small pass: ncnt <= kListsLight and totals below 2^31 (three launches and
// more otherwise, each a few microseconds).  items: at most item_cap are
// written; nitems[ntiles] is the item total.
constexpr int64_t kListsLight = 131072;
void launch_lists_light(int64_t *cnt, int64_t ncnt, const TileMap *tmaps, int nmaps, int ntiles,
                        int64_t gmin, int64_t target, int64_t gmax, int64_t tmax,
                        const int64_t *total, int64_t *nitems, int4 *items, int64_t item_cap,
                        int64_t *tile_items, hipStream_t s);
// flag = (a map's large list outgrew nch * csz entries) | 2 * (pair total >
// pair_cap), for a replayed pass sized at creation
void launch_plan_check(const int64_t *lbase, int nmaps, const TileMap *tmaps,
                       const int64_t *pair_total, int64_t pair_cap, int *flag, hipStream_t s);
// fill == false: nitems (ntiles+1, last = total) ; fill == true: items + tile_items.
// items[i] = (global tile, first pair, count, map).  A tile's list is cut into
// items of at most G entries, G = ceil(*total / target) capped at gmax (if
// gmax > 0), raised to ceil(*total / tmax) (if tmax > 0; then at most
// ntiles + tmax items) and to gmin; G = gmin if total is null.  *total is
// read on the device.
void launch_items(const int64_t *off, const TileMap *tmaps, int nmaps, int ntiles,
                  int64_t gmin, int64_t target, const int64_t *total, int64_t *nitems,
                  int64_t *scan_tmp, int4 *items_or_null, int64_t *tile_items, bool fill,
                  hipStream_t s, int64_t gmax = 0, int64_t tmax = 0);

// index of the last table entry whose key is <= v (keys ascending, key[0] <= v)
template <typename E, typename K, typename F>
__device__ __forceinline__ int find_entry(const E *tab, int n, K v, F key)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (key(tab[mid]) <= v)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

}  // namespace s2g
