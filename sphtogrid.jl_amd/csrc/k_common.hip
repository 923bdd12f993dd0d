// k_common.hip -- dimension-independent stages of the deposits:
//   * stable (particle-order) partition of the particle classes into lists
//   * the (tile, particle) counting sort into per-tile lists
//   * splitting tile lists into work items
// All offsets come from deterministic exclusive scans, so the lists are
// bit-reproducible.
#include "k_common.h"

namespace s2g {

// ---------------------------------------------------------------------------
// Stable partition into three particle-order lists from a class array.
//   pass 1: per-block class counts          (the setup kernels)
//   scan  : exclusive over [class][block] (+ a sentinel: the grand total)
//   pass 2: ballot ranks inside the block    (k_part_scatter)
// list 0 = small, list 1 = large (An + Ex), list 2 = exact (Ex only)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kPartBlock) void k_part_scatter(
    const int32_t *__restrict__ cls, int64_t n, const int64_t *__restrict__ offs,
    int32_t *__restrict__ l0, int32_t *__restrict__ l1, int32_t *__restrict__ l2)
{
    __shared__ int s[3][kPartBlock / kWave];
    const int64_t p = (int64_t)blockIdx.x * kPartBlock + threadIdx.x;
    const int c = p < n ? cls[p] : kClsSkip;
    int f[3];
    part_flags(c, f[0], f[1], f[2]);
    const int wv = threadIdx.x / kWave, ln = threadIdx.x % kWave;
    const uint64_t below = (ln == 0) ? 0ull : (~0ull >> (64 - ln));
    const uint64_t b[3] = {__ballot(f[0]), __ballot(f[1]), __ballot(f[2])};
    if (ln == 0)
        for (int k = 0; k < 3; ++k)
            s[k][wv] = __popcll(b[k]);
    __syncthreads();
    int32_t *lists[3] = {l0, l1, l2};
    for (int k = 0; k < 3; ++k) {
        if (!f[k])
            continue;
        // the scan runs over [class][block]: subtract the class base so the
        // position is local to list k (each list holds at most n entries)
        int64_t pos = offs[(int64_t)k * gridDim.x + blockIdx.x] - offs[(int64_t)k * gridDim.x];
        for (int w = 0; w < wv; ++w)
            pos += s[k][w];
        pos += __popcll(b[k] & below);
        lists[k][pos] = (int32_t)p;
    }
}

// The same lists for a small pass: each block adds up the counts of the blocks
// before it (at most kPartLight, 24 KB from the cache), so no scan runs, and
// the block that holds a map's first particle writes the map's bounds.  The
// first block also adds up the pairs.
__global__ __launch_bounds__(kPartBlock) void k_part_light(
    const int32_t *__restrict__ cls, int64_t n, const int64_t *__restrict__ counts,
    const int64_t *__restrict__ pbase, int nmaps, int32_t *__restrict__ l0,
    int32_t *__restrict__ l1, int32_t *__restrict__ l2, int64_t *__restrict__ out)
{
    constexpr int kW = kPartBlock / kWave;
    __shared__ int s_pre[3][kW], s_tot[3][kW];
    __shared__ uint32_t s_pairs[kW];
    __shared__ uint64_t s_bal[3][kW];
    const int nb = gridDim.x;
    const int wv = threadIdx.x / kWave, ln = threadIdx.x % kWave;
    // the counts of the blocks before this one, all counts, and in the first
    // block the pairs (at most kPartLight / kPartBlock blocks a thread: a wave's
    // sum fits); the loads and the reductions overlap
    int spre[3] = {}, stot[3] = {};
    uint32_t spairs = 0;
    for (int b = threadIdx.x; b < nb; b += kPartBlock) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int v = (int)counts[(int64_t)k * nb + b];
            spre[k] += b < (int)blockIdx.x ? v : 0;
            stot[k] += v;
        }
        if (blockIdx.x == 0)
            spairs += (uint32_t)counts[3 * (int64_t)nb + 1 + b];
    }
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            spre[k] += __shfl_xor(spre[k], o, kWave);
            stot[k] += __shfl_xor(stot[k], o, kWave);
        }
        spairs += __shfl_xor(spairs, o, kWave);
    }
    if (ln == 0) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            s_pre[k][wv] = spre[k];
            s_tot[k][wv] = stot[k];
        }
        s_pairs[wv] = spairs;
    }
    static_assert((int64_t)kWave * (kPartLight / kPartBlock) * kPairsMost < ((int64_t)1 << 32));
    const int64_t p = (int64_t)blockIdx.x * kPartBlock + threadIdx.x;
    int f[3];
    part_flags(p < n ? cls[p] : kClsSkip, f[0], f[1], f[2]);
    const uint64_t below = (ln == 0) ? 0ull : (~0ull >> (64 - ln));
    const uint64_t bal[3] = {__ballot(f[0]), __ballot(f[1]), __ballot(f[2])};
    if (ln == 0)
        for (int k = 0; k < 3; ++k)
            s_bal[k][wv] = bal[k];
    __syncthreads();
    int pre[3], tot[3];
    for (int k = 0; k < 3; ++k) {
        pre[k] = tot[k] = 0;
        for (int w = 0; w < kW; ++w) {
            pre[k] += s_pre[k][w];
            tot[k] += s_tot[k][w];
        }
    }
    int32_t *lists[3] = {l0, l1, l2};
    for (int k = 0; k < 3; ++k) {
        if (!f[k])
            continue;
        int pos = pre[k];
        for (int w = 0; w < wv; ++w)
            pos += __popcll(s_bal[k][w]);
        lists[k][pos + __popcll(bal[k] & below)] = (int32_t)p;
    }
    // class offsets, and the first small / large entry of every map
    if (blockIdx.x == 0 && threadIdx.x < 4) {
        int64_t v = 0;
        for (int k = 0; k < (int)threadIdx.x; ++k)
            v += tot[k];
        out[threadIdx.x] = v;
    } else if (blockIdx.x == 0 && threadIdx.x == 4) {
        int64_t v = 0;
        for (int w = 0; w < kW; ++w)
            v += s_pairs[w];
        out[2 * nmaps + 6] = v;
    }
    for (int m = threadIdx.x; m <= nmaps; m += kPartBlock) {
        const int64_t p0 = m < nmaps ? pbase[m] : n;
        if (p0 >= n) {
            if (blockIdx.x == 0) {
                out[4 + m] = tot[1];
                out[5 + nmaps + m] = tot[0];
            }
        } else if (p0 / kPartBlock == (int64_t)blockIdx.x) {
            const int r = (int)(p0 % kPartBlock);
            int c[2] = {pre[0], pre[1]};
            for (int k = 0; k < 2; ++k) {
                for (int w = 0; w < r / kWave; ++w)
                    c[k] += __popcll(s_bal[k][w]);
                if (r % kWave)
                    c[k] += __popcll(s_bal[k][r / kWave] & (~0ull >> (64 - r % kWave)));
            }
            out[4 + m] = c[1];
            out[5 + nmaps + m] = c[0];
        }
    }
}

int64_t partition_blocks(int64_t n) { return (n + kPartBlock - 1) / kPartBlock; }

void launch_partition(const int32_t *cls, int64_t n, int64_t *counts, int64_t *scan_tmp,
                      int32_t *l0, int32_t *l1, int32_t *l2, hipStream_t s)
{
    if (n == 0)
        return;
    const unsigned nb = (unsigned)partition_blocks(n);
    exclusive_scan_i64(counts, 3 * (int64_t)nb + 1, scan_tmp, s);
    hipLaunchKernelGGL(k_part_scatter, dim3(nb), dim3(kPartBlock), 0, s, cls, n, counts, l0,
                       l1, l2);
}

void launch_partition_light(const int32_t *cls, int64_t n, const int64_t *counts,
                            const int64_t *pbase, int nmaps, int32_t *l0, int32_t *l1,
                            int32_t *l2, int64_t *out, hipStream_t s)
{
    if (n == 0)
        return;
    hipLaunchKernelGGL(k_part_light, dim3((unsigned)partition_blocks(n)), dim3(kPartBlock), 0, s,
                       cls, n, counts, pbase, nmaps, l0, l1, l2, out);
}

// first entry of a particle-order list (len entries) whose particle index is
// >= key
__device__ __forceinline__ int64_t list_lower_bound(const int32_t *__restrict__ list, int64_t len,
                                                    int64_t key)
{
    int64_t lo = 0, hi = len;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int64_t)list[mid] < key)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// class offsets and the per-map ranges of the large and small lists
__global__ void k_class_bounds(const int64_t *__restrict__ counts, int64_t nb,
                               const int32_t *__restrict__ small,
                               const int32_t *__restrict__ large,
                               const int64_t *__restrict__ pbase, int nmaps,
                               int64_t *__restrict__ out)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t ns = counts[nb] - counts[0];
    const int64_t nl = counts[2 * nb] - counts[nb];
    if (m < 4)
        out[m] = counts[(int64_t)m * nb];
    if (m > nmaps)
        return;
    if (m == nmaps) {
        out[4 + m] = nl;
        out[5 + nmaps + m] = ns;
        return;
    }
    out[4 + m] = list_lower_bound(large, nl, pbase[m]);
    out[5 + nmaps + m] = list_lower_bound(small, ns, pbase[m]);
}

void launch_class_bounds(const int64_t *counts, int64_t nb, const int32_t *small,
                         const int32_t *large, const int64_t *pbase, int nmaps, int64_t *out,
                         hipStream_t s)
{
    const int nt = nmaps + 1 > 4 ? nmaps + 1 : 4;
    hipLaunchKernelGGL(k_class_bounds, dim3((unsigned)((nt + 255) / 256)), dim3(256), 0, s,
                       counts, nb, small, large, pbase, nmaps, out);
}

// ---------------------------------------------------------------------------
// (tile, particle) pair lists: a counting sort with deterministic order.
// Chunks are map-local runs of large-list entries (sized per map); map m's
// counts are tile-major [tile][chunk] at cnt[cbase], so one exclusive scan
// over all maps yields every list offset, ordered by (map, tile, particle).
// Local tiles are t = (a * nt + b) * ntc + c over the map's tile grid
// (ntc = 1 in 2D).
// ---------------------------------------------------------------------------

// Order in which the tile lists take a map's large particles.  The map's
// large-list segment e_0 .. e_{L-1} (particle order) is read as f_j =
// e_{(j r) mod L}, r the integer nearest to L / phi (golden ratio), raised to
// the first value coprime to L, so every entry comes once and consecutive
// entries of a tile's list lie far apart in the input.  Snapshots written in
// Peano-Hilbert order would otherwise give a gather batch of consecutive
// entries footprints that cover the same part of the tile, and the block's
// waves that own the other parts idle until its next barrier (2^24 cluster
// set on 4096^2, particles reordered by the 64-pixel tile of the centre:
// gather 282.6 ms in particle order, 272.8 ms read this way, against 270.7
// ms for the set in its generated order).
// Formed in 32 bits: every block of the counting sort computes it, and with
// 64-bit remainders it was half of the fill kernel's time on a small map.
__device__ __forceinline__ uint32_t large_stride(uint32_t L)
{
    if (L <= 2)
        return 1;
    uint32_t r = (uint32_t)((double)L * 0.6180339887498949 + 0.5);
    for (;; ++r) {
        uint32_t a = L, b = r;
        while (b) {
            const uint32_t t = a % b;
            a = b;
            b = t;
        }
        if (a == 1)
            return r;
    }
}

// (j r) mod L for j, r < L < 2^31: the quotient from FP64 is off by at most one
__device__ __forceinline__ uint32_t stride_index(uint32_t j, uint32_t r, uint32_t L, double inv)
{
    const uint64_t x = (uint64_t)j * r;
    int64_t v = (int64_t)(x - (uint64_t)((double)x * inv) * L);
    v += v < 0 ? L : 0;
    v -= v >= (int64_t)L ? L : 0;
    return (uint32_t)v;
}

// A chunk's list entries [l0, l1): entries lbase[m] + k csz .. of map m
// (lbase: the per-map list starts, on the device; csz = TileMap::csz),
// clipped to the map's list, so that the chunk table does not depend on the
// class counts.
__device__ __forceinline__ void chunk_range(const PairChunk &ch, const TileMap &tm,
                                            const int64_t *__restrict__ lbase, int64_t &l0,
                                            int64_t &l1)
{
    const int64_t a = lbase[ch.map] + (int64_t)ch.k * tm.csz, e = lbase[ch.map + 1];
    l0 = a;
    l1 = a + tm.csz < e ? a + tm.csz : e;
    if (l1 < l0)
        l1 = l0;
}

// the small-footprint bucket of a particle: the kST x kST tile holding the
// first pixel of its footprint (one tile, in the map's small-tile grid)
__device__ __forceinline__ void anchor_tile(const Rec2 &r, int &a, int &b, int &c)
{
    a = r.i0 / kST;
    b = r.j0 / kST;
    c = 0;
}
// in 3D the kST3^3 tile holding the first voxel
__device__ __forceinline__ void anchor_tile(const Rec3 &r, int &a, int &b, int &c)
{
    a = r.i0 / kST3;
    b = r.j0 / kST3;
    c = r.k0 / kST3;
}

template <typename R, bool Anchor>
__device__ __forceinline__ void list_rect(const R &r, int &a0, int &a1, int &b0, int &b1, int &c0,
                                          int &c1)
{
    if constexpr (Anchor) {
        anchor_tile(r, a0, b0, c0);
        a1 = a0;
        b1 = b0;
        c1 = c0;
    } else
        tile_rect(r, a0, a1, b0, b1, c0, c1);
}

template <typename R, bool Anchor = false>
__global__ __launch_bounds__(256) void k_pair_count(const int32_t *__restrict__ large,
                                                    const R *__restrict__ rec,
                                                    const PairChunk *__restrict__ chunks,
                                                    const TileMap *__restrict__ tmaps,
                                                    const int64_t *__restrict__ lbase,
                                                    int64_t ncnt, int64_t *__restrict__ cnt)
{
    extern __shared__ int hist[];
    const PairChunk ch = chunks[blockIdx.x];
    const TileMap tm = tmaps[ch.map];
    int64_t cl0, cl1;
    chunk_range(ch, tm, lbase, cl0, cl1);
    // the pair lists read the map's segment in large_stride order (the
    // anchor buckets in list order)
    const int64_t mb = lbase[ch.map];
    const uint32_t L = (uint32_t)(lbase[ch.map + 1] - mb);
    const uint32_t str = Anchor ? 1 : large_stride(L);
    const double inv = 1.0 / (double)L;
    for (int t = threadIdx.x; t < tm.ntiles; t += blockDim.x)
        hist[t] = 0;
    __syncthreads();
    for (int64_t l = cl0 + threadIdx.x; l < cl1; l += blockDim.x) {
        const R r = rec[large[Anchor ? l : mb + stride_index((uint32_t)(l - mb), str, L, inv)]];
        int a0, a1, b0, b1, c0, c1;
        list_rect<R, Anchor>(r, a0, a1, b0, b1, c0, c1);
        for (int a = a0; a <= a1; ++a)
            for (int b = b0; b <= b1; ++b)
                for (int c = c0; c <= c1; ++c)
                    atomicAdd(&hist[(a * tm.nt + b) * tm.ntc + c], 1);
    }
    __syncthreads();
    for (int t = threadIdx.x; t < tm.ntiles; t += blockDim.x)
        cnt[tm.cbase + (int64_t)t * tm.nch + ch.k] = hist[t];
    if (blockIdx.x == 0 && threadIdx.x == 0)
        cnt[ncnt - 1] = 0;  // becomes the pair total after the scan
}

// one wave per chunk: sequential over the chunk's particles, lanes over the
// particle's tiles (distinct per lane), so every list follows the map's
// large_stride order.
// The records of 64 particles are loaded at once (a lane each) and each
// particle's tile rectangle is broadcast by readlane, so the loads' latency
// is paid once per 64 particles.
// pairs: cap entries; a slot at or past cap is not written (a replayed pass
// whose pair total outgrew its capacity; the caller sees the total)
template <typename R>
__global__ __launch_bounds__(kWave) void k_pair_fill(const int32_t *__restrict__ large,
                                                     const R *__restrict__ rec,
                                                     const PairChunk *__restrict__ chunks,
                                                     const TileMap *__restrict__ tmaps,
                                                     const int64_t *__restrict__ lbase,
                                                     const int64_t *__restrict__ off,
                                                     int32_t *__restrict__ pairs, int64_t cap)
{
    extern __shared__ int cursor[];
    const PairChunk ch = chunks[blockIdx.x];
    const TileMap tm = tmaps[ch.map];
    int64_t cl0, cl1;
    chunk_range(ch, tm, lbase, cl0, cl1);
    const int64_t mb = lbase[ch.map];
    const uint32_t L = (uint32_t)(lbase[ch.map + 1] - mb);
    const uint32_t str = large_stride(L);
    const double inv = 1.0 / (double)L;
    for (int t = threadIdx.x; t < tm.ntiles; t += kWave)
        cursor[t] = (int)off[tm.cbase + (int64_t)t * tm.nch + ch.k];
    __syncthreads();
    for (int64_t lb = cl0; lb < cl1; lb += kWave) {
        const int n = cl1 - lb < kWave ? (int)(cl1 - lb) : kWave;
        int32_t pl = 0;
        int ra0 = 0, ra1 = -1, rb0 = 0, rb1 = -1, rc0 = 0, rc1 = -1;
        if ((int)threadIdx.x < n) {
            pl = large[mb + stride_index((uint32_t)(lb + threadIdx.x - mb), str, L, inv)];
            tile_rect(rec[pl], ra0, ra1, rb0, rb1, rc0, rc1);
        }
        for (int e = 0; e < n; ++e) {
            const int32_t p = __builtin_amdgcn_readlane(pl, e);
            const int a0 = __builtin_amdgcn_readlane(ra0, e), a1 = __builtin_amdgcn_readlane(ra1, e);
            const int b0 = __builtin_amdgcn_readlane(rb0, e), b1 = __builtin_amdgcn_readlane(rb1, e);
            const int c0 = __builtin_amdgcn_readlane(rc0, e), c1 = __builtin_amdgcn_readlane(rc1, e);
            const int wb = b1 - b0 + 1, wc = c1 - c0 + 1;
            const int ntr = (a1 - a0 + 1) * wb * wc;
            for (int k = threadIdx.x; k < ntr; k += kWave) {
                const int a = a0 + k / (wb * wc);
                const int rem = k % (wb * wc);
                const int b = b0 + rem / wc, c = c0 + rem % wc;
                const int slot = atomicAdd(&cursor[(a * tm.nt + b) * tm.ntc + c], 1);
                if (slot < cap)
                    pairs[slot] = p;
            }
        }
    }
}

template <typename R>
void launch_pairs(const int32_t *large, const R *rec, const PairChunk *chunks, int nchunks,
                  const TileMap *tmaps, int max_tiles, int64_t *cnt, int64_t ncnt,
                  int64_t *scan_tmp, int32_t *pairs_or_null, bool fill, hipStream_t s,
                  const int64_t *lbase, int64_t cap, bool scan)
{
    const size_t lds = sizeof(int) * (size_t)(max_tiles > 0 ? max_tiles : 1);
    if (!fill) {
        hipLaunchKernelGGL((k_pair_count<R, false>), dim3((unsigned)nchunks), dim3(256), lds, s, large,
                           rec, chunks, tmaps, lbase, ncnt, cnt);
        if (scan)
            exclusive_scan_i64(cnt, ncnt, scan_tmp, s);
    } else {
        hipLaunchKernelGGL(k_pair_fill<R>, dim3((unsigned)nchunks), dim3(kWave), lds, s, large,
                           rec, chunks, tmaps, lbase, cnt, pairs_or_null, cap);
    }
}

template void launch_pairs<Rec2>(const int32_t *, const Rec2 *, const PairChunk *, int,
                                 const TileMap *, int, int64_t *, int64_t, int64_t *, int32_t *,
                                 bool, hipStream_t, const int64_t *, int64_t, bool);
template void launch_pairs<Rec3>(const int32_t *, const Rec3 *, const PairChunk *, int,
                                 const TileMap *, int, int64_t *, int64_t, int64_t *, int32_t *,
                                 bool, hipStream_t, const int64_t *, int64_t, bool);

// Small-footprint buckets as lists over the maps' small-tile grids: counts
// per (tile, chunk) as for the pair lists (k_pair_count with the anchor
// tile), one exclusive scan, then one block per chunk placing its particles
// at LDS cursors.  Within a chunk the order in a tile follows the LDS
// atomics, which only reorders the small scatter's additions.
template <typename R>
__global__ __launch_bounds__(256) void k_anchor_fill(const int32_t *__restrict__ list,
                                                     const R *__restrict__ rec,
                                                     const PairChunk *__restrict__ chunks,
                                                     const TileMap *__restrict__ tmaps,
                                                     const int64_t *__restrict__ lbase,
                                                     const int64_t *__restrict__ off,
                                                     int32_t *__restrict__ out)
{
    extern __shared__ int cursor[];
    const PairChunk ch = chunks[blockIdx.x];
    const TileMap tm = tmaps[ch.map];
    int64_t cl0, cl1;
    chunk_range(ch, tm, lbase, cl0, cl1);
    for (int t = threadIdx.x; t < tm.ntiles; t += blockDim.x)
        cursor[t] = (int)off[tm.cbase + (int64_t)t * tm.nch + ch.k];
    __syncthreads();
    for (int64_t l = cl0 + threadIdx.x; l < cl1; l += blockDim.x) {
        const int32_t p = list[l];
        int a, b, c;
        anchor_tile(rec[p], a, b, c);
        const int slot = atomicAdd(&cursor[(a * tm.nt + b) * tm.ntc + c], 1);
        out[slot] = p;
    }
}

template <typename R>
void launch_anchor_lists(const int32_t *list, const R *rec, const PairChunk *chunks,
                         int nchunks, const TileMap *tmaps, int max_tiles, int64_t *cnt,
                         int64_t ncnt, int64_t *scan_tmp, int32_t *out, bool fill,
                         const int64_t *lbase, hipStream_t s, bool scan)
{
    const size_t lds = sizeof(int) * (size_t)(max_tiles > 0 ? max_tiles : 1);
    if (!fill) {
        hipLaunchKernelGGL((k_pair_count<R, true>), dim3((unsigned)nchunks), dim3(256), lds, s,
                           list, rec, chunks, tmaps, lbase, ncnt, cnt);
        if (scan)
            exclusive_scan_i64(cnt, ncnt, scan_tmp, s);
    } else {
        hipLaunchKernelGGL(k_anchor_fill<R>, dim3((unsigned)nchunks), dim3(256), lds, s, list, rec,
                           chunks, tmaps, lbase, cnt, out);
    }
}
template void launch_anchor_lists<Rec2>(const int32_t *, const Rec2 *, const PairChunk *, int,
                                        const TileMap *, int, int64_t *, int64_t, int64_t *,
                                        int32_t *, bool, const int64_t *, hipStream_t, bool);
template void launch_anchor_lists<Rec3>(const int32_t *, const Rec3 *, const PairChunk *, int,
                                        const TileMap *, int, int64_t *, int64_t, int64_t *,
                                        int32_t *, bool, const int64_t *, hipStream_t, bool);

// Capacity flag of a replayed pass (written whole, one block): bit 0, a
// map's large list is longer than its chunks cover (nch * csz entries; the
// rest of the list was neither counted nor placed); bit 1, the pair total
// passed the pair capacity (the pairs past it were not written).
__global__ __launch_bounds__(256) void k_plan_check(const int64_t *__restrict__ lbase, int nmaps,
                                                    const TileMap *__restrict__ tmaps,
                                                    const int64_t *__restrict__ pair_total,
                                                    int64_t pair_cap, int *__restrict__ flag)
{
    __shared__ int f;
    if (threadIdx.x == 0)
        f = 0;
    __syncthreads();
    for (int m = threadIdx.x; m < nmaps; m += blockDim.x)
        if (lbase[m + 1] - lbase[m] > (int64_t)tmaps[m].nch * tmaps[m].csz)
            atomicOr(&f, 1);
    __syncthreads();
    if (threadIdx.x == 0)
        *flag = f | (*pair_total > pair_cap ? 2 : 0);
}

void launch_plan_check(const int64_t *lbase, int nmaps, const TileMap *tmaps,
                       const int64_t *pair_total, int64_t pair_cap, int *flag, hipStream_t s)
{
    hipLaunchKernelGGL(k_plan_check, dim3(1), dim3(256), 0, s, lbase, nmaps, tmaps, pair_total,
                       pair_cap, flag);
}

// ---------------------------------------------------------------------------
// Work items: tile t's list [start, start+count) is split into ceil(count/G)
// items (global tile, first pair, count, map).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void tile_list(const int64_t *__restrict__ off,
                                          const TileMap *__restrict__ tmaps, int nmaps, int t,
                                          int &m, int64_t &s, int64_t &e)
{
    m = find_entry(tmaps, nmaps, t, [](const TileMap &x) { return x.tbase; });
    const TileMap tm = tmaps[m];
    const int64_t tl = t - tm.tbase;
    // a map without chunks has an empty block: both ends read the same entry
    s = off[tm.cbase + tl * tm.nch];
    e = off[tm.cbase + (tl + 1) * tm.nch];
}

// item size with the total read on the device (so no host round trip is
// needed between the count and the items), or gmin when total is null:
// ceil(total / target), at most gmax (gmax > 0: a large pass is cut into more
// items than target, which shortens the launch's tail), at least
// ceil(total / tmax) (tmax > 0: the items allocated, ntiles + tmax, suffice
// whatever the total) and at least gmin
__device__ __forceinline__ int64_t item_size_of(int64_t gmin, int64_t target, int64_t gmax,
                                                int64_t tmax, int64_t t)
{
    int64_t g = (t + target - 1) / target;
    if (gmax > 0 && g > gmax)
        g = gmax;
    if (tmax > 0) {
        const int64_t gb = (t + tmax - 1) / tmax;
        g = g > gb ? g : gb;
    }
    return g > gmin ? g : gmin;
}

__device__ __forceinline__ int64_t item_size(int64_t gmin, int64_t target, int64_t gmax,
                                             int64_t tmax, const int64_t *__restrict__ total)
{
    return total ? item_size_of(gmin, target, gmax, tmax, *total) : gmin;
}

__global__ void k_item_count(const int64_t *__restrict__ off, const TileMap *__restrict__ tmaps,
                             int nmaps, int ntiles, int64_t gmin, int64_t target, int64_t gmax,
                             int64_t tmax, const int64_t *__restrict__ total,
                             int64_t *__restrict__ nitems)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t == ntiles)
        nitems[t] = 0;  // becomes the item total after the scan
    if (t >= ntiles)
        return;
    const int64_t G = item_size(gmin, target, gmax, tmax, total);
    int m;
    int64_t s, e;
    tile_list(off, tmaps, nmaps, t, m, s, e);
    nitems[t] = (e - s + G - 1) / G;
}

__global__ void k_item_fill(const int64_t *__restrict__ off, const TileMap *__restrict__ tmaps,
                            int nmaps, int ntiles, int64_t gmin, int64_t target, int64_t gmax,
                            int64_t tmax, const int64_t *__restrict__ total,
                            const int64_t *__restrict__ ibase,
                            int4 *__restrict__ items, int64_t *__restrict__ tile_items)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ntiles)
        return;
    const int64_t G = item_size(gmin, target, gmax, tmax, total);
    int m;
    int64_t s, e;
    tile_list(off, tmaps, nmaps, t, m, s, e);
    const int64_t b = ibase[t];
    int64_t k = 0;
    for (int64_t q = s; q < e; q += G, ++k) {
        const int64_t len = e - q < G ? e - q : G;
        items[b + k] = make_int4(t, (int)q, (int)len, m);
    }
    tile_items[2 * t] = b;
    tile_items[2 * t + 1] = k;
}

// The counts' exclusive scan and the items in one block of 16 waves: eight
// counts per thread and step, then a tile per thread and step.
constexpr int kLightThreads = 1024;
constexpr int kLightPer = 8;

// exclusive prefix of v over the block (run: carried from step to step)
__device__ __forceinline__ int light_scan(int v, int *s_wave, int &run)
{
    const int wv = threadIdx.x / kWave, ln = threadIdx.x % kWave;
    int incl = v;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int t = __shfl_up(incl, o, kWave);
        incl += ln >= o ? t : 0;
    }
    __syncthreads();  // the previous step's readers are done
    if (ln == kWave - 1)
        s_wave[wv] = incl;
    __syncthreads();
    int before = 0, all = 0;
    for (int w = 0; w < kLightThreads / kWave; ++w) {
        before += w < wv ? s_wave[w] : 0;
        all += s_wave[w];
    }
    const int excl = run + before + incl - v;
    run += all;
    return excl;
}

__global__ __launch_bounds__(kLightThreads) void k_lists_light(
    int64_t *cnt, int64_t ncnt, const TileMap *__restrict__ tmaps, int nmaps, int ntiles,
    int64_t gmin, int64_t target, int64_t gmax, int64_t tmax, const int64_t *total,
    int64_t *__restrict__ nitems, int4 *__restrict__ items, int64_t item_cap,
    int64_t *__restrict__ tile_items)
{
    __shared__ int s_wave[kLightThreads / kWave];
    int run = 0;
    const int64_t step = kLightThreads * kLightPer;
    for (int64_t base = 0; base < ncnt; base += step) {
        const int64_t i0 = base + (int64_t)threadIdx.x * kLightPer;
        int v[kLightPer], sum = 0;
#pragma unroll
        for (int k = 0; k < kLightPer; ++k) {
            v[k] = i0 + k < ncnt ? (int)cnt[i0 + k] : 0;
            sum += v[k];
        }
        int e = light_scan(sum, s_wave, run);
#pragma unroll
        for (int k = 0; k < kLightPer; ++k) {
            if (i0 + k < ncnt)
                cnt[i0 + k] = e;
            e += v[k];
        }
    }
    __threadfence_block();
    __syncthreads();
    // the counts' own total is the scan's (its last entry is 0)
    const int64_t G = total == cnt + ncnt - 1 ? item_size_of(gmin, target, gmax, tmax, run)
                                              : item_size(gmin, target, gmax, tmax, total);
    run = 0;
    for (int base = 0; base < ntiles; base += kLightThreads) {
        const int t = base + threadIdx.x;
        int m = 0;
        int64_t s = 0, e = 0;
        if (t < ntiles)
            tile_list(cnt, tmaps, nmaps, t, m, s, e);
        const int ni = (int)((e - s + G - 1) / G);
        const int64_t b = light_scan(ni, s_wave, run);
        if (t < ntiles) {
            int64_t k = 0;
            for (int64_t q = s; q < e; q += G, ++k) {
                const int64_t len = e - q < G ? e - q : G;
                if (b + k < item_cap)
                    items[b + k] = make_int4(t, (int)q, (int)len, m);
            }
            tile_items[2 * t] = b;
            tile_items[2 * t + 1] = k;
        }
    }
    if (threadIdx.x == 0)
        nitems[ntiles] = run;
}

void launch_lists_light(int64_t *cnt, int64_t ncnt, const TileMap *tmaps, int nmaps, int ntiles,
                        int64_t gmin, int64_t target, int64_t gmax, int64_t tmax,
                        const int64_t *total, int64_t *nitems, int4 *items, int64_t item_cap,
                        int64_t *tile_items, hipStream_t s)
{
    hipLaunchKernelGGL(k_lists_light, dim3(1), dim3(kLightThreads), 0, s, cnt, ncnt, tmaps, nmaps,
                       ntiles, gmin, target, gmax, tmax, total, nitems, items, item_cap,
                       tile_items);
}

void launch_items(const int64_t *off, const TileMap *tmaps, int nmaps, int ntiles,
                  int64_t gmin, int64_t target, const int64_t *total, int64_t *nitems,
                  int64_t *scan_tmp, int4 *items_or_null, int64_t *tile_items, bool fill,
                  hipStream_t s, int64_t gmax, int64_t tmax)
{
    const unsigned nb = (unsigned)((ntiles + 1 + 255) / 256);
    if (!fill) {
        hipLaunchKernelGGL(k_item_count, dim3(nb), dim3(256), 0, s, off, tmaps, nmaps, ntiles,
                           gmin, target, gmax, tmax, total, nitems);
        exclusive_scan_i64(nitems, ntiles + 1, scan_tmp, s);
    } else {
        hipLaunchKernelGGL(k_item_fill, dim3(nb), dim3(256), 0, s, off, tmaps, nmaps, ntiles,
                           gmin, target, gmax, tmax, total, nitems, items_or_null, tile_items);
    }
}

}  // namespace s2g
