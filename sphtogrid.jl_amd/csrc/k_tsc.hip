// k_tsc.hip -- triangular-shaped-cloud deposit onto an npix^3 grid (textbook
// TSC, Hockney & Eastwood; the reference's TSC path is commented out,
// tsc_interpolation/tsc_interpolation.jl:1-182).
//
// Grid units follow the 3D deposit (get_xyz, cic_shared.jl:85-100):
// g = x*len2pix + npix/2, cell c has its centre at c + 1/2.  Per axis the
// weights of the nearest cell and its two neighbours are
//   W(d) = 3/4 - d^2          |d| < 1/2
//        = (3/2 - |d|)^2 / 2  1/2 <= |d| < 3/2
// and they sum to one.  Plane 0 accumulates q*W, plane 1 accumulates W.
//
// Pipeline (a gather: every cell is written once with a plain store, no
// atomics and no memset, and the result is bit-reproducible):
//   k_tsc_keys     brick of each particle's nearest cell (bricks of
//                  kTX x kTY x kTZ cells, row-major; dropped particles last)
//                  and, in the key's low six bits, whether that cell is the
//                  first or last of its brick along each axis
//                  (and the particle's record, where the output grid has
//                  room for it until the gather)
//   (radix sort)   on the brick bits, stable, so particles keep their input
//                  order in a brick
//   k_tsc_offsets  first sorted particle of every brick
//   k_tsc_prep     grid coordinates (FP64) and quantity in sorted order, and
//                  each particle's nearest cell packed into one word
//   k_tsc_gather   one wave per brick: scans the sorted keys of the (up to)
//                  27 neighbouring bricks, queues the particles whose 3^3
//                  stencil reaches the brick and deposits them into LDS seven
//                  at a time (9 lanes per particle, one stencil row each), in
//                  queue order; then writes the brick's cells.
#include "k_tsc.h"

#include <climits>

namespace s2g {

__device__ __forceinline__ double tsc_w(double d)
{
    const double a = fabs(d);
    if (a < 0.5)
        return 0.75 - a * a;
    if (a < 1.5) {
        const double b = 1.5 - a;
        return 0.5 * b * b;
    }
    return 0.0;
}

__host__ __device__ __forceinline__ int64_t tsc_wrap(int64_t c, int64_t npix)
{
    return ((c % npix) + npix) % npix;
}

// nearest cell of particle p along each axis; false if the particle is
// dropped (a non-finite coordinate, or far outside a non-periodic grid)
template <typename T>
__device__ __forceinline__ bool tsc_cell(const T *__restrict__ pos, int64_t p, int64_t npix,
                                         double len2pix, int periodic, double g[3],
                                         int64_t c[3])
{
    for (int d = 0; d < 3; ++d) {
        g[d] = add_rn(mul_rn(ld(pos, 3 * p + d), len2pix), 0.5 * (double)npix);
        const double fg = floor(g[d]);
        if (!isfinite(fg) || ((fg < -2.0 || fg > (double)npix + 2.0) && !periodic))
            return false;
        c[d] = (int64_t)fg;
    }
    return true;
}

// the brick grid of an npix^3 grid
__host__ __device__ __forceinline__ void tsc_bricks(int64_t npix, int64_t nb[3])
{
    nb[0] = (npix + kTX - 1) / kTX;
    nb[1] = (npix + kTY - 1) / kTY;
    nb[2] = (npix + kTZ - 1) / kTZ;
}

int64_t tsc_nbricks(int64_t npix)
{
    int64_t nb[3];
    tsc_bricks(npix, nb);
    return nb[0] * nb[1] * nb[2];
}

// Sort key: the brick of the particle's nearest cell (clamped into the grid,
// or wrapped when periodic) above kTscFlagBits bits, two per axis: the cell is
// the brick's first (bit 2 d), its last (bit 2 d + 1).  Dropped particles get
// brick nbricks, after all bricks.
constexpr int kTscFlagBits = 6;
template <typename T>
__global__ __launch_bounds__(256) void k_tsc_keys(const T *__restrict__ pos,
                                                  const T *__restrict__ binq, int64_t n,
                                                  int64_t npix, double len2pix, int periodic,
                                                  uint32_t *__restrict__ keys,
                                                  int32_t *__restrict__ vals,
                                                  double4 *__restrict__ rec)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n)
        return;
    int64_t nb[3];
    tsc_bricks(npix, nb);
    double g[3] = {0.0, 0.0, 0.0};
    int64_t c[3];
    uint32_t key = (uint32_t)(nb[0] * nb[1] * nb[2]), flags = 0;
    if (tsc_cell(pos, p, npix, len2pix, periodic, g, c)) {
        const int side[3] = {kTX, kTY, kTZ};
        int b[3];
        for (int d = 0; d < 3; ++d) {
            int64_t xl = periodic ? tsc_wrap(c[d], npix) : c[d];
            const int x = (int)(xl < 0 ? 0 : xl > npix - 1 ? npix - 1 : xl);
            b[d] = x / side[d];
            const int lx = x - b[d] * side[d];
            flags |= lx == 0 ? 1u << (2 * d) : 0u;
            flags |= lx == side[d] - 1 || x == npix - 1 ? 2u << (2 * d) : 0u;
        }
        key = (uint32_t)((b[0] * nb[1] + b[1]) * nb[2] + b[2]);
    }
    keys[p] = key << kTscFlagBits | flags;
    vals[p] = (int32_t)p;
    if (rec)
        rec[p] = make_double4(g[0], g[1], g[2], ld(binq, p));
}

// off[b] = first sorted entry of brick >= b, b in [0, nbricks]
__global__ __launch_bounds__(256) void k_tsc_offsets(const uint32_t *__restrict__ keys,
                                                     int64_t n, int64_t nbricks,
                                                     int64_t *__restrict__ off)
{
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b > nbricks)
        return;
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int64_t)(keys[mid] >> kTscFlagBits) < b)
            lo = mid + 1;
        else
            hi = mid;
    }
    off[b] = lo;
}

// packed nearest cell: 16 bits per axis, each stored as c + kCellBias (c is
// in [-2, npix + 2] when not periodic, wrapped into [0, npix) when periodic;
// npix <= 2048)
constexpr int kCellBias = 4;
__device__ __forceinline__ uint64_t tsc_pack(const int64_t c[3])
{
    return (uint64_t)(c[0] + kCellBias) << 32 | (uint64_t)(c[1] + kCellBias) << 16 |
           (uint64_t)(c[2] + kCellBias);
}
__device__ __forceinline__ int tsc_unpack(uint64_t v, int d)
{
    return (int)((v >> (32 - 16 * d)) & 0xFFFF) - kCellBias;
}

// sorted grid coordinates and quantity (gq) and packed cells (cell) of the
// particles that are not dropped (the first off[nbricks] sorted entries).
// Bound by the cache lines of the particles' random reads: two or three of
// them (a position that may straddle two, the quantity), one where the keys'
// kernel has packed the record (rec): 303 -> 143 us for 2^22 particles in
// FP64, and the keys' kernel 40 -> 77 us.
template <typename T>
__global__ __launch_bounds__(256) void k_tsc_prep(const T *__restrict__ pos,
                                                  const T *__restrict__ binq,
                                                  const double4 *__restrict__ rec,
                                                  const int32_t *__restrict__ order,
                                                  const int64_t *__restrict__ off,
                                                  int64_t nbricks, int64_t npix, double len2pix,
                                                  int periodic, double4 *__restrict__ gq,
                                                  uint64_t *__restrict__ cell)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= off[nbricks])
        return;
    const int64_t p = order[k];
    double4 e;
    int64_t c[3];
    if (rec) {
        e = rec[p];
        c[0] = (int64_t)floor(e.x);
        c[1] = (int64_t)floor(e.y);
        c[2] = (int64_t)floor(e.z);
    } else {
        double g[3];
        tsc_cell(pos, p, npix, len2pix, periodic, g, c);
        e = make_double4(g[0], g[1], g[2], ld(binq, p));
    }
    if (periodic)
        for (int d = 0; d < 3; ++d)
            c[d] = tsc_wrap(c[d], npix);
    gq[k] = e;
    cell[k] = tsc_pack(c);
}

// particles per deposit step: 9 lanes each, one stencil row (o0, o1) per
// lane and its three cells along z
constexpr int kTscPerStep = kWave / 9;
// candidates per lane and scan chunk
constexpr int kTscPer = 4;
// Deposit queue of the gather: the candidates whose stencil reaches the
// brick, as sorted particle indices in a ring of LDS slots.  It holds at most
// kTscPerStep - 1 leftovers plus one chunk of candidates.
constexpr int kTscQueue = 264;
static_assert(kTscQueue >= kTscPerStep - 1 + kTscPer * kWave,
              "queue holds one chunk and the leftovers");

// a particle's record as the deposit step takes it
struct TscRec {
    double4 e;    // grid coordinates, quantity
    uint64_t cv;  // packed nearest cell
};

// One deposit step: a particle per nine lanes (cnt of them), r the particle of
// lane group `slot`.  The weights are formed as the oracle forms them: per
// axis W(g - (c + o) - 1/2) with c = floor(g), and the product (wx * wy) * wz.
__device__ __forceinline__ void tsc_step(const TscRec &r, int cnt, int slot, int o0, int o1,
                                         const int b0[3], int npix, int periodic,
                                         double (*acc)[kTX * kTY * kTZ])
{
    if (slot >= cnt)
        return;
    const double4 e = r.e;
    const uint64_t cv = r.cv;
    auto wrap = [&](int x) {
        return periodic ? (x < 0 ? x + npix : x >= npix ? x - npix : x) : x;
    };
    const int x = wrap(tsc_unpack(cv, 0) + o0), y = wrap(tsc_unpack(cv, 1) + o1);
    const int lx = x - b0[0], ly = y - b0[1];
    if (x >= npix || (unsigned)lx >= (unsigned)kTX || y >= npix || (unsigned)ly >= (unsigned)kTY)
        return;
    const double wx = tsc_w(sub_rn(e.x, floor(e.x) + (double)o0 + 0.5));
    const double wy = tsc_w(sub_rn(e.y, floor(e.y) + (double)o1 + 0.5));
    const double wxy = wx * wy, fz = floor(e.z);
    const int cz = tsc_unpack(cv, 2), row = (lx * kTY + ly) * kTZ;
#pragma unroll
    for (int o2 = -1; o2 <= 1; ++o2) {
        const int z = wrap(cz + o2), lz = z - b0[2];
        const double ww = wxy * tsc_w(sub_rn(e.z, fz + (double)o2 + 0.5));
        if (z < npix && (unsigned)lz < (unsigned)kTZ && ww != 0.0) {
            unsafeAtomicAdd(&acc[0][row + lz], e.w * ww);
            unsafeAtomicAdd(&acc[1][row + lz], ww);
        }
    }
}

// Brick of a block: block x runs on XCD x % 8, and the XCDs take runs of
// kTscRun consecutive bricks in turn, so that the two halves of a cache line
// and the reads of neighbouring bricks meet in one L2 (2^22 particles at
// 512^3: 1.17 -> 1.06 ms; runs of 16 / 512 bricks 1.28 / 1.37 ms, 32 and 128
// as 64).
constexpr int kTscRun = 64;
__device__ __forceinline__ int tsc_brick()
{
    const int x = blockIdx.x, l = x / 8;
    const int whole = (int)gridDim.x / (8 * kTscRun) * (8 * kTscRun);
    return x < whole ? (l / kTscRun * 8 + x % 8) * kTscRun + l % kTscRun : x;
}

// One wave per brick.  Lane j < 27 takes neighbouring brick j (offsets
// (j/9 - 1, (j/3)%3 - 1, j%3 - 1), each brick once), reads its particle range
// and forms the key flags a particle of it needs to reach this brick (the last
// cell along an axis whose offset is -1, the first one for +1).  The ranges,
// cut into groups of kTscPer entries, are laid end to end (wave prefix sum)
// and scanned 64 groups at a time, a group of sorted keys per lane; the
// entries with the needed flags go to the LDS queue, and the queue is
// deposited kTscPerStep particles per step.  The order of the additions to a
// cell follows the scan, so the sums are reproducible.
//
// What bounds it: the round trips to memory of a brick (ranges, keys,
// records; 0.52 ms without the keys and the records, 0.81 without the records)
// beside the stores of the planes (2.1 GB, 0.34 ms at the fill rate); the
// arithmetic and the LDS atomics are hidden (skipping the deposit steps saves
// 0.08 of 1.17 ms).  2^22 particles at 512^3: 1.30 ms with a packed 64-bit
// cell tested per candidate, one range search per 64 candidates and 4x8x8
// bricks, 1.17 with key flags tested four per lane, 0.97 with runs per XCD
// and bricks as long in z as a cache line.  Tried and dropped: two to sixteen
// waves per block (1.26 - 1.81 ms), waves that take bricks in turn and load
// the next brick's ranges and keys ahead (128 VGPRs, 1.51 ms).
__global__ __launch_bounds__(kWave) void k_tsc_gather(const double4 *__restrict__ gq,
                                                      const uint64_t *__restrict__ cell,
                                                      const uint32_t *__restrict__ keys,
                                                      const int64_t *__restrict__ off, int npix,
                                                      int periodic, double *__restrict__ grid)
{
    __shared__ double acc[2][kTX * kTY * kTZ];
    __shared__ int32_t queue[kTscQueue];
    __shared__ int4 s_rng[32];  // first group, first entry, end, needed flags
    const int nb[3] = {(npix + kTX - 1) / kTX, (npix + kTY - 1) / kTY, (npix + kTZ - 1) / kTZ};
    const int side[3] = {kTX, kTY, kTZ};
    const int b = tsc_brick();
    const int bi[3] = {b / (nb[1] * nb[2]), (b / nb[2]) % nb[1], b % nb[2]};
    int b0[3];
    for (int d = 0; d < 3; ++d)
        b0[d] = bi[d] * side[d];
    const int ln = threadIdx.x;
    // neighbour brick of lane ln, if it exists and is not a repeat of an
    // earlier offset on some axis (periodic grids of one or two bricks, whose
    // bricks are reached from either side: no flags needed there)
    int start = 0, end = 0, need = 0;
    if (ln < 27) {
        const int o[3] = {ln / 9 - 1, (ln / 3) % 3 - 1, ln % 3 - 1};
        bool valid = true;
        int x[3];
        for (int d = 0; d < 3; ++d) {
            auto nbr = [&](int oo) {
                int v = bi[d] + oo;
                if (periodic)
                    v = v < 0 ? v + nb[d] : v >= nb[d] ? v - nb[d] : v;
                return v;
            };
            x[d] = nbr(o[d]);
            if (!periodic && (x[d] < 0 || x[d] >= nb[d]))
                valid = false;
            for (int oo = -1; oo < o[d]; ++oo)
                valid = valid && nbr(oo) != x[d];
            if (!(periodic && nb[d] <= 2))
                need |= o[d] < 0 ? 2 << (2 * d) : o[d] > 0 ? 1 << (2 * d) : 0;
        }
        if (valid) {
            const int nbrick = (x[0] * nb[1] + x[1]) * nb[2] + x[2];
            start = (int)off[nbrick];
            end = (int)off[nbrick + 1];
        }
    }
    // exclusive prefix of the ranges' group counts over the lanes
    const int len = (end - start + kTscPer - 1) / kTscPer;
    int incl = len;
#pragma unroll
    for (int sh = 1; sh < 32; sh <<= 1) {
        const int t = __shfl_up(incl, sh);
        incl += ln >= sh ? t : 0;
    }
    const int total = __builtin_amdgcn_readlane(incl, 26);
    const int64_t nd = (int64_t)npix * npix * npix;
    // lane ln writes cells (t, ln / kTZ, ln % kTZ) of the brick, t < kTX
    static_assert(kTY * kTZ == kWave, "one x plane of a brick per wave");
    const int j = b0[1] + ln / kTZ, k = b0[2] + ln % kTZ;
    const bool in = j < npix && k < npix;
    const int64_t plane = (int64_t)npix * npix;
    double *out = grid + ((int64_t)b0[0] * npix + j) * npix + k;
    if (total == 0) {  // wave-uniform: no particle reaches the brick
        for (int t = 0; t < kTX && b0[0] + t < npix; ++t)
            if (in) {
                out[t * plane] = 0.0;
                out[nd + t * plane] = 0.0;
            }
        return;
    }
    for (int e = ln; e < 2 * kTX * kTY * kTZ; e += kWave)
        (&acc[0][0])[e] = 0.0;
    if (ln < 32)  // the lanes past the 27 ranges: bases past every group
        s_rng[ln] = ln < 27 ? make_int4(incl - len, start, end, need)
                            : make_int4(INT_MAX, 0, 0, 0);
    __syncthreads();

    const uint64_t below = ln == 0 ? 0ull : (~0ull >> (kWave - ln));
    const int slot = ln / 9, srow = ln - 9 * slot;
    const int o0 = srow / 3 - 1, o1 = srow % 3 - 1;
    int head = 0, fill = 0;  // first queued slot of the ring, entries queued (wave-uniform)
    // the record of queue entry head + ahead + slot, if it is queued; the
    // loop below loads a step's records while the previous step is deposited
    auto fetch = [&](int ahead) {
        TscRec r = {};
        if (slot < kTscPerStep && ahead + slot < fill) {
            int at = head + ahead + slot;
            at -= at >= kTscQueue ? kTscQueue : 0;
            const int q = queue[at];
            r.e = gq[q];
            r.cv = cell[q];
        }
        return r;
    };
    for (int v0 = 0; v0 < total; v0 += kWave) {
        const int v = v0 + ln;
        int k0 = 0, k1 = 0;
        uint32_t nf = 0;
        if (v < total) {
            // the last range whose first group is <= v (an empty range after
            // the one holding v starts after v)
            int lo = 0;
#pragma unroll
            for (int step = 16; step >= 1; step >>= 1)
                if (s_rng[lo + step].x <= v)
                    lo += step;
            const int4 r = s_rng[lo];
            k0 = r.y + (v - r.x) * kTscPer;
            k1 = r.z;
            nf = (uint32_t)r.w;
        }
        uint32_t kv[kTscPer];
#pragma unroll
        for (int i = 0; i < kTscPer; ++i)
            kv[i] = k0 + i < k1 ? keys[k0 + i] : 0u;
#pragma unroll
        for (int i = 0; i < kTscPer; ++i) {
            const bool use = k0 + i < k1 && (kv[i] & nf) == nf;
            const uint64_t mask = __ballot(use);
            if (use) {
                int at = head + fill + (int)__popcll(mask & below);
                at -= at >= kTscQueue ? kTscQueue : 0;
                queue[at] = k0 + i;
            }
            fill += (int)__popcll(mask);
        }
        __builtin_amdgcn_wave_barrier();
        // after the last chunk the leftovers follow as a short step
        const int keep = v0 + kWave < total ? kTscPerStep - 1 : 0;
        TscRec cur = fetch(0);
        while (fill > keep) {
            const TscRec next = fetch(kTscPerStep);
            const int cnt = fill < kTscPerStep ? fill : kTscPerStep;
            tsc_step(cur, cnt, slot, o0, o1, b0, npix, periodic, acc);
            fill -= cnt;
            head += cnt;
            head -= head >= kTscQueue ? kTscQueue : 0;
            cur = next;
        }
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    for (int t = 0; t < kTX && b0[0] + t < npix; ++t)
        if (in) {
            out[t * plane] = acc[0][t * kWave + ln];
            out[nd + t * plane] = acc[1][t * kWave + ln];
        }
}

int tsc_key_bits(int64_t npix)
{
    const int64_t nbr = tsc_nbricks(npix);
    int bits = 1;
    while (bits < 32 - kTscFlagBits && ((int64_t)1 << bits) <= nbr)
        ++bits;
    return kTscFlagBits + bits;
}

void launch_tsc_keys(int dtype, const void *pos, const void *binq, int64_t n, int64_t npix,
                     double len2pix, int periodic, uint32_t *keys, int32_t *vals, double4 *rec,
                     hipStream_t s)
{
    if (n == 0)
        return;
    const dim3 g((unsigned)((n + 255) / 256)), blk(256);
    if (dtype == S2G_F32)
        hipLaunchKernelGGL(k_tsc_keys<float>, g, blk, 0, s, (const float *)pos,
                           (const float *)binq, n, npix, len2pix, periodic, keys, vals, rec);
    else
        hipLaunchKernelGGL(k_tsc_keys<double>, g, blk, 0, s, (const double *)pos,
                           (const double *)binq, n, npix, len2pix, periodic, keys, vals, rec);
}

void launch_tsc_offsets(const uint32_t *sorted_keys, int64_t n, int64_t npix, int64_t *off,
                        hipStream_t s)
{
    const int64_t nbr = tsc_nbricks(npix);
    hipLaunchKernelGGL(k_tsc_offsets, dim3((unsigned)((nbr + 1 + 255) / 256)), dim3(256), 0, s,
                       sorted_keys, n, nbr, off);
}

void launch_tsc_prep(int dtype, const void *pos, const void *binq, const double4 *rec,
                     const int32_t *order, const int64_t *off, int64_t n, int64_t npix, double len2pix, int periodic,
                     double4 *gq, uint64_t *cell, hipStream_t s)
{
    if (n == 0)
        return;
    const int64_t nbr = tsc_nbricks(npix);
    const dim3 g((unsigned)((n + 255) / 256)), blk(256);
    if (dtype == S2G_F32)
        hipLaunchKernelGGL(k_tsc_prep<float>, g, blk, 0, s, (const float *)pos,
                           (const float *)binq, rec, order, off, nbr, npix, len2pix, periodic, gq,
                           cell);
    else
        hipLaunchKernelGGL(k_tsc_prep<double>, g, blk, 0, s, (const double *)pos,
                           (const double *)binq, rec, order, off, nbr, npix, len2pix, periodic, gq,
                           cell);
}

int tsc_key_begin_bit() { return kTscFlagBits; }

void launch_tsc_gather(const double4 *gq, const uint64_t *cell, const uint32_t *sorted_keys,
                       const int64_t *off, int64_t npix, int periodic, double *grid,
                       hipStream_t s)
{
    const int64_t nbr = tsc_nbricks(npix);
    hipLaunchKernelGGL(k_tsc_gather, dim3((unsigned)nbr), dim3(kWave), 0, s, gq, cell,
                       sorted_keys, off, (int)npix, periodic, grid);
}

}  // namespace s2g
