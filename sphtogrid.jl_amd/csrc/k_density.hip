// k_density.hip -- mass_density (effects/mass_density.jl:30-99) on gfx950:
// SPH density and smoothing length of an arbitrary particle set from its
// k = Nneighbors + 1 nearest neighbours (the particle itself included).
//
// Neighbour search without a tree build: particles are sorted by a 63-bit
// Morton key (21 bits per axis over the domain), so the cells of every level
// of the implicit octree are contiguous ranges of the sorted order.  A table
// of cell offsets at one level (8 at most, 8^8 cells) turns a cell into its range
// with two loads; finer cells are found by binary search inside their table
// cell.
//
//   k_md_prep      FP64 (x, y, z, m), positions wrapped into a periodic box,
//                  per-block bounding boxes
//   k_md_keys      Morton key per particle -> radix sort
//   k_md_sorted    particles in key order
//   k_md_table     cell offsets at the table level (binary search per cell)
//   k_md_knn       one wave per particle:
//                  1. a first bound T0 >= the true k-th distance: the k-th
//                     smallest distance to the particles next to it in key
//                     order (they are k real particles);
//                  2. the level whose cells are between T0/2 and T0 wide and
//                     the cube of <= 5^3 cells around the particle that covers
//                     the ball of radius T0;
//                  3. the particle ranges of the cells within T0, once, two
//                     cells a lane;
//                     every particle in the cube at distance <= T goes to a
//                     per-wave LDS buffer (T shrinks as the buffer is cut back
//                     to the k nearest), the cells within T0/2 first: the
//                     k-th nearest of those gives T1, and of the other cells
//                     only those within T1 are read; the search works on
//                     squared distances, and the exact k-th smallest is a
//                     bisection on their FP64 bit patterns (its square
//                     root is hsml);
//                  4. the kernel sum over the buffer and the bias correction
//                     of Dehnen & Aly (2012, eqs. 18-19).
// The cube holds the whole ball of radius T0 and T0 is an upper bound, so the
// k nearest neighbours are all found: the result is exact, and the work per
// particle follows the local density (clustered sets cost what uniform ones
// cost).  Distances are FP64 without contraction, minimum image per
// dimension in a periodic box.
#include "k_density.h"

namespace s2g {

constexpr int kMdCap = 596;     // candidate buffer per wave (20 waves of 8 KB per CU)
constexpr int kMdBits = 21;     // Morton bits per axis
constexpr int kMdMaxCells = 2 * kWave;  // cube cells per particle

template <typename T>
__global__ __launch_bounds__(256) void k_md_prep(const T *__restrict__ pos,
                                                 const T *__restrict__ mass, int64_t n,
                                                 MdGrid g, double4 *__restrict__ P,
                                                 double *__restrict__ bbox)
{
    __shared__ double s_lo[3][256], s_hi[3][256];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    if (i < n) {
        double x[3];
        for (int d = 0; d < 3; ++d) {
            double v = (double)pos[3 * i + d];
            if (g.periodic) {
                v = v - g.box[d] * floor(v / g.box[d]);
                if (v >= g.box[d])
                    v -= g.box[d];
            }
            x[d] = v;
            lo[d] = hi[d] = v;
            if (!isfinite(v)) {  // reported by the host as an invalid input
                lo[d] = -INFINITY;
                hi[d] = INFINITY;
            }
        }
        P[i] = make_double4(x[0], x[1], x[2], (double)mass[i]);
    }
    for (int d = 0; d < 3; ++d) {
        s_lo[d][threadIdx.x] = lo[d];
        s_hi[d][threadIdx.x] = hi[d];
    }
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            for (int d = 0; d < 3; ++d) {
                s_lo[d][threadIdx.x] = fmin(s_lo[d][threadIdx.x], s_lo[d][threadIdx.x + s]);
                s_hi[d][threadIdx.x] = fmax(s_hi[d][threadIdx.x], s_hi[d][threadIdx.x + s]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 3) {
        bbox[6 * blockIdx.x + threadIdx.x] = s_lo[threadIdx.x][0];
        bbox[6 * blockIdx.x + 3 + threadIdx.x] = s_hi[threadIdx.x][0];
    }
}

// spread the low 21 bits of a over every third bit
__host__ __device__ __forceinline__ uint64_t md_split3(uint32_t a)
{
    uint64_t x = a & 0x1fffffu;
    x = (x | x << 32) & 0x1f00000000ffffull;
    x = (x | x << 16) & 0x1f0000ff0000ffull;
    x = (x | x << 8) & 0x100f00f00f00f00full;
    x = (x | x << 4) & 0x10c30c30c30c30c3ull;
    x = (x | x << 2) & 0x1249249249249249ull;
    return x;
}

__device__ __forceinline__ uint64_t md_morton(uint32_t x, uint32_t y, uint32_t z)
{
    return md_split3(x) | md_split3(y) << 1 | md_split3(z) << 2;
}

__device__ __forceinline__ uint32_t md_quant(double v, const MdGrid &g, int d)
{
    const double t = (v - g.lo[d]) * g.inv_ext[d] * (double)(1u << kMdBits);
    const double c = floor(t);
    return c < 0.0 ? 0u : (c >= (double)((1u << kMdBits) - 1) ? (1u << kMdBits) - 1 : (uint32_t)c);
}

__global__ void k_md_keys(const double4 *__restrict__ P, int64_t n, MdGrid g,
                          uint64_t *__restrict__ keys, int32_t *__restrict__ vals)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    const double4 p = P[i];
    keys[i] = md_morton(md_quant(p.x, g, 0), md_quant(p.y, g, 1), md_quant(p.z, g, 2));
    vals[i] = (int32_t)i;
}

__global__ void k_md_sorted(const double4 *__restrict__ P, const int32_t *__restrict__ idx,
                            int64_t n, double4 *__restrict__ S)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        S[i] = P[idx[i]];
}

__device__ __forceinline__ int64_t md_lower_bound(const uint64_t *__restrict__ K, int64_t lo,
                                                  int64_t hi, uint64_t key)
{
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (K[mid] < key)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

__device__ __forceinline__ int md_lower_bound32(const uint64_t *__restrict__ K, int lo, int hi,
                                                uint64_t key)
{
    while (lo < hi) {
        const int mid = lo + (hi - lo) / 2;
        if (K[mid] < key)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// offsets of the 8^lt cells of level lt (+ the end)
__global__ void k_md_table(const uint64_t *__restrict__ K, int64_t n, int lt,
                           int32_t *__restrict__ tab)
{
    const int64_t ncell = (int64_t)1 << (3 * lt);
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e > ncell)
        return;
    tab[e] = e == ncell ? (int32_t)n
                        : (int32_t)md_lower_bound(K, 0, n, (uint64_t)e << (3 * (kMdBits - lt)));
}

// minimum-image component (mass_density.jl:45-52, Distances.jl PeriodicEuclidean)
__device__ __forceinline__ double md_comp(double a, double b, double box, int periodic)
{
    double x = fabs(a - b);
    if (periodic && x > 0.5 * box)
        x = box - x;
    return x;
}

// squared distance, rounded as the reference rounds it before the square
// root (no contraction).  The search selects on these: the k-th smallest
// squared distance is the square of the k-th smallest distance, because a
// correctly rounded sqrt is monotone, so sqrt of it is the reference's hsml.
__device__ __forceinline__ double md_dist2(const double4 &a, const double4 &b, const MdGrid &g)
{
    const double dx = md_comp(a.x, b.x, g.box[0], g.periodic);
    const double dy = md_comp(a.y, b.y, g.box[1], g.periodic);
    const double dz = md_comp(a.z, b.z, g.box[2], g.periodic);
    return add_rn(add_rn(mul_rn(dx, dx), mul_rn(dy, dy)), mul_rn(dz, dz));
}

// value of another lane (DPP lane pattern) on the rows of the mask, else 0
template <int kCtrl, int kRows = 0xF>
__device__ __forceinline__ int dpp_or_0(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, kCtrl, kRows, 0xF, true);
}

// inclusive prefix sum over the lanes of a fully active wave
__device__ __forceinline__ int wave_incl_scan(int v)
{
    v += dpp_or_0<0x111>(v);       // row_shr 1, 2, 4, 8
    v += dpp_or_0<0x112>(v);
    v += dpp_or_0<0x114>(v);
    v += dpp_or_0<0x118>(v);
    v += dpp_or_0<0x142, 0xA>(v);  // row_bcast 15 into rows 1 and 3
    v += dpp_or_0<0x143, 0xC>(v);  // row_bcast 31 into rows 2 and 3
    return v;
}

// keys (NR a lane) below c, over the wave
template <int NR>
__device__ __forceinline__ int md_count_below(const uint32_t (&key)[NR], uint32_t c)
{
    int m = 0;
#pragma unroll
    for (int r = 0; r < NR; ++r)
        m += (int)__popcll(__ballot(key[r] < c));
    return m;
}

// The k-th smallest of the keys between lo and last, of which `under` are
// below lo and `upto` at most last (under < k <= upto): halves the interval
// until it is no wider than `width` or holds one key, counting with ballots:
// NR compares and scalar additions a step, no LDS and no prefix sums.
template <int NR>
__device__ __forceinline__ void md_bisect(const uint32_t (&key)[NR], int k, uint32_t width,
                                          uint32_t &lo, uint32_t &last, int &under, int &upto)
{
    while (last - lo >= width && upto - under > 1) {
        const uint32_t mid = lo + (last - lo) / 2 + 1;
        const int m = md_count_below<NR>(key, mid);
        if (m < k) {
            lo = mid;
            under = m;
        } else {
            last = mid - 1;
            upto = m;
        }
    }
}

// k-th smallest (1-based) of the doubles buf[0..cnt) (each +0 or positive and
// finite), cnt <= 64 NR, exactly: by the high words first (the sign is 0; keys
// that a lane does not hold are all ones), then, if several entries share the
// k-th's high word, by their low words.  The search starts from the two
// binades up to T, which no entry exceeds (for T = infinity, from the three on
// either side of a sample), and widens where the k-th is not in there.
// kExact == false: an upper bound of it instead, within 1/16, for thresholds
// that only have to keep at least k entries.
template <int NR, bool kExact>
__device__ __forceinline__ double md_select_of(const double *buf, int cnt, int k, double T, int ln)
{
    uint32_t hi[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r)
        hi[r] = r * kWave + ln < cnt ? (uint32_t)__double2hiint(buf[r * kWave + ln]) : ~0u;
    constexpr uint32_t kInf = 0x7ff00000u, kBinade = 1u << 20;
    uint32_t last = (uint32_t)__builtin_amdgcn_readfirstlane(__double2hiint(T));
    uint32_t lo = last > 2 * kBinade ? last - 2 * kBinade : 0;
    int upto = cnt;
    if (last == kInf) {
        const uint32_t g =
            (uint32_t)__builtin_amdgcn_readfirstlane(__double2hiint(buf[cnt / 4]));
        lo = g > 3 * kBinade ? g - 3 * kBinade : 0;
        last = g + 3 * kBinade;
        upto = md_count_below<NR>(hi, last + 1);
        if (upto < k) {
            last = kInf;
            upto = cnt;
        }
    }
    int under = md_count_below<NR>(hi, lo);
    if (under >= k) {
        last = lo - 1;
        upto = under;
        lo = 0;
        under = 0;
    }
    md_bisect<NR>(hi, k, kExact ? 1 : kBinade / 16, lo, last, under, upto);
    // the only entry for which `in` holds
    const auto one = [&](auto &&in) -> double {
        double v = 0.0;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const uint64_t bt = __ballot(in(r));
            if (bt)  // wave-uniform
                v = buf[r * kWave + __ffsll((unsigned long long)bt) - 1];
        }
        return v;
    };
    if (upto - under == 1)
        return one([&](int r) { return hi[r] - lo <= last - lo; });
    if (!kExact)
        return __hiloint2double((int)last, -1);
    // several with the high word lo == last
    uint32_t low[NR], l0 = 0, l1 = ~0u;
#pragma unroll
    for (int r = 0; r < NR; ++r)
        low[r] = hi[r] == lo ? (uint32_t)__double2loint(buf[r * kWave + ln]) : ~0u;
    k -= under;
    upto -= under;
    under = 0;
    md_bisect<NR>(low, k, 1, l0, l1, under, upto);
    if (l0 == l1)
        return __hiloint2double((int)lo, (int)l0);
    return one([&](int r) { return hi[r] == lo && low[r] - l0 <= l1 - l0; });
}

template <bool kExact>
__device__ __forceinline__ double md_select(const double *buf, int cnt, int k, double T, int ln)
{
    static_assert(kMdCap <= 10 * kWave, "the buffer in ten registers a lane");
    const double v = cnt <= 3 * kWave   ? md_select_of<3, kExact>(buf, cnt, k, T, ln)
                     : cnt <= 6 * kWave ? md_select_of<6, kExact>(buf, cnt, k, T, ln)
                                        : md_select_of<10, kExact>(buf, cnt, k, T, ln);
    // the same on every lane: keeps what follows from it in scalar registers
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// keep the entries below T and, of those equal to T, as many as make k in
// total (they are at u = 1, W = 0); returns the new count
__device__ int md_compact(double *buf, int *jb, int cnt, double T, int k, int ln)
{
    int nless = 0;
    for (int e0 = 0; e0 < cnt; e0 += kWave) {
        const int e = e0 + ln;
        nless += __popcll(__ballot(e < cnt && buf[e] < T));
    }
    int quota = k - nless;  // entries equal to T to keep
    int out = 0;
    const uint64_t below = ln == 0 ? 0ull : (~0ull >> (kWave - ln));
    for (int e0 = 0; e0 < cnt; e0 += kWave) {
        const int e = e0 + ln;
        const double d = e < cnt ? buf[e] : 0.0;
        const int j = e < cnt ? jb[e] : 0;
        const bool less = e < cnt && d < T;
        const bool eq = e < cnt && d == T;
        const uint64_t beq = __ballot(eq);
        const bool keep_eq = eq && (int)__popcll(beq & below) < quota;
        const bool keep = less || keep_eq;
        const uint64_t bk = __ballot(keep);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        if (keep) {
            const int at = out + (int)__popcll(bk & below);
            buf[at] = d;
            jb[at] = j;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        out += (int)__popcll(bk);
        const int taken = (int)__popcll(beq);
        quota -= taken < quota ? taken : (quota > 0 ? quota : 0);
    }
    return out;
}

// Append the candidates (lane's j, squared distance d, valid flag) with
// d <= T to the buffer; when it is about to overflow, cut it back to the k
// nearest.
__device__ __forceinline__ void md_offer(bool valid, double d, int j, double &T, int &cnt,
                                         double *buf, int *jb, int k1, int ln, uint64_t below)
{
    const bool take = valid && d <= T;
    const uint64_t bt = __ballot(take);
    if (take) {
        const int at = cnt + (int)__popcll(bt & below);
        buf[at] = d;
        jb[at] = j;
    }
    cnt += (int)__popcll(bt);
    if (cnt > kMdCap - kWave) {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        T = md_select<true>(buf, cnt, k1, T, ln);
        cnt = md_compact(buf, jb, cnt, T, k1, ln);
    }
}

// The hardware hands consecutive blocks to the eight XCDs in turn; here each
// XCD takes runs of kMdXcdRun consecutive particles in key order, whose cells
// are the same few, through its own L2 (runs of 256 to 8192 time alike).  The
// last n mod (8 kMdXcdRun) particles keep their own order.
constexpr int kXcds = 8, kMdXcdRun = 1024;
__device__ __forceinline__ int64_t md_xcd_query(int64_t i, int64_t n)
{
    const int64_t span = (int64_t)kXcds * kMdXcdRun;
    if (i >= n / span * span)
        return i;
    const int64_t x = i % kXcds, t = i / kXcds;
    return t / kMdXcdRun * span + x * kMdXcdRun + t % kMdXcdRun;
}

// Bound by instruction issue, vector and scalar alike, and by the latency of
// the cells' searches and candidates, so by the waves in flight: one wave a
// block, which is replaced as soon as it ends (four in a block waited for the
// slowest), and 8 KB of LDS, 20 waves per CU.  A particle's cell ranges are
// searched once for both passes; the selects bisect with ballots from a guessed
// interval in place of radix passes over LDS histograms; what is the same on
// all lanes is kept in scalar registers.  2^20 particles in halos, 64
// neighbours: 9.18 -> 4.95 ms (3,700 -> about 2,000 vector instructions a
// particle).  A bound from the last particle's neighbours instead of the key
// order's (median 1.35 times the true distance against 1.27) measured slower,
// and so did a search of the ranges by quarters (5.57 -> 5.88 ms).
template <int K>
__global__ __launch_bounds__(kWave, 4) void k_md_knn(
    const double4 *__restrict__ S, const uint64_t *__restrict__ SK,
    const int32_t *__restrict__ order, const int32_t *__restrict__ tab, int lt, int64_t n,
    MdGrid g, int k1, int dim, int nneigh, double norm, double *__restrict__ rho_out,
    double *__restrict__ hsml_out)
{
    __shared__ double buf[kMdCap];
    __shared__ int jb[kMdCap];
    __shared__ int cstart[kMdMaxCells];  // cube cell: first particle
    __shared__ int cpre[kMdMaxCells];    // prefix of the cells' counts
    const int ln = threadIdx.x;
    const uint64_t below = ln == 0 ? 0ull : (~0ull >> (kWave - ln));
    for (int64_t i = blockIdx.x; i < n; i += gridDim.x) {
        const int64_t q = md_xcd_query(i, n);
        const double4 me = S[q];
        // 1. first bound: the k-th nearest of the particles next in key
        //    order, k on each side (where the particles on one side are far,
        //    as at the edge of a cluster in key order, the other side alone
        //    still holds k)
        int cnt = 0;
        double T;  // squared distances from here on
        {
            const int w = k1 < kMdCap / 2 ? k1 : kMdCap / 2 - 1;
            int64_t a = q - w > 0 ? q - w : 0;
            int64_t b = q + w < n - 1 ? q + w : n - 1;
            if (b - a + 1 < k1) {  // a large k near either end
                a = a < n - k1 ? a : n - k1;
                b = a + k1 - 1;
            }
            cnt = (int)(b - a) + 1;  // in [k1, kMdCap)
            for (int t = ln; t < cnt; t += kWave)
                buf[t] = md_dist2(me, S[a + t], g);
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            T = md_select<false>(buf, cnt, k1, __builtin_inf(), ln);  // >= the k-th of these
        }
        const double T20 = T, T0 = sqrt(T20);
        // 2. level with cells in [T0/2, T0) along the narrowest axis; per
        //    axis the cells that meet [x - T0, x + T0], found with the
        //    particles' own quantisation widened by one quantum: the span is
        //    2 T0 + 2 quanta < 5 cells (cells are >= T0 / 2 wide and a
        //    quantum is at most half a cell below level 21, where the cell
        //    exceeds T0), so at most six cells per axis
        int lev = kMdBits;
        if (T0 > 0.0) {
            const int l = __builtin_amdgcn_frexp_exp(g.min_ext / T0);  // floor(log2) + 1
            lev = l < 0 ? 0 : (l > kMdBits ? kMdBits : l);
        }
        uint32_t ncl;
        int ca[3], cl[3], ncube;  // first cell (unwrapped) and cell count per axis
        const double mv[3] = {me.x, me.y, me.z};
        int qlo[3], qhi[3];
        for (int d = 0; d < 3; ++d) {
            const double qs = (double)(1u << kMdBits);
            // far outside the domain (a narrow axis) means all of its cells:
            // the clamp to 2^28 quanta, 128 domains, keeps that
            const double far = 268435456.0;
            const double l = (mv[d] - T0 - g.lo[d]) * g.inv_ext[d] * qs;
            const double h = (mv[d] + T0 - g.lo[d]) * g.inv_ext[d] * qs;
            qlo[d] = (int)floor(fmax(l, -far)) - 1;
            qhi[d] = (int)floor(fmin(h, far)) + 1;
        }
        for (;; --lev) {
            ncl = 1u << lev;
            const int sh = kMdBits - lev;
            for (int d = 0; d < 3; ++d) {
                int clo = qlo[d] >> sh, chi = qhi[d] >> sh;  // floor division
                if (g.periodic) {
                    if (chi - clo + 1 >= (int)ncl) {
                        clo = 0;
                        chi = (int)ncl - 1;
                    }
                } else {
                    clo = clo < 0 ? 0 : clo;
                    chi = chi > (int)ncl - 1 ? (int)ncl - 1 : chi;
                }
                ca[d] = clo;
                cl[d] = chi - clo + 1;
            }
            ncube = cl[0] * cl[1] * cl[2];
            // two cells a lane: 6 x 6 x 4 cells and more take the next
            // coarser level, at most 4^3
            if (ncube <= kMdMaxCells)
                break;
        }
        // cells whose nearest point is farther than T0 (with a margin of two
        // quanta per axis) hold no candidate
        const double T0m = T0 * (1.0 + 1e-12);
        // 3. the cube's particles; cells are ranges of the sorted order.  The
        //    cells whose nearest point lies within T0/2 go first: the k-th
        //    nearest of their particles is a bound T1 close to the true k-th
        //    distance (T0 is often half as large again), and of the other
        //    cells only those within T1 are read
        // per axis: unwrapped cell o spans [o, o + 1) * cw around x; the
        // distance to it is taken eps = two quanta short
        double cw[3], xlo[3], xhi[3];
        float rcl[3];
        for (int d = 0; d < 3; ++d) {
            const double eps = 2.0 * g.ext[d] / (double)(1u << kMdBits);
            const double xr = mv[d] - g.lo[d];
            cw[d] = ldexp(g.ext[d], -lev);
            xlo[d] = xr + eps;
            xhi[d] = xr - eps;
            rcl[d] = 1.0f / (float)cl[d];
        }
        // the cube's cells, two a lane: squared nearest distance (above T0's:
        // not read), first particle and count
        double cdd[2];
        int cs[2], cn[2];
#pragma unroll
        for (int z = 0; z < 2; ++z) {
            const int t = z * kWave + ln;
            cdd[z] = 1e300;
            cs[z] = cn[z] = 0;
            if (z * kWave < ncube && t < ncube) {
                uint32_t cc[3];
                int r = t;
                double dd = 0.0;
                for (int d = 0; d < 3; ++d) {
                    // r = q cl + rem with r < 128, cl <= 6: the float
                    // quotient of r + 1/2 is at least 1/12 from an integer
                    const int qd = d < 2 ? (int)(((float)r + 0.5f) * rcl[d]) : 0;
                    int o = ca[d] + (r - qd * cl[d]);
                    r = qd;
                    if (cl[d] < (int)ncl || !g.periodic) {
                        const double a = (double)o * cw[d] - xlo[d];
                        const double b = xhi[d] - (double)(o + 1) * cw[d];
                        const double dx = a > 0.0 ? a : (b > 0.0 ? b : 0.0);
                        dd += dx * dx;
                    }
                    o = o < 0 ? o + (int)ncl : (o >= (int)ncl ? o - (int)ncl : o);
                    cc[d] = (uint32_t)o;
                }
                if (dd <= T0m * T0m) {
                    const uint64_t pre = md_morton(cc[0], cc[1], cc[2]);  // 3*lev bits
                    int s, e;
                    if (lev <= lt) {
                        s = tab[pre << (3 * (lt - lev))];
                        e = tab[(pre + 1) << (3 * (lt - lev))];
                    } else {
                        const uint64_t par = pre >> (3 * (lev - lt));
                        const int ksh = 3 * (kMdBits - lev);
                        s = tab[par];
                        e = tab[par + 1];
                        s = md_lower_bound32(SK, s, e, pre << ksh);
                        // the cell holds few of the parent's particles
                        const uint64_t end = (pre + 1) << ksh;
                        const bool more = s + 32 < e && SK[s + 32] < end;
                        e = md_lower_bound32(SK, more ? s + 33 : s,
                                            more || e < s + 32 ? e : s + 32, end);
                    }
                    cdd[z] = dd;
                    cs[z] = s;
                    cn[z] = e - s;
                }
            }
        }
        int ncells = 0;  // uniform
        auto list_cells = [&](double lo2, double hi2) -> int {
            // the non-empty cells with lo2 < (nearest distance)^2 <= hi2, in
            // cube order, into cstart/cpre (first particle, number of the
            // first candidate) and ncells; returns their particle count
            // (uniform)
            int C = 0, nc = 0;
#pragma unroll
            for (int z = 0; z < 2; ++z) {
                if (z * kWave >= ncube)
                    break;
                const int len = cdd[z] > lo2 && cdd[z] <= hi2 ? cn[z] : 0;
                const int in = wave_incl_scan(len);
                const uint64_t bne = __ballot(len > 0);
                if (len > 0) {
                    const int at = nc + (int)__popcll(bne & below);
                    cstart[at] = cs[z];
                    cpre[at] = C + in - len;
                }
                nc += (int)__popcll(bne);
                C += __builtin_amdgcn_readlane(in, kWave - 1);
            }
            ncells = nc;
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            return C;
        };
        auto offer_cells = [&](int C) {
            // candidate u lies in the last cell c with cpre[c] <= u.  Of a
            // chunk of 64 candidates from u0, the cells after cp (the cell
            // of u0 - 1) that start in it are the next ones in the list:
            // their starts are flagged (in the 64 entries of jb that the
            // chunk may fill afterwards), and a lane's cell is cp plus the
            // flags at or below its position
            int cp = -1;  // uniform
            for (int u0 = 0; u0 < C; u0 += kWave) {
                int *start = jb + cnt;
                start[ln] = 0;
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                const int ci = cp + 1 + ln;
                if (ci < ncells) {
                    const int st = cpre[ci] - u0;  // >= 0
                    if (st < kWave)
                        start[st] = 1;
                }
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                const uint64_t bf = __ballot(start[ln] != 0);
                const int u = u0 + ln;
                const bool valid = u < C;
                double d = 0.0;
                int j = 0;
                if (valid) {
                    const int c = cp + (int)__popcll(bf & (below | (1ull << ln)));
                    j = cstart[c] + (u - cpre[c]);
                    d = md_dist2(me, S[j], g);
                }
                cp += (int)__popcll(bf);
                md_offer(valid, d, j, T, cnt, buf, jb, k1, ln, below);
            }
            // the next pass rewrites cstart/cpre
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        };
        cnt = 0;  // fresh buffer, threshold T0 (inclusive)
        T = T20;
        const double inner2 = 0.25 * T0m * T0m;
        for (int pass = 0; pass < 2; ++pass) {
            double lo2 = -1.0, hi2 = inner2;
            if (pass == 1) {
                const double T1m = sqrt(T) * (1.0 + 1e-12);
                lo2 = inner2;
                hi2 = T1m * T1m;
            }
            offer_cells(list_cells(lo2, hi2));
            // after the inner cells a bound T1 <= T0 of the k-th (at least
            // k entries are within it); at the end the exact k-th, with
            // every particle nearer than it in the buffer, each once
            if (cnt >= k1)
                T = pass == 0 ? md_select<false>(buf, cnt, k1, T, ln)
                              : md_select<true>(buf, cnt, k1, T, ln);
        }
        // 4. mass_density.jl:70-86: kernel sum over the neighbours, bias correction
        const double h = sqrt(T), h_inv = 1.0 / h;
        double rho = 0.0;
        for (int e = ln; e < cnt; e += kWave) {
            const double d2 = buf[e];
            if (d2 <= T) {
                const double d = sqrt(d2);
                if (d < h)
                    rho += S[jb[e]].w * shape_of<K, double>(d * h_inv);
            }
        }
        rho = wave_sum(rho);
        double hd = h_inv;
        for (int d = 1; d < dim; ++d)
            hd *= h_inv;
        rho *= norm * hd;
        rho = md_bias_correction(K, rho, me.w, norm * hd, nneigh);
        if (ln == 0) {
            const int oi = order[q];
            rho_out[oi] = rho;
            hsml_out[oi] = h;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
int64_t md_prep_blocks(int64_t n) { return (n + 255) / 256; }


int md_max_neighbours()
{
    static_assert(471 + 1 <= kMdCap - kWave, "k entries and a chunk of candidates fit");
    return 471;
}

int md_bits() { return kMdBits; }

void launch_md_prep(int dtype, const void *pos, const void *mass, int64_t n, const MdGrid &g,
                    double4 *P, double *bbox, hipStream_t s)
{
    const dim3 grid((unsigned)md_prep_blocks(n)), blk(256);
    if (dtype == S2G_F32)
        hipLaunchKernelGGL(k_md_prep<float>, grid, blk, 0, s, (const float *)pos,
                           (const float *)mass, n, g, P, bbox);
    else
        hipLaunchKernelGGL(k_md_prep<double>, grid, blk, 0, s, (const double *)pos,
                           (const double *)mass, n, g, P, bbox);
}

void launch_md_keys(const double4 *P, int64_t n, const MdGrid &g, uint64_t *keys, int32_t *vals,
                    hipStream_t s)
{
    hipLaunchKernelGGL(k_md_keys, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, P, n, g,
                       keys, vals);
}

void launch_md_sorted(const double4 *P, const int32_t *idx, int64_t n, double4 *S,
                      hipStream_t s)
{
    hipLaunchKernelGGL(k_md_sorted, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, P, idx,
                       n, S);
}

void launch_md_table(const uint64_t *K, int64_t n, int lt, int32_t *tab, hipStream_t s)
{
    const int64_t ne = ((int64_t)1 << (3 * lt)) + 1;
    hipLaunchKernelGGL(k_md_table, dim3((unsigned)((ne + 255) / 256)), dim3(256), 0, s, K, n, lt,
                       tab);
}

void launch_md_knn(int kernel, const double4 *S, const uint64_t *SK, const int32_t *order,
                   const int32_t *tab, int lt, int64_t n, const MdGrid &g, int k1, int dim,
                   int nneigh, double norm, double *rho, double *hsml, hipStream_t s)
{
    int64_t blocks = n;
    if (blocks > (1 << 18))
        blocks = 1 << 18;
    const dim3 grid((unsigned)blocks), blk(kWave);
#define S2G_MD_CASE(KK)                                                                      \
    hipLaunchKernelGGL(k_md_knn<KK>, grid, blk, 0, s, S, SK, order, tab, lt, n, g, k1, dim, \
                       nneigh, norm, rho, hsml)
    switch (kernel) {
    case S2G_KERNEL_CUBIC: S2G_MD_CASE(S2G_KERNEL_CUBIC); break;
    case S2G_KERNEL_QUINTIC: S2G_MD_CASE(S2G_KERNEL_QUINTIC); break;
    case S2G_KERNEL_WENDLAND_C2: S2G_MD_CASE(S2G_KERNEL_WENDLAND_C2); break;
    case S2G_KERNEL_WENDLAND_C4: S2G_MD_CASE(S2G_KERNEL_WENDLAND_C4); break;
    case S2G_KERNEL_WENDLAND_C6: S2G_MD_CASE(S2G_KERNEL_WENDLAND_C6); break;
    default: S2G_MD_CASE(S2G_KERNEL_WENDLAND_C8); break;
    }
#undef S2G_MD_CASE
}

}  // namespace s2g
