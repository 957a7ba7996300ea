// fb_sort.hip -- the sort stage: fields of few points in one launch (k_field_sort), all others by
// row buckets (scan of the row counts, scatter into the rows, row sorts).
//
// Used to order the injection's points by base cell while keeping, inside a cell, the point
// order of the input (the order in which the reference's _inject_data_*d loop adds them,
// interpolation.py:246-270): both sorts order the composite (cell key, point index), so the
// result does not depend on timing.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "fb_internal.h"
#include "fb_launch.h"
#include "fb_points.h"

namespace fb {

namespace {

constexpr int kThreads = 256;
constexpr int kItems = 4;
constexpr int kTile = kThreads * kItems;   // 1024 elements per workgroup of the scan
constexpr int kLocalSortThreads = 1024;

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Sum of v over the workgroup's earlier threads; total: over all of them.  wsum: one word per wave
// (nobody may still read it).
__device__ __forceinline__ uint32_t block_before(uint32_t v, uint32_t *wsum, uint32_t &total)
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
    uint32_t inc = v;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(inc, d);
        if (lane >= d) inc += o;
    }
    if (lane == 63) wsum[wv] = inc;
    __syncthreads();
    uint32_t before = 0;
    total = 0;
    for (int w = 0; w < nw; ++w) {
        const uint32_t x = wsum[w];
        before += w < wv ? x : 0u;
        total += x;
    }
    return before + inc - v;
}

// ---- scan ----------------------------------------------------------------

// out = exclusive scan of in within each tile of kTile words, and tiles[t] = the sum of all tiles before tile
// t: up to kFewTiles tiles each workgroup sums the words before its own, which spares a launch (16 tiles 4.0 us,
// 33 5.1, 64 7.2; two launches 3.0 + 3.0 and the gap between them); beyond that tiles[t] is left the sum of
// tile t, which k_scan_sums makes it of.  (In one launch, the workgroup that ends last taking the sums, each
// workgroup's release before its count writes back its L2: 50 ns a tile, 98 us for 2 million rows and 10.9 for
// 200 thousand; two launches take 9.1 and 5.6.)
constexpr int kFewTiles = 48;

__global__ __launch_bounds__(kThreads) void k_scan_tiles(const uint32_t *__restrict__ in, uint32_t *__restrict__ out,
                                                         int64_t n, uint32_t *__restrict__ tiles)
{
    __shared__ uint32_t wsum[kThreads / 64], wpre[kThreads / 64];
    const int tid = threadIdx.x;
    const int64_t base = (int64_t)blockIdx.x * kTile + (int64_t)tid * kItems;
    uint32_t v[kItems] = {}, sum = 0, total, before = 0;
    if (base + kItems <= n) {
        const uint4 x = *reinterpret_cast<const uint4 *>(in + base);
        v[0] = x.x, v[1] = x.y, v[2] = x.z, v[3] = x.w;
    } else {
#pragma unroll
        for (int i = 0; i < kItems; ++i) v[i] = base + i < n ? in[base + i] : 0u;
    }
    const bool few = gridDim.x <= kFewTiles;
    if (few) {
        constexpr int kLoads = 16;   // in flight
        uint32_t pre = 0;
        for (int t0 = 0; t0 < (int)blockIdx.x; t0 += kLoads) {
            uint4 x[kLoads];
#pragma unroll
            for (int u = 0; u < kLoads; ++u)
                x[u] = t0 + u < (int)blockIdx.x ? reinterpret_cast<const uint4 *>(in + (int64_t)(t0 + u) * kTile)[tid]
                                                : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
            for (int u = 0; u < kLoads; ++u) pre += x[u].x + x[u].y + x[u].z + x[u].w;
        }
        block_before(pre, wpre, before);
    }
#pragma unroll
    for (int i = 0; i < kItems; ++i) sum += v[i];
    uint32_t run = block_before(sum, wsum, total);
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        if (base + i < n) out[base + i] = run;
        run += v[i];
    }
    if (tid == 0) tiles[blockIdx.x] = few ? before : total;
}

static_assert(kTile == kThreads * 4, "a thread reads 16 bytes of a tile");

constexpr int kSumThreads = 1024;

// The exclusive scan of the tiles' sums in place, by one workgroup, kSumThreads * kItems of them a round.
__global__ __launch_bounds__(kSumThreads) void k_scan_sums(uint32_t *__restrict__ tiles, int64_t n)
{
    __shared__ uint32_t wsum[kSumThreads / 64];
    uint32_t carry = 0;
    for (int64_t t0 = 0; t0 < n; t0 += kSumThreads * kItems) {
        const int64_t base = t0 + (int64_t)threadIdx.x * kItems;
        uint32_t v[kItems], sum = 0, total;
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            v[i] = base + i < n ? tiles[base + i] : 0u;
            sum += v[i];
        }
        uint32_t run = carry + block_before(sum, wsum, total);
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            if (base + i < n) tiles[base + i] = run;
            run += v[i];
        }
        carry += total;
        __syncthreads();   // wsum is rewritten
    }
}

// Bitonic network over sk[0, np2) (np2 a power of two) in LDS by the whole workgroup, ascending.
// Pair t of a stage is (i, i + j) with i = t with a zero bit inserted at bit log2(j).  A thread
// takes pairs t = tid + m*blockDim.x, so for j <= 64 wave w touches only the 128-element blocks
// w + (waves per workgroup)*m: consecutive stages that both have j <= 64 depend on the wave's own
// program order only; a barrier follows every stage where this stage or the next one has j > 64.
// Ends with a workgroup barrier.
__device__ __forceinline__ void block_bitonic(unsigned long long *sk, int np2)
{
    const int tid = threadIdx.x, nt = blockDim.x;
    for (int k = 2; k <= np2; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int t = tid; t < (np2 >> 1); t += nt) {
                const int i = ((t & ~(j - 1)) << 1) | (t & (j - 1));
                const int l = i + j;
                const unsigned long long a = sk[i], b = sk[l];
                const bool up = (i & k) == 0;
                if ((a > b) == up) {
                    sk[i] = b;
                    sk[l] = a;
                }
            }
            const int jn = j > 1 ? (j >> 1) : k;   // the next stage's distance
            if (j > 64 || jn > 64) __syncthreads();
            else __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
    }
    __syncthreads();
}

// ---- fields of at most kLocalSortMax points and kLocalRowsMax rows ----------------------------
// One workgroup per field takes its whole sort stage: the value offset; each point's base cell; the
// rows' counts and starts (absolute: a field's list begins at its first point index, pt_prefix[f], and
// its in-grid points fill the first of its slots); and the points in (cell key, point index) order.
// The points are counted in LDS by buckets, 2^ls column ranges of each row, and dropped into the
// buckets' ranges; when no bucket holds more than kRankMax points each point's place is its bucket's
// start plus the number of the bucket's entries below its own.  Otherwise a bitonic network sorts the
// 64-bit composites in LDS.  Both give the same order.
//
// EXACT: the list is written as FP64 injection records (irec), else as point indices (out_vals),
// with each point's position in rec.  The workgroups after the fields' zero the FP64 grids meanwhile.
//
// Bound by latency, one workgroup's chain of loads, divisions and LDS steps.  kBuckets buckets, as
// many as there may be points, keep the last step short: with one bucket per row (12 to 40 points) it
// took 6 us more.  5001 points on 601x299: zero fill, keys with the offset and sort took 1.9 + 5.5 +
// 15.6 us in launches of their own, this takes 14.8.
//
// THREADS (1024 or 256): a workgroup takes up to 8 points and 8 rows per thread and has as many buckets.
struct FieldSortArgs {
    const FieldDev *fields;
    const int64_t *pt_prefix;
    const double *pts, *val;
    double *offsets;
    uint32_t *row_count, *row_start, *out_vals;
    PointRec *rec;
    InjectRec *irec;
    ZeroRange zero[2];
    int nfields, np2, raw;   // np2: the LDS composites; raw: offset 0
};

constexpr int kSortPerThread = kLocalSortMax / kLocalSortThreads;   // points, rows and buckets per thread
static_assert(kLocalRowsMax <= kLocalSortMax, "a row has at least one bucket");
constexpr int kRankMax = 64;                                        // largest bucket placed by rank
constexpr int kSortZeroPer = 8;   // 16-byte stores of a zeroing thread
constexpr int kRankStep = 4;      // LDS reads in flight of a rank; sk has as many entries to spare

template <int DIM, bool EXACT, int THREADS>
__global__ __launch_bounds__(THREADS) void k_field_sort(FieldSortArgs A)
{
    constexpr int kBuckets = kSortPerThread * THREADS, kBucketsPerThread = kSortPerThread;
    constexpr int kSortWaves = THREADS / 64;
    extern __shared__ __align__(16) unsigned char smem[];   // composites
    __shared__ __align__(16) uint32_t start[kBuckets + 4];  // the buckets' counts, then their starts
    __shared__ uint32_t wsum[kSortWaves], wmax[kSortWaves];
    __shared__ double dmin[kSortWaves], dmax[kSortWaves];
    __shared__ int dnan[kSortWaves];
    if ((int64_t)blockIdx.x >= A.nfields) {
        int64_t b = (int64_t)blockIdx.x - A.nfields;
        if (!zero_block<THREADS, kSortZeroPer>(A.zero[0], b))
            zero_block<THREADS, kSortZeroPer>(A.zero[1], b);
        return;
    }
    const int f = blockIdx.x, tid = threadIdx.x, wv = tid >> 6;
    FieldDev F = A.fields[f];   // by value: the stores below cannot change it
    F.dim = DIM;
    const int64_t p0 = A.pt_prefix[f];
    const int n = (int)(A.pt_prefix[f + 1] - p0);
    const int nr = (int)(F.size[1] * F.size[2]);   // x-lines (rows) of the field
    const uint32_t dst = (uint32_t)p0;
    unsigned long long *const sk = reinterpret_cast<unsigned long long *>(smem);
    // bucket = row << ls | column range; the range ascends with the column
    int ls = 0;
    while (nr << (ls + 1) <= kBuckets) ++ls;
    const float bscale = (float)(1 << ls) / (float)F.size[0];

    uint4 *const quads = reinterpret_cast<uint4 *>(start);
    double mn = INFINITY, mx = -INFINITY;
    int isn = 0;
    int xi[kSortPerThread];            // base column, -1 outside the grid
    uint32_t bs[kSortPerThread];       // bucket, slot in it << 16
    double v[kSortPerThread], w[EXACT ? kSortPerThread : 1][DIM];
    // coordinates and values of kGroup points in flight together (as many as there are registers for)
    constexpr int kGroup = EXACT && DIM >= 3 ? kSortPerThread / 4 : kSortPerThread;
#pragma unroll
    for (int g = 0; g < kSortPerThread; g += kGroup) {
        double c[kGroup][DIM];
#pragma unroll
        for (int u = 0; u < kGroup; ++u) {
            const int i = tid + (g + u) * THREADS;
            if (i < n) {
                v[g + u] = A.val[p0 + i];
#pragma unroll
                for (int m = 0; m < DIM; ++m) c[u][m] = A.pts[(p0 + i) * DIM + m];
            }
        }
        if (g == 0) {
#pragma unroll
            for (int q = 0; q < kBucketsPerThread / 4; ++q)
                quads[tid + q * THREADS] = make_uint4(0u, 0u, 0u, 0u);
            __syncthreads();
        }
#pragma unroll
        for (int u = 0; u < kGroup; ++u) {
            const int k = g + u, i = tid + k * THREADS;
            xi[k] = -1;
            if (i < n) {
                if (v[k] != v[k]) isn = 1;
                mn = fmin(mn, v[k]);
                mx = fmax(mx, v[k]);
                PointPos pp;
                if (point_pos(F, c[u], pp)) {
                    const int row = (int)(DIM >= 3 ? pp.i[2] * F.size[1] + pp.i[1] : pp.i[1]);
                    xi[k] = (int)pp.i[0];
                    const uint32_t b = (uint32_t)row << ls | min((uint32_t)((float)xi[k] * bscale), (1u << ls) - 1u);
                    bs[k] = b | atomicAdd(&start[b], 1u) << 16;
                    if constexpr (EXACT) {
#pragma unroll
                        for (int m = 0; m < DIM; ++m) w[k][m] = pp.w[m];
                    } else {
                        A.rec[p0 + i] = PointRec{{pp.w[0], pp.w[1], DIM >= 3 ? pp.w[2] : v[k]}, xi[k], 0};
                    }
                }
            }
        }
    }
    minmax_wave(mn, mx, isn);
    if ((tid & 63) == 0) {
        dmin[wv] = mn;
        dmax[wv] = mx;
        dnan[wv] = isn;
    }
    __syncthreads();

    // the buckets' starts (consecutive buckets per thread) and the largest bucket
    uint32_t rc[kBucketsPerThread], sum = 0, big = 0, total;
#pragma unroll
    for (int q = 0; q < kBucketsPerThread; q += 4) {
        const uint4 x = quads[tid * (kBucketsPerThread / 4) + q / 4];
        rc[q] = x.x, rc[q + 1] = x.y, rc[q + 2] = x.z, rc[q + 3] = x.w;
    }
#pragma unroll
    for (int q = 0; q < kBucketsPerThread; ++q) {
        sum += rc[q];
        big = max(big, rc[q]);
    }
    for (int d = 32; d >= 1; d >>= 1) big = max(big, (uint32_t)__shfl_xor((int)big, d));
    if ((tid & 63) == 0) wmax[wv] = big;
    uint32_t run = block_before(sum, wsum, total);
#pragma unroll
    for (int q = 0; q < kBucketsPerThread; ++q) {
        const uint32_t x = rc[q];
        rc[q] = run;
        run += x;
    }
#pragma unroll
    for (int q = 0; q < kBucketsPerThread; q += 4)
        quads[tid * (kBucketsPerThread / 4) + q / 4] = make_uint4(rc[q], rc[q + 1], rc[q + 2], rc[q + 3]);
    if (tid == THREADS - 1) start[kBuckets] = run;
#pragma unroll
    for (int q = 0; q < kSortWaves; ++q) {
        big = max(big, wmax[q]);
        mn = fmin(mn, dmin[q]);
        mx = fmax(mx, dmax[q]);
        isn |= dnan[q];
    }
    const double off = A.raw ? 0.0 : field_offset(mn, mx, isn);
    if (tid == 0) A.offsets[f] = off;
    __syncthreads();
    for (int r = tid; r < nr; r += THREADS) {
        const uint32_t s0 = start[r << ls];
        A.row_start[F.xline_off + r] = dst + s0;
        A.row_count[F.xline_off + r] = start[(r + 1) << ls] - s0;
    }
    if constexpr (EXACT)
        for (int i = (int)total + tid; i < n; i += THREADS) A.irec[dst + i].row = kInvalidKey;

    if (big <= (uint32_t)kRankMax) {
#pragma unroll
        for (int k = 0; k < kSortPerThread; ++k)
            if (xi[k] >= 0)
                sk[start[bs[k] & 0xffffu] + (bs[k] >> 16)] =
                    ((unsigned long long)(uint32_t)xi[k] << 32) | (uint32_t)(p0 + tid + k * THREADS);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kSortPerThread; ++k) {
            if (xi[k] < 0) continue;
            const uint32_t p = (uint32_t)(p0 + tid + k * THREADS);
            const unsigned long long e = ((unsigned long long)(uint32_t)xi[k] << 32) | p;
            const uint32_t b = bs[k] & 0xffffu, s0 = start[b], s1 = start[b + 1];
            uint32_t at = s0;
            for (uint32_t j = s0; j < s1; j += kRankStep) {
                unsigned long long x[kRankStep];
#pragma unroll
                for (int u = 0; u < kRankStep; ++u) x[u] = sk[j + u];
#pragma unroll
                for (int u = 0; u < kRankStep; ++u) at += j + u < s1 && x[u] < e ? 1u : 0u;
            }
            if constexpr (EXACT) {
                // (three axes leave no registers for the values)
                InjectRec R{xi[k], p, (uint32_t)(F.xline_off + (b >> ls)), f, 0.0, 0.0, 0.0,
                            (DIM >= 3 ? A.val[p] : v[k]) - off};
                R.wx = w[k][0];
                if constexpr (DIM >= 2) R.wy = w[k][1];
                if constexpr (DIM >= 3) R.wz = w[k][2];
                A.irec[dst + at] = R;
            } else {
                A.out_vals[dst + at] = p;
            }
        }
        return;
    }

    const uint32_t W = (uint32_t)F.size[0];
    for (int i = n + tid; i < A.np2; i += THREADS) sk[i] = ~0ull;
#pragma unroll
    for (int k = 0; k < kSortPerThread; ++k) {
        const int i = tid + k * THREADS;
        if (i < n)
            sk[i] = xi[k] < 0 ? ~0ull
                              : ((unsigned long long)(((bs[k] & 0xffffu) >> ls) * W + (uint32_t)xi[k]) << 32) |
                                    (uint32_t)(p0 + i);
    }
    __syncthreads();
    block_bitonic(sk, A.np2);
    for (int i = tid; i < (int)total; i += THREADS) {
        const uint32_t p = (uint32_t)sk[i];
        if constexpr (EXACT) {
            PointPos pp;
            point_pos(F, A.pts + (int64_t)p * DIM, pp);
            A.irec[dst + i] = InjectRec{(int)pp.i[0], p, (uint32_t)(F.xline_off + pp.i[2] * F.size[1] + pp.i[1]), f,
                                        pp.w[0], pp.w[1], pp.w[2], A.val[p] - off};
        } else {
            A.out_vals[dst + i] = p;
        }
    }
}

// ---- row buckets (all other plans) ------------------------------------------------------------
// The order of a stable sort of the (cell key, point index) pairs: every in-grid point
// has a slot in its base row (k_point_keys' atomic count), the rows start at the exclusive scan
// of the counts, and each row's entries are then sorted by the composite (key, point index).

constexpr int kRowSmall = 16;      // rows of at most this many entries: one thread, in registers
constexpr int kRowWave = 512;      // rows of at most this many entries: one wave, in LDS ...
constexpr int kRankWave = 256;     // ... by rank up to this many, by a bitonic network above
constexpr int kRowThreads = 1024;  // workgroup of the row sorts: 16 waves share kLocalSortMax composites
constexpr int kRowGrid = 512;      // ... and their number, at most

__global__ __launch_bounds__(kThreads) void k_row_scatter(const FieldDev *__restrict__ fields,
                                                          const int64_t *__restrict__ pt_prefix, int nfields, int64_t n,
                                                          const uint32_t *__restrict__ keys,
                                                          const uint32_t *__restrict__ slot,
                                                          const uint32_t *__restrict__ row_start,
                                                          const uint32_t *__restrict__ tiles,
                                                          unsigned long long *__restrict__ comp)
{
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const uint32_t key = keys[i], sl = slot[i];
    if (key == kInvalidKey) return;   // outside its grid
    const FieldDev &F = fields[find_seg(pt_prefix, nfields, i)];
    const int64_t r = F.xline_off + (key - (uint32_t)F.cell_off) / (uint32_t)F.size[0];
    comp[row_start[r] + tiles[r / kTile] + sl] = ((unsigned long long)key << 32) | (unsigned long long)(uint32_t)i;
}

// One thread sorts a row of n <= M entries by a bitonic network in registers (padded with the
// largest composite).
template <int M>
__device__ __forceinline__ void small_row(const unsigned long long *__restrict__ comp, uint32_t *__restrict__ list,
                                          uint32_t s0, uint32_t n)
{
    unsigned long long e[M];
#pragma unroll
    for (int q = 0; q < M; ++q) e[q] = (uint32_t)q < n ? comp[s0 + q] : ~0ull;
#pragma unroll
    for (int k = 2; k <= M; k <<= 1)
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1)
#pragma unroll
            for (int i = 0; i < M; ++i) {
                const int l = i ^ j;
                if (l > i) {
                    const bool up = (i & k) == 0;
                    const unsigned long long a = e[i], b = e[l];
                    if ((a > b) == up) {
                        e[i] = b;
                        e[l] = a;
                    }
                }
            }
#pragma unroll
    for (int q = 0; q < M; ++q)
        if ((uint32_t)q < n) list[s0 + q] = (uint32_t)e[q];
}

// One wave sorts the row of n <= 64*NU entries at s0 by rank: each entry's slot is the number of
// the row's composites below it (all differ), counted against the row's copy in LDS `sk`, two
// composites per read (every lane reads the same pair at a time: broadcast reads; an odd row
// is padded with ~0, which no composite exceeds).  NU = ceil(n/64) keeps the compares to the
// registers that hold entries.
template <int NU>
__device__ __forceinline__ void rank_row(const unsigned long long *__restrict__ comp, uint32_t *__restrict__ list,
                                         uint32_t s0, uint32_t n, unsigned long long *__restrict__ sk, int lane)
{
    unsigned long long e[NU];
    uint32_t rk[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        const uint32_t i = lane + 64 * u;
        e[u] = i < n ? comp[s0 + i] : ~0ull;
        if (i < n) sk[i] = e[u];
        rk[u] = 0u;
    }
    if (lane == 0 && (n & 1u)) sk[n] = ~0ull;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const ulonglong2 *sk2 = reinterpret_cast<const ulonglong2 *>(sk);
#pragma unroll 4
    for (uint32_t j = 0; j < (n + 1) >> 1; ++j) {
        const ulonglong2 x = sk2[j];
#pragma unroll
        for (int u = 0; u < NU; ++u) rk[u] += (x.x < e[u] ? 1u : 0u) + (x.y < e[u] ? 1u : 0u);
    }
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        if (lane + 64 * u < (int)n) list[s0 + rk[u]] = (uint32_t)e[u];
    }
}

// The rows of workgroup b are the groups b, b + gridDim.x, ... of 1 << shift rows: neighbouring rows, which tend
// to be of a size, go to different workgroups, one by one while a workgroup's threads take all of its rows at
// once, else 16 by 16, so that a wave reads whole 64-byte pieces of the counts and starts (2 million rows
// 40 -> 13 us).  A thread completes its row's start and sorts it if it is
// small; the workgroup's waves then take its rows of up to kRowWave entries, each wave in its own
// slice of the LDS, by rank or by the bitonic network (within one wave every step only needs its LDS
// operations complete: a wavefront fence, never a barrier); then the whole workgroup its larger rows:
// up to kLocalSortMax entries by the bitonic network in LDS, more by rank (each entry counts the row's
// smaller composites; all composites differ).
//
// Bound by latency: each row a load, its sort and a store.  One launch instead of three (a global list
// of rows for each kind) and the composites in one 64-bit array instead of two of 32: 16 fields of
// 2400x1200 (19200 rows, 1.6 million points), scatter 25 + sorts 40 us, now 21 + 32; 65536 rows of 3 points
// 7.1 + 14.3 us, now 6.2 + 9.0.  Of 512 threads with slices of 1024 composites it took 41 and 8.9.
__global__ __launch_bounds__(kRowThreads) void k_row_sort(int64_t nrows, int shift,
                                                          const uint32_t *__restrict__ row_count,
                                                          uint32_t *__restrict__ row_start,
                                                          const uint32_t *__restrict__ tiles,
                                                          const unsigned long long *__restrict__ comp,
                                                          uint32_t *__restrict__ list)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ uint32_t s_n[kRowThreads], s_at[kRowThreads];   // rows for a wave from the front, larger ones from the end
    __shared__ uint32_t s_count[2];
    unsigned long long *const skb = reinterpret_cast<unsigned long long *>(smem);
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    unsigned long long *const sk = skb + wv * kRowWave;
    for (int64_t q0 = 0; q0 * gridDim.x < nrows; q0 += kRowThreads) {
        const int64_t q = q0 + tid;
        const int64_t r = ((blockIdx.x + (q >> shift) * gridDim.x) << shift) + (q & ((1 << shift) - 1));
        if (tid < 2) s_count[tid] = 0u;
        __syncthreads();
        uint32_t n = 0, s0 = 0;
        if (r < nrows) {
            n = row_count[r];
            s0 = row_start[r] + tiles[r / kTile];
            row_start[r] = s0;
        }
        if (n > (uint32_t)kRowSmall) {
            const bool big = n > (uint32_t)kRowWave;
            const uint32_t k = atomicAdd(&s_count[big], 1u), at = big ? kRowThreads - 1 - k : k;
            s_n[at] = n;
            s_at[at] = s0;
            n = 0;
        }
        if (__any(n > 8)) small_row<16>(comp, list, s0, n);
        else if (__any(n > 4)) small_row<8>(comp, list, s0, n);
        else if (__any(n > 2)) small_row<4>(comp, list, s0, n);
        else if (__any(n > 0)) small_row<2>(comp, list, s0, n);
        __syncthreads();
        const int nwave = s_count[0], nbig = s_count[1];
        for (int b = wv; b < nwave; b += kRowThreads / 64) {
            const uint32_t m = s_n[b], a = s_at[b];
            if (m <= (uint32_t)kRankWave) {
                switch ((m + 63) >> 6) {
                case 1: rank_row<1>(comp, list, a, m, sk, lane); break;
                case 2: rank_row<2>(comp, list, a, m, sk, lane); break;
                case 3: rank_row<3>(comp, list, a, m, sk, lane); break;
                default: rank_row<kRankWave / 64>(comp, list, a, m, sk, lane); break;
                }
            } else {
                int np2 = 1;
                while ((uint32_t)np2 < m) np2 <<= 1;
                for (int i = lane; i < np2; i += 64) sk[i] = (uint32_t)i < m ? comp[a + i] : ~0ull;
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                for (int k = 2; k <= np2; k <<= 1)
                    for (int j = k >> 1; j > 0; j >>= 1) {
                        for (int t = lane; t < (np2 >> 1); t += 64) {
                            const int i = ((t & ~(j - 1)) << 1) | (t & (j - 1));
                            const int l = i + j;
                            const unsigned long long x = sk[i], y = sk[l];
                            const bool up = (i & k) == 0;
                            if ((x > y) == up) {
                                sk[i] = y;
                                sk[l] = x;
                            }
                        }
                        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                    }
                for (int i = lane; (uint32_t)i < m; i += 64) list[a + i] = (uint32_t)sk[i];
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");   // before the next row reuses sk
        }
        for (int b = 0; b < nbig; ++b) {
            const uint32_t m = s_n[kRowThreads - 1 - b], a = s_at[kRowThreads - 1 - b];
            __syncthreads();   // the LDS is free
            if (m <= (uint32_t)kLocalSortMax) {
                int np2 = 1;
                while ((uint32_t)np2 < m) np2 <<= 1;
                for (int i = tid; i < np2; i += kRowThreads) skb[i] = (uint32_t)i < m ? comp[a + i] : ~0ull;
                __syncthreads();
                block_bitonic(skb, np2);
                for (int i = tid; (uint32_t)i < m; i += kRowThreads) list[a + i] = (uint32_t)skb[i];
            } else {
                for (uint32_t i = tid; i < m; i += kRowThreads) {
                    const unsigned long long e = comp[a + i];
                    uint32_t rank = 0;
                    for (uint32_t j = 0; j < m; ++j) rank += comp[a + j] < e;
                    list[a + rank] = (uint32_t)e;
                }
            }
        }
        __syncthreads();   // the lists and the LDS are reused
    }
}

}  // namespace

int64_t scan_tiles(int64_t n) { return n > 0 ? cdiv(n, kTile) : 1; }

int row_bucket_sort(const FieldDev *d_fields, const int64_t *d_pt_prefix, int nfields, const uint32_t *d_keys,
                    const uint32_t *d_slot, int64_t npoints, uint32_t *d_row_start, const uint32_t *d_row_count,
                    int64_t nrows, uint32_t *d_tiles, unsigned long long *d_comp, uint32_t *d_list, hipStream_t stream)
{
    if (nrows <= 0) return FB_OK;
    hipLaunchKernelGGL(k_scan_tiles, dim3((unsigned)scan_tiles(nrows)), dim3(kThreads), 0, stream, d_row_count,
                       d_row_start, nrows, d_tiles);
    FB_HIP_CHECK(hipGetLastError());
    if (scan_tiles(nrows) > kFewTiles) {
        hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(kSumThreads), 0, stream, d_tiles, scan_tiles(nrows));
        FB_HIP_CHECK(hipGetLastError());
    }
    if (npoints > 0) {
        hipLaunchKernelGGL(k_row_scatter, dim3((unsigned)cdiv(npoints, kThreads)), dim3(kThreads), 0, stream, d_fields,
                           d_pt_prefix, nfields, npoints, d_keys, d_slot, (const uint32_t *)d_row_start,
                           (const uint32_t *)d_tiles, d_comp);
        FB_HIP_CHECK(hipGetLastError());
    }
    const int shift = nrows > (int64_t)kRowGrid * kRowThreads ? 4 : 0;
    hipLaunchKernelGGL(k_row_sort, dim3((unsigned)std::min<int64_t>(nrows, kRowGrid)), dim3(kRowThreads),
                       (size_t)kLocalSortMax * sizeof(unsigned long long), stream, nrows, shift, d_row_count, d_row_start,
                       (const uint32_t *)d_tiles, (const unsigned long long *)d_comp, d_list);
    FB_HIP_CHECK(hipGetLastError());
    return FB_OK;
}

int field_sort_init()
{
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [] {
        const int lds = (kLocalSortMax + kRankStep) * (int)sizeof(unsigned long long);
        constexpr int T = kLocalSortThreads;   // (the smaller workgroups' LDS needs no raised limit)
        const void *fns[] = {(const void *)k_field_sort<1, false, T>, (const void *)k_field_sort<2, false, T>,
                             (const void *)k_field_sort<3, false, T>, (const void *)k_field_sort<1, true, T>,
                             (const void *)k_field_sort<2, true, T>,  (const void *)k_field_sort<3, true, T>,
                             (const void *)k_row_sort};
        for (const void *fn : fns)
            if (err == hipSuccess) err = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    });
    if (err != hipSuccess) {
        (void)hipGetLastError();
        set_error(std::string("hipFuncSetAttribute failed: ") + hipGetErrorString(err));
        return FB_ERR_HIP;
    }
    return FB_OK;
}

int launch_field_sort(const FieldDev *d_fields, const int64_t *d_pt_prefix, int nfields, int dim, int max_n,
                      int max_rows, const double *d_pts, const double *d_val, bool raw, double *d_offsets,
                      uint32_t *d_row_count, uint32_t *d_row_start, uint32_t *d_out_vals, PointRec *d_rec,
                      InjectRec *d_irec, const ZeroRange (&zero)[2], hipStream_t stream)
{
    if (nfields <= 0) return FB_OK;
    if (max_n > kLocalSortMax || max_rows > kLocalRowsMax) {
        set_error("field sort: a field has more than " + std::to_string(kLocalSortMax) + " points or " +
                  std::to_string(kLocalRowsMax) + " x-lines");
        return FB_ERR_UNSUPPORTED;
    }
    int np2 = 1;
    while (np2 < max_n) np2 <<= 1;
    FieldSortArgs A{d_fields,   d_pt_prefix, d_pts, d_val,  d_offsets,          d_row_count, d_row_start,
                    d_out_vals, d_rec,       d_irec, {zero[0], zero[1]}, nfields, np2, raw ? 1 : 0};
    const size_t lds = (size_t)(np2 + kRankStep) * 8;
    auto launch = [&](auto kernel, int threads, int64_t zero_wgs) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)(nfields + zero_wgs)), dim3(threads), lds, stream, A);
    };
    auto run = [&](auto threads) {
        constexpr int T = decltype(threads)::value;
        int64_t zero_wgs = 0;
        for (const ZeroRange &z : zero) zero_wgs += zero_blocks<T, kSortZeroPer>(z);
        if (d_irec) {
            if (dim == 1) launch(k_field_sort<1, true, T>, T, zero_wgs);
            else if (dim == 2) launch(k_field_sort<2, true, T>, T, zero_wgs);
            else launch(k_field_sort<3, true, T>, T, zero_wgs);
        } else {
            if (dim == 1) launch(k_field_sort<1, false, T>, T, zero_wgs);
            else if (dim == 2) launch(k_field_sort<2, false, T>, T, zero_wgs);
            else launch(k_field_sort<3, false, T>, T, zero_wgs);
        }
    };
    // One workgroup of 1024 threads runs on a CU at a time.  Where there are more fields than CUs, small ones
    // take 256 threads each: 2000 fields of 50 points on 30x20 nodes 47.8 -> 14.3 us (zero fill, keys and sort
    // in launches of their own took 31.5), 300 fields of 2000 points 24.8 -> 20.0.  Fewer fields gain a tenth
    // by it, but points crowded into few buckets, for the bitonic network, lose: one field of 406 12.5 -> 17.8.
    constexpr int kSmall = 256;
    if (nfields > 256 && max_n <= kSmall * kSortPerThread && max_rows <= kSmall * kSortPerThread)
        run(std::integral_constant<int, kSmall>());
    else
        run(std::integral_constant<int, kLocalSortThreads>());
    FB_HIP_CHECK(hipGetLastError());
    return FB_OK;
}

}  // namespace fb
