// fb_kernels.hip -- device kernels of fast Barnes interpolation on gfx950.
//
// Pipeline of one batch (every stage covers all fields of the batch):
//   sort stage      value offset (min+max)/2 per field           interpolation.py:204-212
//                   and the points in (base cell, point index) order, interpolation.py:218-322: fields of
//                   few points in one launch (k_field_sort, fb_sort.hip); larger ones k_sort_begin,
//                   k_point_keys (cells and row counts), then the row buckets of fb_sort.hip
//   FP64 path:      k_inject_cells, k_exact_stream (fb_lines.hip) along each axis, the last one
//                   with the quotient -- the reference's operation order; k_exact_lines (one
//                   thread per line) and k_exact_finalize for kernels too wide for the LDS and
//                   for short columns of large grids
//   FP32C path:     k_fast_pass<inject> along x, k_fast_pass along y (and z);
//                   quotient, offset and NaN mask fused into the last pass
#include <algorithm>
#include <climits>
#include <cmath>
#include <mutex>
#include <string>

#include "fb_launch.h"
#include "fb_points.h"

namespace fb {

namespace {

constexpr int kBlock = 256;

// ---------------------------------------------------------------------------
// value offsets: (min + max)/2 over all values of a field, NaN if any value is NaN
// (numpy's amin/amax propagate NaN), interpolation.py:209.  The smallest, the largest and the NaN
// flag do not depend on the order of the reduction.

// (min, max, NaN flag) of the workgroup's threads, valid in thread 0
__device__ __forceinline__ void minmax_block(double &mn, double &mx, int &isn)
{
    __shared__ double smin[kBlock / 64], smax[kBlock / 64];
    __shared__ int snan[kBlock / 64];
    minmax_wave(mn, mx, isn);
    if ((threadIdx.x & 63) == 0) {
        smin[threadIdx.x >> 6] = mn;
        smax[threadIdx.x >> 6] = mx;
        snan[threadIdx.x >> 6] = isn;
    }
    __syncthreads();
    for (int w = 0; w < kBlock / 64; ++w) {
        mn = fmin(mn, smin[w]);
        mx = fmax(mx, smax[w]);
        isn |= snan[w];
    }
}

__global__ __launch_bounds__(kBlock) void k_offsets(const FieldDev *__restrict__ fields,
                                                    const double *__restrict__ val, double *__restrict__ offsets)
{
    const FieldDev &F = fields[blockIdx.x];
    double mn = INFINITY, mx = -INFINITY;
    int isn = 0;
    minmax_range(val + F.pt_off, threadIdx.x, F.n, kBlock, mn, mx, isn);
    minmax_block(mn, mx, isn);
    if (threadIdx.x == 0) offsets[blockIdx.x] = field_offset(mn, mx, isn);
}

// The same over many workgroups per field (large fields): each reduces one chunk of kOffChunk values
// to (min, max, NaN flag); offsets_final combines a field's chunks.  The chunks of field f begin at
// workgroup pt_off / kOffChunk + f: at least as many as it has, and at most one more, so that one
// large field among many small ones costs its own chunks only (4 million points beside 2000 fields of
// 100, as many workgroups for each field as for the largest: sort stage 4.6 ms, now 0.37).
constexpr int kOffChunk = 2048;     // values of a chunk
constexpr int kOffSingle = 8192;    // fields of up to this many values: one workgroup each

__host__ __device__ inline int64_t first_chunk(int64_t pt_off, int64_t f) { return pt_off / kOffChunk + f; }

__device__ __forceinline__ void offsets_part(const FieldDev *__restrict__ fields, int nfields,
                                             const double *__restrict__ val, double *__restrict__ part, int64_t blk)
{
    int lo = 0, hi = nfields - 1;   // the last field that begins at blk or before
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (first_chunk(fields[mid].pt_off, mid) <= blk) lo = mid; else hi = mid - 1;
    }
    const FieldDev &F = fields[lo];
    const int64_t b0 = (blk - first_chunk(F.pt_off, lo)) * kOffChunk;
    if (b0 >= F.n) return;
    double mn = INFINITY, mx = -INFINITY;
    int isn = 0;
    minmax_range(val + F.pt_off, b0 + threadIdx.x, min(F.n, b0 + kOffChunk), kBlock, mn, mx, isn);
    minmax_block(mn, mx, isn);
    if (threadIdx.x == 0) {
        part[3 * blk] = mn;
        part[3 * blk + 1] = mx;
        part[3 * blk + 2] = isn ? 1.0 : 0.0;
    }
}

// One wave per field.
__device__ __forceinline__ void offsets_final(const FieldDev *__restrict__ fields, int nfields,
                                              const double *__restrict__ part, double *__restrict__ offsets,
                                              int64_t blk)
{
    const int64_t f = blk * (kBlock / 64) + (threadIdx.x >> 6);
    if (f >= nfields) return;
    double mn = INFINITY, mx = -INFINITY;
    int isn = 0;
    const int64_t c0 = first_chunk(fields[f].pt_off, f), c1 = c0 + (fields[f].n + kOffChunk - 1) / kOffChunk;
    for (int64_t c = c0 + (threadIdx.x & 63); c < c1; c += 64) {
        const double *o = part + c * 3;
        mn = fmin(mn, o[0]);
        mx = fmax(mx, o[1]);
        if (o[2] != 0.0) isn = 1;
    }
    minmax_wave(mn, mx, isn);
    if ((threadIdx.x & 63) == 0) offsets[f] = field_offset(mn, mx, isn);
}

__global__ __launch_bounds__(kBlock) void k_offsets_part(const FieldDev *__restrict__ fields, int nfields,
                                                         const double *__restrict__ val, double *__restrict__ part)
{
    offsets_part(fields, nfields, val, part, blockIdx.x);
}

__global__ __launch_bounds__(kBlock) void k_offsets_final(const FieldDev *__restrict__ fields, int nfields,
                                                          const double *__restrict__ part,
                                                          double *__restrict__ offsets)
{
    offsets_final(fields, nfields, part, offsets, blockIdx.x);
}

// The first launch of the row-bucket sort stage: the offsets' chunks (the first noff workgroups) and
// the zero fills, which do not depend on each other: the row counts and the FP64 grids.
constexpr int kZeroPer = 4;   // 16-byte stores of a thread

__global__ __launch_bounds__(kBlock) void k_sort_begin(const FieldDev *__restrict__ fields, int nfields,
                                                       const double *__restrict__ val, double *__restrict__ part,
                                                       int64_t noff, ZeroRange z0, ZeroRange z1, ZeroRange z2)
{
    if (blockIdx.x < noff) {
        offsets_part(fields, nfields, val, part, blockIdx.x);
        return;
    }
    int64_t b = blockIdx.x - noff;
    if (zero_block<kBlock, kZeroPer>(z0, b) || zero_block<kBlock, kZeroPer>(z1, b)) return;
    zero_block<kBlock, kZeroPer>(z2, b);
}

// ---------------------------------------------------------------------------
// bilinear / trilinear corner weight of corner (bx, by, bz), formed left to right as
// in the reference, e.g. (1.0-xw)*(1.0-yw) at interpolation.py:256
__device__ __forceinline__ double corner_weight(int dim, const PointPos &pp, int64_t bx, int64_t by, int64_t bz)
{
    double w = bx ? pp.w[0] : (1.0 - pp.w[0]);
    if (dim >= 2) w = w * (by ? pp.w[1] : (1.0 - pp.w[1]));
    if (dim >= 3) w = w * (bz ? pp.w[2] : (1.0 - pp.w[2]));
    return w;
}

// A point's sort key is its base cell (the grid cell of its lower corner), kInvalidKey for points
// the injection drops.  The corners of a point lie in the base row (x-line) and the rows above it;
// counts per base row (integer atomics) give, after the scan, each row's range in the sorted list,
// and slot is the point's position among its row's points as the atomics handed them out.  The
// workgroups from nkb on take the fields' offsets from their chunks.
__global__ __launch_bounds__(kBlock) void k_point_keys(const FieldDev *__restrict__ fields,
                                                       const int64_t *__restrict__ pt_prefix, int nfields,
                                                       int64_t npoints, const double *__restrict__ pts,
                                                       const double *__restrict__ val,
                                                       uint32_t *__restrict__ keys, uint32_t *__restrict__ row_count,
                                                       uint32_t *__restrict__ slot, PointRec *__restrict__ rec,
                                                       int64_t nkb, const double *__restrict__ part,
                                                       double *__restrict__ offsets)
{
    if (blockIdx.x >= nkb) {
        offsets_final(fields, nfields, part, offsets, blockIdx.x - nkb);
        return;
    }
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= npoints) return;
    const FieldDev &F = fields[find_seg(pt_prefix, nfields, i)];
    PointPos pp;
    if (!point_pos(F, pts + i * F.dim, pp)) {
        keys[i] = kInvalidKey;
        return;
    }
    const int64_t row = pp.i[2] * F.size[1] + pp.i[1];
    keys[i] = (uint32_t)(F.cell_off + row * F.size[0] + pp.i[0]);
    if (rec) rec[i] = PointRec{{pp.w[0], pp.w[1], F.dim >= 3 ? pp.w[2] : val[i]}, (int32_t)pp.i[0], 0};
    slot[i] = atomicAdd(&row_count[F.xline_off + row], 1u);
}

// k_point_keys for large point sets: each workgroup takes ppt*kBlock consecutive points and,
// when the rows of the fields they belong to number at most nbins, counts them per row in
// LDS first; one global atomic per row the workgroup touches then reserves the row's slots for
// all of them (instead of one contended atomic per point), and each point's slot is that base
// plus its rank among the workgroup's points of the row.  The slots come in another order than
// with one atomic per point; the row sort orders every row by (base cell, point index), so the
// sorted list is the same.  Workgroups whose rows do not fit count with one atomic per point.
constexpr int kKeysMaxPpt = 16;     // points per thread, at most
constexpr int kKeysBins = 8192;     // LDS row counters of a workgroup (32 KB) ...
constexpr int kKeysBinsMax = 16384; // ... or, for plans with fields of up to this many rows, 64 KB

__global__ __launch_bounds__(kBlock) void k_point_keys_hist(const FieldDev *__restrict__ fields,
                                                            const int64_t *__restrict__ pt_prefix, int nfields,
                                                            int64_t npoints, int ppt, int nbins,
                                                            const double *__restrict__ pts,
                                                            const double *__restrict__ val,
                                                            uint32_t *__restrict__ keys,
                                                            uint32_t *__restrict__ row_count,
                                                            uint32_t *__restrict__ slot, PointRec *__restrict__ rec,
                                                            int64_t nkb, const double *__restrict__ part,
                                                            double *__restrict__ offsets)
{
    extern __shared__ uint32_t hist[];   // nbins row counters (dynamic LDS)
    if (blockIdx.x >= nkb) {
        offsets_final(fields, nfields, part, offsets, blockIdx.x - nkb);
        return;
    }
    __shared__ int64_t s_rbase;
    __shared__ int s_span;
    const int64_t p0 = (int64_t)blockIdx.x * ppt * kBlock;
    const int64_t p1 = min(p0 + (int64_t)ppt * kBlock, npoints);
    if (threadIdx.x == 0) {
        const FieldDev &A = fields[find_seg(pt_prefix, nfields, p0)];
        const FieldDev &B = fields[find_seg(pt_prefix, nfields, p1 - 1)];
        const int64_t r0 = A.xline_off;
        const int64_t span = B.xline_off + B.size[1] * B.size[2] - r0;
        s_rbase = r0;
        s_span = span <= nbins ? (int)span : -1;
    }
    __syncthreads();
    const int64_t rbase = s_rbase;
    const int span = s_span;
    for (int b = threadIdx.x; b < span; b += kBlock) hist[b] = 0u;
    __syncthreads();
    int rr[kKeysMaxPpt];
    uint32_t lr[kKeysMaxPpt];
    // a thread's points ascend: its field is found once and then advanced, and the field's
    // geometry stays in registers until its points pass into the next field
    int f = p0 + threadIdx.x < p1 ? find_seg(pt_prefix, nfields, p0 + threadIdx.x) : 0;
    int64_t fnext = f + 1 < nfields ? pt_prefix[f + 1] : INT64_MAX;
    const int dim = fields[0].dim;   // the same for every field of a plan
    double gx0[3], gst[3];
    int64_t gsz[3], gcell = 0, gxl = 0;
    auto geometry = [&](int ff) {
        const FieldDev &F = fields[ff];
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            gx0[m] = F.x0[m];
            gst[m] = F.step[m];
            gsz[m] = F.size[m];
        }
        gcell = F.cell_off;
        gxl = F.xline_off;
    };
    geometry(f);
    // kKeysGrp points at a time: their coordinates are loaded first, all in flight together
    constexpr int kKeysGrp = 4;
#pragma unroll
    for (int k0 = 0; k0 < kKeysMaxPpt; k0 += kKeysGrp) {
        double c[kKeysGrp][3];
#pragma unroll
        for (int u = 0; u < kKeysGrp; ++u) {
            const int64_t i = p0 + (int64_t)(k0 + u) * kBlock + threadIdx.x;
            const bool ok = k0 + u < ppt && i < p1;
#pragma unroll
            for (int m = 0; m < 3; ++m) c[u][m] = ok && m < dim ? pts[i * dim + m] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < kKeysGrp; ++u) {
            const int k = k0 + u;
            rr[k] = -1;
            lr[k] = 0u;
            const int64_t i = p0 + (int64_t)k * kBlock + threadIdx.x;
            if (k >= ppt || i >= p1) continue;
            if (i >= fnext) {
                while (i >= fnext) {
                    ++f;
                    fnext = f + 1 < nfields ? pt_prefix[f + 1] : INT64_MAX;
                }
                geometry(f);
            }
            // point_pos on the cached geometry
            bool inside = true;
            int64_t ci[3] = {0, 0, 0};
            double w[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                if (m < dim) {
                    const double cc = (c[u][m] - gx0[m]) / gst[m];
                    if (!(cc >= 0.0) || cc >= (double)(gsz[m] - 1)) inside = false;
                    const int64_t q = inside ? (int64_t)cc : 0;
                    ci[m] = q;
                    w[m] = cc - (double)q;
                }
            }
            if (!inside) {
                keys[i] = kInvalidKey;
                continue;
            }
            const int64_t row = ci[2] * gsz[1] + ci[1];
            keys[i] = (uint32_t)(gcell + row * gsz[0] + ci[0]);
            if (rec) rec[i] = PointRec{{w[0], w[1], dim >= 3 ? w[2] : val[i]}, (int32_t)ci[0], 0};
            const int64_t grow = gxl + row;
            if (span >= 0) {
                rr[k] = (int)(grow - rbase);
                lr[k] = atomicAdd(&hist[rr[k]], 1u);
            } else {
                slot[i] = atomicAdd(&row_count[grow], 1u);
            }
        }
    }
    if (span < 0) return;   // uniform for the workgroup
    __syncthreads();
    // one global atomic per touched row; the LDS counter becomes the row's first slot
    for (int b = threadIdx.x; b < span; b += kBlock) {
        const uint32_t c = hist[b];
        if (c) hist[b] = atomicAdd(&row_count[rbase + b], c);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kKeysMaxPpt; ++k) {
        if (rr[k] < 0) continue;
        const int64_t i = p0 + (int64_t)k * kBlock + threadIdx.x;
        slot[i] = hist[rr[k]] + lr[k];
    }
}

// ---------------------------------------------------------------------------
// FP64 path, reference operation order

// Each sorted entry's injection record, in list order: base column and row, point, field,
// position within the base cell and value minus the offset, as point_pos forms them.  The
// row-bucket sort packs all fields' entries by row; slots past the list's last entry get row
// kInvalidKey.  (k_field_sort writes its fields' records itself.)
__global__ __launch_bounds__(kBlock) void k_inject_records(
    const FieldDev *__restrict__ fields, const int64_t *__restrict__ pt_prefix, int nfields, int64_t npoints,
    int64_t nxlines, const uint32_t *__restrict__ vals, const uint32_t *__restrict__ row_start,
    const uint32_t *__restrict__ row_count, const double *__restrict__ pts, const double *__restrict__ val,
    const double *__restrict__ offsets, InjectRec *__restrict__ irec)
{
    const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e >= npoints) return;
    const int64_t last = nxlines - 1;   // the list's last row
    if (e >= (int64_t)row_start[last] + row_count[last]) {
        irec[e].row = kInvalidKey;
        return;
    }
    const uint32_t p = vals[e];
    const int f = find_seg(pt_prefix, nfields, p);
    const FieldDev &F = fields[f];
    PointPos pp;
    point_pos(F, pts + (int64_t)p * F.dim, pp);
    irec[e] = InjectRec{(int)pp.i[0], p, (uint32_t)(F.xline_off + pp.i[2] * F.size[1] + pp.i[1]), f,
                        pp.w[0], pp.w[1], pp.w[2], val[p] - offsets[f]};
}

// The injection, cell by cell: a grid cell t receives corner s (its bits: x, y, z) of the points of
// base cell t - s, s < 2^DIM, in increasing point index, which is the order of the reference's
// point loop.  One thread per sorted entry and corner: the first entry of a base cell's run takes
// the cell at that corner of it, unless a base cell of a smaller s has points too (then that one's
// thread takes it), finds the runs of the cell's other base cells in their rows by bisection, all
// of them in step, and merges the runs by point index.  The cell's sums start at 0.0 when the grids
// were cleared (ZEROED), else at the grids' values, and are stored once.
//
// Bound by latency: about six reads per bisection, one per contribution, each depending on the one
// before.  A thread per x line that merged the rows' entries took as long as the line had entries:
// 3490 points on 300x150 (23 to a row) 139 us, here 12; on 2400x1200 27 us, here 8; 20000 on
// 151x133x61 73 us, here 17; 24 fields of 3490 on 600x300 99 us, here 16.
template <int DIM, bool ZEROED>
__global__ __launch_bounds__(kBlock) void k_inject_cells(
    const FieldDev *__restrict__ fields, int64_t first, int64_t npoints, const InjectRec *__restrict__ irec,
    const uint32_t *__restrict__ row_start, const uint32_t *__restrict__ row_count, double *__restrict__ vg,
    double *__restrict__ wg)
{
    constexpr int NC = 1 << DIM;
    const int64_t i = (first + blockIdx.x) * kBlock + threadIdx.x;
    const uint32_t e = (uint32_t)(i >> DIM);
    if ((i >> DIM) >= npoints) return;
    const int own = (int)i & (NC - 1);
    const uint32_t row = irec[e].row;
    if (row == kInvalidKey) return;
    const int bx = irec[e].x;
    const FieldDev &F = fields[irec[e].f];
    const uint32_t rs = row_start[row];
    if (e > rs && irec[e - 1].x == bx) return;
    const int64_t H = F.size[1], lrow = (int64_t)row - F.xline_off;
    const int64_t y = DIM >= 3 ? (uint32_t)lrow % (uint32_t)H : lrow;   // a 2D line is its row
    const int64_t z = DIM >= 3 ? (uint32_t)lrow / (uint32_t)H : 0;

    // the sources' rows; source s starts at its first entry of column tx - (s & 1) or beyond
    const int tx = bx + (own & 1);
    uint32_t lo[NC], end[NC];
#pragma unroll
    for (int s = 0; s < NC; ++s) {
        const int dy = ((own >> 1) & 1) - ((s >> 1) & 1), dz = (own >> 2) - (s >> 2);
        lo[s] = end[s] = 0;
        if (tx - (s & 1) >= 0 && y + dy >= 0 && z + dz >= 0) {
            const uint32_t r = (uint32_t)((int64_t)row + dy + dz * H);
            lo[s] = row_start[r];
            end[s] = lo[s] + row_count[r];
        }
    }
    uint32_t hi[NC];
#pragma unroll
    for (int s = 0; s < NC; ++s) {
        hi[s] = end[s];
        if (s == own) lo[s] = hi[s] = e;
    }
    for (bool more = true; more;) {
        more = false;
#pragma unroll
        for (int s = 0; s < NC; ++s) {
            if (lo[s] < hi[s]) {
                const uint32_t mid = (lo[s] + hi[s]) >> 1;
                if (irec[mid].x < tx - (s & 1)) lo[s] = mid + 1;
                else hi[s] = mid;
                more = more || lo[s] < hi[s];
            }
        }
    }
    // the next entry's point of each source, kInvalidKey when the run has ended
    uint32_t head[NC];
#pragma unroll
    for (int s = 0; s < NC; ++s) {
        head[s] = lo[s] < end[s] && irec[lo[s]].x == tx - (s & 1) ? irec[lo[s]].p : kInvalidKey;
        if (s < own && head[s] != kInvalidKey) return;
    }
    const int64_t cell = F.cell_off + tx + (int64_t)F.size[0] * (lrow + ((own >> 1) & 1) + (own >> 2) * H);
    double av = ZEROED ? 0.0 : vg[cell];
    double aw = ZEROED ? 0.0 : wg[cell];
    while (true) {
        int best = 0;
        uint32_t p = head[0], at = lo[0], stop = end[0];
#pragma unroll
        for (int s = 1; s < NC; ++s)
            if (head[s] < p) {
                best = s;
                p = head[s];
                at = lo[s];
                stop = end[s];
            }
        if (p == kInvalidKey) break;
        const InjectRec &r = irec[at];
        const uint32_t nx = at + 1 < stop && irec[at + 1].x == r.x ? irec[at + 1].p : kInvalidKey;
        PointPos pp;
        pp.w[0] = r.wx;
        pp.w[1] = r.wy;
        pp.w[2] = r.wz;
        const double w = corner_weight(DIM, pp, best & 1, (best >> 1) & 1, best >> 2);
        av += w * r.vc;
        aw += w;
#pragma unroll
        for (int s = 0; s < NC; ++s)
            if (s == best) {
                head[s] = nx;
                lo[s] = at + 1;
            }
    }
    vg[cell] = av;
    wg[cell] = aw;
}

// _accumulate_tail_array (interpolation.py:484-533) and _accumulate_array (:729-772)
// on one strided line, ping-ponging between the grid line G and a scratch line S.
constexpr int kExactBlk = 32;  // interior steps of exact_line whose loads are issued together

// UNIT: element stride 1 (rows), known at compile time so that adjacent loads merge
template <bool UNIT>
__device__ void exact_line(double *__restrict__ G, double *__restrict__ S, int64_t L, int64_t st_, int64_t rect_len,
                           int num_iter, int tail, double alpha)
{
    const int64_t st = UNIT ? 1 : st_;
    const int64_t h0 = (rect_len - 1) / 2;
    const int64_t h0_1 = h0 + 1;
    const int64_t h1 = rect_len - h0;
    double *in = G;
    double *h = S;
#define IN(i) in[(i) * st]
#define H_(i) h[(i) * st]
    for (int it = 0; it < num_iter; ++it) {
        double accu = 0.0;
        int64_t k;
        if (tail) {
            for (k = -h0; k < 0; ++k) accu += IN(k + h0);
            for (k = 0; k < h1; ++k) {
                accu += IN(k + h0);
                H_(k) = accu + alpha * IN(k + h0_1);
            }
            // the interior in blocks of kExactBlk steps: the block's input terms are loaded
            // first (they do not depend on accu; `in` and `h` are different arrays), then the
            // steps run in the reference's order, so the memory latency is paid once per block
            for (k = h1; k + kExactBlk <= L - h0_1; k += kExactBlk) {
                double a[kExactBlk], b[kExactBlk + 1];
#pragma unroll
                for (int j = 0; j < kExactBlk; ++j) {
                    a[j] = IN(k + j + h0);
                    b[j] = IN(k + j - h1);
                }
                b[kExactBlk] = IN(k + kExactBlk + h0);   // IN(k + j + h0_1) is a[j + 1]
#pragma unroll
                for (int j = 0; j < kExactBlk; ++j) {
                    const double nxt = j + 1 < kExactBlk ? a[j + 1] : b[kExactBlk];
                    accu += (a[j] - b[j]);
                    H_(k + j) = accu + alpha * (b[j] + nxt);
                }
            }
            for (; k < L - h0_1; ++k) {
                accu += (IN(k + h0) - IN(k - h1));
                H_(k) = accu + alpha * (IN(k - h1) + IN(k + h0_1));
            }
            k = L - h0_1;
            accu += (IN(k + h0) - IN(k - h1));
            H_(k) = accu + alpha * IN(k - h1);
            for (k = L - h0; k < L; ++k) {
                accu -= IN(k - h1);
                H_(k) = accu + alpha * IN(k - h1);
            }
        } else {
            for (k = -h0; k < 0; ++k) accu += IN(k + h0);
            for (k = 0; k < h1; ++k) {
                accu += IN(k + h0);
                H_(k) = accu;
            }
            for (k = h1; k + kExactBlk <= L - h0; k += kExactBlk) {
                double a[kExactBlk], b[kExactBlk];
#pragma unroll
                for (int j = 0; j < kExactBlk; ++j) {
                    a[j] = IN(k + j + h0);
                    b[j] = IN(k + j - h1);
                }
#pragma unroll
                for (int j = 0; j < kExactBlk; ++j) {
                    accu += (a[j] - b[j]);
                    H_(k + j) = accu;
                }
            }
            for (; k < L - h0; ++k) {
                accu += (IN(k + h0) - IN(k - h1));
                H_(k) = accu;
            }
            for (k = L - h0; k < L; ++k) {
                accu -= IN(k - h1);
                H_(k) = accu;
            }
        }
        double *t = in; in = h; h = t;
    }
    if (in != G)
        for (int64_t i = 0; i < L; ++i) G[i * st] = in[i * st];
#undef IN
#undef H_
}

// One wave per workgroup: a field's few thousand line chains then spread over as many CUs as
// they have waves instead of sharing a quarter as many CUs' memory pipelines.
constexpr int kExactLineThreads = 64;

__global__ __launch_bounds__(kExactLineThreads) void k_exact_lines(const FieldDev *__restrict__ fields,
                                                        const int64_t *__restrict__ line_prefix, int nfields,
                                                        int64_t nslots, int axis, int rect_override,
                                                        double *__restrict__ vg, double *__restrict__ wg,
                                                        double *__restrict__ vs, double *__restrict__ ws)
{
    const int64_t g = (int64_t)blockIdx.x * kExactLineThreads + threadIdx.x;
    if (g >= nslots) return;
    const int f = find_seg(line_prefix, nfields, g);
    const FieldDev &F = fields[f];
    const int64_t r = g - line_prefix[f];
    const int which = (int)(r & 1);
    const int64_t l = r >> 1;
    const int64_t W = F.size[0], H = F.size[1], D = F.size[2];
    int64_t L, st, base;
    if (axis == 0) {
        L = W; st = 1; base = l * W;
    } else if (axis == 1) {
        L = H; st = W; base = (l / W) * W * H + (l % W);
    } else {
        L = D; st = W * H; base = l;
    }
    const int64_t rect = rect_override > 0 ? rect_override : 2 * (int64_t)F.T[axis] + 1;
    double *G = (which ? wg : vg) + F.cell_off + base;
    double *S = (which ? ws : vs) + F.cell_off + base;
    if (st == 1) exact_line<true>(G, S, L, st, rect, F.num_iter, F.tail, F.alpha[axis]);
    else exact_line<false>(G, S, L, st, rect, F.num_iter, F.tail, F.alpha[axis]);
}

// wg[wg < thr] = NaN, then (vg/wg + offset).astype(float32): interpolation.py:428-430, :367
__global__ __launch_bounds__(kBlock) void k_exact_finalize(const FieldDev *__restrict__ fields,
                                                           const int64_t *__restrict__ cell_prefix, int nfields,
                                                           int64_t ncells, const double *__restrict__ vg,
                                                           const double *__restrict__ wg,
                                                           const double *__restrict__ offsets, float *__restrict__ out)
{
    const int64_t g = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (g >= ncells) return;
    const int f = find_seg(cell_prefix, nfields, g);
    const FieldDev &F = fields[f];
    const int64_t i = g - F.cell_off;
    if (i >= F.size[0] * F.size[1] * F.size[2]) return;   // alignment gap between fields
    const double w = wg[g];
    const double v = vg[g];
    out[F.out_off + i] = (w < F.thr) ? __builtin_nanf("") : (float)(v / w + offsets[f]);
}

__global__ __launch_bounds__(kBlock) void k_mask(const FieldDev *__restrict__ fields,
                                                 const int64_t *__restrict__ cell_prefix, int nfields, int64_t ncells,
                                                 double *__restrict__ wg, int fast)
{
    const int64_t g = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (g >= ncells) return;
    const FieldDev &F = fields[find_seg(cell_prefix, nfields, g)];
    if (g - F.cell_off >= F.size[0] * F.size[1] * F.size[2]) return;   // alignment gap between fields
    const double thr = fast ? F.thr_fast : F.thr;
    if (wg[g] < thr) wg[g] = __builtin_nan("");
}

// ---------------------------------------------------------------------------
// FP32C path
//
// One workgroup processes `nlines` lines of one field held in LDS as float32,
// with T+1 zeros of padding on both sides of every line (the reference's zero
// padding, interpolation.py:503-523).  A line is split into lpl contiguous
// segments, one per lane; each lane re-anchors its window sum at its segment
// start with a direct (2T+1)-term sum in FP64 and slides it across the segment
// in FP64, so no running sum ever spans more than one segment and no FP32 sum
// is ever formed.  Each iteration is computed into registers (one field at a
// time) and written back in place after a barrier.  The last iteration scales
// by (1/(K+2*alpha))^n and, on the last pass, forms the masked FP64 quotient
// directly from the FP64 window sums of both fields.

// Segment lengths (elements per lane) the fast pass is instantiated for; odd, so the LDS
// lane stride is conflict-free.  The host picks one per pass and line length.
#define FB_FAST_SEGS(X) X(19) X(21) X(23) X(25) X(29) X(33) X(37) X(39) X(41) X(45) X(49)
constexpr int kFastBlock = 512;   // threads of a fast-pass workgroup: 256 per field
constexpr int kBlk = 4;           // add-stream block (LDS loads in flight)

// One iteration of the tailed box filter over the lane's segment starting at s of one
// field's line `lin`.  The subtract stream lin[s-T+j] (j < kSegArr) is read in one burst
// into registers and doubles as the first part of the initial window sum lin[s-T .. s+T];
// the add stream lin[s+T+1+j] is read in blocks of kBlk with one block of lookahead, so
// many LDS loads are in flight.  All kSegArr steps run unconditionally; steps past the
// lane's segment read in-bounds LDS (next line or the tail reserve) and their outputs are
// discarded by stage_store.  Results replace sb[j] (dead after step j: its value lives on
// in p), so the register array doubles as the staging buffer of the in-place update.
//   SCALE: multiply the results by `scale` (last iteration of a pass).
// Masked FP32C quotient v/w + offset of one node (interpolation.py:367, :428-430): a
// float32 reciprocal refined by one Newton step on the quotient (~1 ulp of v/w; w is
// normalised, well inside the float32 range), the offset added in FP64 before the final
// rounding to float32, and w < thr decided exactly as in FP64 through the float32 threshold.
__device__ __forceinline__ float fast_quotient(float vf, float wf, double off, float thr_f)
{
    const float r = __builtin_amdgcn_rcpf(wf);
    float q = vf * r;
    q = fmaf(fmaf(-q, wf, vf), r, q);
    return wf < thr_f ? __builtin_nanf("") : (float)((double)q + off);
}

template <int SEG, bool SCALE>
__device__ __forceinline__ void slide1(const float *__restrict__ lin, int s, int T, double alpha, double scale,
                                       float (&sb)[SEG])
{
    constexpr int kSegArr = SEG;
    constexpr int kNBlk = (SEG + kBlk - 1) / kBlk;   // blocks covering the SEG steps
    const int K = 2 * T + 1;
    const float *subp = lin + s - T;
#pragma unroll
    for (int j = 0; j < kSegArr; ++j) sb[j] = subp[j];
    const float p0 = lin[s - T - 1];
    // window sum: the first min(K, kSegArr) terms are sb[], the rest (K > kSegArr) from LDS,
    // four at a time without per-term conditions (K is the same for the whole workgroup)
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    if (K >= kSegArr) {
        int i = kSegArr;
        for (; i + 4 <= K; i += 4) {
            float x[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) x[u] = subp[i + u];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] += (double)x[u];
        }
        for (; i < K; ++i) v[0] += (double)subp[i];
#pragma unroll
        for (int j = 0; j < kSegArr; ++j) v[j & 3] += (double)sb[j];
    } else {
        // short kernels (2T+1 < kSegArr): direct sum from LDS
        int i = 0;
        for (; i + 4 <= K; i += 4) {
            float x[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) x[u] = subp[i + u];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] += (double)x[u];
        }
        for (; i < K; ++i) v[0] += (double)subp[i];
    }
    double a = (v[0] + v[1]) + (v[2] + v[3]);
    // Each step: output = a + alpha*(left + right tail), then a slides by the entering minus
    // the leaving term, exactly in FP64.  The output rounds a to float32 and adds the tails
    // in float32 (one float32 FMA; a float32 operation costs half an FP64 one): it is stored
    // as float32 anyway, and the tails are a small part of it.  The scaling iteration
    // multiplies by the float32 scale, whose rounding is the same for the v and w fields of
    // an axis and cancels in their quotient.
    float pf = p0;
    const float alpha_f = (float)alpha;
    const float scale_f = (float)scale;
    const float *addp = lin + s + T + 1;
    float cur[kBlk], nxt[kBlk];
#pragma unroll
    for (int u = 0; u < kBlk; ++u) cur[u] = addp[u];
#pragma unroll
    for (int b = 0; b < kNBlk; ++b) {
        if (b + 1 < kNBlk) {
#pragma unroll
            for (int u = 0; u < kBlk; ++u)
                if ((b + 1) * kBlk + u < kSegArr) nxt[u] = addp[(b + 1) * kBlk + u];
        }
#pragma unroll
        for (int u = 0; u < kBlk; ++u) {
            const int j = b * kBlk + u;
            if (j < kSegArr) {
                const float svf = sb[j];
                float r = fmaf(alpha_f, pf + cur[u], (float)a);
                if (SCALE) r *= scale_f;
                pf = svf;
                a += (double)cur[u] - (double)svf;
                // the empty asm pins each float32 result at its step; otherwise the compiler
                // sinks all conversions to the store and keeps kSegArr doubles live
                asm volatile("" : "+v"(r));
                sb[j] = r;
            }
        }
        if (b + 1 < kNBlk) {
#pragma unroll
            for (int u = 0; u < kBlk; ++u) cur[u] = nxt[u];
        }
    }
}

// n: elements of the segment inside the line; full: the line's right padding holds at
// least kSegArr-1 floats, so the whole segment may be stored (the caller re-zeroes the padding)
template <int SEG>
__device__ __forceinline__ void stage_store(float *__restrict__ lin, int s, int n, bool full,
                                            const float (&sb)[SEG])
{
    constexpr int kSegArr = SEG;
    if (full || n == kSegArr) {
#pragma unroll
        for (int j = 0; j < kSegArr; ++j) lin[s + j] = sb[j];
    } else {
#pragma unroll
        for (int j = 0; j < kSegArr; ++j)
            if (j < n) lin[s + j] = sb[j];
    }
}

// Four floats that this pass reads once, from a line that no other workgroup reads: nontemporal.
__device__ __forceinline__ float4 load_once(const float *p)
{
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    const f32x4 x = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(p));
    return make_float4(x.x, x.y, x.z, x.w);
}

__device__ __forceinline__ bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

// global tile <-> LDS.  Tile: nl lines of length L; element (l, j) at g[l*ls + j*es] maps
// to lds[l*lstride + j].  Either ls == 1 (columns: rows of nl contiguous floats) or es == 1
// (rows of L contiguous floats); float4 global accesses when the layout allows.  All
// threads of the workgroup take part.  Pointers advance by increments (no 64-bit index
// products per element).  A store takes the value of each LDS element through `src`: the
// element itself, or the masked quotient of the v element and the w element `wdiff` floats
// after it (the last pass's result, formed on the way out).
struct LdsValue {
    __device__ __forceinline__ float operator()(const float *d) const { return *d; }
};
struct LdsQuotient {
    int wdiff;
    double off;
    float thr_f;
    __device__ __forceinline__ float operator()(const float *d) const { return fast_quotient(d[0], d[wdiff], off, thr_f); }
};

template <bool LOAD, class SRC = LdsValue>
__device__ __forceinline__ void tile_copy(float *__restrict__ g, int64_t ls, int64_t es, int nl, int L,
                                          float *__restrict__ lds, int lstride, SRC src = SRC())
{
    const int tid = threadIdx.x, nthr = blockDim.x;
    if (ls == 1) {
        if ((nl & 3) == 0 && (es & 3) == 0 && aligned16(g)) {
            const int nq = nl >> 2;
            const int rstep = nthr / nq;
            const int q = tid % nq;
            const int r0 = tid / nq;
            if (r0 < rstep) {
                float *gp = g + (int64_t)r0 * es + 4 * q;
                const int64_t gstep = (int64_t)rstep * es;
                float *d = lds + (4 * q) * lstride + r0;
#pragma unroll 4
                for (int r = r0; r < L; r += rstep, gp += gstep, d += rstep) {
                    if (LOAD) {
                        const float4 x = *reinterpret_cast<const float4 *>(gp);
                        d[0] = x.x;
                        d[lstride] = x.y;
                        d[2 * lstride] = x.z;
                        d[3 * lstride] = x.w;
                    } else {
                        *reinterpret_cast<float4 *>(gp) =
                            make_float4(src(d), src(d + lstride), src(d + 2 * lstride), src(d + 3 * lstride));
                    }
                }
            }
        } else {
            const int rstep = nthr / nl;
            const int l = tid % nl;
            const int r0 = tid / nl;
            if (r0 < rstep) {
                float *gp = g + (int64_t)r0 * es + l;
                const int64_t gstep = (int64_t)rstep * es;
                float *d = lds + l * lstride + r0;
#pragma unroll 4
                for (int r = r0; r < L; r += rstep, gp += gstep, d += rstep) {
                    if (LOAD) *d = *gp;
                    else *gp = src(d);
                }
            }
        }
    } else {
        if ((L & 3) == 0 && (ls & 3) == 0 && aligned16(g)) {
            const int Lq = L >> 2;
            for (int l = 0; l < nl; ++l) {
                float4 *gp = reinterpret_cast<float4 *>(g + l * ls) + tid;
                float4 *d = reinterpret_cast<float4 *>(lds + l * lstride) + tid;
#pragma unroll 4
                for (int q = tid; q < Lq; q += nthr, gp += nthr, d += nthr) {
                    // LDS rows start at pad offsets: float4 LDS access only when 16-byte aligned
                    float *dd = reinterpret_cast<float *>(d);
                    if (LOAD) {
                        const float4 x = *gp;
                        dd[0] = x.x;
                        dd[1] = x.y;
                        dd[2] = x.z;
                        dd[3] = x.w;
                    } else {
                        *gp = make_float4(src(dd), src(dd + 1), src(dd + 2), src(dd + 3));
                    }
                }
            }
        } else {
            for (int l = 0; l < nl; ++l) {
                float *gp = g + l * ls + (int64_t)tid * es;
                const int64_t gstep = (int64_t)nthr * es;
                float *d = lds + l * lstride + tid;
#pragma unroll 4
                for (int j = tid; j < L; j += nthr, gp += gstep, d += nthr) {
                    if (LOAD) *d = *gp;
                    else *gp = src(d);
                }
            }
        }
    }
}

// Columns of a width that float4 cannot take (tile_copy's scalar columns), both fields' elements of
// kColRows rows per thread in flight together: the y pass of 96 uneven fields, half of them of odd
// widths, 812 -> 772 us against four rows of one field at a time.
constexpr int kColRows = 8;

__device__ __forceinline__ void load_columns(const float *__restrict__ gv, const float *__restrict__ gw, int64_t es,
                                             int nl, int L, float *__restrict__ dv, float *__restrict__ dw, int lstride)
{
    const int rstep = blockDim.x / nl;
    const int l = threadIdx.x % nl, r0 = threadIdx.x / nl;
    if (r0 >= rstep) return;
    const float *pv = gv + (int64_t)r0 * es + l, *pw = gw + (int64_t)r0 * es + l;
    const int64_t step = (int64_t)rstep * es;
    dv += l * lstride;
    dw += l * lstride;
    for (int r = r0; r < L; r += kColRows * rstep, pv += kColRows * step, pw += kColRows * step) {
        float a[kColRows], b[kColRows];
#pragma unroll
        for (int k = 0; k < kColRows; ++k)
            if (r + k * rstep < L) {
                a[k] = pv[k * step];
                b[k] = pw[k * step];
            }
#pragma unroll
        for (int k = 0; k < kColRows; ++k)
            if (r + k * rstep < L) {
                dv[r + k * rstep] = a[k];
                dw[r + k * rstep] = b[k];
            }
    }
}

// x-pass store of nl rows (y0 ..) of a 2D field into the blocked intermediate: consecutive
// threads take the rows of one 4-column group, so a 2-row tile writes 32-byte pieces.
__device__ __forceinline__ void blocked_store_rows(float *__restrict__ g, int64_t W, int64_t y0, int nl, int L,
                                                   const float *__restrict__ lds, int lstride)
{
    const int nq = L >> 2;
    const int nthr = blockDim.x;
    if (nthr % nl == 0) {
        // thread t keeps row t % nl and steps through the 4-column groups t / nl + k*(nthr/nl):
        // consecutive groups of a row are 32 floats apart in the blocked layout
        const int l = threadIdx.x % nl;
        const int qstep = nthr / nl;
        const float *d = lds + l * lstride;
        float *gp = g + blocked_index(y0 + l, 0, W);
        for (int q = threadIdx.x / nl; q < nq; q += qstep)
            *reinterpret_cast<float4 *>(gp + 32 * (int64_t)q) =
                make_float4(d[4 * q], d[4 * q + 1], d[4 * q + 2], d[4 * q + 3]);
    } else {
        for (int i = threadIdx.x; i < nl * nq; i += nthr) {
            const int l = i % nl, q = i / nl;
            const float *d = lds + l * lstride + 4 * q;
            *reinterpret_cast<float4 *>(g + blocked_index(y0 + l, 4 * q, W)) = make_float4(d[0], d[1], d[2], d[3]);
        }
    }
}

// y-pass load of the columns x0 .. x0+nl-1 (nl a multiple of 4) of both intermediate fields
// from the blocked layout into LDS lines (line l, element j at lds[l*lstride + j]).  Thread t
// takes column group t % (nl/4) and rows t / (nl/4) + k*rstep, k < kBlkRows (the host checks
// that they cover the column); all loads are issued before the first LDS write.  A 128-byte line of
// the layout is read by one wave, once: nontemporal, so that it does not push the partly written
// lines of the results (16 bytes of each from this workgroup, the rest from its neighbours) out of
// the L2 (64 fields of 2400x1200: y pass 725 -> 697 us; row-major columns, whose lines several
// workgroups read, lose by it: 156 -> 203 us for 512x512x128).
__device__ __forceinline__ void blocked_load_cols(const float *__restrict__ gv, const float *__restrict__ gw,
                                                  int64_t W, int64_t x0, int nl, int L, float *__restrict__ dv,
                                                  float *__restrict__ dw, int lstride)
{
    const int nq = nl >> 2;
    const int rstep = blockDim.x / nq;
    const int q = threadIdx.x % nq, r0 = threadIdx.x / nq;
    if (r0 >= rstep) return;
    float4 rv[kBlkRows], rw[kBlkRows];
#pragma unroll
    for (int k = 0; k < kBlkRows; ++k) {
        const int r = r0 + k * rstep;
        if (r < L) {
            const int64_t o = blocked_index(r, x0 + 4 * q, W);
            rv[k] = load_once(gv + o);
            rw[k] = load_once(gw + o);
        }
    }
    float *a = dv + (4 * q) * lstride + r0, *b = dw + (4 * q) * lstride + r0;
#pragma unroll
    for (int k = 0; k < kBlkRows; ++k)
        if (r0 + k * rstep < L) {
            const int e = k * rstep;
            a[e] = rv[k].x;
            a[lstride + e] = rv[k].y;
            a[2 * lstride + e] = rv[k].z;
            a[3 * lstride + e] = rv[k].w;
            b[e] = rw[k].x;
            b[lstride + e] = rw[k].y;
            b[2 * lstride + e] = rw[k].z;
            b[3 * lstride + e] = rw[k].w;
        }
}

// Store of a y pass that is not the last one (the adjoint's, whose v and w lines hold A and
// B): in place, as (A, B) pairs (adj_pair_index), within the 8-row blocks of the columns
// x0 .. x0+nl-1 it read, so no other workgroup's nodes are touched.  Thread (q, r) writes the
// pairs of row r, columns x0+4q .. x0+4q+3: 32 contiguous bytes.
__device__ __forceinline__ void blocked_store_cols(float *__restrict__ gv, float *__restrict__ gw, int64_t W,
                                                   int64_t x0, int nl, int L, const float *__restrict__ dv,
                                                   const float *__restrict__ dw, int lstride)
{
    const int nq = nl >> 2;
    const int rstep = blockDim.x / nq;
    const int q = threadIdx.x % nq, r0 = threadIdx.x / nq;
    if (r0 >= rstep) return;
    const float *a = dv + (4 * q) * lstride + r0, *b = dw + (4 * q) * lstride + r0;
#pragma unroll
    for (int k = 0; k < kBlkRows; ++k) {
        const int r = r0 + k * rstep;
        if (r < L) {
            const int e = k * rstep;
            float4 *p = reinterpret_cast<float4 *>(((r & 4) ? gw : gv) + adj_pair_index(r, x0 + 4 * q, W));
            p[0] = make_float4(a[e], b[e], a[lstride + e], b[lstride + e]);
            p[1] = make_float4(a[2 * lstride + e], b[2 * lstride + e], a[3 * lstride + e], b[3 * lstride + e]);
        }
    }
}

// Load of the adjoint's first pass (rows, element stride 1): from the forward output f, the
// saved normalised weights W and dL/df = g of a row tile it forms a = g / W and
// b = -a (f - offset) (the two fields the adjoint filters; zero where f or g is NaN) straight
// into the v and w lines, instead of a separate pass writing them to HBM.  float32
// arithmetic: the quotient with one Newton step, and f - offset as (f - hi) - lo with the
// offset split into float32 hi + lo (f - hi is exact while f is within a factor 2 of hi).
// float4 global loads when the rows allow, nontemporal: they are read once (the three passes of a
// backward of 16 fields of 2400x1200 703 -> 674 us, the gather after them 73 -> 80).
__device__ __forceinline__ void adjoint_ab(float fo, float go, float wv, float hi, float lo, float &a, float &b)
{
    a = 0.f;
    b = 0.f;
    if (fo == fo && go == go) {
        const float r = __builtin_amdgcn_rcpf(wv);
        float q = go * r;
        q = fmaf(fmaf(-q, wv, go), r, q);
        a = q;
        b = -q * ((fo - hi) - lo);
    }
}

__device__ __forceinline__ void adjoint_load(const float *__restrict__ f, const float *__restrict__ w,
                                             const float *__restrict__ g, double off, int64_t ls, int nl, int L,
                                             float *__restrict__ sa, float *__restrict__ sb, int lstride)
{
    const float hi = (float)off;
    const float lo = (float)(off - (double)hi);
    const int tid = threadIdx.x, nthr = blockDim.x;
    if ((L & 3) == 0 && (ls & 3) == 0 && aligned16(f) && aligned16(w) && aligned16(g)) {
        const int Lq = L >> 2;
        for (int l = 0; l < nl; ++l) {
            float *da = sa + l * lstride, *db = sb + l * lstride;
            for (int q = tid; q < Lq; q += nthr) {
                const float4 fo = load_once(f + l * ls + 4 * q), go = load_once(g + l * ls + 4 * q),
                             wv = load_once(w + l * ls + 4 * q);
                float a, b;
                adjoint_ab(fo.x, go.x, wv.x, hi, lo, a, b);
                da[4 * q] = a;
                db[4 * q] = b;
                adjoint_ab(fo.y, go.y, wv.y, hi, lo, a, b);
                da[4 * q + 1] = a;
                db[4 * q + 1] = b;
                adjoint_ab(fo.z, go.z, wv.z, hi, lo, a, b);
                da[4 * q + 2] = a;
                db[4 * q + 2] = b;
                adjoint_ab(fo.w, go.w, wv.w, hi, lo, a, b);
                da[4 * q + 3] = a;
                db[4 * q + 3] = b;
            }
        }
    } else {
        for (int l = 0; l < nl; ++l) {
            const float *fl = f + l * ls, *wl = w + l * ls, *gl = g + l * ls;
            for (int j = tid; j < L; j += nthr) {
                float a, b;
                adjoint_ab(fl[j], gl[j], wl[j], hi, lo, a, b);
                sa[l * lstride + j] = a;
                sb[l * lstride + j] = b;
            }
        }
    }
}

// Lane i receives lane i+1's value (from_next) or lane i-1's (from_prev) by a DPP wave shift;
// the lane without a source keeps its own value.
__device__ __forceinline__ int dpp_from_next(int v) { return __builtin_amdgcn_update_dpp(v, v, 0x130, 0xf, 0xf, false); }
__device__ __forceinline__ int dpp_from_prev(int v) { return __builtin_amdgcn_update_dpp(v, v, 0x138, 0xf, 0xf, false); }
__device__ __forceinline__ double dpp_from_next(double v)
{
    return __hiloint2double(dpp_from_next(__double2hiint(v)), dpp_from_next(__double2loint(v)));
}

// Deterministic fused injection of one line's points into its float32 row.  For s < 4 (2 without
// planes), the points of base row (y - dy, z - dz), dy = s & 1, dz = s >> 1, contribute their corners
// (0, dy, dz) and (1, dy, dz) at x = base x and base x + 1: two sub-streams, in which the points
// ascend in base x (point order for equal x) and so in target cell.  The line's sub-streams,
// concatenated, are taken in chunks of up to 64 entries by the line's first `iw` lanes
// (`injector`).  A run sum over adjacent lanes of equal target cell (in lane order) gives
// each run's total to its first lane.  Equal cells adjacent in one
// sub-stream form one run; a cell can head two runs of a chunk only from different
// sub-streams, so the heads add their totals in one round per sub-stream of the head
// (program order), without conflicts.  The result does not depend on timing.  Called by
// every thread of the workgroup (wave-wide ballots).
//
// Bound by its instructions, some hundred per chunk and wave, which every line pays at least once: the
// x pass without it 548 us of 650 (64 fields of 2400x1200, 6 points to a row), 534 of 733 (96 uneven
// fields).  Row ranges without a division, entries found row by row, chunks counted by ballots, runs
// summed up to their ends and the value beside the position (1D, 2D): x 650 -> 625, 733 -> 670 us, and
// 162 -> 157 for 512x512x128 with 200000 points.
struct LineInjection {
    uint32_t start[4], count[4];   // the base rows' ranges of the sorted list
    uint32_t total;                // entries of the line

    // the row ranges, before the line is cleared
    __device__ __forceinline__ void begin(const PassWork &wk, int my_line, bool injector,
                                          const uint32_t *__restrict__ line_start,
                                          const uint32_t *__restrict__ line_count)
    {
        const uint32_t line = wk.line + my_line, row = wk.row + my_line, H = wk.plane;
        const uint32_t y = H ? line % H : line, z = H ? line / H : 0u;   // a 2D line is y itself
        total = 0;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const uint32_t dy = s & 1, dz = s >> 1;
            start[s] = count[s] = 0;
            if (s < 2 || H) {
                if (injector && y >= dy && z >= dz) {
                    const uint32_t r = row - dy - dz * H;
                    start[s] = line_start[r];
                    count[s] = line_count[r];
                }
                total += 2 * count[s];
            }
        }
    }

    // row[x - lo] receives cell x of the line for x in [lo, lo + len) (a chunk of a long line);
    // cells outside are skipped
    __device__ __forceinline__ void add(int dim, bool planes, int iw, int sid, int fsel, double off,
                                        const uint32_t *__restrict__ vals, const PointRec *__restrict__ rec,
                                        const double *__restrict__ val, float *row, int lo, int len)
    {
        // This lane's entry e: its sub-stream (2 * row + corner column) and its slot in the sorted
        // point list.
        auto entry = [&](uint32_t e, int &hq, uint32_t &src) {
            uint32_t st = start[0], ct = count[0];
            hq = 0;
#pragma unroll
            for (int s = 1; s < 4; ++s)
                if (s < 2 || planes) {
                    const bool on = hq == 2 * (s - 1) && e >= 2 * ct;   // past row s - 1
                    e -= on ? 2 * ct : 0u;
                    st = on ? start[s] : st;
                    ct = on ? count[s] : ct;
                    hq = on ? 2 * s : hq;
                }
            const bool bx = e >= ct;
            src = st + e - (bx ? ct : 0u);
            hq += bx;
        };
        // Software pipeline over the chunks: while chunk ch is summed, the point data of chunk ch+1
        // and the point index of chunk ch+2 are in flight.
        auto fetch_index = [&](uint32_t e, bool &ok, int &hq, uint32_t &p) {
            ok = e < total;
            hq = 0;
            p = 0;
            if (ok) {
                uint32_t src;
                entry(e, hq, src);
                p = vals[src];
            }
        };
        struct PointData {
            PointRec r;
            double v;
        };
        auto load_point = [&](bool ok, uint32_t p, PointData &o) {
            o.r = PointRec{{0.0, 0.0, 0.0}, 0, 0};
            o.v = 0.0;
            if (!ok) return;
            o.r = rec[p];
            if (planes) o.v = val[p];
        };
        const int lane = threadIdx.x & 63;
        bool ok_a, ok_b;
        int hq_a, hq_b;
        uint32_t p_a, p_b, e = sid;
        PointData pd_a;
        fetch_index(e, ok_a, hq_a, p_a);
        load_point(ok_a, p_a, pd_a);
        fetch_index(e += iw, ok_b, hq_b, p_b);
        while (__any(ok_a)) {   // the chunks ascend: a lane without an entry has none in later ones
            const bool valid = ok_a;
            const int hq = hq_a;
            const PointData pd = pd_a;
            ok_a = ok_b;
            hq_a = hq_b;
            load_point(ok_b, p_b, pd_a);
            fetch_index(e += iw, ok_b, hq_b, p_b);
            int x = -1;
            double c = 0.0;
            if (valid) {
                PointPos pp;
#pragma unroll
                for (int m = 0; m < 3; ++m) {
                    pp.i[m] = 0;
                    pp.w[m] = pd.r.w[m];
                }
                x = pd.r.xi + (hq & 1);
                const double w = corner_weight(dim, pp, hq & 1, (hq >> 1) & 1, hq >> 2);
                c = fsel ? w : w * ((planes ? pd.v : pd.r.w[2]) - off);
            }
            // runs: maximal groups of adjacent lanes with equal cell (the concatenated stream is
            // not sorted, so equal cells further apart belong to different runs), each up to the
            // next run's first lane
            const int px = dpp_from_prev(x);
            const bool start = sid == 0 || px != x;
            // The run sum only where some run of this wave's chunk has more than one entry:
            // otherwise every lane is its own run and keeps c.  Each run's first lane adds the
            // contributions of the run's next lanes one at a time (DPP wave shifts, no LDS
            // round trips), in lane order, until the longest run ends.
            if (__any(valid && !start)) {
                const unsigned long long next = (__ballot(start) >> lane) >> 1;
                const int left = valid ? (next ? __builtin_ctzll(next) + 1 : 64 - lane) : 0;   // this lane's run from here on
                double o = c;
                for (int t = 1; __any(t < left); ++t) {
                    o = dpp_from_next(o);
                    if (t < left) c += o;
                }
            }
            const bool here = valid && start && x >= lo && x < lo + len;
            float *cell = row + (here ? x - lo : 0);
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if (q < 4 || planes)
                    if (here && hq == q) *cell = (float)((double)*cell + c);
        }
    }
};

// Orders the LDS accesses of one phase of a line pass before the next: a workgroup
// barrier when a line spans several waves; a line within one wave needs only program order
// (a wave's LDS instructions execute in order), kept by a compiler fence.
__device__ __forceinline__ void line_sync(int lpl)
{
    if (lpl > 64) __syncthreads();
    else __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

// One workgroup = 128, 256 or 512 threads: the first half works on the v field, the second
// half on the w field of the same nlines lines (each half: up to lines_cap lines of lpl
// lanes).  LDS holds the v lines, then the w lines, each padded by zeros on both sides.
template <bool INJECT, int SEG>
__global__ __launch_bounds__(kFastBlock, 1) void k_fast_pass(
    const FieldDev *__restrict__ fields, const double *__restrict__ offsets, const PassWork *__restrict__ work,
    const PassField *__restrict__ passes, const PointRec *__restrict__ rec, const uint32_t *__restrict__ vals,
    const uint32_t *__restrict__ line_start, const uint32_t *__restrict__ line_count,
    const double *__restrict__ val, float *__restrict__ gv, float *__restrict__ gw, float *__restrict__ out,
    float *__restrict__ wsave, int final_pass, const float *__restrict__ adj_g)
{
    constexpr int kSegArr = SEG;
    extern __shared__ __align__(16) unsigned char smem[];
    // The waves that fill their tile go first, those that filter it give way (64 fields of 2400x1200,
    // us: x 640 -> 625, y 705 -> 685; the adjoint's passes of 16 fields 250 -> 235).  Not where columns
    // are read in pieces of lines that other workgroups read too: y of 512x512x128 156 -> 161.
    if (INJECT || adj_g) __builtin_amdgcn_s_setprio(2);
    const PassWork wk = work[blockIdx.x];
    const FieldDev &F = fields[wk.field];
    const PassField P = passes[wk.field];
    if (P.blocked == kBlockedIn) __builtin_amdgcn_s_setprio(2);
    const int tid = threadIdx.x;
    const int nthr = blockDim.x;
    const int half = nthr >> 1;
    const int fsel = tid >= half;            // 0: v worker, 1: w worker
    const int ltid = tid - fsel * half;
    // line range of this work item: the whole line, or for a chunked field the chunk's nodes
    // [lo + so, lo + so + sc) with their halos, [lo, lo + L); the LDS is laid out for P.len
    int L = (int)P.len;
    int lo = 0, so = 0, sc = L;
    if (P.chunk) {
        const int64_t c0 = (int64_t)wk.chunk * P.chunk;
        const int64_t c1 = min(c0 + (int64_t)P.chunk, P.full_len);
        const int64_t a0 = max(c0 - (int64_t)P.halo, (int64_t)0);
        lo = (int)a0;
        L = (int)(min(c1 + (int64_t)P.halo, P.full_len) - a0);
        so = (int)(c0 - a0);
        sc = (int)(c1 - c0);
    }
    const int T = P.T;
    const int lpl = P.lpl;
    const int lines_cap = P.lines;
    // LDS: T+1 zeros, then per line its P.len cells and a gap of P.rpad floats: line l's
    // overflow area (full stores, below) followed by zeros, whose last T+1 are line l+1's
    // left padding.  The w lines follow the v lines, their first left padding the end of the
    // last v line's gap.
    const int pad = T + 1;
    const int rpad = P.rpad;
    const int lstride = (int)P.len + rpad;
    const int nl = wk.nlines;
    const int64_t es = P.elem_stride;
    float *sv = reinterpret_cast<float *>(smem);
    float *sw = sv + (size_t)lines_cap * lstride;
    float *mine = fsel ? sw : sv;
    const int my_line = ltid / lpl;
    const int sid = ltid - my_line * lpl;
    const bool line_ok = my_line < nl;
    const double off = offsets[wk.field];

    // injection: the first (up to 64) lanes of each line
    const int iw = lpl < 64 ? lpl : 64;
    const bool injector = INJECT && line_ok && sid < iw;
    LineInjection inj;

    if (INJECT) {
        inj.begin(wk, my_line, injector, line_start, line_count);
        // each line's lanes zero the line's left padding, cells and gap (the left padding is
        // the previous line's gap end, which that line also zeroes and never writes again:
        // zeros over zeros); lines past nl and the reserve after the w lines feed only
        // discarded steps
        if (line_ok) {
            float *z = mine + (size_t)my_line * lstride;
            const int zlen = pad + lstride;
            const int head = (int)((16 - ((uintptr_t)z & 15u)) & 15u) >> 2;   // floats before a 16-byte boundary
            const int nq = (zlen - head) >> 2;
            float4 *z4 = reinterpret_cast<float4 *>(z + head);
            for (int i = sid; i < head; i += lpl) z[i] = 0.f;
            for (int i = sid; i < nq; i += lpl) z4[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            for (int i = head + 4 * nq + sid; i < zlen; i += lpl) z[i] = 0.f;
        }
        line_sync(lpl);
    } else {
        // zero what follows each line's cells (the rest of a chunk's cells and the gap) and the
        // left padding of the v lines
        const int nz = lstride - L;
        if (nz <= 64) {
            // wave w zeroes the gaps of lines w, w + waves, ... (lane = position in the gap)
            const int lane = tid & 63;
            if (lane < nz) {
                for (int l = tid >> 6; l < lines_cap; l += nthr >> 6) {
                    sv[pad + l * lstride + L + lane] = 0.f;
                    sw[pad + l * lstride + L + lane] = 0.f;
                }
            }
        } else {
            for (int i = tid; i < lines_cap * nz; i += nthr) {
                const int l = i / nz, r = i - l * nz;
                const int o = pad + l * lstride + L + r;
                sv[o] = 0.f;
                sw[o] = 0.f;
            }
        }
        for (int i = tid; i < pad; i += nthr) sv[i] = 0.f;
        if (adj_g)
            adjoint_load(out + F.out_off + wk.base + lo, wsave + F.out_off + wk.base + lo,
                         adj_g + F.out_off + wk.base + lo, off, P.line_stride, nl, L, sv + pad, sw + pad, lstride);
        else if (P.blocked == kBlockedIn)
            blocked_load_cols(gv + F.cell_off, gw + F.cell_off, F.size[0], wk.base, nl, L, sv + pad, sw + pad,
                              lstride);
        else if (P.line_stride == 1 && ((nl | es) & 3))
            load_columns(gv + F.cell_off + wk.base + lo * es, gw + F.cell_off + wk.base + lo * es, es, nl, L, sv + pad,
                         sw + pad, lstride);
        else {
            tile_copy<true>(gv + F.cell_off + wk.base + lo * es, P.line_stride, es, nl, L, sv + pad, lstride);
            tile_copy<true>(gw + F.cell_off + wk.base + lo * es, P.line_stride, es, nl, L, sw + pad, lstride);
        }
        __syncthreads();
    }

    if (INJECT) {
        // a line's injection writes cells 0..L-1 of that line only
        inj.add(F.dim, wk.plane != 0, iw, sid, fsel, off, vals, rec, val, mine + my_line * lstride + pad, lo, L);
        line_sync(lpl);
    }

    // n-fold tailed box filter, in place.  Every lane owns kSegArr consecutive elements;
    // the host picks lpl with lpl*kSegArr >= L and reserves 64 floats past the w lines so
    // that the branch-free slides never read out of bounds.
    const int s0 = sid * kSegArr;
    int myseg = L - s0;
    myseg = myseg < 0 ? 0 : (myseg > kSegArr ? kSegArr : myseg);
    const bool act = line_ok && myseg > 0;
    float *ln = mine + (size_t)(line_ok ? my_line : 0) * lstride + pad;
    const double alpha = P.alpha;
    const int niter = F.num_iter;
    // whole-segment stores (when the host widened the gap by the overflow of the last
    // segment): the segment crossing the line end writes `over` floats into the gap's
    // overflow area, short of the next line's left padding; the line's lanes then re-zero
    // those of them the next iteration reads (within the first T+1), after the stores: by the
    // wave's program order when the line lies in one wave, else after a workgroup barrier
    const int over = (kSegArr - L % kSegArr) % kSegArr;
    const bool full = L > kSegArr && rpad - pad >= over;   // the overflow stays clear of the next left padding
    const int nclr = full ? min(pad, over) : 0;
    // An iteration reads and writes only its own line and its left padding, which no lane
    // writes after the zeroing (reads past the line feed discarded steps),
    // so the lines synchronise on their own: by wave order when a line's lanes lie in one
    // wave (lpl <= 64, a power of two; each field's half of the workgroup is whole waves),
    // else by workgroup barriers.  The tile IO after the loop spans all lines.
    float sb[kSegArr];
    __builtin_amdgcn_s_setprio(0);
    for (int it = 0; it < niter; ++it) {
        const bool last = it + 1 == niter;
        const bool grp = (it + 1) % P.sgroup == 0;
        if (act) {
            if (last || grp) slide1<SEG, true>(ln, s0, T, alpha, last ? P.slast : P.sgscale, sb);
            else slide1<SEG, false>(ln, s0, T, alpha, 1.0, sb);
        }
        line_sync(lpl);
        // an opaque copy of the lane's element count keeps the compiler from hoisting the
        // kSegArr store predicates of the partial case out of the loop (into spilled SGPRs)
        int nst = myseg;
        asm volatile("" : "+v"(nst));
        if (act) stage_store(ln, s0, nst, full, sb);
        // the lane whose segment crosses the line end stores into the padding; in a line of
        // several waves it is not in the wave of the lanes that re-zero the padding, so a
        // barrier orders its stores before theirs (nclr and lpl are the same for the whole
        // workgroup)
        if (lpl > 64 && nclr > 0) __syncthreads();
        if (line_ok)
            for (int e = sid; e < nclr; e += lpl) ln[L + e] = 0.f;
        line_sync(lpl);
    }
    __syncthreads();

    if (final_pass) {
        // masked quotient + offset (interpolation.py:367, :428-430), formed as the v lines are stored
        tile_copy<false>(out + F.out_off + wk.base + (lo + so) * es, P.line_stride, es, nl, sc, sv + pad + so, lstride,
                         LdsQuotient{(int)(sw - sv), off, F.thr_fast_f});
        // training forward: keep the normalised weight field for the adjoint
        if (wsave)
            tile_copy<false>(wsave + F.out_off + wk.base + (lo + so) * es, P.line_stride, es, nl, sc, sw + pad + so,
                             lstride);
    } else if (P.blocked == kBlockedOut) {
        const int64_t y0 = wk.base / F.size[0];
        blocked_store_rows(gv + F.cell_off, F.size[0], y0, nl, L, sv + pad, lstride);
        blocked_store_rows(gw + F.cell_off, F.size[0], y0, nl, L, sw + pad, lstride);
    } else if (P.blocked == kBlockedIn) {
        blocked_store_cols(gv + F.cell_off, gw + F.cell_off, F.size[0], wk.base, nl, L, sv + pad, sw + pad, lstride);
    } else {
        tile_copy<false>(gv + F.cell_off + wk.base + (lo + so) * es, P.line_stride, es, nl, sc, sv + pad + so,
                         lstride);
        tile_copy<false>(gw + F.cell_off + wk.base + (lo + so) * es, P.line_stride, es, nl, sc, sw + pad + so,
                         lstride);
    }
}

// ---------------------------------------------------------------------------
// FP32C prefix pass.  The same n-fold tailed box filter (interpolation.py:484-533), computed
// on FP64 prefix sums of the line held in LDS.  With P_m = sum of the line's elements
// before position m (zero padding outside the line), one iteration is
//   o_k = (1 - alpha) (P_{k+T+1} - P_{k-T}) + alpha (P_{k+T+2} - P_{k-T-1})
// (the window of 2T+1 terms plus the two tail terms).  Each lane owns SEG consecutive
// positions: it chains the FP64 prefix of its outputs, the line's lanes scan their segment
// totals, and the lanes store the next iteration's P = base + chain.  Nothing is rounded to
// float32 between iterations; the last iteration writes float32 outputs into the line's
// tile.  5 FP64 operations per element and iteration, no conversions.
//
// LDS per (field, line): prefix_line_stride(lpl, SEG, T) doubles holding positions
// -T-1 .. lpl*SEG+T+1 (position m at index m+T+1): zero for m <= 0, P_L for m >= L.  The
// float32 tile of the line (tile IO, injection, results) aliases the same storage.  After
// all lines: one double per wave for the segment-total scan of lines wider than a wave.

// Segment lengths the prefix pass is instantiated for; odd, so the 8-byte LDS lane stride is
// conflict-free.
#define FB_PFX_SEGS(X) X(15) X(17) X(19) X(21) X(23)
constexpr int kPfxBlk = 4;   // prefix reads in flight per stream

// x + (x of the lane CTRL selects), as a DPP move of both halves; lanes whose source is
// outside the row, and rows outside ROWMASK, add 0
template <int CTRL, int ROWMASK>
__device__ __forceinline__ double dpp_add(double x)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, ROWMASK, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, ROWMASK, 0xf, false);
    return x + __hiloint2double(hi, lo);
}

// Exclusive scan of the lanes' segment totals t along each line (lpl lanes of consecutive
// threads) and the line total.  Lines of 16 or more lanes scan with DPP row shifts and row
// broadcasts (a row is 16 lanes), shorter ones with shuffles.  For lines of several waves it
// contains the workgroup barrier that ends the read phase; every thread of the workgroup
// calls it.
__device__ __forceinline__ void line_scan(double t, int sid, int lpl, double *wtot, double &base, double &total)
{
    const int w = lpl < 64 ? lpl : 64;
    const int li = sid & (w - 1);
    double inc = t;
    if (w >= 16) {
        inc = dpp_add<0x111, 0xf>(inc);   // row_shr:1
        inc = dpp_add<0x112, 0xf>(inc);   // row_shr:2
        inc = dpp_add<0x114, 0xf>(inc);   // row_shr:4
        inc = dpp_add<0x118, 0xf>(inc);   // row_shr:8
        if (w >= 32) inc = dpp_add<0x142, 0xa>(inc);   // row_bcast:15 into rows 1, 3
        if (w >= 64) inc = dpp_add<0x143, 0xc>(inc);   // row_bcast:31 into rows 2, 3
    } else {
        for (int d = 1; d < w; d <<= 1) {
            const double o = __shfl_up(inc, d, w);
            if (li >= d) inc += o;
        }
    }
    const double ex = inc - t;
    if (lpl > 64) {
        // lines of several waves: wave totals through LDS
        if ((threadIdx.x & 63) == 63) wtot[threadIdx.x >> 6] = inc;
        __syncthreads();
        const int wv = sid >> 6;
        const int w0 = (int)(threadIdx.x >> 6) - wv;   // first wave of the line
        double pre = 0.0, tot = 0.0;
        for (int k = 0; k < (lpl >> 6); ++k) {
            const double x = wtot[w0 + k];
            pre += k < wv ? x : 0.0;
            tot += x;
        }
        base = pre + ex;
        total = tot;
    } else {
        base = ex;
        total = __shfl(inc, w - 1, w);
    }
}

// One iteration over the lane's segment: pl[j] = P_{s+j-T-1}, pr[j] = P_{s+j+T+1} for
// j = 0..SEG.  OUT: o_j = c1 D_j + c2 E_j into res[]; else the chain
// q[j+1] = q[j] + o_j, and q[nvp] is returned (the partial lane's total).
template <int SEG, bool OUT>
__device__ __forceinline__ double prefix_step(const double *pl, const double *pr, double c1, double c2, int nvp,
                                              double (&q)[SEG + 1], float (&res)[SEG])
{
    constexpr int NB = (SEG + kPfxBlk - 1) / kPfxBlk;
    double la = pl[0], ra = pr[0];
    double lc[kPfxBlk], rc[kPfxBlk], ln[kPfxBlk], rn[kPfxBlk];
#pragma unroll
    for (int u = 0; u < kPfxBlk; ++u) {
        lc[u] = pl[1 + u];
        rc[u] = pr[1 + u];
    }
    double snap = 0.0;
    q[0] = 0.0;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if (b + 1 < NB) {
#pragma unroll
            for (int u = 0; u < kPfxBlk; ++u) {
                const int j = (b + 1) * kPfxBlk + u;
                if (j < SEG) {
                    ln[u] = pl[1 + j];
                    rn[u] = pr[1 + j];
                }
            }
        }
#pragma unroll
        for (int u = 0; u < kPfxBlk; ++u) {
            const int j = b * kPfxBlk + u;
            if (j < SEG) {
                const double D = ra - lc[u];   // P_{k+T+1} - P_{k-T}
                const double E = rc[u] - la;   // P_{k+T+2} - P_{k-T-1}
                if (OUT) {
                    res[j] = (float)fma(c1, D, c2 * E);
                } else {
                    q[j + 1] = fma(c1, D, fma(c2, E, q[j]));
                }
                la = lc[u];
                ra = rc[u];
            }
        }
        if (b + 1 < NB) {
#pragma unroll
            for (int u = 0; u < kPfxBlk; ++u) {
                lc[u] = ln[u];
                rc[u] = rn[u];
            }
        }
    }
    if (!OUT) {
        // q[nvp] with the wave-uniform nvp: scalar branches, no per-element selects
        switch (nvp) {
#define FB_SNAP(J) case J: if (J <= SEG) snap = q[J <= SEG ? J : 0]; break;
            FB_SNAP(1) FB_SNAP(2) FB_SNAP(3) FB_SNAP(4) FB_SNAP(5) FB_SNAP(6) FB_SNAP(7) FB_SNAP(8)
            FB_SNAP(9) FB_SNAP(10) FB_SNAP(11) FB_SNAP(12) FB_SNAP(13) FB_SNAP(14) FB_SNAP(15) FB_SNAP(16)
            FB_SNAP(17) FB_SNAP(18) FB_SNAP(19) FB_SNAP(20) FB_SNAP(21) FB_SNAP(22) FB_SNAP(23) FB_SNAP(24)
#undef FB_SNAP
        default: break;
        }
    }
    return snap;
}

template <bool INJECT, int SEG>
__global__ __launch_bounds__(kFastBlock, 1) void k_prefix_pass(
    const FieldDev *__restrict__ fields, const double *__restrict__ offsets, const PassWork *__restrict__ work,
    const PassField *__restrict__ passes, const PointRec *__restrict__ rec, const uint32_t *__restrict__ vals,
    const uint32_t *__restrict__ line_start, const uint32_t *__restrict__ line_count,
    const double *__restrict__ val, float *__restrict__ gv, float *__restrict__ gw, float *__restrict__ out,
    float *__restrict__ wsave, int final_pass, const float *__restrict__ adj_g)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const PassWork wk = work[blockIdx.x];
    const FieldDev &F = fields[wk.field];
    const PassField P = passes[wk.field];
    const int tid = threadIdx.x;
    const int nthr = blockDim.x;
    const int half = nthr >> 1;
    const int fsel = tid >= half;            // 0: v worker, 1: w worker
    const int ltid = tid - fsel * half;
    const int L = (int)P.len;
    const int T = P.T;
    const int lpl = P.lpl;
    const int lines_cap = P.lines;
    const int lstride = prefix_line_stride(lpl, SEG, T);
    const int fstride = 2 * lstride;         // floats per line of the float32 tiles
    const int pad = T + 1;                   // index of position 0
    const int nl = wk.nlines;
    double *pall = reinterpret_cast<double *>(smem);
    double *wtot = pall + (size_t)2 * lines_cap * lstride;
    float *tv = reinterpret_cast<float *>(smem);
    float *tw = tv + (size_t)lines_cap * fstride;
    const int my_line = ltid / lpl;
    const int sid = ltid - my_line * lpl;
    const bool line_ok = my_line < nl;
    double *myP = pall + (size_t)(fsel * lines_cap + (line_ok ? my_line : 0)) * lstride;
    float *myX = reinterpret_cast<float *>(myP);
    const double off = offsets[wk.field];

    if (INJECT) {
        const int iw = lpl < 64 ? lpl : 64;
        LineInjection inj;
        inj.begin(wk, my_line, line_ok && sid < iw, line_start, line_count);
        float4 *z = reinterpret_cast<float4 *>(smem);
        const int nz = (2 * lines_cap * fstride) >> 2;
        for (int i = tid; i < nz; i += nthr) z[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        __syncthreads();
        inj.add(F.dim, wk.plane != 0, iw, sid, fsel, off, vals, rec, val, myX, 0, L);
    } else {
        if (adj_g)
            adjoint_load(out + F.out_off + wk.base, wsave + F.out_off + wk.base, adj_g + F.out_off + wk.base, off,
                         P.line_stride, nl, L, tv, tw, fstride);
        else {
            tile_copy<true>(gv + F.cell_off + wk.base, P.line_stride, P.elem_stride, nl, L, tv, fstride);
            tile_copy<true>(gw + F.cell_off + wk.base, P.line_stride, P.elem_stride, nl, L, tw, fstride);
        }
    }
    __syncthreads();

    // lane classes: nfull lanes of SEG positions, then (when L mod SEG != 0) one partial lane
    // of nvp positions, then lanes past the line end
    const int s0 = sid * SEG;
    const int nfull = L / SEG;
    const int nvp = L - nfull * SEG;
    const int nv = !line_ok ? 0 : (sid < nfull ? SEG : (sid == nfull ? nvp : 0));
    const bool partial = line_ok && nvp > 0 && sid == nfull;
    double q[SEG + 1];
    float res[SEG];
    double base, total;

    // prefix of the input line
    q[0] = 0.0;
#pragma unroll
    for (int j = 0; j < SEG; ++j) {
        const float xv = j < nv ? myX[s0 + j] : 0.f;
        q[j + 1] = q[j] + (double)xv;
    }
    line_scan(q[SEG], sid, lpl, wtot, base, total);
    line_sync(lpl);   // the float32 reads above end before the prefix stores alias them
    if (line_ok) {
#pragma unroll
        for (int j = 0; j < SEG; ++j) myP[pad + s0 + j] = base + q[j];
        for (int e = sid; e < pad; e += lpl) myP[e] = 0.0;
        for (int e = sid; e < T + 2; e += lpl) myP[pad + lpl * SEG + e] = total;
    }
    line_sync(lpl);

    const double alpha = P.alpha;
    const int niter = F.num_iter;
    const double *pl = myP + s0;                 // P_{s0-T-1}
    const double *pr = myP + s0 + 2 * T + 2;     // P_{s0+T+1}
    for (int it = 0; it < niter; ++it) {
        const bool last = it + 1 == niter;
        const bool grp = (it + 1) % P.sgroup == 0;
        const double sc = last ? P.slast : (grp ? P.sgscale : 1.0);
        const double c1 = nv > 0 ? sc * (1.0 - alpha) : 0.0;
        const double c2 = nv > 0 ? sc * alpha : 0.0;
        if (!last) {
            const double snap = prefix_step<SEG, false>(pl, pr, c1, c2, nvp, q, res);
            line_scan(partial ? snap : q[SEG], sid, lpl, wtot, base, total);
            line_sync(lpl);
            if (line_ok) {
#pragma unroll
                for (int j = 0; j < SEG; ++j) myP[pad + s0 + j] = base + q[j];
                // the partial lane's chain ran on past the line end: its positions after L
                // hold P_L (program order after its own stores above)
                if (partial)
                    for (int e = nvp + 1; e < SEG; ++e) myP[pad + s0 + e] = total;
                for (int e = sid; e < T + 2; e += lpl) myP[pad + lpl * SEG + e] = total;
            }
            line_sync(lpl);
        } else {
            prefix_step<SEG, true>(pl, pr, c1, c2, nvp, q, res);
            line_sync(lpl);
            if (line_ok) {
#pragma unroll
                for (int j = 0; j < SEG; ++j) myX[s0 + j] = res[j];
            }
            __syncthreads();   // the tile IO below spans all lines
        }
    }

    if (final_pass) {
        // masked quotient + offset (interpolation.py:367, :428-430), formed as the v tiles are stored
        tile_copy<false>(out + F.out_off + wk.base, P.line_stride, P.elem_stride, nl, L, tv, fstride,
                         LdsQuotient{(int)(tw - tv), off, F.thr_fast_f});
        if (wsave) tile_copy<false>(wsave + F.out_off + wk.base, P.line_stride, P.elem_stride, nl, L, tw, fstride);
    } else {
        tile_copy<false>(gv + F.cell_off + wk.base, P.line_stride, P.elem_stride, nl, L, tv, fstride);
        tile_copy<false>(gw + F.cell_off + wk.base, P.line_stride, P.elem_stride, nl, L, tw, fstride);
    }
}

// ---------------------------------------------------------------------------
// elementwise helpers

// zero fill by kernel (a fill kernel instead of hipMemsetAsync keeps the batch graph free
// of memset nodes)
__global__ __launch_bounds__(kBlock) void k_zero_u32(uint32_t *__restrict__ p, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// the same for a 16-byte aligned buffer of n words: four words per thread (one 16-byte store),
// the last thread's remainder word by word
__global__ __launch_bounds__(kBlock) void k_zero_u32x4(uint32_t *__restrict__ p, int64_t n)
{
    const int64_t i = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * 4;
    if (i + 4 <= n) {
        *reinterpret_cast<uint4 *>(p + i) = make_uint4(0u, 0u, 0u, 0u);
    } else {
        for (int64_t k = i; k < n; ++k) p[k] = 0u;
    }
}

__global__ __launch_bounds__(kBlock) void k_f64_to_f32(const double *__restrict__ in, float *__restrict__ out,
                                                       int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) out[i] = (float)in[i];
}

__global__ __launch_bounds__(kBlock) void k_f32_to_f64(const float *__restrict__ in, double *__restrict__ out,
                                                       int64_t n, double scale)
{
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) out[i] = (double)in[i] * scale;
}

// ---------------------------------------------------------------------------
// Adjoint of the FP32C batch (no counterpart in the reference, which has no gradient).
//
// On unmasked nodes f = V/W + offset with V = B S (val - offset), W = B S 1, where S is
// the bilinear injection and B the product of the per-axis n-fold tailed box filters
// (zero-padded banded symmetric matrices, so B is self-adjoint).  For g = dL/df:
//   a = g/W,  b = -g V/W^2 = -a (f - offset),  A = B a,  Bb = B b
//   dL/dval_k  = sum_c w_c(p_k) A[c]
//   dL/dp_k,m  = sum_c (dw_c/dp_m) ((val_k - offset) A[c] + Bb[c])
// The offset drops out (V/W does not depend on it).  The FP32C passes carry the
// normalisation (1/(K+2 alpha))^n per axis in both V and W; applying the same scaled
// operator to a = g/W_scaled gives the same A, so the gradient needs no rescaling.

// Transposed injection: one thread per point gathers A and Bb at its 2^DIM corners.
// Points dropped by the injection (outside the grid, NaN) get zero gradients.  (Taking the
// points in the forward's sorted order makes the A, Bb reads local but the point reads and
// gradient writes scattered; measured slower.)
//
// Bound by the random reads' latency: all corners of a point are loaded before the first is used.
// 1.6 million points on 16 fields of 2400x1200: corner by corner 99 us, now 67.
template <int DIM>
__global__ __launch_bounds__(kBlock) void k_adj_gather(const FieldDev *__restrict__ fields,
                                                       const int64_t *__restrict__ pt_prefix, int nfields,
                                                       int64_t npoints, const double *__restrict__ pts,
                                                       const double *__restrict__ val,
                                                       const double *__restrict__ offsets,
                                                       const float *__restrict__ A, const float *__restrict__ Bb,
                                                       const PassField *__restrict__ pass_y,
                                                       double *__restrict__ gval, double *__restrict__ gpts)
{
    constexpr int NC = 1 << DIM;
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= npoints) return;
    double c[DIM];
#pragma unroll
    for (int m = 0; m < DIM; ++m) c[m] = pts[i * DIM + m];
    const double v = val[i];
    const int f = find_seg(pt_prefix, nfields, i);
    const FieldDev &F = fields[f];
    // A and B of a 2D field whose y pass ran on the blocked intermediate are (A, B) pairs
    // (adj_pair_index), the pairs of rows y % 8 < 4 in A's field and the others in Bb's
    const bool blocked = DIM == 2 && pass_y[f].blocked == kBlockedIn;
    PointPos pp;
    double gv = 0.0, gp[3] = {0.0, 0.0, 0.0};
    if (point_pos(F, c, pp)) {
        const double vk = v - offsets[f];
        const int64_t W = F.size[0], H = F.size[1];
        float ca[NC], cb[NC];
        if (blocked) {
#pragma unroll
            for (int q = 0; q < NC; ++q) {
                const int64_t y = pp.i[1] + ((q >> 1) & 1);
                const float2 ab = *reinterpret_cast<const float2 *>((y & 4 ? Bb : A) + F.cell_off +
                                                                    adj_pair_index(y, pp.i[0] + (q & 1), W));
                ca[q] = ab.x;
                cb[q] = ab.y;
            }
        } else {
#pragma unroll
            for (int q = 0; q < NC; ++q) {
                const int64_t cell = F.cell_off + ((pp.i[2] + (q >> 2)) * H + (pp.i[1] + ((q >> 1) & 1))) * W +
                                     (pp.i[0] + (q & 1));
                ca[q] = A[cell];
                cb[q] = Bb[cell];
            }
        }
#pragma unroll
        for (int q = 0; q < NC; ++q) {
            const int bx = q & 1, by = (q >> 1) & 1, bz = q >> 2;
            const double a = (double)ca[q], b = (double)cb[q];
            const double fx = bx ? pp.w[0] : 1.0 - pp.w[0];
            const double fy = DIM >= 2 ? (by ? pp.w[1] : 1.0 - pp.w[1]) : 1.0;
            const double fz = DIM >= 3 ? (bz ? pp.w[2] : 1.0 - pp.w[2]) : 1.0;
            const double sx = bx ? 1.0 : -1.0, sy = by ? 1.0 : -1.0, sz = bz ? 1.0 : -1.0;
            gv += corner_weight(DIM, pp, bx, by, bz) * a;
            const double t = vk * a + b;
            gp[0] += sx * fy * fz * t;
            gp[1] += fx * sy * fz * t;
            gp[2] += fx * fy * sz * t;
        }
    }
    gval[i] = gv;
    if (gpts) {
#pragma unroll
        for (int m = 0; m < DIM; ++m) gpts[i * DIM + m] = gp[m] / F.step[m];
    }
}

inline unsigned nblocks(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

}  // namespace

// ---------------------------------------------------------------------------
// launchers

int64_t offsets_part_elems(int nfields, int64_t npoints) { return 3 * first_chunk(npoints, nfields); }

int launch_offsets(const FieldDev *d_fields, int nfields, int64_t max_n, int64_t npoints, const double *d_val,
                   double *d_part, double *d_offsets, hipStream_t s)
{
    if (!d_part || max_n <= kOffSingle) {
        hipLaunchKernelGGL(k_offsets, dim3(nfields), dim3(kBlock), 0, s, d_fields, d_val, d_offsets);
    } else {
        hipLaunchKernelGGL(k_offsets_part, dim3((unsigned)first_chunk(npoints, nfields)), dim3(kBlock), 0, s, d_fields,
                           nfields, d_val, d_part);
        FB_HIP_CHECK(hipGetLastError());
        hipLaunchKernelGGL(k_offsets_final, dim3(nblocks((int64_t)nfields * 64)), dim3(kBlock), 0, s, d_fields,
                           nfields, (const double *)d_part, d_offsets);
    }
    FB_HIP_CHECK(hipGetLastError());
    return FB_OK;
}

int launch_sort_begin(const FieldDev *d_fields, int nfields, int64_t npoints, const double *d_val, double *d_part,
                      const ZeroRange (&zero)[3], hipStream_t s)
{
    const int64_t noff = first_chunk(npoints, nfields);
    int64_t nz = 0;
    for (const ZeroRange &z : zero) nz += zero_blocks<kBlock, kZeroPer>(z);
    hipLaunchKernelGGL(k_sort_begin, dim3((unsigned)(noff + std::max<int64_t>(nz, 1))), dim3(kBlock), 0, s, d_fields,
                       nfields, d_val, d_part, noff, zero[0], zero[1], zero[2]);
    FB_HIP_CHECK(hipGetLastError());
    return FB_OK;
}

int launch_point_keys(const FieldDev *d_fields, const int64_t *d_pt_prefix, int nfields, int64_t npoints,
                      const double *d_pts, const double *d_val, uint32_t *d_keys, uint32_t *d_row_count,
                      uint32_t *d_slot, int64_t max_rows, PointRec *d_rec, const double *d_part, double *d_offsets,
                      hipStream_t s)
{
    if (nfields <= 0) return FB_OK;
    const unsigned nfin = nblocks((int64_t)nfields * 64);
    // points per thread: enough for each workgroup to see many points per row, while keeping
    // at least ~512 workgroups; small point sets, and fields with more rows than the LDS
    // counters (a workgroup of k_point_keys_hist over them would take one atomic per point, for
    // several points per thread), take one atomic per point and one point per thread
    const int64_t q = npoints / (512 * (int64_t)kBlock);
    const int64_t ppt = q < kKeysMaxPpt ? q : kKeysMaxPpt;
    if (ppt >= 4 && max_rows <= kKeysBinsMax) {
        // 64 KB of counters only where the fields need them (they halve the workgroups per CU;
        // fast_pass_init raised the kernel's dynamic-LDS limit)
        const int nbins = max_rows <= kKeysBins ? kKeysBins : kKeysBinsMax;
        const int64_t per = ppt * kBlock, nkb = (npoints + per - 1) / per;
        hipLaunchKernelGGL(k_point_keys_hist, dim3((unsigned)(nkb + nfin)), dim3(kBlock), (size_t)nbins * 4, s,
                           d_fields, d_pt_prefix, nfields, npoints, (int)ppt, nbins, d_pts, d_val, d_keys, d_row_count, d_slot,
                           d_rec, nkb, d_part, d_offsets);
    } else {
        const int64_t nkb = npoints > 0 ? nblocks(npoints) : 0;
        hipLaunchKernelGGL(k_point_keys, dim3((unsigned)(nkb + nfin)), dim3(kBlock), 0, s, d_fields, d_pt_prefix,
                           nfields, npoints, d_pts, d_val, d_keys, d_row_count, d_slot, d_rec, nkb, d_part, d_offsets);
    }
    FB_HIP_CHECK(hipGetLastError());
    return FB_OK;
}

int launch_inject_records(const FieldDev *d_fields, const int64_t *d_pt_prefix, int nfields, int64_t npoints,
                          int64_t nxlines, const uint32_t *d_vals, const uint32_t *d_row_start,
                          const uint32_t *d_row_count, const double *d_pts, const double *d_val,
                          const double *d_offsets, InjectRec *d_irec, hipStream_t s)
{
    if (npoints <= 0 || nxlines <= 0) return FB_OK;
    if (!d_irec) {
        set_error("FP64 injection: the plan has no record array");
        return FB_ERR_INVALID_ARGUMENT;
    }
    hipLaunchKernelGGL(k_inject_records, dim3((unsigned)((npoints + kBlock - 1) / kBlock)), dim3(kBlock), 0, s,
                       d_fields, d_pt_prefix, nfields, npoints, nxlines, d_vals, d_row_start,
                       d_row_count, d_pts, d_val, d_offsets, d_irec);
    FB_HIP_CHECK(hipGetLastError());
    return FB_OK;
}

int launch_inject_cells(const FieldDev *d_fields, int64_t npoints, const InjectRec *d_irec,
                        const uint32_t *d_row_start, const uint32_t *d_row_count, double *d_vg, double *d_wg, int dim,
                        bool zeroed, hipStream_t s)
{
    if (npoints <= 0) return FB_OK;
    if (!d_irec) {
        set_error("FP64 injection: the plan has no record array");
        return FB_ERR_INVALID_ARGUMENT;
    }
    return launch_parts(((npoints << dim) + kBlock - 1) / kBlock, kBlock, [&](int64_t first, unsigned count) {
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(count), dim3(kBlock), 0, s, d_fields, first, npoints, d_irec, d_row_start,
                               d_row_count, d_vg, d_wg);
        };
        if (dim == 1) zeroed ? launch(k_inject_cells<1, true>) : launch(k_inject_cells<1, false>);
        else if (dim == 2) zeroed ? launch(k_inject_cells<2, true>) : launch(k_inject_cells<2, false>);
        else zeroed ? launch(k_inject_cells<3, true>) : launch(k_inject_cells<3, false>);
        FB_HIP_CHECK(hipGetLastError());
        return FB_OK;
    });
}

int launch_exact_lines(const FieldDev *d_fields, const int64_t *d_line_prefix, int nfields, int64_t nslots,
                       int axis, int rect_len, double *d_vg, double *d_wg, double *d_vs, double *d_ws, hipStream_t s)
{
    if (nslots <= 0) return FB_OK;
    hipLaunchKernelGGL(k_exact_lines, dim3((unsigned)((nslots + kExactLineThreads - 1) / kExactLineThreads)),
                       dim3(kExactLineThreads), 0, s, d_fields, d_line_prefix, nfields, nslots, axis, rect_len, d_vg,
                       d_wg, d_vs, d_ws);
    FB_HIP_CHECK(hipGetLastError());
    return FB_OK;
}

int launch_exact_finalize(const FieldDev *d_fields, const int64_t *d_cell_prefix, int nfields, int64_t ncells,
                          const double *d_vg, const double *d_wg, const double *d_offsets, float *d_out,
                          hipStream_t s)
{
    if (ncells <= 0) return FB_OK;
    hipLaunchKernelGGL(k_exact_finalize, dim3(nblocks(ncells)), dim3(kBlock), 0, s, d_fields, d_cell_prefix,
                       nfields, ncells, d_vg, d_wg, d_offsets, d_out);
    FB_HIP_CHECK(hipGetLastError());
    return FB_OK;
}

int launch_mask(const FieldDev *d_fields, const int64_t *d_cell_prefix, int nfields, int64_t ncells, double *d_wg,
                int fast, hipStream_t s)
{
    if (ncells <= 0) return FB_OK;
    hipLaunchKernelGGL(k_mask, dim3(nblocks(ncells)), dim3(kBlock), 0, s, d_fields, d_cell_prefix, nfields, ncells,
                       d_wg, fast);
    FB_HIP_CHECK(hipGetLastError());
    return FB_OK;
}

int fast_pass_max_lds() { return 160 * 1024; }

// Raises the dynamic-LDS limit of the line passes and of k_point_keys_hist once per process
// (before any stream capture, where attribute calls are not allowed).
int fast_pass_init()
{
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [] {
        const void *fns[] = {
#define FB_FN(S) (const void *)k_fast_pass<true, S>, (const void *)k_fast_pass<false, S>,
            FB_FAST_SEGS(FB_FN)
#undef FB_FN
#define FB_FN(S) (const void *)k_prefix_pass<true, S>, (const void *)k_prefix_pass<false, S>,
            FB_PFX_SEGS(FB_FN)
#undef FB_FN
        };
        for (const void *fn : fns) {
            err = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, fast_pass_max_lds());
            if (err != hipSuccess) break;
        }
        if (err == hipSuccess)   // the point keys' row counters
            err = hipFuncSetAttribute((const void *)k_point_keys_hist, hipFuncAttributeMaxDynamicSharedMemorySize,
                                      kKeysBinsMax * (int)sizeof(uint32_t));
    });
    if (err != hipSuccess) {
        (void)hipGetLastError();
        set_error(std::string("hipFuncSetAttribute failed: ") + hipGetErrorString(err));
        return FB_ERR_HIP;
    }
    return exact_stream_init();
}

bool fast_pass_seg_supported(int kind, int seg)
{
    if (kind == kPassPrefix) {
        switch (seg) {
#define FB_CASE(S) case S:
            FB_PFX_SEGS(FB_CASE)
#undef FB_CASE
            return true;
        default:
            return false;
        }
    }
    switch (seg) {
#define FB_CASE(S) case S:
        FB_FAST_SEGS(FB_CASE)
#undef FB_CASE
        return true;
    default:
        return false;
    }
}

int launch_fast_pass(int kind, bool inject, int seg, const FieldDev *d_fields, const double *d_offsets,
                     const PassWork *d_work, int nwork, const PassField *d_pass, int threads, size_t lds_bytes,
                     const PointRec *d_rec, const uint32_t *d_vals, const uint32_t *d_line_start,
                     const uint32_t *d_line_count, const double *d_val, float *d_v, float *d_w,
                     float *d_out, float *d_wsave, int final_pass, const float *d_adj_g, hipStream_t s)
{
    if (nwork <= 0) return FB_OK;
    if (threads != 128 && threads != 256 && threads != kFastBlock) {
        set_error("fast pass: unsupported workgroup size");
        return FB_ERR_UNSUPPORTED;
    }
    if (!fast_pass_seg_supported(kind, seg)) {
        set_error("fast pass: unsupported segment length " + std::to_string(seg));
        return FB_ERR_UNSUPPORTED;
    }
#define FB_LAUNCH(K, S)                                                                                            \
    case S:                                                                                                        \
        if (inject)                                                                                                \
            hipLaunchKernelGGL((K<true, S>), dim3(nwork), dim3(threads), lds_bytes, s, d_fields, d_offsets, d_work, \
                               d_pass, d_rec, d_vals, d_line_start, d_line_count, d_val, d_v, d_w, d_out,           \
                               d_wsave, final_pass, d_adj_g);                                                      \
        else                                                                                                       \
            hipLaunchKernelGGL((K<false, S>), dim3(nwork), dim3(threads), lds_bytes, s, d_fields, d_offsets,        \
                               d_work, d_pass, d_rec, d_vals, d_line_start, d_line_count, d_val, d_v, d_w,          \
                               d_out, d_wsave, final_pass, d_adj_g);                                               \
        break;
#define FB_LAUNCH_SLIDE(S) FB_LAUNCH(k_fast_pass, S)
#define FB_LAUNCH_PFX(S) FB_LAUNCH(k_prefix_pass, S)
    if (kind == kPassPrefix) {
        switch (seg) { FB_PFX_SEGS(FB_LAUNCH_PFX) default: break; }
    } else {
        switch (seg) { FB_FAST_SEGS(FB_LAUNCH_SLIDE) default: break; }
    }
#undef FB_LAUNCH_PFX
#undef FB_LAUNCH_SLIDE
#undef FB_LAUNCH
    FB_HIP_CHECK(hipGetLastError());
    return FB_OK;
}

int launch_adj_gather(const FieldDev *d_fields, const int64_t *d_pt_prefix, int nfields, int dim, int64_t npoints,
                      const double *d_pts, const double *d_val, const double *d_offsets, const float *d_A,
                      const float *d_Bb, const PassField *d_pass_y, double *d_gval, double *d_gpts, hipStream_t s)
{
    if (npoints <= 0) return FB_OK;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(nblocks(npoints)), dim3(kBlock), 0, s, d_fields, d_pt_prefix, nfields, npoints,
                           d_pts, d_val, d_offsets, d_A, d_Bb, d_pass_y, d_gval, d_gpts);
    };
    if (dim == 1) launch(k_adj_gather<1>);
    else if (dim == 2) launch(k_adj_gather<2>);
    else launch(k_adj_gather<3>);
    FB_HIP_CHECK(hipGetLastError());
    return FB_OK;
}

int launch_zero(void *p, int64_t bytes, hipStream_t s)
{
    const int64_t n = bytes / 4;
    if (n <= 0) return FB_OK;
    if (((uintptr_t)p & 15) == 0 && n >= 4 * kBlock)
        hipLaunchKernelGGL(k_zero_u32x4, dim3(nblocks((n + 3) / 4)), dim3(kBlock), 0, s, (uint32_t *)p, n);
    else
        hipLaunchKernelGGL(k_zero_u32, dim3(nblocks(n)), dim3(kBlock), 0, s, (uint32_t *)p, n);
    FB_HIP_CHECK(hipGetLastError());
    return FB_OK;
}

int launch_f64_to_f32(const double *in, float *out, int64_t n, hipStream_t s)
{
    if (n <= 0) return FB_OK;
    hipLaunchKernelGGL(k_f64_to_f32, dim3(nblocks(n)), dim3(kBlock), 0, s, in, out, n);
    FB_HIP_CHECK(hipGetLastError());
    return FB_OK;
}

int launch_f32_to_f64(const float *in, double *out, int64_t n, double scale, hipStream_t s)
{
    if (n <= 0) return FB_OK;
    hipLaunchKernelGGL(k_f32_to_f64, dim3(nblocks(n)), dim3(kBlock), 0, s, in, out, n, scale);
    FB_HIP_CHECK(hipGetLastError());
    return FB_OK;
}

}  // namespace fb
