// fb_naive.hip -- the exact Gaussian sums: method 'naive' (interpolation.py:861-938) and 'radius'
// (:809-855, brute force in place of the kd-tree, same inclusion test sqr_dist <= radius^2), FP64.
//
// The naive weight of station k at node (x, y, z) is a product of one factor per axis,
// exp(-dx^2/(2 sx^2)) exp(-dy^2/(2 sy^2)) exp(-dz^2/(2 sz^2)), so the two sums over the stations
// are matrix products of the factors: with A[m][k] = the y (and z) factors of grid row m and
// B[k][x] = the x factors, sum_k w = A B and sum_k w (val - offset) = A (B scaled by the values).
// The factors are tabulated (n (W + H + D) exponentials instead of n W H D) and the products run
// on the FP64 matrix cores.
#include <algorithm>
#include <climits>
#include <string>

#include "fb_launch.h"

namespace fb {

namespace {

constexpr int kBlock = 256;

typedef double dvec4 __attribute__((ext_vector_type(4)));

// The sums ws and wt of a workgroup's nodes by the reference's own formula, in station order: thread by
// thread the node g (`on`: its thread wants them), the stations in tiles through LDS.  Called by every
// thread of the workgroup.  FAR: most stations are so far that their weight is 0.0 (exp(-d) from d = 745.2
// on), which need no exponential.
constexpr double kZeroWeight = 750.0;

template <bool RADIUS, bool FAR>
__device__ __forceinline__ void node_sums(const FieldDev &F, double r2, const double *__restrict__ pts,
                                          const double *__restrict__ val, double off, int64_t g, bool on, double &ws,
                                          double &wt)
{
    __shared__ double sp[3][kBlock];
    __shared__ double sval[kBlock];
    const int tid = threadIdx.x;
    const int dim = F.dim;
    const int64_t W = F.size[0], H = F.size[1];
    const int64_t x = g % W, y = (g / W) % H, z = g / (W * H);
    const double c0 = F.x0[0] + (double)x * F.step[0];
    const double c1 = dim > 1 ? F.x0[1] + (double)y * F.step[1] : 0.0;
    const double c2 = dim > 2 ? F.x0[2] + (double)z * F.step[2] : 0.0;
    // scale = 2*sigma**2 per axis (interpolation.py:872)
    const double s0 = 2 * (F.sigma[0] * F.sigma[0]);
    const double s1 = 2 * (F.sigma[1] * F.sigma[1]);
    const double s2 = 2 * (F.sigma[2] * F.sigma[2]);
    ws = wt = 0.0;
    for (int64_t b = 0; b < F.n; b += kBlock) {
        __syncthreads();
        const int64_t k = b + tid;
        if (k < F.n) {
            for (int m = 0; m < dim; ++m) sp[m][tid] = pts[k * dim + m];
            sval[tid] = val[k] - off;
        }
        __syncthreads();
        const int cnt = (int)min((int64_t)kBlock, F.n - b);
        if (on) {
            if (!RADIUS) {
                for (int t = 0; t < cnt; ++t) {
                    const double d0 = sp[0][t] - c0;
                    double d = d0 * d0 / s0;
                    if (dim > 1) {
                        const double d1 = sp[1][t] - c1;
                        d = d + d1 * d1 / s1;
                    }
                    if (dim > 2) {
                        const double d2 = sp[2][t] - c2;
                        d = d + d2 * d2 / s2;
                    }
                    if (FAR && d > kZeroWeight) continue;
                    const double w = exp(-d);
                    ws += w * sval[t];
                    wt += w;
                }
            } else {
                for (int t = 0; t < cnt; ++t) {
                    const double dx = c0 - sp[0][t];
                    const double dy = c1 - sp[1][t];
                    const double d2 = dx * dx + dy * dy;
                    if (d2 <= r2) {
                        const double w = exp(-d2 / s0);
                        ws += w * sval[t];
                        wt += w;
                    }
                }
            }
        }
    }
}

// Both methods node by node, one thread each.
template <bool RADIUS>
__global__ __launch_bounds__(kBlock) void k_naive(const FieldDev *__restrict__ fp, double r2, double mdw,
                                                  const double *__restrict__ pts, const double *__restrict__ val,
                                                  const double *__restrict__ offsets, double *__restrict__ out,
                                                  int64_t ncells)
{
    const FieldDev F = *fp;
    const int64_t g = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const double off = offsets[0];
    double ws, wt;
    node_sums<RADIUS, false>(F, r2, pts, val, off, g, g < ncells, ws, wt);
    if (g < ncells) {
        if (!RADIUS) out[g] = wt > 0.0 ? ws / wt + off : __builtin_nan("");
        else out[g] = wt >= mdw ? ws / wt + off : __builtin_nan("");
    }
}

// ---- naive sums as matrix products ------------------------------------------

// Weights below this are summed again by the reference's formula: a sum this small may come from
// factors that underflow one by one, and the node is NaN where the sum itself does.  k_naive_finish does
// that, a thread per node; without parts it knows the nodes by kAgain, which k_naive_product leaves there
// (a NaN of that payload which came from a station's would be summed again as well, to the same NaN).
constexpr double kTinyWeight = 1e-280;
constexpr long long kAgain = 0x7ff8616761696e21ll;
constexpr int kTile = 64;    // rows and columns of a workgroup's tile, 32 x 32 to each of its 4 waves
constexpr int kStep = 4;     // stations of one matrix instruction
constexpr int kGroup = 16;   // stations whose factors a wave loads together

struct NaiveArgs {
    const FieldDev *field;
    const double *pts, *val, *offset;
    double *tx, *ty, *tz;    // factors of the station block, [station][node], rows of wp, hp, dp
    double *tv;              // the block's values minus the offset
    int64_t wp, hp, dp;
    int64_t k0;              // first station of the block
    int nk;                  // stations of the block, a multiple of kGroup (zeros past the last)
    int split, kper;         // parts of the block's stations, stations per part
    int first;               // the first block: the partial sums start here
    int tn;                  // tiles along x
    int64_t M;               // grid rows: H*D
    int64_t ntiles;
    double *part;            // partial sums, [part][w, v][row][x] with wp columns; NULL: none needed
    int64_t plane;           // doubles of one of them
    double *out;
};

// the factor tables of one station block: a thread takes one node of one axis for kGroup stations
__global__ __launch_bounds__(kBlock) void k_naive_factors(NaiveArgs A)
{
    const FieldDev &F = *A.field;
    const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const int kk0 = blockIdx.y * kGroup;
    if (blockIdx.x == 0 && threadIdx.x < kGroup) {
        const int64_t k = A.k0 + kk0 + threadIdx.x;
        A.tv[kk0 + threadIdx.x] = k < F.n ? A.val[k] - A.offset[0] : 0.0;
    }
    if (c >= A.wp + A.hp + A.dp) return;
    const int m = c < A.wp ? 0 : c < A.wp + A.hp ? 1 : 2;
    const int64_t j = m == 0 ? c : m == 1 ? c - A.wp : c - A.wp - A.hp;
    const int64_t len = m == 0 ? A.wp : m == 1 ? A.hp : A.dp;
    double *const t = (m == 0 ? A.tx : m == 1 ? A.ty : A.tz) + kk0 * len + j;
    const double x = F.x0[m] + (double)j * F.step[m];
    const double scale = 2 * (F.sigma[m] * F.sigma[m]);   // interpolation.py:872
    const bool node = j < F.size[m];
    for (int i = 0; i < kGroup; ++i) {
        const int64_t k = A.k0 + kk0 + i;
        double e = 0.0;
        if (node && k < F.n) {
            const double d = A.pts[k * F.dim + m] - x;
            e = exp(-(d * d / scale));
        }
        t[i * len] = e;
    }
}

// One 64 x 64 tile of grid rows and columns over one part of the block's stations.  A wave holds
// 2 x 2 tiles of 16 x 16 of both sums (64 registers); an instruction takes 4 stations, each lane
// one factor of a row (lane & 15) and one of a column of station lane >> 4.  The operands come
// straight from the tables, 16 stations ahead of the products: 32 rows and columns of 4 stations
// feed 8 instructions.  Lane l holds rows l/16 + 4 r, column l & 15 of a 16 x 16 result.
//
// Bound by the FP64 matrix rate.  3490 stations on 600x300 nodes (2.5 GFLOP): 65 us, 39 TFLOP/s
// (one group of 4 stations ahead: 89 us), with 15 us for the factors and 6 us for the parts' sums; a
// thread per node with an exponential per station took 1583 us.
template <int DIM>
__global__ __launch_bounds__(kBlock) void k_naive_product(NaiveArgs A)
{
    const FieldDev &F = *A.field;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r = lane & 15, kq = lane >> 4;
    const int64_t t = blockIdx.x % A.ntiles;
    const int part = (int)(blockIdx.x / A.ntiles);
    const int64_t m0 = t / A.tn * kTile + (wave >> 1) * 32, n0 = t % A.tn * kTile + (wave & 1) * 32;
    const int kbeg = part * A.kper, kend = min(kbeg + A.kper, A.nk);

    // this lane's factors: rows m0 + r and m0 + 16 + r (clamped; rows past the grid are not
    // stored), columns n0 + r and n0 + 16 + r (the tables have whole tiles of columns)
    const double *py[2], *pz[2];
    const double *px = A.tx + n0 + r;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int64_t m = min(m0 + 16 * i + r, A.M - 1);
        py[i] = A.ty + (DIM == 3 ? m % F.size[1] : m);
        pz[i] = DIM == 3 ? A.tz + m / F.size[1] : nullptr;
    }
    dvec4 aw[2][2], av[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) aw[i][j] = av[i][j] = (dvec4)(0.0);

    constexpr int G = kGroup / kStep;
    struct Group {
        double a[G][2], b[G][2], v[G];
    };
    auto load = [&](int k, Group &g) {
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const int64_t kk = k + kStep * u + kq;
            g.v[u] = A.tv[kk];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                g.a[u][i] = py[i][kk * A.hp];
                if (DIM == 3) g.a[u][i] *= pz[i][kk * A.dp];
                g.b[u][i] = px[kk * A.wp + 16 * i];
            }
        }
    };
    auto multiply = [&](const Group &g) {
#pragma unroll
        for (int u = 0; u < G; ++u)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const double bv = g.b[u][j] * g.v[u];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    aw[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(g.a[u][i], g.b[u][j], aw[i][j], 0, 0, 0);
                    av[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(g.a[u][i], bv, av[i][j], 0, 0, 0);
                }
            }
    };
    // two groups in turn, the next one's loads in flight under the products (past the part's end
    // the block's last group is loaded again and not used)
    Group g0, g1;
    if (kbeg < kend) load(kbeg, g0);
    for (int k = kbeg; k < kend; k += 2 * kGroup) {
        load(min(k + kGroup, A.nk - kGroup), g1);
        multiply(g0);
        if (k + kGroup >= kend) break;
        load(min(k + 2 * kGroup, A.nk - kGroup), g0);
        multiply(g1);
    }

    const int64_t W = F.size[0];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t m = m0 + 16 * i + kq + 4 * e, x = n0 + 16 * j + r;
                if (m >= A.M || x >= W) continue;
                if (!A.part) {
                    const double wt = aw[i][j][e];
                    A.out[m * W + x] = wt < kTinyWeight ? __longlong_as_double(kAgain) : av[i][j][e] / wt + A.offset[0];
                    continue;
                }
                double *const pw = A.part + (int64_t)(2 * part) * A.plane + m * A.wp + x, *const pv = pw + A.plane;
                *pw = A.first ? aw[i][j][e] : *pw + aw[i][j][e];
                *pv = A.first ? av[i][j][e] : *pv + av[i][j][e];
            }
}

// The parts' sums and the result of every node; without parts the nodes of tiny weight alone.  Where a
// workgroup has any, its threads sum them as k_naive does.  3490 stations of sigma 0.25 in a corner of a field
// of 75 degrees, a call on 600x300 nodes 1290 us, on 2400x1200 9.8 ms; node by node throughout 1700 us and 19.6
// ms; with a lane of k_naive_product for its 16 nodes one after the other, or a thread here without the LDS
// tiles, 2200 us and 22 ms.
__global__ __launch_bounds__(kBlock) void k_naive_finish(NaiveArgs A)
{
    const FieldDev &F = *A.field;
    const int64_t W = F.size[0], g = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const bool on = g < W * A.M;
    const double off = A.offset[0];
    double ws = 0.0, wt = 0.0;
    bool again = false;
    if (on && A.part) {
        const double *p = A.part + g / W * A.wp + g % W;
        for (int s = 0; s < A.split; ++s) {
            wt += p[(int64_t)(2 * s) * A.plane];
            ws += p[(int64_t)(2 * s + 1) * A.plane];
        }
        again = wt < kTinyWeight;
    } else if (on) {
        again = __double_as_longlong(A.out[g]) == kAgain;
    }
    if (__syncthreads_or(again)) {
        double s, t;
        node_sums<false, true>(F, 0.0, A.pts, A.val, off, g, again, s, t);
        if (again) {
            ws = s;
            wt = t;
        }
    }
    if (again || (on && A.part)) A.out[g] = wt > 0.0 ? ws / wt + off : __builtin_nan("");
}

int64_t up(int64_t a, int64_t b) { return (a + b - 1) / b * b; }

// How a field's naive sums run as products.  Stations are taken in blocks whose tables hold at
// most 64 MB; a block's stations are split over as many workgroups as 512 need, each part of at
// least 64 stations.
struct NaivePlan {
    int64_t wp, hp, dp, M, tn, ntiles, kb, plane;
    int split;
    bool parts;
};

NaivePlan naive_plan(int dim, const int64_t *size, int64_t n)
{
    NaivePlan p;
    p.wp = up(size[0], kTile);
    p.hp = size[1];
    p.dp = dim == 3 ? size[2] : 0;
    p.M = size[1] * (dim == 3 ? size[2] : 1);
    p.tn = p.wp / kTile;
    p.ntiles = p.tn * ((p.M + kTile - 1) / kTile);
    const int64_t fit = std::max<int64_t>(64, (64ll << 20) / (8 * (p.wp + p.hp + p.dp)) / 64 * 64);
    p.kb = std::min(up(n, kGroup), fit);
    p.split = (int)std::max<int64_t>(1, std::min<int64_t>(512 / std::max<int64_t>(1, p.ntiles), p.kb / 64));
    p.parts = p.split > 1 || p.kb < n;
    p.plane = p.M * p.wp;
    return p;
}

}  // namespace

// Products need a few rows and columns to fill their tiles; fields of one axis or of fewer than 16
// nodes along x or 16 rows run node by node (there is no more than an exponential per node and
// station to save, and little work in all).  So do few stations: node by node each takes 0.22 us, or 2 ps a
// node where those fill the chip, and the products' further launches 38 us more than the one (64 stations on
// 64x64 nodes 75 us a call, as products 105; 128 on 600x300 196 and 179, 16 on 1200x600 308 and 297).
int64_t naive_work_elems(int radius, int dim, const int64_t *size, int64_t n)
{
    const int64_t rows = size[1] * (dim == 3 ? size[2] : 1);
    if (radius || dim < 2 || size[0] < 16 || rows < 16) return 0;
    if ((double)n * std::max(0.22, 2e-6 * (double)size[0] * (double)rows) < 38.0) return 0;
    const NaivePlan p = naive_plan(dim, size, n);
    if (p.ntiles * p.split > INT32_MAX) return 0;
    return p.kb * (p.wp + p.hp + p.dp + 1) + (p.parts ? 2 * p.split * p.plane : 0);
}

int launch_naive(const FieldDev *d_field, int radius, double radius_sqr, double max_dist_weight, int dim,
                 const int64_t *size, int64_t n, const double *d_pts, const double *d_val, const double *d_offsets,
                 double *d_work, double *d_out, hipStream_t s)
{
    int64_t ncells = 1;
    for (int m = 0; m < dim; ++m) ncells *= size[m];
    if (ncells <= 0) return FB_OK;
    auto blocks = [](int64_t c) { return dim3((unsigned)((c + kBlock - 1) / kBlock)); };
    if (!d_work) {
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, blocks(ncells), dim3(kBlock), 0, s, d_field, radius_sqr, max_dist_weight, d_pts,
                               d_val, d_offsets, d_out, ncells);
        };
        radius ? launch(k_naive<true>) : launch(k_naive<false>);
        FB_HIP_CHECK(hipGetLastError());
        return FB_OK;
    }
    const NaivePlan p = naive_plan(dim, size, n);
    NaiveArgs a{};
    a.field = d_field;
    a.pts = d_pts;
    a.val = d_val;
    a.offset = d_offsets;
    a.tx = d_work;
    a.ty = a.tx + p.kb * p.wp;
    a.tz = a.ty + p.kb * p.hp;
    a.tv = a.tz + p.kb * p.dp;
    a.part = p.parts ? a.tv + p.kb : nullptr;
    a.wp = p.wp;
    a.hp = p.hp;
    a.dp = p.dp;
    a.split = p.split;
    a.tn = (int)p.tn;
    a.M = p.M;
    a.ntiles = p.ntiles;
    a.plane = p.plane;
    a.out = d_out;
    for (a.k0 = 0; a.k0 < n; a.k0 += p.kb) {
        a.nk = (int)std::min(p.kb, up(n - a.k0, kGroup));
        a.kper = (int)up((a.nk + p.split - 1) / p.split, kGroup);
        a.first = a.k0 == 0;
        const dim3 fgrid(blocks(p.wp + p.hp + p.dp).x, (unsigned)(a.nk / kGroup));
        hipLaunchKernelGGL(k_naive_factors, fgrid, dim3(kBlock), 0, s, a);
        const dim3 grid((unsigned)(p.ntiles * p.split));
        if (dim == 3) hipLaunchKernelGGL(k_naive_product<3>, grid, dim3(kBlock), 0, s, a);
        else hipLaunchKernelGGL(k_naive_product<2>, grid, dim3(kBlock), 0, s, a);
    }
    hipLaunchKernelGGL(k_naive_finish, blocks(ncells), dim3(kBlock), 0, s, a);
    FB_HIP_CHECK(hipGetLastError());
    return FB_OK;
}

}  // namespace fb
