// fb_lines.hip -- FP64 line passes in the reference's operation order, all iterations of a
// pass streaming through LDS at once.
//
// _accumulate_tail_array (interpolation.py:484-533) runs num_iter iterations over a line, each a
// running sum: step k adds in[k+h0], subtracts in[k-h1] and writes the sum plus alpha times the
// two tail terms.  Iteration i's step k needs iteration i-1 only up to k+h0+1, so the iterations
// of one line overlap in time: k_exact_stream gives every iteration lanes of its own, four iterations
// of 16 slots to a wave, and they pass blocks of kLineStep outputs through LDS rings, each iteration
// h0/kLineStep + 2 blocks behind the one before it.  Every running sum still adds its terms in the reference's order, so
// the results are the reference's bits; the line's chain of dependent steps is num_iter times
// shorter, and the grids are read and written once per pass instead of once per iteration.
//
// Bound by the issue of one wave per 16 slots: a tick of 16 steps takes about 1150 cycles, of which
// the 80 FP64 operations take 320 (4 cycles each from one wave), the 18 16-byte LDS reads 200 and
// the 8 to 16 writes 220 to 430; LDS instructions cost the same for any number of active lanes,
// so the iterations of 16 slots share one wave.  Measured against a wave per 16 or 32 x lines that
// ran one iteration after the other through an LDS ring, and a thread per y or z line: one 2400x1200
// field, n = 4, T = 27: x 384 -> 89 us, y 300 -> 58 us (with the quotient, 15 us of its own before);
// 300x150: 77 -> 20 and 45 -> 17 us; 24 fields of 600x300: 158 -> 69 and 153 -> 75 us.  32 slots
// with two iterations to a wave: x 96, y 58 us for the large field, 65 and 86 us for the 24; a wave
// per iteration: 113 and 66, 73 and 92.  Reading the next tick's terms ahead of the steps (183 VGPRs
// instead of 101): 88 and 60 us, and 71 instead of 51 us for the lines of a 151x133x61 field.
#include <mutex>
#include <string>

#include "fb_launch.h"

namespace fb {

namespace {

constexpr int B = kLineStep;
constexpr int S = kLineSlots;
constexpr int kAhead = 8;      // blocks that the loader has in flight

// Orders this wave's LDS accesses before the barrier; global loads and stores stay in flight
// across it (they are never shared between the waves of a workgroup).
__device__ __forceinline__ void tick_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

struct StreamArgs {
    const FieldDev *fields;
    const int64_t *wg_prefix;   // first workgroup of each field
    int nfields;
    int axis;
    int rect_override;          // > 0: the kernel's length, else 2*T[axis]+1
    int it0;                    // iterations [it0, it0 + ni) of each field
    int ni;
    int R;                      // blocks per ring
    double *vg, *wg;
    const double *offsets;
    float *out;                 // last axis: the masked quotient goes here instead of vg, wg
    int64_t wg0;                // first workgroup of the launch (PARTS)
};

// LDS position of (position, slot) of a block or ring: pairs of positions adjacent, so that a
// wave's terms are read two per instruction; the pairs' stride keeps the loader's row-wise writes
// on different banks.
__device__ __forceinline__ int at_pos(int pos, int slot)
{
    return (pos >> 1) * (2 * S + 2) + 2 * slot + (pos & 1);
}

// N terms of a lane's ring from position `from` (its parity ODD): aligned 16-byte reads.
template <int N, int ODD>
__device__ __forceinline__ void read_terms(const double *in, int from, double (&r)[B + 2])
{
    const double2 *p = (const double2 *)(in + ((from - ODD) >> 1) * (2 * S + 2));
#pragma unroll
    for (int j = 0; j < (N + ODD + 1) / 2; ++j) {
        const double2 x = p[j * (S + 1)];
        r[2 * j] = x.x;
        r[2 * j + 1] = x.y;
    }
}

// What a lane of the iterations' waves needs of its workgroup: its own iteration of its slot.
struct IterLane {
    const double *in;     // ring read, at the lane's slot
    double *out;          // ring or output blocks written, at the lane's slot
    int h0, h1, L;
    int lag, qend;        // first tick, end of the blocks it writes
    int ticks, R;
    int nout;             // blocks of the output ring (2: the output blocks, which have no mirror)
    double alpha;
};

// The lane's iteration over its line, B steps per tick.  OA, OB: the parities of the first
// entering and leaving positions of a block (h0 and h1).
template <bool TAIL, int OA, int OB>
__device__ void run_iterations(const IterLane &I)
{
    const int ringlen = I.R * B;
    double accu = 0.0;
    int pa = I.h0 % ringlen;              // ring positions of the next block's first terms
    int pb = (ringlen - I.h1 % ringlen) % ringlen;
    int blk = 0;                          // the next block in the output
    for (int t = 0; t < I.ticks; ++t) {
        const int q = t - I.lag;
        if (q >= 0 && q < I.qend) {
            if (q == 0)
                for (int k = 0; k < I.h0; ++k) accu += I.in[at_pos(k, 0)];   // h0 <= ringlen
            double a[B + 2], b[B + 2], o[B];
            read_terms<B + 1, OA>(I.in, pa, a);
            read_terms<B, OB>(I.in, pb, b);
            pa += B;
            pb += B;
            if (pa >= ringlen) pa -= ringlen;
            if (pb >= ringlen) pb -= ringlen;
            const int left = I.L - q * B;
            double *const w = I.out + at_pos(blk * B, 0);
#pragma unroll
            for (int j = 0; j < B; ++j) {
                accu += (a[j + OA] - b[j + OB]);
                o[j] = TAIL ? accu + I.alpha * (b[j + OB] + a[j + 1 + OA]) : accu;
                if (j & 1) *(double2 *)(w + at_pos(j - 1, 0)) = make_double2(o[j - 1], o[j]);
            }
            if (left < B) {   // the line ends within the block, or before it
#pragma unroll
                for (int j = 0; j < B; ++j)
                    if (j >= left) w[at_pos(j, 0)] = o[j] = 0.0;
            }
            if (blk == 0 && I.nout > 2) {
                double *const wm = I.out + at_pos(ringlen, 0);
#pragma unroll
                for (int j = 0; j < B; j += 2)
                    *(double2 *)(wm + at_pos(j, 0)) = make_double2(o[j], o[j + 1]);
            }
            blk = blk + 1 == I.nout ? 0 : blk + 1;
        }
        tick_barrier();
    }
}

// One workgroup: S/2 lines of one field, v and w of each (slot = c*S/2 + l).
//   wave 0          loads the lines' blocks, kAhead blocks in flight, into ring 0
//   next waves      the iterations i = 1..nf, 64/S to a wave: lane = (iteration, slot), ring i-1
//                   in, ring i out
//   last two waves  store iteration nf's blocks, half each, or form the float32 result from them
// nf: the field's share of the launch's ni iterations.  A tick ends with a barrier; in tick t
// the loader writes block t, iteration i runs block t - i*(d+1) with d = 1 + h0/B (its terms
// reach d blocks ahead, finished the tick before), the storing waves run one block later.
//
// A ring holds R blocks of B positions and its first block once more past its end, so that a
// wave's terms take immediate offsets from two addresses.  Positions outside the line read as
// zeros: the rings start cleared and every writer sends zeros for positions past the end.  Adding
// or subtracting +0.0 leaves a running sum that started from 0.0 unchanged, so the reference's
// phases at the line ends need no code of their own.
//
// PARTS: the launch takes the workgroups from A.wg0 on.  Of its own, since the offset in every launch's
// code cost the steps of all (another register order): 2400x1200, T = 27, x 90.5 -> 95.0, y 58.6 -> 61.1 us.
template <bool ROWS, bool PARTS>
__global__ __launch_bounds__(kLineWavesMax * 64) void k_exact_stream(StreamArgs A)
{
    constexpr int HL = S / 2;
    constexpr int M = B * S / 64;          // doubles per lane of a loaded block
    extern __shared__ __attribute__((aligned(16))) double lds[];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int64_t b = PARTS ? A.wg0 + blockIdx.x : blockIdx.x;
    const int f = find_seg(A.wg_prefix, A.nfields, b);
    const FieldDev &F = A.fields[f];
    const int nf = min(A.ni, F.num_iter - A.it0);
    if (nf <= 0) return;
    const int axis = ROWS ? 0 : A.axis;
    const int64_t W = F.size[0], H = F.size[1], D = F.size[2];
    const int L = (int)F.size[axis];
    const int64_t nlines = axis == 0 ? H * D : axis == 1 ? W * D : W * H;
    const int64_t l0 = (b - A.wg_prefix[f]) * HL;
    const int nl = (int)min((int64_t)HL, nlines - l0);
    const int rect = A.rect_override > 0 ? A.rect_override : 2 * F.T[axis] + 1;
    const int h0 = (rect - 1) / 2, h1 = rect - h0;
    const int d = 1 + h0 / B;
    const int NT = (L + B - 1) / B;
    const int ring_doubles = line_ring_doubles(A.R);
    double *const obuf = lds + nf * ring_doubles;       // two blocks
    const bool fin = A.out && A.it0 + nf == F.num_iter;
    const int last = nf * (d + 1) + 1;                  // the storing waves' lag
    const int ticks = (NT + last + kAhead - 1) / kAhead * kAhead;

    for (int i = threadIdx.x; i < nf * ring_doubles; i += blockDim.x) lds[i] = 0.0;
    __syncthreads();

    // offset of a line's first element in the field, and between its elements
    auto line_base = [&](int l) -> int64_t {
        const int64_t g = l0 + l;
        if (axis == 0) return g * W;
        if (axis == 2) return g;
        const uint32_t z = (uint32_t)g / (uint32_t)W;   // a plan's cells are counted in 32 bits
        return g + (int64_t)z * W * (H - 1);
    };
    const int64_t st = ROWS ? 1 : axis == 1 ? W : W * H;

    if (wave == 0) {
        // element m of a block as this lane loads it: along rows its neighbours are the next
        // positions, else the next lines
        auto pos_of = [&](int m) { return ROWS ? (lane & (B - 1)) : (m * 64 + lane) / S; };
        auto slot_of = [&](int m) { return ROWS ? (m * 64 + lane) / B : (lane & (S - 1)); };
        const double *src[M];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int sl = slot_of(m), l = min(sl & (HL - 1), nl - 1);
            src[m] = (sl >= HL ? A.wg : A.vg) + F.cell_off + line_base(l);
        }
        double pre[kAhead][M];
        // block q's elements (past the line's end: any of its elements, sent as zeros below)
        auto fetch = [&](double (&p)[M], int q) {
            if ((q + 1) * B <= L) {
                const int64_t at = (int64_t)(q * B + pos_of(0)) * st;
                const int64_t next = ROWS ? 0 : (64 / S) * st;
#pragma unroll
                for (int m = 0; m < M; ++m) p[m] = src[m][at + m * next];
            } else {
#pragma unroll
                for (int m = 0; m < M; ++m) p[m] = src[m][(int64_t)min(q * B + pos_of(m), L - 1) * st];
            }
            // the loads stay in block order, so that the wait for one block leaves the next in flight
            asm volatile("" ::: "memory");
        };
#pragma unroll
        for (int u = 0; u < kAhead; ++u) fetch(pre[u], u);
        int blk = 0;   // t mod R
        for (int t0 = 0; t0 < ticks; t0 += kAhead) {
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int t = t0 + u;
                double *const o = lds + at_pos(blk * B, 0);
                const int mirror = at_pos(A.R * B, 0);
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    if (!(t * B + pos_of(m) < L)) pre[u][m] = 0.0;
                    o[at_pos(pos_of(m), slot_of(m))] = pre[u][m];
                }
                if (blk == 0) {
#pragma unroll
                    for (int m = 0; m < M; ++m) o[at_pos(pos_of(m), slot_of(m)) + mirror] = pre[u][m];
                }
                fetch(pre[u], t + kAhead);
                blk = blk + 1 == A.R ? 0 : blk + 1;
                tick_barrier();
            }
        }
        return;
    }

    const int iter_waves = (A.ni + 64 / S - 1) / (64 / S);
    if (wave <= iter_waves) {
        const int i = (wave - 1) * (64 / S) + lane / S + 1;
        const bool to_ring = i < nf;
        IterLane I;
        I.in = lds + (i - 1) * ring_doubles + 2 * (lane & (S - 1));
        I.out = (to_ring ? lds + i * ring_doubles : obuf) + 2 * (lane & (S - 1));
        I.h0 = h0;
        I.h1 = h1;
        I.L = L;
        I.lag = i * (d + 1);
        I.qend = i > nf ? 0 : to_ring ? NT + d : NT;   // the next iteration reads d blocks past the line
        I.ticks = ticks;
        I.R = A.R;
        I.nout = to_ring ? A.R : 2;
        I.alpha = F.alpha[axis];
        const int par = (h0 & 1) | (h1 & 1) << 1;
#define FB_ITER(T_)                                       \
    if (par == 1) run_iterations<T_, 1, 0>(I);         \
    else if (par == 2) run_iterations<T_, 0, 1>(I);    \
    else if (par == 3) run_iterations<T_, 1, 1>(I);    \
    else run_iterations<T_, 0, 0>(I)
        if (F.tail) {
            FB_ITER(true);
        } else {
            FB_ITER(false);
        }
#undef FB_ITER
        return;
    }

    const int half = wave - (iter_waves + 1);
    const double off = fin ? A.offsets[f] : 0.0;
    const double thr = F.thr;
    // This wave's values of a block: (position, line) pairs, every other group of 64, with v and w
    // of each; the lane's neighbours as in the loader.
    constexpr int MS = B * HL / 128;
    const double *ob[MS];
    int64_t base[MS];
    int pos[MS];
#pragma unroll
    for (int m = 0; m < MS; ++m) {
        const int i = (2 * m + half) * 64 + lane;
        const int l = ROWS ? i / B : (i & (HL - 1));
        pos[m] = ROWS ? (i & (B - 1)) : i / HL;
        ob[m] = obuf + at_pos(pos[m], l);
        base[m] = l < nl ? line_base(l) + pos[m] * st : 0;
        if (l >= nl) pos[m] = L;          // stores nothing
    }
    double *const gv = A.vg + F.cell_off, *const gw = A.wg + F.cell_off;
    float *const go = fin ? A.out + F.out_off : nullptr;
    for (int t = 0; t < ticks; ++t) {
        const int q = t - last;
        if (q >= 0 && q < NT) {
            const int64_t at = (int64_t)(q * B) * st;
            const int ofs = (q & 1) * at_pos(B, 0);
#pragma unroll
            for (int m = 0; m < MS; ++m) {
                const double v = ob[m][ofs], w = ob[m][ofs + 2 * HL];
                if (q * B + pos[m] < L) {
                    if (fin) {   // wg[wg < thr] = NaN, then (vg/wg + offset).astype(float32): :428-430, :367
                        go[base[m] + at] = (w < thr) ? __builtin_nanf("") : (float)(v / w + off);
                    } else {
                        gv[base[m] + at] = v;
                        gw[base[m] + at] = w;
                    }
                }
            }
        }
        tick_barrier();
    }
}

}  // namespace

int exact_stream_init()
{
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [] {
        for (const void *fn : {(const void *)k_exact_stream<true, false>, (const void *)k_exact_stream<false, false>,
                               (const void *)k_exact_stream<true, true>, (const void *)k_exact_stream<false, true>})
            if (err == hipSuccess)
                err = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kLineLdsMax);
    });
    FB_HIP_CHECK(err);
    return FB_OK;
}

int launch_exact_stream(const FieldDev *d_fields, const int64_t *d_wg_prefix, int nfields, int64_t nwg, int axis,
                        int rect_override, const LineGeom &g, int max_iter, double *d_vg, double *d_wg,
                        const double *d_offsets, float *d_out, hipStream_t s)
{
    if (nwg <= 0) return FB_OK;
    if (!g.ni) {
        set_error("FP64 lines: the kernel is too wide for the LDS rings");
        return FB_ERR_UNSUPPORTED;
    }
    StreamArgs a{d_fields, d_wg_prefix, nfields, axis, rect_override, 0, g.ni, g.R, d_vg, d_wg, d_offsets, d_out, 0};
    const int threads = 64 * ((g.ni + 64 / S - 1) / (64 / S) + 3);
    for (a.it0 = 0; a.it0 < max_iter; a.it0 += g.ni) {
        const int rc = launch_parts(nwg, threads, [&](int64_t first, unsigned count) {
            a.wg0 = first;
            auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(count), dim3(threads), g.lds, s, a); };
            if (count == nwg) axis == 0 ? launch(k_exact_stream<true, false>) : launch(k_exact_stream<false, false>);
            else axis == 0 ? launch(k_exact_stream<true, true>) : launch(k_exact_stream<false, true>);
            FB_HIP_CHECK(hipGetLastError());
            return FB_OK;
        });
        if (rc) return rc;
    }
    return FB_OK;
}

}  // namespace fb
