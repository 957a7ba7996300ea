// fb_launch.h -- host-side launchers shared between translation units.
#pragma once

#include "fastbarnes.h"
#include <algorithm>

#include "fb_internal.h"

namespace fb {

// A launch holds fewer than 2^32 work-items; larger grids run in parts.  launch(first, count) takes the
// workgroups [first, first + count) of nwg and returns its status.
template <class F>
inline int launch_parts(int64_t nwg, int threads, F launch)
{
    const int64_t most = 0xFFFFFFFFll / threads;
    for (int64_t first = 0; first < nwg; first += most)
        if (const int rc = launch(first, (unsigned)std::min(most, nwg - first))) return rc;
    return FB_OK;
}

// fb_sort.hip
// The whole sort stage of fields of at most kLocalSortMax points and kLocalRowsMax x-lines, one
// workgroup each: the value offset (0 with `raw`), the rows' counts and starts (the range of field f
// begins at pt_prefix[f]) and the in-grid points in the row buckets' order: the point list (d_out_vals)
// with each point's PointRec (d_rec), or, with d_irec, the list of FP64 injection records, whose
// unused slots get row kInvalidKey.  Further workgroups zero the ranges.
int field_sort_init();
int launch_field_sort(const FieldDev *d_fields, const int64_t *d_pt_prefix, int nfields, int dim, int max_n,
                      int max_rows, const double *d_pts, const double *d_val, bool raw, double *d_offsets,
                      uint32_t *d_row_count, uint32_t *d_row_start, uint32_t *d_out_vals, PointRec *d_rec,
                      InjectRec *d_irec, const ZeroRange (&zero)[2], hipStream_t stream);
// fb_sort.hip -- row buckets for all other plans: the row starts from the row counts (scan_tiles(nrows)
// words of d_tiles), the in-grid points into their rows (d_comp), each
// row sorted by (key, point index) into d_list, which may be d_keys' memory.
int64_t scan_tiles(int64_t n);
int row_bucket_sort(const FieldDev *d_fields, const int64_t *d_pt_prefix, int nfields, const uint32_t *d_keys,
                    const uint32_t *d_slot, int64_t npoints, uint32_t *d_row_start, const uint32_t *d_row_count,
                    int64_t nrows, uint32_t *d_tiles, unsigned long long *d_comp, uint32_t *d_list, hipStream_t stream);

// fb_kernels.hip -- injection front end
// (min+max)/2 per field; with d_part (offsets_part_elems doubles) large fields are reduced
// by many workgroups
int64_t offsets_part_elems(int nfields, int64_t npoints);
int launch_offsets(const FieldDev *d_fields, int nfields, int64_t max_n, int64_t npoints, const double *d_val,
                   double *d_part, double *d_offsets, hipStream_t stream);
// The row buckets' first two launches.  launch_sort_begin: the offsets' chunks (d_part) and the ranges
// zeroed.  launch_point_keys: the offsets from the chunks; each point's base cell,
// its base row's count (row = x-line index, integer atomics on zeroed counts) and its slot there.
// max_rows: the most x-lines of any field.  d_rec (may be NULL): each in-grid point's PointRec, for
// the FP32C injection
int launch_sort_begin(const FieldDev *d_fields, int nfields, int64_t npoints, const double *d_val, double *d_part,
                      const ZeroRange (&zero)[3], hipStream_t stream);
int launch_point_keys(const FieldDev *d_fields, const int64_t *d_pt_prefix, int nfields, int64_t npoints,
                      const double *d_pts, const double *d_val, uint32_t *d_keys, uint32_t *d_row_count,
                      uint32_t *d_slot, int64_t max_rows, PointRec *d_rec, const double *d_part, double *d_offsets,
                      hipStream_t stream);

// fb_kernels.hip -- FP64 path with the reference's operation order
// Each sorted entry's FP64 injection record (row buckets).
int launch_inject_records(const FieldDev *d_fields, const int64_t *d_pt_prefix, int nfields, int64_t npoints,
                          int64_t nxlines, const uint32_t *d_vals, const uint32_t *d_row_start,
                          const uint32_t *d_row_count, const double *d_pts, const double *d_val,
                          const double *d_offsets, InjectRec *d_irec, hipStream_t stream);
// The injection sums of every cell that receives any, in point order; the grids must be cleared
// (zeroed) or are added to.
int launch_inject_cells(const FieldDev *d_fields, int64_t npoints, const InjectRec *d_irec,
                        const uint32_t *d_row_start, const uint32_t *d_row_count, double *d_vg, double *d_wg, int dim,
                        bool zeroed, hipStream_t stream);
// One thread per (line, field component); lines of axis `axis` of every field.
// line_prefix[f] = first (2*line) slot of field f; total = line_prefix[nfields].
// rect_len < 0 selects 2*T[axis]+1 from the field.
int launch_exact_lines(const FieldDev *d_fields, const int64_t *d_line_prefix, int nfields, int64_t nslots,
                       int axis, int rect_len, double *d_vg, double *d_wg, double *d_vs, double *d_ws,
                       hipStream_t stream);
// fb_lines.hip -- FP64 lines through LDS rings, all iterations at once (k_exact_stream), the same
// bits as launch_exact_lines: d_wg_prefix[f] = first workgroup of field f (ceil(lines / (kLineSlots/2))
// each, nwg in all), g = line_geom of the fields' widest kernel (2T+1 or rect_override) and
// max_iter = their most iterations.  d_out (last axis, may be NULL): the masked quotient is
// written there and the grids are left undefined.  FB_ERR_UNSUPPORTED when the rings do not fit
// the LDS (g.ni == 0): take launch_exact_lines then.
int exact_stream_init();
int launch_exact_stream(const FieldDev *d_fields, const int64_t *d_wg_prefix, int nfields, int64_t nwg, int axis,
                        int rect_override, const LineGeom &g, int max_iter, double *d_vg, double *d_wg,
                        const double *d_offsets, float *d_out, hipStream_t stream);
int launch_exact_finalize(const FieldDev *d_fields, const int64_t *d_cell_prefix, int nfields, int64_t ncells,
                          const double *d_vg, const double *d_wg, const double *d_offsets, float *d_out,
                          hipStream_t stream);
int launch_mask(const FieldDev *d_fields, const int64_t *d_cell_prefix, int nfields, int64_t ncells, double *d_wg,
                int fast, hipStream_t stream);

// fb_kernels.hip -- FP32C path
int fast_pass_max_lds();
int fast_pass_init();
bool fast_pass_seg_supported(int kind, int seg);
// kind: kPassSlide (k_fast_pass) or kPassPrefix (k_prefix_pass).  Injecting passes: d_vals is the
// sorted point list (rows' ranges d_line_start/d_line_count), d_rec and d_val each point's
// injection record and value by point index.  d_adj_g (first pass of the adjoint): the tile
// load forms a = g/W, b = -a(f - offset) from d_out = f, d_wsave = W, d_adj_g = g.
int launch_fast_pass(int kind, bool inject, int seg, const FieldDev *d_fields, const double *d_offsets, const PassWork *d_work,
                     int nwork, const PassField *d_pass, int threads, size_t lds_bytes, const PointRec *d_rec,
                     const uint32_t *d_vals, const uint32_t *d_line_start, const uint32_t *d_line_count,
                     const double *d_val, float *d_v, float *d_w, float *d_out,
                     float *d_wsave, int final_pass, const float *d_adj_g, hipStream_t stream);

// fb_kernels.hip -- adjoint of the FP32C batch
int launch_adj_gather(const FieldDev *d_fields, const int64_t *d_pt_prefix, int nfields, int dim, int64_t npoints,
                      const double *d_pts, const double *d_val, const double *d_offsets, const float *d_A,
                      const float *d_Bb, const PassField *d_pass_y, double *d_gval, double *d_gpts,
                      hipStream_t stream);

// fb_s2.hip -- spherical variant (proj = center_lon, n, n_inv, F, rho0)
int launch_lambert_points(const double *d_pts, double *d_out, int64_t n, const double *proj, hipStream_t stream);
int launch_resample(const float *d_lam, const int64_t *lam_size, const double *lam_x0, const double *x0,
                    const double *step, const int64_t *size, const double *proj, float *d_out, hipStream_t stream);
int launch_naive_s2(const double *d_pts, const double *d_val, const double *d_offset, int64_t n, double sigma,
                    const double *x0, const double *step, const int64_t *size, double *d_out, hipStream_t stream);

// fb_kernels.hip -- elementwise helpers
int launch_zero(void *p, int64_t bytes, hipStream_t stream);   // bytes: multiple of 4
int launch_f64_to_f32(const double *in, float *out, int64_t n, hipStream_t stream);
int launch_f32_to_f64(const float *in, double *out, int64_t n, double scale, hipStream_t stream);

// fb_naive.hip -- naive / radius sums in FP64.  naive_work_elems: doubles of workspace with which
// the naive sums run as matrix products (0: node by node); with d_work = NULL they run node by node.
int64_t naive_work_elems(int radius, int dim, const int64_t *size, int64_t n);
int launch_naive(const FieldDev *d_field, int radius, double radius_sqr, double max_dist_weight, int dim,
                 const int64_t *size, int64_t n, const double *d_pts, const double *d_val, const double *d_offsets,
                 double *d_work, double *d_out, hipStream_t stream);

}  // namespace fb
