// fb_line_choice.h -- how an axis of the FP64 path runs (host code): through LDS rings (k_exact_stream) and with
// how many iterations to a launch, or a thread per line (k_exact_lines).
#pragma once

#include <algorithm>
#include <vector>

#include "fb_internal.h"

namespace fb {

// A ring pass takes its ticks per workgroup of 8 lines, the blocks of a line and the iterations' lag, as often
// as workgroups follow each other on the LDS that their rings leave them.  More iterations to a launch
// spare passes over the grids; fewer let more workgroups run at once, which counts where there are many of short
// lines: 8 iterations of 400000 y lines of 64 nodes 3228 us in one launch, 1673 in two, 1689 in three, 2793 in
// eight; 4 iterations of 2400 lines of 1200 nodes (T = 27) 59 in one, 106 in two.  A thread per line runs every iteration over memory and needs many
// neighbouring lines to hide its chain of dependent steps, so the shortest lines of large grids are left to the
// threads: z lines of 1000x1000x6 at 4 iterations 1991 us through rings, 209 by threads, of 512x512x16 474
// and 141; but of 151x133x61 64 and 74.  Along x its accesses are strided and cost more the longer the lines:
// 128000 lines of 6 nodes at 8 iterations 1034 and 59, of 12 1008 and 252, of 22 1053 and 860 (all iterations in
// one launch; of 30 nodes 1008 so, 350 in launches of fewer).
//
// The times are estimated, from a least-squares fit to what was measured of 2260 ring passes (lines of 6 to 2400
// nodes, 1000 to 400000 of them, T = 0 to 100, 2 to 12 iterations of which 1 to 8 to a launch; 17 % off
// in the mean) and of 600 passes by threads (lines of up to 256 nodes, along x up to 16; 20 % off).  A choice other
// than the most iterations to a launch through rings is taken where its estimate is clearly lower: 0.85 of it
// for fewer iterations, and 0.7 (y, z) or 0.6 (x) of the rings' best for the threads.  Of the shapes measured
// one lost more than 5 % by that (8000 lines of 1000 nodes at 12 iterations, 464 us instead of 419).
class AxisLines {
public:
    explicit AxisLines(int axis) : x_(axis == 0) {}
    // one field's lines; rect: the kernel's terms
    void add(int64_t len, int64_t lines, int64_t rect, int num_iter)
    {
        max_len_ = std::max(max_len_, len);
        max_rect_ = std::max(max_rect_, rect);
        max_iter_ = std::max(max_iter_, num_iter);
        cells_ += (len * lines + 63) / 64 * 64;
        const Lines l{len, lines, (rect - 1) / 2, num_iter, 1};
        if (!lines_.empty() && lines_.back().same(l)) ++lines_.back().fields;
        else lines_.push_back(l);
    }
    // the rings' geometry; ni = 0: a thread per line
    LineGeom geom() const
    {
        const LineGeom most = line_geom(max_rect_, max_iter_, max_len_);
        if (!most.ni || max_iter_ > kMostIter) return most;
        const double most_us = rings(most);
        LineGeom g = most;
        double us = most_us;
        for (int ni = most.ni - 1; ni >= 1; --ni) {
            const LineGeom c = line_geom(max_rect_, ni, max_len_);
            const double t = rings(c);
            if (t < us && t < 0.85 * most_us) {
                g = c;
                us = t;
            }
        }
        // (k_exact_lines and k_exact_finalize have a work-item per line and per cell in one launch: 2^32)
        if (max_len_ <= (x_ ? 16 : 256) && cells_ <= 0xFFFFFF00ll && threads() < (x_ ? 0.6 : 0.7) * us)
            return LineGeom();
        return g;
    }

private:
    static constexpr int kMostIter = 1000;   // iterations up to which the estimates, a sum over launches, are formed
    struct Lines {
        int64_t len, lines, T;
        int num_iter;
        int64_t fields;
        bool same(const Lines &o) const
        {
            return len == o.len && lines == o.lines && T == o.T && num_iter == o.num_iter;
        }
    };
    double rings(const LineGeom &g) const
    {
        const int waves = (g.ni + 64 / kLineSlots - 1) / (64 / kLineSlots) + 3;
        // registers leave a SIMD 4 waves, 5 along x
        const int resident = std::min(kLineLdsMax / (int)g.lds, 4 * (x_ ? 5 : 4) / waves);
        const int64_t launch_lds = line_ring_doubles(g.R) * (int64_t)sizeof(double);
        double us = 6.9;
        for (int it0 = 0; it0 < max_iter_; it0 += g.ni) {
            double ticks = 0, wg_ticks = 0, lds = 0, cells = 0;
            for (const Lines &l : lines_) {
                const int64_t nf = std::min(g.ni, l.num_iter - it0);
                if (nf <= 0) continue;
                const double wgs = (double)((l.lines + kLineSlots / 2 - 1) / (kLineSlots / 2)) * l.fields;
                const double t = (double)(((l.len + kLineStep - 1) / kLineStep + nf * (2 + l.T / kLineStep) + 8) / 8 * 8);
                ticks = std::max(ticks, t);
                wg_ticks += wgs * t;
                lds += wgs * (double)(nf * launch_lds);
                cells += (double)l.len * l.lines * l.fields;
            }
            us += 0.7 + 0.546 * std::max(ticks, wg_ticks / (256.0 * resident)) + 31e-6 / 256 * lds + 2.45e-6 * cells;
        }
        return us;
    }
    double threads() const
    {
        double steps = 0, us = 0;
        for (const Lines &l : lines_) {
            const double cells = (double)l.len * l.lines * l.fields;
            const int sweeps = l.num_iter + (l.num_iter & 1);   // an odd number ends with a copy
            steps = std::max(steps, (double)l.num_iter * (l.len + l.T));
            us += cells * (x_ ? 3.6e-6 + 1.29e-6 * l.len * sweeps : 5.9e-6 + (5.2e-6 + 0.1e-6 * l.T) * sweeps);
        }
        return us + (x_ ? 6.1 + 0.116 * steps : 18.9 + 0.081 * steps);
    }

    bool x_;
    int64_t max_len_ = 1, max_rect_ = 1, cells_ = 0;
    int max_iter_ = 0;
    std::vector<Lines> lines_;
};

}  // namespace fb
