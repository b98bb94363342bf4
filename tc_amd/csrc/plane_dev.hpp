// plane_dev.hpp -- device pieces of the plane-first pair pipeline (kernels_plane.hip): the
// workgroup shapes, the column runs and the row loads.
#pragma once

#include "kernels_common.hpp"

namespace tcx {

// Workgroups of the plane passes: R tiles (planes of a pair in pass A, pairs of a plane in
// pass C) of NP lines each, line t of tile r on thread r NP + t.
template <typename T, int NP>
struct PlaneWg {
    static constexpr int tile_bytes = (int)sizeof(PlaneTile<T, NP>);
    // tiles that fill w wavefronts, and the share of the lanes that they use in percent
    static constexpr int fit(int w) { return 64 * w / NP < NP ? 64 * w / NP : NP; }
    static constexpr int fill(int w)
    {
        const int lanes = fit(w) * NP;
        return 100 * lanes / (64 * ((lanes + 63) / 64));
    }
};

// Pass A has no work that tiles share: the fewest wavefronts whose lanes are 84% used, so that
// a workgroup waits for little but its own transpose.  Against filling the lanes best (FP32, per
// apply): 36^3 4.4 -> 3.9 ms with 3 planes for 7; 32^3, 30^3 two planes 31 and 1.7 ms against 42
// and 2.3 ms with eight.
template <typename T, int NP>
struct PlaneWgA : PlaneWg<T, NP> {
    using B = PlaneWg<T, NP>;
    static constexpr int pick()
    {
        int best = 0, best_fill = 0;
        for (int w = 1; w <= 4; ++w) {
            const int r = B::fit(w);
            if (r < 1 || r * B::tile_bytes > 80 * 1024 || best_fill >= 84) continue;
            if (B::fill(w) > best_fill) {
                best = r;
                best_fill = B::fill(w);
            }
        }
        return best;
    }
    static constexpr int R = pick();
    static constexpr int threads = ((R * NP + 63) / 64) * 64;
    static_assert(R >= 1 && threads <= 256, "plane pass A workgroup");
};

// Pass C sums the points of a plane over its R tiles, so every tile more also takes accumulators
// off a thread: two wavefronts, and more only where they use over a tenth more of their lanes
// (36^3: 7 pairs, 48^3: 4).  One wavefront, 15 and 16 accumulators a thread, took 4.1 ms at
// 30^3 and 67 ms at 32^3 where two take 2.3 and 39 ms; 24^3 with one 21, with two 11.3, with
// four 12.0 ms; 40^3 with two 21, with four 23 ms.
template <typename T, int NP>
struct PlaneWgC : PlaneWg<T, NP> {
    using B = PlaneWg<T, NP>;
    static constexpr int pick()
    {
        int best = 0, best_fill = -11;
        for (int w = 2; w <= 4; ++w) {
            const int r = B::fit(w);
            if (r < 1 || r * B::tile_bytes > 80 * 1024) continue;
            if (B::fill(w) > best_fill + 10) {
                best = r;
                best_fill = B::fill(w);
            }
        }
        return best;
    }
    static constexpr int R = pick();
    static constexpr int threads = ((R * NP + 63) / 64) * 64;
    static constexpr int rows = (NP + R - 1) / R;  // plane rows a thread sums
    static_assert(R >= 1 && R <= NP && rows <= 16 && threads <= 256, "plane pass C workgroup");
};

// The runs of a column set, read once per workgroup into scalar registers.
template <int NP>
struct PlaneRuns {
    int run[NP];
    __device__ __forceinline__ explicit PlaneRuns(const int* __restrict__ p)
    {
        static_for<0, NP>([&](auto xc) { run[decltype(xc)::value] = p[decltype(xc)::value]; });
    }
    // column (kx = x, row t) is kept, at base(x) + t
    __device__ __forceinline__ bool has(int x, int t) const
    {
        return (unsigned)(t - (run[x] & 0xff)) < (unsigned)((run[x] >> 8) & 0xff);
    }
    __device__ __forceinline__ int base(int x) const { return (run[x] >> 16) - (run[x] & 0xff); }
};

// Row t of the record plane at `plane` (uniform) + off (the lane's plane and t), zero outside the
// support.  The runs are read from memory at every call (the empty asm hides that they do not
// change): held across a loop they would spill.
template <typename T, int NP>
__device__ __forceinline__ void load_row(cpx<T> (&v)[NP], const cpx<T>* plane, unsigned off,
                                         const int* __restrict__ runs, int t)
{
    asm volatile("" : "+s"(runs));
    const PlaneRuns<NP> rr(runs);
    static_for<0, NP>([&](auto xc) {
        constexpr int x = decltype(xc)::value;
        v[x] = cpx<T>{T(0), T(0)};
        if (rr.has(x, t)) v[x] = ld_nt<T>(plane + rr.base(x), off);
    });
}

}  // namespace tcx
