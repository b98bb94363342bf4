// plane_dev.hpp -- device pieces of the plane-first pair pipelines (kernels_plane.hip,
// kernels_plane_tc2x.hip): the workgroup shape, the column runs and the row loads.
#pragma once

#include "kernels_common.hpp"

namespace tcx {

// Workgroup of the plane passes: R tiles (planes of a pair in pass A, pairs of a plane in
// pass C) of NP lines each, line t of tile r on thread r NP + t.  R fills the wavefronts best
// among those that leave 8 wavefronts (2 per SIMD) of workgroups in a CU's 160 KB of LDS, with
// at most 16 accumulators a thread (a single 48-line tile would hold 48 of them: 48^3 ran at two
// thirds of the z-first speed).
template <typename T, int NP>
struct PlaneWg {
    static constexpr int tile_bytes = (int)sizeof(PlaneTile<T, NP>);
    static constexpr int pick()
    {
        int best = (NP + 15) / 16;
        double best_score = 0.0;
        for (int r = (NP + 15) / 16; r <= 16 && r * NP <= 256 && r * tile_bytes <= 80 * 1024; ++r) {
            const int waves = (r * NP + 63) / 64;
            const int per_cu = (160 * 1024) / (r * tile_bytes) * waves;
            const double score = double(r * NP) / (64 * waves) * (per_cu >= 8 ? 1.0 : per_cu / 8.0);
            if (score > best_score + 1e-9) {
                best_score = score;
                best = r;
            }
        }
        return best;
    }
    static constexpr int R = pick();
    static constexpr int threads = ((R * NP + 63) / 64) * 64;
    static constexpr int rows = (NP + R - 1) / R;  // plane rows a thread sums in pass C
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

template <typename T, int NZ>
__device__ __forceinline__ void ld_column(cpx<T> (&v)[NZ], const cpx<T>* base, unsigned off, int cstride)
{
    static_for<0, NZ>([&](auto zc) {
        constexpr int z = decltype(zc)::value;
        v[z] = ld_nt<T>(base + (size_t)z * cstride, off);
    });
}
template <typename T, int NZ>
__device__ __forceinline__ void st_column(const cpx<T> (&v)[NZ], cpx<T>* base, unsigned off, int cstride)
{
    static_for<0, NZ>([&](auto zc) {
        constexpr int z = decltype(zc)::value;
        st_nt<T>(base + (size_t)z * cstride, off, v[z]);
    });
}
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
template <typename T, int NP>
__device__ __forceinline__ void store_row(const cpx<T> (&v)[NP], cpx<T>* plane, unsigned off,
                                          const int* __restrict__ runs, int t)
{
    asm volatile("" : "+s"(runs));
    const PlaneRuns<NP> rr(runs);
    static_for<0, NP>([&](auto xc) {
        constexpr int x = decltype(xc)::value;
        if (rr.has(x, t)) st_nt<T>(plane + rr.base(x), off, v[x]);
    });
}

}  // namespace tcx
