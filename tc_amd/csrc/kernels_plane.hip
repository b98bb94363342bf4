// kernels_plane.hip -- plane-first pair pipeline of the Fock exchange (hf2x), FP32-split.
//
// The same operator as kernels_hf2x.hip (src/calc_hamiltonian_hf2x.cpp:123-135):
//     rho(r) = conj(phi_qi(r)) phi_kj(r),  rho~ = FFT_forward(rho) v(G)/N,
//     W_kj(r) += f_qi phi_qi(r) FFT_backward(rho~)(r),
// with the two 3D transforms split the other way round:
//   A  (xy planes):  rho on plane z, FFT along y and x, store the plane's
//                    support columns;
//   Z  (z pencils):  one per support column (kx, ky): FFT along z, x v(G)/N,
//                    inverse FFT along z, store in place;
//   C  (xy planes):  inverse FFT along x and y, x phi_qi, accumulate over the
//                    pairs of the target in FP64 registers, add once into W_kj.
// rho has G-space support only inside |G + k - q| < 2 G_w (the sum of the two
// orbitals' cutoff spheres), and so has every quantity between the passes.  A z
// pencil after a first pass along z covers every (kx, ky) column, but between xy
// and z only the columns in the support's projection on the (kx, ky) plane are
// non-zero: about two thirds of them at 40^3 (fcc, 4x4x4 k).  The pair record holds
// just those (73% of the grid with their padding), 30% fewer bytes than z-first by counters: at
// 40^3, 4x4x4 k, 16 bands (1,048,576 pairs) A 128, Z 132 and C 147 ms per apply against 166,
// 206 and 143 ms (535 -> 428 ms with the host copies).  Z runs at the HBM copy rate; A writes its
// records at 3.1 and C reads them at 2.7 TB/s (by counters A moves 5.0, Z 6.0, C 3.4 TB/s),
// bound by the latency of one workgroup's load, transform and store phases at the two waves per
// SIMD that their tiles leave.
//
// Columns (PlaneCols): one set for all pairs, the union over the (k, q) of the bases, so
// that every index below is uniform over a launch.  kx by kx, a contiguous run of rotated
// ky (t = (i2 - rot) mod n2), run[kx] = lo | len << 8 | first << 16; record [z][c].  A lane
// owns one row t, so the lanes of a load or store of one kx are consecutive columns.
#include "plane_dev.hpp"
#include "size_switch.hpp"

namespace tcx {

namespace {
using PT = float;  // precision of the pair records
}

// Pass A: R planes of one pair; pair = target tg x source s, nsrc sources per target.  Column
// x = t of rho -> FFT_y -> LDS transpose -> row ky -> FFT_x -> the row's support columns.
// Consecutive workgroups go to the 8 XCDs in turn, each with its own L2; the items of a target
// are padded to a multiple of 8, so the same planes of the same source are read on the same XCD
// for every target and stay in its L2 (40^3 FP32: 125 ms per apply with 32 or 48 sources per
// launch, 149-161 ms where the count made them wander or with 96, whose planes exceed the L2).
// Plane-group-fastest order also keeps the record writes in flight close together: a
// plane-slowest order, which gives each XCD a fixed set of planes too, took 139 ms.
template <typename T, int NP>
__global__ __launch_bounds__((PlaneWgA<T, NP>::threads), 2) void k_plane_A(const cpx<T>* __restrict__ phiR_app,
                                                                     const cpx<T>* __restrict__ phiR_occ,
                                                                     const PairEntry* __restrict__ pairs, int nsrc,
                                                                     const int* __restrict__ runs, PlaneCols pc,
                                                                     cpx<T>* __restrict__ rec, int nz)
{
    using Wg = PlaneWgA<T, NP>;
    __shared__ PlaneTile<T, NP> tiles[Wg::R];
    const int ngrp = (nz + Wg::R - 1) / Wg::R, per = (nsrc * ngrp + 7) & ~7;
    const int tg = blockIdx.x / per, i = blockIdx.x - tg * per;
    if (i >= nsrc * ngrp) return;
    const int p = tg * nsrc + i / ngrp, grp = i % ngrp;
    const int r = threadIdx.x / NP, t = threadIdx.x % NP;
    const int z = grp * Wg::R + r;
    const bool active = r < Wg::R && z < nz;
    int row = t + pc.rot;
    row = row >= NP ? row - NP : row;
    const PairEntry pe = pairs[p];
    const size_t ng = (size_t)NP * NP * nz, o = (size_t)z * (NP * NP) + t;
    cpx<T> v[NP];
    if (active) {
        // per-lane pointers here and in the stores: with a uniform base per access and 32-bit lane
        // offsets, as in pass C, the pass ran 7% (40^3) to 14% (48^3) longer
        const cpx<T>* a = phiR_app + (size_t)pe.app * ng + o;
        const cpx<T>* b = phiR_occ + (size_t)pe.occ * ng + o;
        static_for<0, NP>([&](auto yc) {
            constexpr int y = decltype(yc)::value;
            v[y] = cmulc(b[y * NP], a[y * NP]);
        });
        fft<T, NP, -1>(v);
    }
    cols_to_rows<T, NP>(tiles[active ? r : 0], v, t, row, active);
    if (active) {
        fft<T, NP, -1>(v);
        const PlaneRuns<NP> rr(runs);
        cpx<T>* out = rec + ((size_t)p * nz + z) * pc.cstride + t;
        static_for<0, NP>([&](auto xc) {
            constexpr int x = decltype(xc)::value;
            if (rr.has(x, t)) st_nt<T>(out + rr.base(x), 0, v[x]);
        });
    }
}

// v(G)/N at the support columns of every k-q row of a launch (hf2x.cpp:91-104: 1/(N |k-q+G|^2),
// 0 below 1e-8; the 1/N is FFT_forward's), evaluated in FP64 and rounded once: tab[row][kz][c].
template <typename T>
__global__ __launch_bounds__(256) void k_plane_coulomb(T* __restrict__ tab, const double* __restrict__ kqcart, int row0,
                                                       PlaneCols pc, Geom g, double invN)
{
    const int c = blockIdx.x * 256 + threadIdx.x, kz = blockIdx.y;
    if (c >= pc.ncol) return;
    const int xy = pc.colxy[c];
    const int m1 = centered(xy & 0xffff, g.n1), m2 = centered(xy >> 16, g.n2), m3 = centered(kz, g.n3);
    const double* kq = kqcart + 3 * (row0 + blockIdx.z);
    double g2 = 0.0;
    for (int d = 0; d < 3; ++d) {
        const double x = kq[d] + g.b[d] * m1 + g.b[3 + d] * m2 + g.b[6 + d] * m3;
        g2 += x * x;
    }
    tab[((size_t)blockIdx.z * g.n3 + kz) * pc.cstride + c] = static_cast<T>(g2 < 1e-8 ? 0.0 : invN / g2);
}

// Pass Z: one lane per support column of a pair, its whole z pencil in registers.
template <typename T, int NZ>
__global__ __launch_bounds__(kPencilBlock, 2) void k_plane_Z(cpx<T>* __restrict__ rec, const PairEntry* __restrict__ pairs,
                                                          const T* __restrict__ tab, int kq0, PlaneCols pc)
{
    const int c = blockIdx.x * kPencilBlock + threadIdx.x;
    if (c >= pc.ncol) return;
    cpx<T>* col = rec + (size_t)blockIdx.y * NZ * pc.cstride + c;
    const T* v = tab + (size_t)(pairs[blockIdx.y].kq - kq0) * NZ * pc.cstride + c;
    cpx<T> x[NZ];
    load_pencil_nt<T, NZ>(x, col, pc.cstride);
    fft<T, NZ, -1>(x);
    static_for<0, NZ>([&](auto zc) {
        constexpr int z = decltype(zc)::value;
        x[z] = scale(x[z], v[(size_t)z * pc.cstride]);
    });
    fft<T, NZ, 1>(x);
    store_pencil_nt<T, NZ>(x, col, pc.cstride);
}

// Pass C: plane z of one target, R pairs at a time, pair r in tile r.  Row ky = t from the
// record -> inverse FFT_x -> tile -> column x = t -> inverse FFT_y -> x phi_qi -> tile; then
// every thread adds its points of the plane over the R tiles into FP64 registers.  Summing by
// points and not by lines keeps the accumulators at rows() complex values a thread (14 at
// 40^3) with whole lines per lane: split lines (4 lanes each, the accumulators by line) cost
// twice the instructions and ran 2.7 times longer.
template <typename T, int NP>
__global__ __launch_bounds__((PlaneWgC<T, NP>::threads), 2) void k_plane_C(
    const cpx<T>* __restrict__ rec, const cpx<T>* __restrict__ phiR_occ, const PairEntry* __restrict__ pairs,
    const TargetEntry* __restrict__ targets, const int* __restrict__ runs, PlaneCols pc,
    const double* __restrict__ fill, cpx<double>* __restrict__ W, float2* __restrict__ Wc, int nz)
{
    using Wg = PlaneWgC<T, NP>;
    constexpr int R = Wg::R, ROWS = Wg::rows;
    __shared__ PlaneTile<T, NP> tiles[R];
    const int z = blockIdx.x;
    const TargetEntry te = targets[blockIdx.y];
    const int r = threadIdx.x / NP, t = threadIdx.x % NP;
    int row = t + pc.rot;
    row = row >= NP ? row - NP : row;
    const size_t ng = (size_t)NP * NP * nz, pz = (size_t)z * (NP * NP);
    PlaneTile<T, NP>& tile = tiles[r < R ? r : 0];
    cpx<double> acc[ROWS];  // points x = t, y = r + i R
    static_for<0, ROWS>([&](auto ic) { acc[decltype(ic)::value] = cpx<double>{0.0, 0.0}; });
    const int pend = te.pair0 + te.npair;
    auto plane_of = [&](int pp) { return rec + ((size_t)pp * nz + z) * pc.cstride; };  // uniform
    const unsigned off = (unsigned)(r * nz * pc.cstride + t) * sizeof(cpx<T>);           // pair r of the group
    // the rows of the next group are loaded while the points of this one are summed (152 -> 147 ms
    // per apply at 40^3)
    cpx<T> v[NP];
    if (r < R && te.pair0 + r < pend) load_row<T, NP>(v, plane_of(te.pair0), off, runs, t);
#pragma unroll 1
    for (int p0 = te.pair0; p0 < pend; p0 += R) {
        const bool on = r < R && p0 + r < pend, next = r < R && p0 + R + r < pend;
        if (on) fft<T, NP, 1>(v);
        rows_to_cols<T, NP>(tile, v, row, t, on);
        if (on) {
            fft<T, NP, 1>(v);
            const cpx<T>* q = phiR_occ + (size_t)pairs[p0 + r].occ * ng + pz + t;
            static_for<0, NP>([&](auto yc) {
                constexpr int y = decltype(yc)::value;
                v[y] = v[y] * q[y * NP];
            });
        }
        const int nr = pend - p0 < R ? pend - p0 : R;
        if (on) tile_put_col<T, NP>(tile, v, t);  // column t was read by this thread alone
        if (next) load_row<T, NP>(v, plane_of(p0 + R), off, runs, t);
        __syncthreads();
        if (r < R)
            for (int s = 0; s < nr; ++s) {
                const double f = fill[pairs[p0 + s].occ];
                static_for<0, ROWS>([&](auto ic) {
                    constexpr int i = decltype(ic)::value;
                    if (i * R + R <= NP || i * R + r < NP) {
                        const cpx<T> x = tiles[s].a[i * R + r][t];
                        acc[i].re += f * static_cast<double>(x.re);
                        acc[i].im += f * static_cast<double>(x.im);
                    }
                });
            }
        __syncthreads();
    }
    if (r >= R) return;
    const size_t o = (size_t)te.app * ng + pz + t;
    static_for<0, ROWS>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if (i * R + R <= NP || i * R + r < NP) {
            const size_t e = o + (size_t)(i * R + r) * NP;
            add_partial((double2*)(W + e), Wc ? Wc + e : nullptr, acc[i].re, acc[i].im);
        }
    });
}

// ----------------------------------------------------------------- launchers
PlaneShape plane_shape(int n1)
{
    PlaneShape ps{1, 256};
#define TCX_L(NP)                                                                              \
    {                                                                                          \
        using Wg = PlaneWgC<PT, NP>;                                                             \
        const int by_lds = (160 * 1024) / (Wg::R * Wg::tile_bytes), by_waves = 8 / (Wg::threads / 64); \
        ps = {Wg::R, 256 * (by_lds < by_waves ? by_lds : by_waves)};                           \
    }
    TCX_SIZE_SWITCH(n1, TCX_L)
#undef TCX_L
    return ps;
}

void launch_plane_A(const Geom& g, const void* app, const void* occ, const PairEntry* pairs, int ntargets,
                    int nsrc, const PlaneCols& pc, void* rec, hipStream_t s)
{
    if (ntargets == 0 || nsrc == 0) return;
#define TCX_L(NP)                                                                                                \
    {                                                                                                            \
        using Wg = PlaneWgA<PT, NP>;                                                                               \
        const unsigned per = ((unsigned)((g.n3 + Wg::R - 1) / Wg::R) * nsrc + 7) / 8 * 8;                        \
        hipLaunchKernelGGL((k_plane_A<PT, NP>), dim3(per * ntargets), dim3(Wg::threads), 0, s, (const cpx<PT>*)app, \
                           (const cpx<PT>*)occ, pairs, nsrc, pc.run, pc, (cpx<PT>*)rec, g.n3);                   \
    }
    TCX_SIZE_SWITCH(g.n1, TCX_L)
#undef TCX_L
    TCX_HIP_CHECK(hipGetLastError());
}

void launch_plane_coulomb(void* tab, const double* kqcart, int row0, int nrows, const PlaneCols& pc,
                          const Geom& g, hipStream_t s)
{
    if (nrows == 0 || pc.ncol == 0) return;
    const double invN = 1.0 / ((double)g.n1 * g.n2 * g.n3);
    const dim3 grid((pc.ncol + 255) / 256, g.n3, nrows);
    hipLaunchKernelGGL(k_plane_coulomb<float>, grid, dim3(256), 0, s, (float*)tab, kqcart, row0, pc, g, invN);
    TCX_HIP_CHECK(hipGetLastError());
}

void launch_plane_Z(const Geom& g, void* rec, const PairEntry* pairs, int npairs, const void* tab, int kq0,
                    const PlaneCols& pc, hipStream_t s)
{
    if (npairs == 0 || pc.ncol == 0) return;
    if (npairs > 65535) throw Error(TCX_ERR_INTERNAL, "plane pipeline: too many pairs in one launch");
#define TCX_L(NZ)                                                                                               \
    hipLaunchKernelGGL((k_plane_Z<PT, NZ>), dim3((pc.ncol + kPencilBlock - 1) / kPencilBlock, npairs),           \
                       dim3(kPencilBlock), 0, s, (cpx<PT>*)rec, pairs, (const PT*)tab, kq0, pc);
    TCX_SIZE_SWITCH(g.n3, TCX_L)
#undef TCX_L
    TCX_HIP_CHECK(hipGetLastError());
}

void launch_plane_C(const Geom& g, const void* rec, const void* occ, const PairEntry* pairs,
                    const TargetEntry* targets, int ntargets, const PlaneCols& pc, const double* fill, double* W,
                    float* Wc, hipStream_t s)
{
    if (ntargets == 0) return;
    if (ntargets > 65535) throw Error(TCX_ERR_INTERNAL, "plane pipeline: too many targets in one launch");
#define TCX_L(NP)                                                                                                \
    {                                                                                                            \
        using Wg = PlaneWgC<PT, NP>;                                                                               \
        hipLaunchKernelGGL((k_plane_C<PT, NP>), dim3(g.n3, ntargets), dim3(Wg::threads), 0, s,                    \
                           (const cpx<PT>*)rec, (const cpx<PT>*)occ, pairs, targets, pc.run, pc, fill,             \
                           (cpx<double>*)W, (float2*)Wc, g.n3);                                                  \
    }
    TCX_SIZE_SWITCH(g.n1, TCX_L)
#undef TCX_L
    TCX_HIP_CHECK(hipGetLastError());
}

}  // namespace tcx
