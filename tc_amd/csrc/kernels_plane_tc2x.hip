// kernels_plane_tc2x.hip -- plane-first pair pipeline of the TC/BITC two-body exchange (tc2x),
// FP32-split, and the orbital sets and gather of its two-channel form.
//
// The reference sums, per pair (k,j | q,i) (src/calc_hamiltonian_tc2x.cpp:253-401), with
// K = k-q+G, u = u(K), g_d = FFT_backward((q+G)_d phi),
//     b   = FFT_backward(rho~ V2 + sum_d K_d u FFT_forward(conj(chi_qi) g_kj,d)),
//     a_d = FFT_backward(K_d u rho~),       W += f (b phi_qi - sum_d a_d g_qi,d):
// eight 3D FFTs on four channels.  For plane waves p of phi_kj, p' of chi_qi and p'' of phi_qi,
// where K = p - p' and the output wave is P = K + p'' (no aliasing, see Context::tc2x_form):
//     K.p   = (K^2 + p^2 - p'^2) / 2,       -K.p'' = p''^2 - P.p'',
// so with L phi = FFT_backward(p^2 phi) the same operator is, to rounding,
//     rho = conj(chi_qi) phi_kj,  tau = conj(chi_qi) L phi_kj - conj(L chi_qi) phi_kj,
//     b = FFT_backward(rho~ (V2 + K^2 u / 2) + tau~ u / 2),   U = FFT_backward(rho~ u),
//     W_0 += f (b phi_qi + U L phi_qi),  W_d += f U g_qi,d,   H phi_P += W_0~ - sum_d P_d W_d~:
// four FFTs on two channels; U is never multiplied by K in the working precision, as
// K.p'' = (P^2 - K^2 - p''^2) / 2 with one accumulator P^2 W would (its FP32 error is 1.4 times
// the four-channel form's at 40^3; this form's is 0.86 times it).
// Passes as in kernels_plane.hip (A: rho and tau, xy planes; Z: z pencils and the map; C: xy
// planes and the sums); the pair densities' support columns are the only ones in the records.
#include "jastrow_dev.hpp"
#include "plane_dev.hpp"
#include "size_switch.hpp"

namespace tcx {

// ----------------------------------------------------------------- orbital sets
// [orbital][component][N] FP64 -> [orbital][N][component] in the working precision
template <typename T, int NC>
__global__ __launch_bounds__(256) void k_interleave(const double2* __restrict__ in, cpx<T>* __restrict__ out,
                                                    long long N)
{
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= N) return;
    const double2* p = in + (size_t)blockIdx.y * NC * N + e;
    cpx<T>* q = out + ((size_t)blockIdx.y * N + e) * NC;
    for (int c = 0; c < NC; ++c) {
        const double2 v = p[(size_t)c * N];
        q[c] = cpx<T>{(T)v.x, (T)v.y};
    }
}

void launch_interleave(int prec, int nc, const double* in, void* out, int norb, long long N, hipStream_t s)
{
    for (int a = 0; a < norb; a += 65535) {
        const int n = norb - a < 65535 ? norb - a : 65535;
        const dim3 grid((unsigned)((N + 255) / 256), n);
        const double2* p = (const double2*)in + (size_t)a * nc * N;
        const size_t o = (size_t)a * nc * N;
        if (prec == TCX_PREC_FP64 && nc == 2)
            hipLaunchKernelGGL((k_interleave<double, 2>), grid, dim3(256), 0, s, p, (cpx<double>*)out + o, N);
        else if (prec == TCX_PREC_FP64)
            hipLaunchKernelGGL((k_interleave<double, 5>), grid, dim3(256), 0, s, p, (cpx<double>*)out + o, N);
        else if (nc == 2)
            hipLaunchKernelGGL((k_interleave<float, 2>), grid, dim3(256), 0, s, p, (cpx<float>*)out + o, N);
        else
            hipLaunchKernelGGL((k_interleave<float, 5>), grid, dim3(256), 0, s, p, (cpx<float>*)out + o, N);
        TCX_HIP_CHECK(hipGetLastError());
    }
}

// out[l] += factor (W_0~ - sum_d (k+G)_d W_d~) on the sphere of each applied band; W holds four
// grids per band in G space
__global__ __launch_bounds__(256) void k_gather_tc2x(const double2* __restrict__ W, const int* __restrict__ gindex,
                                                     const OrbEntry* __restrict__ jobs, double2* __restrict__ out,
                                                     long long N, const double* __restrict__ kcart, Geom g,
                                                     double factor)
{
    const OrbEntry e = jobs[blockIdx.y];
    const int l = blockIdx.x * 256 + threadIdx.x;
    if (l >= e.npw) return;
    const int idx = gindex[e.gidx_off + l];
    const int m1 = centered(idx % g.n1, g.n1), m2 = centered((idx / g.n1) % g.n2, g.n2),
              m3 = centered(idx / (g.n1 * g.n2), g.n3);
    const double2* w = W + (size_t)blockIdx.y * 4 * N + idx;
    double2 a = w[0];
    for (int d = 0; d < 3; ++d) {
        const double P = kcart[3 * e.kidx + d] + g.b[d] * m1 + g.b[3 + d] * m2 + g.b[6 + d] * m3;
        const double2 x = w[(size_t)(1 + d) * N];
        a.x -= P * x.x;
        a.y -= P * x.y;
    }
    double2 o = out[e.coef_off + l];
    o.x += factor * a.x;
    o.y += factor * a.y;
    out[e.coef_off + l] = o;
}

void launch_gather_tc2x(const double* W, const int* gindex, const OrbEntry* jobs, int njobs, int max_npw, double* out,
                        long long N, const double* kcart, const Geom& g, double factor, hipStream_t s)
{
    if (njobs == 0 || max_npw == 0) return;
    for (int j0 = 0; j0 < njobs; j0 += 65535) {
        const int nj = njobs - j0 < 65535 ? njobs - j0 : 65535;
        hipLaunchKernelGGL(k_gather_tc2x, dim3((max_npw + 255) / 256, nj), dim3(256), 0, s,
                           (const double2*)W + (size_t)j0 * 4 * N, gindex, jobs + j0, (double2*)out, N, kcart, g, factor);
        TCX_HIP_CHECK(hipGetLastError());
    }
}

namespace {

// Workgroup of pass C: R tiles, tile 2 s + c = channel c of pair s of the group.  At most 8 plane
// rows a thread (four FP64 accumulators per point), two wavefronts or more where a plane has
// them, and more tiles only for clearly more of the lanes in use (FP32, per apply: 16^3 0.16 ->
// 0.13 ms with 8 tiles for 4; 20^3 1.61 -> 1.01 ms with 6 for 16).
template <int NP>
struct Tc2xWg {
    static constexpr int tile_bytes = (int)sizeof(PlaneTile<float, NP>);
    static constexpr int pick()
    {
        int best = 0;
        double best_score = 0.0;
        for (int r = 2; r <= 16 && r <= NP && r * NP <= 512 && r * tile_bytes <= 160 * 1024; r += 2) {
            if (r * 8 < NP || (NP >= 16 && r * NP <= 64)) continue;
            const int waves = (r * NP + 63) / 64;
            const int per_cu = (160 * 1024) / (r * tile_bytes) * waves;
            const double score = double(r * NP) / (64 * waves) * (per_cu >= 8 ? 1.0 : per_cu / 8.0) *
                                 (per_cu >= 2 * waves ? 1.0 : 0.8);  // one workgroup alone waits at its barriers
            if (score > best_score + 0.145) {
                best_score = score;
                best = r;
            }
        }
        return best;
    }
    static constexpr int R = pick();
    static constexpr int threads = ((R * NP + 63) / 64) * 64;
    static constexpr int rows = (NP + R - 1) / R;
    static_assert(R >= 2 && R <= NP, "row r < R of a tile is read by every thread of tile r");
};

struct Bra {
    cpx<float> c, l;  // phi and L phi (or chi and L chi) at a point
};
struct Ket {
    cpx<float> c, l, g[3];  // phi, L phi and g_d at a point
};

}  // namespace

// The map's coefficients at the support columns of every k-q row of a launch, 1/N folded in:
// tab[row][kz][c] = (V2 + K^2 u / 2, u) / N, in FP64, rounded once.
template <bool kPoly>
__global__ __launch_bounds__(256) void k_plane_tc_table(cpx<float>* __restrict__ tab, const double* __restrict__ kqcart,
                                                        int row0, PlaneCols pc, Geom g, JastrowPair jp, double invN)
{
    const int c = blockIdx.x * 256 + threadIdx.x, kz = blockIdx.y;
    if (c >= pc.ncol) return;
    const int xy = pc.colxy[c];
    const int m1 = centered(xy & 0xffff, g.n1), m2 = centered(xy >> 16, g.n2), m3 = centered(kz, g.n3);
    const double* kq = kqcart + 3 * (row0 + blockIdx.z);
    double k2 = 0.0;
    for (int d = 0; d < 3; ++d) {
        const double x = kq[d] + g.b[d] * m1 + g.b[3 + d] * m2 + g.b[6 + d] * m3;
        k2 += x * x;
    }
    const double u = jastrow_uk<kPoly>(jp, k2);
    tab[((size_t)blockIdx.z * g.n3 + kz) * pc.cstride + c] =
        cpx<float>{(float)((jastrow_tc2body<kPoly>(jp, k2) + 0.5 * k2 * u) * invN), (float)(u * invN)};
}

// Pass A: R planes of one pair, rho and then tau through the same tiles (both at once would take
// the registers of a wave per SIMD from 36 points a line on).
template <int NP>
__global__ __launch_bounds__((PlaneWgA<float, NP>::threads), 2) void k_plane_tc2x_A(
    const Bra* __restrict__ app, const Bra* __restrict__ bra, const PairEntry* __restrict__ pairs, int nsrc,
    const int* __restrict__ runs, PlaneCols pc, cpx<float>* __restrict__ rec, int nz)
{
    using Wg = PlaneWgA<float, NP>;
    __shared__ PlaneTile<float, NP> tiles[Wg::R];
    const int ngrp = (nz + Wg::R - 1) / Wg::R, per = (nsrc * ngrp + 7) & ~7;  // as k_plane_A
    const int tg = blockIdx.x / per, i = blockIdx.x - tg * per;
    if (i >= nsrc * ngrp) return;
    const int p = tg * nsrc + i / ngrp, grp = i % ngrp;
    const int r = threadIdx.x / NP, t = threadIdx.x % NP;
    const int z = grp * Wg::R + r;
    const bool active = r < Wg::R && z < nz;
    int row = t + pc.rot;
    row = row >= NP ? row - NP : row;
    const PairEntry pe = pairs[p];
    const size_t ng = (size_t)NP * NP * nz, o = (size_t)grp * Wg::R * (NP * NP);
    const Bra* a = app + (size_t)pe.app * ng + o;
    const Bra* b = bra + (size_t)pe.occ * ng + o;
    const unsigned off = (unsigned)(r * (NP * NP) + t) * sizeof(Bra);
    static_for<0, 2>([&](auto cc) {
        constexpr int c = decltype(cc)::value;
        cpx<float> v[NP];
        if (active) {
            static_for<0, NP>([&](auto yc) {
                constexpr int y = decltype(yc)::value;
                if constexpr (c == 0) {
                    v[y] = cmulc(ld<cpx<float>>(b + y * NP, off), ld<cpx<float>>(a + y * NP, off));
                } else {
                    const Bra x = ld<Bra>(a + y * NP, off), w = ld<Bra>(b + y * NP, off);
                    v[y] = cmulc(w.c, x.l) - cmulc(w.l, x.c);
                }
            });
            fft<float, NP, -1>(v);
        }
        if constexpr (c == 1) __syncthreads();  // the rows of rho have been read
        cols_to_rows<float, NP>(tiles[active ? r : 0], v, t, row, active);
        if (active) {
            fft<float, NP, -1>(v);
            store_row<float, NP>(v, rec + (((size_t)p * 2 + c) * nz + grp * Wg::R) * pc.cstride,
                                 (unsigned)(r * pc.cstride + t) * sizeof(cpx<float>), runs, t);
        }
    });
}

// Pass Z: one lane per support column of a pair, both channels' z pencils in registers;
// (rho~, tau~) -> (b~, U~) in place.
template <int NZ>
__global__ __launch_bounds__(kPencilBlock, 2) void k_plane_tc2x_Z(cpx<float>* __restrict__ rec,
                                                                  const PairEntry* __restrict__ pairs,
                                                                  const cpx<float>* __restrict__ tab, int kq0,
                                                                  PlaneCols pc)
{
    const int c = blockIdx.x * kPencilBlock + threadIdx.x;
    if (c >= pc.ncol) return;
    cpx<float>* c0 = rec + (size_t)blockIdx.y * 2 * NZ * pc.cstride;
    cpx<float>* c1 = c0 + (size_t)NZ * pc.cstride;
    const cpx<float>* m = tab + (size_t)(pairs[blockIdx.y].kq - kq0) * NZ * pc.cstride;
    const unsigned off = (unsigned)c * sizeof(cpx<float>);
    cpx<float> x[NZ], y[NZ];
    ld_column<float, NZ>(y, c1, off, pc.cstride);
    fft<float, NZ, -1>(y);
    __builtin_amdgcn_sched_barrier(0);  // the scheduler would hoist every load and spill
    ld_column<float, NZ>(x, c0, off, pc.cstride);
    fft<float, NZ, -1>(x);
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, NZ>([&](auto zc) {
        constexpr int z = decltype(zc)::value;
        const cpx<float> s = ld<cpx<float>>(m + (size_t)z * pc.cstride, off);
        const cpx<float> rho = x[z];
        x[z] = scale(rho, s.re) + scale(y[z], 0.5f * s.im);
        y[z] = scale(rho, s.im);
        if constexpr (z % 8 == 7) __builtin_amdgcn_sched_barrier(0);
    });
    fft<float, NZ, 1>(x);
    st_column<float, NZ>(x, c0, off, pc.cstride);
    __builtin_amdgcn_sched_barrier(0);
    fft<float, NZ, 1>(y);
    st_column<float, NZ>(y, c1, off, pc.cstride);
}

// Pass C: plane z of one target, R/2 pairs at a time; as k_plane_C with (b, U) in tiles 2 s and
// 2 s + 1, and the orbital set read at the points where the sums are formed.
template <int NP>
__global__ __launch_bounds__((Tc2xWg<NP>::threads), 2) void k_plane_tc2x_C(
    const cpx<float>* __restrict__ rec, const Ket* __restrict__ ket, const PairEntry* __restrict__ pairs,
    const TargetEntry* __restrict__ targets, const int* __restrict__ runs, PlaneCols pc,
    const double* __restrict__ fill, double2* __restrict__ W, float2* __restrict__ Wc, int nz)
{
    using Wg = Tc2xWg<NP>;
    constexpr int R = Wg::R, ROWS = Wg::rows, S = R / 2;
    __shared__ PlaneTile<float, NP> tiles[R];
    const int z = blockIdx.x;
    const TargetEntry te = targets[blockIdx.y];
    const int r = threadIdx.x / NP, t = threadIdx.x % NP;
    int row = t + pc.rot;
    row = row >= NP ? row - NP : row;
    const size_t ng = (size_t)NP * NP * nz, pz = (size_t)z * (NP * NP);
    PlaneTile<float, NP>& tile = tiles[r < R ? r : 0];
    double2 acc[4][ROWS];  // points x = t, y = r + i R
    static_for<0, 4 * ROWS>([&](auto ic) {
        acc[decltype(ic)::value / ROWS][decltype(ic)::value % ROWS] = make_double2(0.0, 0.0);
    });
    const int pend = te.pair0 + te.npair;
    auto plane_of = [&](int pp) { return rec + ((size_t)pp * 2 * nz + z) * pc.cstride; };  // uniform
    const unsigned off = (unsigned)(r * nz * pc.cstride + t) * sizeof(cpx<float>);         // pair r/2, channel r&1
    const unsigned koff = (unsigned)(r * NP + t) * sizeof(Ket);
    cpx<float> v[NP];
    if (r < R && te.pair0 + r / 2 < pend) load_row<float, NP>(v, plane_of(te.pair0), off, runs, t);
#pragma unroll 1
    for (int p0 = te.pair0; p0 < pend; p0 += S) {
        const bool on = r < R && p0 + r / 2 < pend, next = r < R && p0 + S + r / 2 < pend;
        if (on) fft<float, NP, 1>(v);
        rows_to_cols<float, NP>(tile, v, row, t, on);
        if (on) {
            fft<float, NP, 1>(v);
            tile_put_col<float, NP>(tile, v, t);  // column t was read by this thread alone
        }
        if (next) load_row<float, NP>(v, plane_of(p0 + S), off, runs, t);
        __syncthreads();
        const int ns = pend - p0 < S ? pend - p0 : S;
        if (r < R)
#pragma unroll 1
            for (int s = 0; s < ns; ++s) {
                const int occ = pairs[p0 + s].occ;
                const double f = fill[occ];
                const Ket* q = ket + (size_t)occ * ng + pz;
                static_for<0, ROWS>([&](auto ic) {
                    constexpr int i = decltype(ic)::value;
                    {
                        // past the last row: row r again, not stored (no branch: it spilled)
                        const bool in = i * R + R <= NP || i * R + r < NP;
                        const Ket k = ld<Ket>(in ? q + i * R * NP : q, koff);
                        const int y0 = in ? i * R + r : r;
                        const cpx<float> b = tiles[2 * s].a[y0][t], U = tiles[2 * s + 1].a[y0][t];
                        const cpx<float> x = b * k.c, y = U * k.l;
                        acc[0][i].x += f * ((double)x.re + (double)y.re);
                        acc[0][i].y += f * ((double)x.im + (double)y.im);
                        static_for<0, 3>([&](auto dc) {
                            constexpr int d = decltype(dc)::value;
                            const cpx<float> w = U * k.g[d];
                            acc[1 + d][i].x += f * (double)w.re;
                            acc[1 + d][i].y += f * (double)w.im;
                        });
                    }
                    if constexpr (i % 2 == 1) __builtin_amdgcn_sched_barrier(0);
                });
            }
        __syncthreads();
    }
    if (r >= R) return;
    const size_t o = (size_t)te.app * 4 * ng + pz + t;
    static_for<0, 4>([&](auto cc) {
        constexpr int c = decltype(cc)::value;
        static_for<0, ROWS>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            if (i * R + R <= NP || i * R + r < NP) {
                const size_t e = o + c * ng + (size_t)(i * R + r) * NP;
                add_partial(W + e, Wc + e, acc[c][i].x, acc[c][i].y);
            }
        });
    });
}

// ----------------------------------------------------------------- launchers
void launch_plane_tc_table(void* tab, const double* kqcart, int row0, int nrows, const PlaneCols& pc, const Geom& g,
                           const JastrowPair& jp, hipStream_t s)
{
    if (nrows == 0 || pc.ncol == 0) return;
    const double invN = 1.0 / ((double)g.n1 * g.n2 * g.n3);
    const dim3 grid((pc.ncol + 255) / 256, g.n3, nrows);
    TCX_POLY_DISPATCH(jp.pdeg > 0, hipLaunchKernelGGL(k_plane_tc_table<kPoly>, grid, dim3(256), 0, s, (cpx<float>*)tab,
                                                      kqcart, row0, pc, g, jp, invN));
    TCX_HIP_CHECK(hipGetLastError());
}

PlaneShape plane_tc2x_shape(int n1)
{
    PlaneShape ps{1, 256};
#define TCX_L(NP)                                                                             \
    {                                                                                         \
        using Wg = Tc2xWg<NP>;                                                                \
        const int by_lds = (160 * 1024) / (Wg::R * Wg::tile_bytes), by_waves = 8 / (Wg::threads / 64); \
        const int wgs = by_lds < by_waves ? by_lds : by_waves;                                \
        ps = {Wg::R / 2, 256 * (wgs > 0 ? wgs : 1)};                                          \
    }
    TCX_SIZE_SWITCH(n1, TCX_L)
#undef TCX_L
    return ps;
}

void launch_plane_tc2x_A(const Geom& g, const void* app, const void* bra, const PairEntry* pairs, int ntargets,
                         int nsrc, const PlaneCols& pc, void* rec, hipStream_t s)
{
    if (ntargets == 0 || nsrc == 0) return;
#define TCX_L(NP)                                                                                             \
    {                                                                                                         \
        using Wg = PlaneWgA<float, NP>;                                                                        \
        const unsigned per = ((unsigned)((g.n3 + Wg::R - 1) / Wg::R) * nsrc + 7) / 8 * 8;                     \
        hipLaunchKernelGGL((k_plane_tc2x_A<NP>), dim3(per * ntargets), dim3(Wg::threads), 0, s, (const Bra*)app, \
                           (const Bra*)bra, pairs, nsrc, pc.run, pc, (cpx<float>*)rec, g.n3);                 \
    }
    TCX_SIZE_SWITCH(g.n1, TCX_L)
#undef TCX_L
    TCX_HIP_CHECK(hipGetLastError());
}

void launch_plane_tc2x_Z(const Geom& g, void* rec, const PairEntry* pairs, int npairs, const void* tab, int kq0,
                         const PlaneCols& pc, hipStream_t s)
{
    if (npairs == 0 || pc.ncol == 0) return;
    if (npairs > 65535) throw Error(TCX_ERR_INTERNAL, "plane pipeline: too many pairs in one launch");
#define TCX_L(NZ)                                                                                             \
    hipLaunchKernelGGL((k_plane_tc2x_Z<NZ>), dim3((pc.ncol + kPencilBlock - 1) / kPencilBlock, npairs),       \
                       dim3(kPencilBlock), 0, s, (cpx<float>*)rec, pairs, (const cpx<float>*)tab, kq0, pc);
    TCX_SIZE_SWITCH(g.n3, TCX_L)
#undef TCX_L
    TCX_HIP_CHECK(hipGetLastError());
}

void launch_plane_tc2x_C(const Geom& g, const void* rec, const void* ket, const PairEntry* pairs,
                         const TargetEntry* targets, int ntargets, const PlaneCols& pc, const double* fill, double* W,
                         float* Wc, hipStream_t s)
{
    if (ntargets == 0) return;
    if (ntargets > 65535) throw Error(TCX_ERR_INTERNAL, "plane pipeline: too many targets in one launch");
#define TCX_L(NP)                                                                                              \
    {                                                                                                          \
        using Wg = Tc2xWg<NP>;                                                                                 \
        hipLaunchKernelGGL((k_plane_tc2x_C<NP>), dim3(g.n3, ntargets), dim3(Wg::threads), 0, s,                \
                           (const cpx<float>*)rec, (const Ket*)ket, pairs, targets, pc.run, pc, fill, (double2*)W, \
                           (float2*)Wc, g.n3);                                                                 \
    }
    TCX_SIZE_SWITCH(g.n1, TCX_L)
#undef TCX_L
    TCX_HIP_CHECK(hipGetLastError());
}

}  // namespace tcx
