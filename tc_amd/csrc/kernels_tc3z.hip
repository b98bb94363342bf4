// kernels_tc3z.hip -- z passes of FFT_backward fused with the real-space consumers of the
// three-body record pipelines.
//
// A record channel arrives inverse-transformed along x and y (the fused combine pass);
// one thread group owns a z pencil of one target and loops over the target's pairs: it
// finishes FFT_backward along z with the pencil split over S lanes (PencilSplit), then
// applies the consumer at the lane's output points, summing in FP64 registers, and adds
// once into the FP64 grids of the target (no atomics, deterministic).  The consumers are
// the reference's real-space steps:
//   tc3a3b3b4b6 (src/calc_hamiltonian_tc3a3b3b4b6.cpp:316-335): qsum_j,d += f P_0,d phi_qi,
//     then P_s,d *= density_s, transformed along z again for the next FFT_forward;
//   tc3a2a4b2b5 (src/calc_hamiltonian_tc3a2a4b2b5.cpp:377-427): the q-sums Q2, Q4, Q5;
//     (:848-913) the apply-phase accumulation into W.
#include "kernels_common.hpp"
#include "size_switch.hpp"

namespace tcx {

namespace {

// lanes per pencil: Want when it divides NZ, else 2
template <int NZ, int Want>
struct SplitFor {
    static constexpr int value = (NZ % Want == 0) ? Want : 2;
};

template <typename T>
__device__ __forceinline__ double2 upd(cpx<T> a)
{
    return make_double2((double)a.re, (double)a.im);
}
__device__ __forceinline__ double2 cmadd(double2 acc, double2 a, double2 b, double s)  // acc + s a b
{
    return make_double2(acc.x + s * (a.x * b.x - a.y * b.y), acc.y + s * (a.x * b.y + a.y * b.x));
}

// Lane geometry of a split pencil.
template <int S>
struct LaneOf {
    int h, xy, ob;
    bool valid;
    __device__ LaneOf(int nxy)
    {
        using Split = PencilSplit<S>;
        h = threadIdx.x / Split::pencils;
        const int xy0 = blockIdx.x * Split::pencils + (threadIdx.x % Split::pencils);
        valid = xy0 < nxy;
        xy = valid ? xy0 : 0;  // out-of-range lanes still join the shuffles
        ob = Split::out_block(h);
    }
};

}  // namespace

// ----------------------------------------------------------------- tc3a3b3b4b6 real-space step
// Per target (k,j) and direction d = blockIdx.z: qsum[j][d] += sum_p f P[p][d] phi_qi (the
// s2 = 0 channel, before the density), and P[p][3s+d] <- FFT_z(density_s * P[p][3s+d]) * sc
// for s = 0, 1 (in place): the real-space step between the z pass of FFT_backward and the
// z pass of the next FFT_forward.  The lanes of a pencil move from the blocked output layout
// of one split transform to the strided input layout of the next through LDS.
template <typename T, int NZ, int S>
__global__ __launch_bounds__(kPencilBlock) void k_za7_mid(cpx<T>* __restrict__ P, const cpx<T>* __restrict__ occR,
                                                          const PairEntry* __restrict__ pairs,
                                                          const TargetEntry* __restrict__ targets,
                                                          const double* __restrict__ fill,
                                                          const double2* __restrict__ dens, size_t dstride,
                                                          double2* __restrict__ qsum, int nxy, T sc)
{
    constexpr int M = NZ / S;
    constexpr int PN = PencilSplit<S>::pencils;
    __shared__ cpx<T> xs[PN][NZ + 1];  // one pencil per row (+1 against bank conflicts)
    const LaneOf<S> L(nxy);
    const int pi = threadIdx.x % PN;
    const TargetEntry te = targets[blockIdx.y];
    const int d = blockIdx.z;
    const size_t ng = (size_t)nxy * NZ;
    const size_t o0 = L.xy + (size_t)L.ob * M * nxy;  // first output point of the lane
    double2 acc[M];
    static_for<0, M>([&](auto kc) { acc[decltype(kc)::value] = make_double2(0.0, 0.0); });
    // steps it = 2 (pair) + s over the target's pairs; the pencil of step it + 1 is
    // loaded before step it is transformed (steps touch distinct grids)
    const int nsteps = 2 * te.npair;
    auto grid_of = [&](int it) { return P + ((size_t)(te.pair0 + (it >> 1)) * 6 + 3 * (it & 1) + d) * ng; };
    constexpr bool kPrefetch = sizeof(T) == 4;  // FP64 instances have no VGPRs to spare
    cpx<T> vn[M];
    if (kPrefetch && nsteps > 0) load_pencil<T, M>(vn, grid_of(0) + L.xy + (size_t)L.h * nxy, S * nxy);
#pragma unroll 1
    for (int it = 0; it < nsteps; ++it) {
        const int pp = te.pair0 + (it >> 1), s = it & 1;
        const int occ = pairs[pp].occ;
        const double f = fill[occ];
        const cpx<T>* ph = occR + (size_t)occ * ng + o0;
        cpx<T>* g = grid_of(it);
        cpx<T> v[M];
        if (kPrefetch) {
            static_for<0, M>([&](auto mc) { v[decltype(mc)::value] = vn[decltype(mc)::value]; });
            if (it + 1 < nsteps) load_pencil<T, M>(vn, grid_of(it + 1) + L.xy + (size_t)L.h * nxy, S * nxy);
        } else {
            load_pencil<T, M>(v, g + L.xy + (size_t)L.h * nxy, S * nxy);  // z = S m + h
        }
        const double2* n = dens + s * dstride + o0;  // dstride 0: one independent spin
        // FP32: the orbital and density points of the step are loaded before the transform,
        // so that their latency overlaps it (FP64 loads them where they are used)
        double2 dnv[kPrefetch ? M : 1];
        cpx<T> phv[kPrefetch ? M : 1];
        if constexpr (kPrefetch)
            static_for<0, M>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                dnv[k] = n[(size_t)k * nxy];
                if (s == 0) phv[k] = ph[(size_t)k * nxy];
            });
        // the exchanges of both transforms use lane swaps here (3.5% faster than ds_bpermute)
        PencilSplit<S>::template fft<T, NZ, 1, true>(v, L.h);  // -> z = ob M + k
        {
            static_for<0, M>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                const double2 x = upd(v[k]);
                double2 dn;
                if constexpr (kPrefetch) {
                    if (s == 0) acc[k] = cmadd(acc[k], x, upd(phv[k]), f);
                    dn = dnv[k];
                } else {
                    if (s == 0) acc[k] = cmadd(acc[k], x, upd(ph[(size_t)k * nxy]), f);
                    dn = n[(size_t)k * nxy];
                }
                xs[pi][L.ob * M + k] = cpx<T>{(T)(x.x * dn.x - x.y * dn.y), (T)(x.x * dn.y + x.y * dn.x)};
            });
            __syncthreads();
            static_for<0, M>([&](auto mc) {
                constexpr int m = decltype(mc)::value;
                v[m] = xs[pi][S * m + L.h];  // z = S m + h
            });
            __syncthreads();
            PencilSplit<S>::template fft<T, NZ, -1, true>(v, L.h);  // -> z = ob M + k
            if (L.valid)
                static_for<0, M>([&](auto kc) {
                    constexpr int k = decltype(kc)::value;
                    g[o0 + (size_t)k * nxy] = scale(v[k], sc);
                });
        }
    }
    if (!L.valid) return;
    double2* q = qsum + ((size_t)te.app * 3 + d) * ng + o0;
    static_for<0, M>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        const double2 a = q[(size_t)k * nxy];
        q[(size_t)k * nxy] = make_double2(a.x + acc[k].x, a.y + acc[k].y);
    });
}

// ----------------------------------------------------------------- tc3a2a4b2b5 q-sums
// Per target t (q2,i2) and direction d = blockIdx.z, over its entries e = {record app, source
// occ (q1,i1), role kq}; v = O_0,s,d and w = O_1,s,d of the record (O[rec][6h + 3s + d], h = 1 only
// for BITC, else w = v):
//   Q2[d] -= f1 sum_s v conj(w)
//   Q4[d] += f1 v_0 phi_q1,   Q5[d] -= f1 conj(w_0 chi_q1)   (s = 0; Q5 for BITC only)
// Role 1: the record is that of the reversed pair (target q1, source q2).  With K odd under the
// exchange and rho_21 = conj of the other side's rho_12, O_0 of (q1, q2) is -conj(O_1) of
// (q2, q1) and the reverse, so v and w change places, conjugated and negated, and v conj(w)
// stays.  One pass reads each channel once and feeds all three sums (before, Q2 and Q4/Q5 read
// and transformed 18 channels per pair in separate passes, now 12).
// 40^3 FP32 BITC, 96 orbitals: 2.30 -> 1.67 us per ordered pair (3.7 TB/s of record reads; the
// FP64 accumulators leave two waves per SIMD).
// Two waves per SIMD where the accumulators leave room (the compiler took one for 36 points).
// kPart 0: all three sums; 1: Q2 only, 2: Q4 and Q5 only (s = 0), for BITC pencils of 15 points a
// lane, whose three accumulators would leave one wave per SIMD.
template <typename T, int NZ, int S, bool kBitc, int kPart>
__global__ __launch_bounds__(kPencilBlock, (NZ / S <= (sizeof(T) == 4 ? 12 : 10) ? 2 : 1)) void k_za8_q(const cpx<T>* __restrict__ O, const cpx<T>* __restrict__ occR,
                                                        const cpx<T>* __restrict__ chiR,
                                                        const PairEntry* __restrict__ entries,
                                                        const TargetEntry* __restrict__ targets,
                                                        const double* __restrict__ fill, double2* __restrict__ Q2,
                                                        size_t q2_slice, double2* __restrict__ Q4,
                                                        double2* __restrict__ Q5, int nxy)
{
    constexpr int M = NZ / S;
    constexpr int nch = kBitc ? 12 : 6;
    const LaneOf<S> L(nxy);
    const TargetEntry te = targets[blockIdx.y];
    const int d = blockIdx.z;
    const size_t ng = (size_t)nxy * NZ;
    const size_t o0 = L.xy + (size_t)L.ob * M * nxy;
    constexpr bool kQ2 = kPart != 2, kQ45 = kPart != 1;
    constexpr int s_first = kQ2 ? 1 : 0;
    double2 q2[kQ2 ? M : 1], q4[kQ45 ? M : 1], q5[kBitc && kQ45 ? M : 1];
    static_for<0, M>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        if constexpr (kQ2) q2[k] = make_double2(0.0, 0.0);
        if constexpr (kQ45) q4[k] = make_double2(0.0, 0.0);
        if constexpr (kBitc && kQ45) q5[k] = make_double2(0.0, 0.0);
    });
    // FP32 up to 40^3: the h = 0 pencil of the next (entry, s) step is loaded before this one is
    // transformed, the h = 1 pencil when v's registers are its own: 15.4 ms against 17.4 without
    // (96 orbitals at 40^3); both pencils ahead would spill
    constexpr bool kPrefetch = sizeof(T) == 4 && M <= 10;
    auto chan = [&](int rec, int h, int s) { return O + ((size_t)rec * nch + 6 * h + 3 * s + d) * ng; };
    const unsigned ioff = (unsigned)(L.xy + L.h * nxy) * sizeof(cpx<T>), ooff = (unsigned)o0 * sizeof(cpx<T>);
    cpx<T> vn[M];
    auto load = [&](int rec, int s) { ld_pencil<T, M>(vn, chan(rec, 0, s), ioff, S * nxy); };  // z = S m + h
    const int end = te.pair0 + te.npair;
    if (kPrefetch && te.npair > 0) load(entries[te.pair0].app, s_first);
#pragma unroll 1
    for (int i = te.pair0; i < end; ++i) {
        const PairEntry e = entries[i];
        const double f1 = fill[e.occ];
        const bool rev = e.kq != 0;
        static_for<0, 1 + s_first>([&](auto sc) {
            constexpr int s = s_first - decltype(sc)::value;
            if constexpr (!kPrefetch) load(e.app, s);
            cpx<T> v[M], w[kBitc ? M : 1];
            static_for<0, M>([&](auto mc) { v[decltype(mc)::value] = vn[decltype(mc)::value]; });
            if constexpr (kPrefetch) {
                if constexpr (s == 1)
                    load(e.app, 0);
                else if (i + 1 < end)
                    load(entries[i + 1].app, s_first);
            }
            PencilSplit<S>::template fft<T, NZ, 1>(v, L.h);  // -> z = ob M + k
            if constexpr (kBitc) { ld_pencil<T, M>(w, chan(e.app, 1, s), ioff, S * nxy); PencilSplit<S>::template fft<T, NZ, 1>(w, L.h); }
            __builtin_amdgcn_sched_barrier(0);  // the orbital points loaded earlier would spill
            const cpx<T>* ph = occR + (size_t)e.occ * ng;
            const cpx<T>* ch = chiR + (size_t)e.occ * ng;
            static_for<0, M>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                const double2 a = upd(v[k]);
                double2 b = a;
                if constexpr (kBitc) b = upd(w[k]);
                if constexpr (kQ2 && kBitc)
                    q2[k] = cmadd(q2[k], a, make_double2(b.x, -b.y), -f1);
                else if constexpr (kQ2)
                    q2[k].x -= f1 * (a.x * a.x + a.y * a.y);
                if constexpr (s == 0 && kQ45) {
                    // v_0 of the target: a, or -conj(b); conj(w_0): conj(b), or -a
                    const double2 x = make_double2(rev ? -b.x : a.x, rev ? b.y : a.y);
                    q4[k] = cmadd(q4[k], x, upd(ld<cpx<T>>(ph + (size_t)k * nxy, ooff)), f1);
                    if constexpr (kBitc) {
                        const double2 y = make_double2(rev ? -a.x : b.x, rev ? -a.y : -b.y), c = upd(ld<cpx<T>>(ch + (size_t)k * nxy, ooff));
                        q5[k] = cmadd(q5[k], y, make_double2(c.x, -c.y), -f1);
                    }
                }
                if constexpr (k % 2 == 1) __builtin_amdgcn_sched_barrier(0);
            });
        });
    }
    if (!L.valid) return;
    auto add = [&](double2* q, const double2 (&acc)[M]) {
        static_for<0, M>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            const double2 a = q[(size_t)k * nxy];
            q[(size_t)k * nxy] = make_double2(a.x + acc[k].x, a.y + acc[k].y);
        });
    };
    if constexpr (kQ2) add(Q2 + d * q2_slice + (size_t)te.app * ng + o0, q2);
    if constexpr (kQ45) add(Q4 + ((size_t)te.app * 3 + d) * ng + o0, q4);
    if constexpr (kBitc && kQ45) add(Q5 + ((size_t)te.app * 3 + d) * ng + o0, q5);
}

// Apply phase: W[t.app] += sum_p Z[p][0] phi_occ(p) + sum_d Z[p][1+d] Q4T[occ(p)][d]
template <typename T, int NZ, int S>
__global__ __launch_bounds__(kPencilBlock) void k_za8_apply(const cpx<T>* __restrict__ Z,
                                                            const cpx<T>* __restrict__ occR,
                                                            const cpx<T>* __restrict__ Q4T,
                                                            const PairEntry* __restrict__ pairs,
                                                            const TargetEntry* __restrict__ targets,
                                                            double2* __restrict__ W, float2* __restrict__ Wc,
                                                            int nxy)
{
    constexpr int M = NZ / S;
    const LaneOf<S> L(nxy);
    const TargetEntry te = targets[blockIdx.y];
    const size_t ng = (size_t)nxy * NZ;
    const size_t o0 = L.xy + (size_t)L.ob * M * nxy;
    double2 acc[M];
    static_for<0, M>([&](auto kc) { acc[decltype(kc)::value] = make_double2(0.0, 0.0); });
    // steps it = 4 (pair) + c; the pencil of step it + 1 is loaded before step it is
    // transformed (FP32)
    constexpr bool kPrefetch = sizeof(T) == 4;
    const int nsteps = 4 * te.npair;
    auto grid_of = [&](int it) { return Z + ((size_t)te.pair0 * 4 + it) * ng + L.xy + (size_t)L.h * nxy; };
    cpx<T> vn[M];
    if (kPrefetch && nsteps > 0) load_pencil<T, M>(vn, grid_of(0), S * nxy);
#pragma unroll 1
    for (int it = 0; it < nsteps; ++it) {
        const int pp = te.pair0 + it / 4, c = it % 4;
        const int o = pairs[pp].occ;
        {
            cpx<T> v[M];
            if (kPrefetch) {
                static_for<0, M>([&](auto mc) { v[decltype(mc)::value] = vn[decltype(mc)::value]; });
                if (it + 1 < nsteps) load_pencil<T, M>(vn, grid_of(it + 1), S * nxy);
            } else {
                load_pencil<T, M>(v, grid_of(it), S * nxy);  // z = S m + h
            }
            PencilSplit<S>::template fft<T, NZ, 1>(v, L.h);  // -> z = ob M + k
            const cpx<T>* m = (c == 0 ? occR + (size_t)o * ng : Q4T + ((size_t)o * 3 + (c - 1)) * ng) + o0;
            static_for<0, M>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                acc[k] = cmadd(acc[k], upd(v[k]), upd(m[(size_t)k * nxy]), 1.0);
            });
        }
    }
    if (!L.valid) return;
    const size_t o = (size_t)te.app * ng + o0;
    static_for<0, M>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        add_partial(W + o + (size_t)k * nxy, Wc ? Wc + o + (size_t)k * nxy : nullptr, acc[k].x, acc[k].y);
    });
}

// ----------------------------------------------------------------- launchers
namespace {

template <typename F>
void for_target_slices(int n, F&& f)
{
    for (int a = 0; a < n; a += 65535) f(a, n - a < 65535 ? n - a : 65535);
}

}  // namespace

#define TCX_Z_DISPATCH(prec, g, LAUNCH)                        \
    do {                                                       \
        if ((prec) == TCX_PREC_FP64) {                         \
            using T = double;                                  \
            TCX_SIZE_SWITCH((g).n3, LAUNCH)                    \
        } else {                                               \
            using T = float;                                   \
            TCX_SIZE_SWITCH((g).n3, LAUNCH)                    \
        }                                                      \
        TCX_HIP_CHECK(hipGetLastError());                      \
    } while (0)

void launch_za7_mid(int prec, const Geom& g, void* P, const void* occR, const PairEntry* pairs,
                    const TargetEntry* targets, int ntargets, const double* fill, const double* dens,
                    long long dens_stride, double* qsum, double sc, hipStream_t s)
{
    const int nxy = g.n1 * g.n2;
    for_target_slices(ntargets, [&](int a, int n) {
#define TCX_L(NZ)                                                                                            \
    {                                                                                                        \
        constexpr int S = SplitFor<NZ, 4>::value;                                                            \
        constexpr int PN = PencilSplit<S>::pencils;                                                          \
        hipLaunchKernelGGL((k_za7_mid<T, NZ, S>), dim3((nxy + PN - 1) / PN, n, 3), dim3(kPencilBlock), 0, s,\
                           (cpx<T>*)P, (const cpx<T>*)occR, pairs, targets + a, fill, (const double2*)dens,  \
                           (size_t)dens_stride, (double2*)qsum, nxy, (T)sc);                                 \
    }
        TCX_Z_DISPATCH(prec, g, TCX_L);
#undef TCX_L
    });
}

void launch_za8_q(int prec, const Geom& g, const void* O, int bitc, const void* occR, const void* chiR,
                  const PairEntry* entries, const TargetEntry* targets, int ntargets, const double* fill, double* Q2,
                  size_t q2_slice, double* Q4, double* Q5, hipStream_t s)
{
    const int nxy = g.n1 * g.n2;
    for_target_slices(ntargets, [&](int a, int n) {
#define TCX_L(NZ)                                                                                              \
    {                                                                                                          \
        constexpr int S = SplitFor<NZ, 4>::value;                                                              \
        constexpr int PN = PencilSplit<S>::pencils;                                                            \
        const dim3 grid((nxy + PN - 1) / PN, n, 3);                                                            \
        constexpr bool kSplit = NZ / S > 12;                                                                   \
        if (bitc) {                                                                                            \
            hipLaunchKernelGGL((k_za8_q<T, NZ, S, true, kSplit ? 1 : 0>), grid, dim3(kPencilBlock), 0, s, (const cpx<T>*)O,        \
                               (const cpx<T>*)occR, (const cpx<T>*)chiR, entries, targets + a, fill, (double2*)Q2,  \
                               q2_slice, (double2*)Q4, (double2*)Q5, nxy);                                          \
            if (kSplit)                                                                                        \
                hipLaunchKernelGGL((k_za8_q<T, NZ, S, true, kSplit ? 2 : 0>), grid, dim3(kPencilBlock), 0, s, (const cpx<T>*)O,        \
                               (const cpx<T>*)occR, (const cpx<T>*)chiR, entries, targets + a, fill, (double2*)Q2,  \
                               q2_slice, (double2*)Q4, (double2*)Q5, nxy);                                      \
        } else                                                                                                 \
            hipLaunchKernelGGL((k_za8_q<T, NZ, S, false, 0>), grid, dim3(kPencilBlock), 0, s, (const cpx<T>*)O,        \
                               (const cpx<T>*)occR, (const cpx<T>*)chiR, entries, targets + a, fill, (double2*)Q2,  \
                               q2_slice, (double2*)Q4, (double2*)Q5, nxy);                                          \
    }
        TCX_Z_DISPATCH(prec, g, TCX_L);
#undef TCX_L
    });
}

void launch_za8_apply(int prec, const Geom& g, const void* Z, const void* occR, const void* Q4T,
                      const PairEntry* pairs, const TargetEntry* targets, int ntargets, double* W, float* Wc,
                      hipStream_t s)
{
    const int nxy = g.n1 * g.n2;
    for_target_slices(ntargets, [&](int a, int n) {
#define TCX_L(NZ)                                                                                              \
    {                                                                                                          \
        constexpr int S = SplitFor<NZ, sizeof(T) == 8 ? 4 : 2>::value;                                         \
        constexpr int PN = PencilSplit<S>::pencils;                                                            \
        hipLaunchKernelGGL((k_za8_apply<T, NZ, S>), dim3((nxy + PN - 1) / PN, n), dim3(kPencilBlock), 0, s,   \
                           (const cpx<T>*)Z, (const cpx<T>*)occR, (const cpx<T>*)Q4T, pairs, targets + a,      \
                           (double2*)W, (float2*)Wc, nxy);                                                     \
    }
        TCX_Z_DISPATCH(prec, g, TCX_L);
#undef TCX_L
    });
}

#undef TCX_Z_DISPATCH

}  // namespace tcx
