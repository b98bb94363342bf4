// tcx_plane.cpp -- host side of the plane-first pair pipeline (kernels_plane.hip): the
// support columns of the basis and the hf2x launch sequence.
//
// The pair density of (k,j | q,i) has G-space components G = G_k - G_q with G_k in the
// basis of k and G_q in the basis of q (src/calc_hamiltonian_hf2x.cpp:123-135 forms it
// from the two orbitals on the FFT grid).  Its (kx, ky) columns are therefore the
// differences of the two bases' columns.
#include <algorithm>
#include <vector>

#include "tcx_terms.hpp"

namespace tcx {

namespace {

int posmod(int a, int n)
{
    const int r = a % n;
    return r < 0 ? r + n : r;
}
int centered_host(int i, int n) { return i <= n / 2 ? i : i - n; }

}  // namespace

// Automatic order: plane-first in FP32-split (40^3, 4x4x4 k, 16 bands: 428 ms per apply against
// 535), z-first in FP64 (36^3: 18.2 ms of pair passes against 18.4; the FP64 line transforms of
// pass C take every register).  Calls that return numbers at the level of rounding keep the z-first
// sums that have given them so far (kFlagZFirst): tcx_davidson, whose eigensolver takes the phases of
// the eigenvectors from rounding-level entries, so another order flips the signs of some returned
// bands, and tcx_grad_exchange, whose imaginary part of E_x is rounding alone (0 by Hermiticity).
// hf2x is the only term with two orders; TC and BITC applies hold none of it.
bool Context::use_plane_first(int prec, unsigned flags) const
{
    if (prec != TCX_PREC_FP32 || hf2x_order == 0) return false;
    return hf2x_order == 1 || !(flags & kFlagZFirst);
}

// One column set for every (k, q): per kx, the hull of the ky differences of all bases.
// With the ky span of the whole set at most n2, ky rotated by the smallest difference makes
// every run contiguous; a run that still wraps (bases that alias on the grid) takes every ky.
// Hulls and the union only add columns, so the record holds every non-zero one.
// Found by tcx_set_basis from the grid points that some basis holds (`seen`): one pass over the
// grid without a division per plane wave.  Returns run[n1] and colxy[ncol]; they go to the device
// behind the grid indices, in the same copy.
std::vector<int> Context::set_columns(const std::vector<unsigned char>& seen)
{
    const int n1 = geo.n1, n2 = geo.n2, n3 = geo.n3, nxy = n1 * n2;
    const int none_lo = 1 << 20, none_hi = -(1 << 20);
    std::vector<unsigned char> col(nxy, 0);
    int mn[3] = {none_lo, none_lo, none_lo}, mx[3] = {none_hi, none_hi, none_hi};  // centred indices held
    auto widen = [&](int d, int m) {
        mn[d] = std::min(mn[d], m);
        mx[d] = std::max(mx[d], m);
    };
    for (int i3 = 0; i3 < n3; ++i3) {
        const unsigned char* p = seen.data() + (size_t)i3 * nxy;
        unsigned char any = 0;
        for (int e = 0; e < nxy; ++e) {
            col[e] |= p[e];
            any |= p[e];
        }
        if (any) widen(2, centered_host(i3, n3));
    }
    // per kx: [lo, hi] of centred ky over all bases (lo > hi: none)
    std::vector<int> lo(n1, none_lo), hi(n1, none_hi);
    for (int i2 = 0; i2 < n2; ++i2)
        for (int i1 = 0; i1 < n1; ++i1) {
            if (!col[(size_t)i2 * n1 + i1]) continue;
            const int m2 = centered_host(i2, n2);
            widen(0, centered_host(i1, n1));
            widen(1, m2);
            lo[i1] = std::min(lo[i1], m2);
            hi[i1] = std::max(hi[i1], m2);
        }
    std::vector<int> dlo(n1, none_lo), dhi(n1, none_hi);
    for (int a = 0; a < n1; ++a) {
        if (lo[a] > hi[a]) continue;
        for (int b = 0; b < n1; ++b) {
            if (lo[b] > hi[b]) continue;
            const int x = posmod(centered_host(a, n1) - centered_host(b, n1), n1);
            dlo[x] = std::min(dlo[x], lo[a] - hi[b]);
            dhi[x] = std::max(dhi[x], hi[a] - lo[b]);
        }
    }
    int first_ky = none_lo;
    for (int x = 0; x < n1; ++x) first_ky = std::min(first_ky, dlo[x]);
    std::vector<int> run(n1), colxy;
    for (int x = 0; x < n1; ++x) {
        int l = 0, len = 0;
        if (dlo[x] <= dhi[x]) {
            l = dlo[x] - first_ky;
            len = dhi[x] - dlo[x] + 1;
            if (l + len > n2) {
                l = 0;
                len = n2;
            }
            // whole 32-byte sectors per run (4 FP32 values): fewer partly written lines
            // (pass A at 40^3 FP32 152 -> 139 ms for 1% more columns)
            len = std::min(n2, (len + 3) / 4 * 4);
            l = std::min(l, n2 - len);
        }
        run[x] = l | (len << 8) | ((int)colxy.size() << 16);
        for (int j = 0; j < len; ++j) colxy.push_back(x | (posmod(first_ky + l + j, n2) << 16));
    }
    cols.ncol = (int)colxy.size();
    // record rows start on 128-byte lines, unless that would make them longer than a grid plane
    cols.cstride = std::min((cols.ncol + 15) / 16 * 16, nxy);
    cols.rot = posmod(first_ky, n2);
    // No difference of two basis vectors reaches the Nyquist index or wraps: with every basis inside a
    // span s of Miller indices per direction, 2 s < n keeps the differences inside (-n/2, n/2), where
    // -G has the index opposite to G's and K(-G) = -K(G).
    const int n[3] = {n1, n2, n3};
    basis_no_alias = true;
    for (int d = 0; d < 3; ++d) basis_no_alias = basis_no_alias && 2 * (mx[d] - mn[d]) < n[d];
    run.insert(run.end(), colxy.begin(), colxy.end());
    return run;
}

// The three plane-first passes of every launch; W (FP64) was cleared by the caller.
void Context::hf2x_plane_first(const Plan& P)
{
    const PlaneCols& pc = cols;
    hf2x_record_cols = pc.ncol;
    const size_t es = 8, plane = (size_t)geo.n3 * pc.cstride;
    d_pairbuf.ensure((size_t)std::max(1, P.max_launch_pairs) * plane * es);
    int max_rows = 1;
    for (const Launch& L : P.launches) max_rows = std::max(max_rows, L.nkq);
    d_ktab.ensure((size_t)max_rows * plane * (es / 2));
    for (const Launch& L : P.launches) {
        const PairEntry* pairs = (const PairEntry*)P.d_pairs.p + L.pair0;
        const TargetEntry* targets = (const TargetEntry*)P.d_targets.p + L.target0;
        launch_plane_coulomb(d_ktab.p, (const double*)P.d_kq.p, L.kq0, L.nkq, pc, geo, stream);
        timed(0, L.npairs, [&] {
            launch_plane_A(geo, d_appR.p, d_occR[TCX_PREC_FP32].p, pairs, L.ntargets, L.npairs / L.ntargets, pc,
                           d_pairbuf.p, stream);  // every source of a launch pairs with every target
        });
        timed(1, L.npairs, [&] {
            launch_plane_Z(geo, d_pairbuf.p, pairs, L.npairs, d_ktab.p, L.kq0, pc, stream);
        });
        timed(2, L.npairs, [&] {
            launch_plane_C(geo, d_pairbuf.p, d_occR[TCX_PREC_FP32].p, pairs, targets, L.ntargets, pc,
                           (const double*)d_fill.p, (double*)d_W.p, (float*)d_Wc.p, stream);
        });
    }
}

}  // namespace tcx
