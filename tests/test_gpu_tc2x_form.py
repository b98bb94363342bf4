"""tc2x on its four record channels, against the oracle and against its own formula in 32 bits.

Every compiled grid size, TC and BITC, both precisions, ragged bands with an empty k; then bases whose
spans go past half the grid, where sums of basis vectors wrap.  FP64 within 1e-10 relative.  FP32-split
per band within the rounding bound of its path (fp32_rounding).

The precision test holds FP32-split to what the reference's formula gives in 32 bits: with
K = k - q + G, the products are K_d (chi* d_d phi_j) and (K_d u) rho, so rounding is relative to K p.
Forms with fewer channels write K.p as a difference of squares; their rounding is relative to p^2, and
grows with p/K (bands that reach the cut-off) and with A: 1.7 to 2.9 times the error of this formula in
complex64 for these inputs.  The library's transforms round no more than plain ones (0.5 to 0.85 times
that error); the bound is 1.5 times, between the two.
"""
import math

import numpy as np
import pytest
import scipy.fft

from oracle import oracle as O
from tc_amd import system as S
from tc_amd import tcx
from test_gpu_hf2x import fp32_rounding, per_band_rel

pytestmark = pytest.mark.gpu


def check(engine, sys_, nb, seed):
    engine.load_system(sys_)
    _, phi = S.applied_bands(sys_, nb=nb, seed=seed)
    ref = O.Oracle(sys_).tc2x(nb, phi)
    for prec, tol in ((tcx.PREC_FP64, 1e-10), (tcx.PREC_FP32, fp32_rounding(sys_.n))):
        got = engine.tc2x(nb, phi, precision=prec)
        rel = per_band_rel(sys_, nb, got, ref).max()
        print(sys_.name, "precision", prec, f"per-band rel max {rel:.3e} (bound {tol:.1e})", flush=True)
        assert rel <= tol


@pytest.mark.parametrize("grid", [6, 8, 10, 12, 16, 18, 20, 24, 30, 32, 36, 40, 48])
@pytest.mark.parametrize("method", ["TC", "BITC"])
def test_grid_sizes(engine, grid, method):
    sys_ = S.build_system(S.fcc_lattice(10.26 if grid > 20 else 6.0), (grid,) * 3, (2, 1, 1), nbands=3, nocc=2,
                          seed_stream=600 + grid, method=method, A=np.full((2, 2), 0.5), name=f"{method} {grid}^3")
    check(engine, sys_, np.array([3, 0] if grid % 4 else [1, 3], np.int32), 601)


@pytest.mark.parametrize("n", [(12, 12, 18), (20, 20, 12)])
@pytest.mark.parametrize("scale", [0.8, 1.0, 1.15, 1.4, 1.9])
def test_bases_that_wrap(engine, n, scale):
    lat = S.fcc_lattice(6.0)
    sys_ = S.build_system(lat, n, (4, 1, 2), nbands=2, nocc=2, seed_stream=640, method="BITC",
                          A=np.full((2, 2), 0.5), gw=scale * S.gw_rule(lat, n), name=f"BITC {n} x{scale}")
    check(engine, sys_, np.full(sys_.nk, 1, np.int32), 641)


def tc2x_plain(sys_, k, coef, ctype, rtype):
    """src/calc_hamiltonian_tc2x.cpp:253-401 for one band at k, products and FFTs in ctype, kernel
    tables rounded to rtype, the pair sum in 64 bits."""
    n1, n2, n3 = sys_.n
    N = n1 * n2 * n3
    G = (S.miller_of_index(sys_.n) @ sys_.recip).T.reshape(3, n3, n2, n1)
    kc = sys_.kfrac @ sys_.recip
    po = np.concatenate([[0], np.cumsum(sys_.npw)])
    A, F = sys_.A[0, 0], sys_.F[0, 0]

    def real(q, c, d=None):  # FP64 transforms of the orbitals, rounded once
        g = np.zeros(N, complex)
        g[sys_.gindex[po[q]:po[q + 1]]] = c
        g = g.reshape(n3, n2, n1)
        return (scipy.fft.ifftn(g if d is None else g * (kc[q, d] + G[d])) * N).astype(ctype)

    def fwd(x):
        return scipy.fft.fftn(x) * rtype(1.0 / N)

    def bwd(x):
        return scipy.fft.ifftn(x, norm="forward")

    a, ga = real(k, coef), [real(k, coef, d) for d in range(3)]
    W = np.zeros((n3, n2, n1), complex)
    o = 0
    for q in range(sys_.nk):
        K = [G[d] + kc[k, d] - kc[q, d] for d in range(3)]
        x2 = K[0] ** 2 + K[1] ** 2 + K[2] ** 2
        z = x2 < 1e-12
        x2 = np.where(z, 1.0, x2)
        u = np.where(z, -4 * math.pi * A * F * F, 4 * math.pi * A / (x2 * (x2 * F * F + 1.0)))
        p, f2, x = math.pi * A * A / F ** 2, F * F * x2, np.sqrt(x2)
        v = 4 * math.pi / x2 - 4 * math.pi * A / (1 + f2) + (p / x) * (
            math.pi * f2 + (4 + 2 * f2) * np.arctan(F * x / 2) - (4 + 4 * f2) * np.arctan(F * x))
        v = np.where(z, -2 * p * F, v).astype(rtype)
        Ku = [(K[d] * u).astype(rtype) for d in range(3)]
        for i in range(sys_.nocc[q]):
            f = sys_.filling[o]
            m = int(np.sum(sys_.nocc[:q] * sys_.npw[:q])) + i * int(sys_.npw[q])
            c, l = sys_.phi_occ[m:m + sys_.npw[q]], sys_.chi_occ[m:m + sys_.npw[q]]
            chi = np.conj(real(q, l))
            rho = fwd(chi * a)
            b = rho * v
            for d in range(3):
                b += fwd(chi * ga[d]) * Ku[d]
            W += f * (bwd(b) * real(q, c)).astype(complex)
            for d in range(3):
                W -= f * (bwd(rho * Ku[d]) * real(q, c, d)).astype(complex)
            o += 1
    w = scipy.fft.fftn(W).reshape(-1)[sys_.gindex[po[k]:po[k + 1]]] / N
    return w * (-0.5 / (sys_.nk * sys_.volume))


@pytest.mark.parametrize("n,mesh", [((40, 40, 40), (2, 2, 2)), ((24, 24, 30), (2, 2, 1))])
@pytest.mark.parametrize("A,flat", [(0.5, True), (4.0, False)])
def test_fp32_precision(engine, n, mesh, A, flat):
    """Bands as heavy at the cut-off as at k = 0, and a strong Jastrow factor (F = sqrt A)."""
    lat = S.fcc_lattice(10.26)
    sys_ = S.build_system(lat, n, mesh, nbands=3, nocc=3, seed_stream=650, method="BITC", A=np.full((2, 2), A),
                          F=np.full((2, 2), math.sqrt(A)), div_corr=False)
    rng = np.random.default_rng(651)
    if flat:
        for k in range(sys_.nk):
            m, w = sys_.npw[k], int(np.sum(sys_.nocc[:k] * sys_.npw[:k]))
            r, x = (np.linalg.qr((rng.standard_normal((m, 3)) + 1j * rng.standard_normal((m, 3))))[0].T for _ in "rl")
            left = r + 0.3 * x
            sys_.phi_occ[w:w + 3 * m] = r.reshape(-1)
            sys_.chi_occ[w:w + 3 * m] = (np.conj(np.linalg.inv(np.conj(left) @ r.T)) @ left).reshape(-1)
    engine.load_system(sys_)
    nb = np.zeros(sys_.nk, np.int32)
    nb[1] = 1
    phi = sys_.phi_occ[3 * sys_.npw[0]:3 * sys_.npw[0] + sys_.npw[1]].copy()
    ref = tc2x_plain(sys_, 1, phi, complex, float)
    scale = np.linalg.norm(ref)
    plain = np.linalg.norm(tc2x_plain(sys_, 1, phi, np.complex64, np.float32) - ref) / scale
    assert np.linalg.norm(engine.tc2x(nb, phi) - ref) <= 1e-11 * scale
    err = np.linalg.norm(engine.tc2x(nb, phi, precision=tcx.PREC_FP32) - ref) / scale
    print(n, A, flat, f"FP32-split {err:.2e}, the formula in complex64 {plain:.2e}", flush=True)
    assert err <= 1.5 * plain
