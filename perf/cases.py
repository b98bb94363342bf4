"""The work that users of this package have it do, as cases that can be timed and checked.

A case is one call (or the short call sequence of one SCF iteration) on one plane-wave
system, through the entry points of `tc_amd.tcx.Engine`.  The sizes are those of the
package's own configurations and tests: homogeneous-electron-gas cells in simple cubic and
fcc lattices, FFT grids of 16 to 48 points per side, one to 64 k-points, 2 to 16 occupied
bands per k (the same number everywhere, or ragged as a metal's are), HF, TC and BITC, the
FP64 pipeline and the FP32-split one.  Bands carry fillings as Gaussian smearing leaves
them: 2, and a fraction in the highest band.

`op` of a case:
  hf2x, tc2x, tc3a3b3b4b6   one term applied to a block of trial bands, as block Davidson does;
  tc3a2a4b2b5               the same after new occupied orbitals were set, as every SCF
                            iteration does (the term's occupied-set sums belong to it);
  apply_all                 new occupied orbitals, then the whole H*phi;
  davidson                  new occupied orbitals, then one block-Davidson call;
  grad_exchange, grad_tc2   energy and orbital gradients of the occupied set (backward).
"""
import math

import numpy as np
import torch

from tc_amd import system as S
from tc_amd import tcx

FOURPI = 4.0 * math.pi
LATTICES = {"fcc": (S.fcc_lattice, 10.26), "sc": (S.sc_lattice, 15.62)}
GRIDS = (16, 18, 20, 24, 30, 32, 36, 40, 48)


def listed():
    def case(name, op, method, prec, lattice, n, n3, mesh, occ, app, ragged=False):
        return {"name": name, "op": op, "method": method, "prec": prec, "lattice": lattice, "n": n, "n3": n3,
                "k1": mesh[0], "k2": mesh[1], "k3": mesh[2], "occ": occ, "app": app, "ragged": ragged}

    return [
        # a cell at Gamma: the smallest apply, where launches and the host path count
        case("hf2x_gamma_16", "hf2x", "HF", "fp64", "sc", 16, 16, (1, 1, 1), 4, 4),
        # one SCF iteration of the simple-cubic HEG (7 of 8 bands occupied) on its 24^3 grid
        case("davidson_hf_24", "davidson", "HF", "fp64", "sc", 24, 24, (2, 2, 2), 7, 8),
        # the whole transcorrelated H*phi at the size of the package's TC and BITC example runs
        case("apply_all_tc_20", "apply_all", "TC", "fp64", "fcc", 20, 20, (2, 2, 2), 4, 6),
        # the same in FP32-split with ragged bands on a non-cubic grid
        case("apply_all_bitc_24x18", "apply_all", "BITC", "fp32", "sc", 24, 18, (2, 2, 1), 6, 6, True),
        # exchange of a converged k-mesh: the headline workload's cell
        case("hf2x_fp32_40", "hf2x", "HF", "fp32", "fcc", 40, 40, (4, 4, 4), 16, 16),
        # exchange in FP64, ragged bands, fewer k
        case("hf2x_fp64_36_ragged", "hf2x", "HF", "fp64", "fcc", 36, 36, (3, 3, 2), 13, 15, True),
        # two-body transcorrelated exchange, BITC, half the headline mesh
        case("tc2x_fp32_40", "tc2x", "BITC", "fp32", "fcc", 40, 40, (4, 4, 2), 14, 14),
        # the same in FP64 on a mixed grid with ragged bands
        case("tc2x_fp64_32x30_ragged", "tc2x", "TC", "fp64", "sc", 32, 30, (2, 2, 2), 11, 9, True),
        # three-body exchange terms at 40^3
        case("tc3a3b3b4b6_fp32_40", "tc3a3b3b4b6", "BITC", "fp32", "fcc", 40, 40, (2, 2, 2), 12, 12),
        case("tc3a2a4b2b5_fp32_40", "tc3a2a4b2b5", "BITC", "fp32", "fcc", 40, 40, (2, 2, 2), 12, 12),
        # one of them in FP64 at a middle grid, TC
        case("tc3a3b3b4b6_fp64_30", "tc3a3b3b4b6", "TC", "fp64", "fcc", 30, 30, (2, 2, 2), 7, 8, True),
        # energy and gradients of the BITC two-body energy on the largest grid
        case("grad_tc2_fp32_48", "grad_tc2", "BITC", "fp32", "fcc", 48, 48, (2, 2, 2), 9, 9),
    ]


# relative cost of one band pair at one grid point
_COST = {"hf2x": 1.0, "davidson": 2.5, "tc2x": 4.0, "tc3a3b3b4b6": 13.0, "tc3a2a4b2b5": 14.0, "apply_all": 32.0,
         "grad_exchange": 1.0, "grad_tc2": 9.0}


def _cost(c):
    nk = c["k1"] * c["k2"] * c["k3"]
    w = _COST["davidson" if c["op"] == "davidson" else c["op"]]
    if c["op"] == "apply_all" and c["method"] == "HF":
        w = 1.2
    pairs = (nk * c["occ"]) * (nk * max(c["occ"], c["app"]))
    return w * (2.0 if c["prec"] == "fp64" else 1.0) * pairs * c["n"] * c["n"] * c["n3"]


def draw(rng):
    biggest = max(_cost(c) for c in listed())
    while True:
        op = rng.choice(["hf2x", "hf2x", "tc2x", "tc2x", "tc3a3b3b4b6", "tc3a2a4b2b5", "apply_all", "davidson",
                         "grad_exchange", "grad_tc2"])
        if op in ("hf2x", "grad_exchange"):
            method = "HF"
        elif op == "davidson":
            method = "HF"
        elif op == "apply_all":
            method = rng.choice(["HF", "TC", "BITC"])
        else:
            method = rng.choice(["TC", "BITC"])
        n = rng.choice(GRIDS)
        n3 = rng.choice([m for m in GRIDS if n / 2 <= m <= 2 * n]) if rng.random() < 0.3 else n
        mesh = rng.choice([(1, 1, 1), (2, 1, 1), (2, 2, 1), (2, 2, 2), (3, 2, 2), (3, 3, 2), (3, 3, 3), (4, 4, 2)])
        occ = rng.randint(2, 16)
        app = occ if op.startswith("grad") else (occ + rng.randint(0, 2) if op == "davidson" else rng.randint(2, 16))
        c = {"op": op, "method": method, "prec": rng.choice(["fp32", "fp64"]), "lattice": rng.choice(["fcc", "sc"]),
             "n": n, "n3": n3, "k1": mesh[0], "k2": mesh[1], "k3": mesh[2], "occ": occ, "app": app,
             "ragged": op != "davidson" and rng.random() < 0.5}
        if _cost(c) <= 0.6 * biggest:  # a drawn case costs no more than the largest listed one
            return c


# ----------------------------------------------------------------------------- inputs
def _counts(case, most, which):
    """Bands per k: part of the case's shape, so the same for every seed."""
    nk = case["k1"] * case["k2"] * case["k3"]
    if not case["ragged"]:
        return np.full(nk, most, np.int32)
    r = np.random.default_rng([7, which, most, nk])
    return r.integers(max(1, most // 3), most + 1, size=nk).astype(np.int32)


def _make(case, seed):
    """The system (occupied orbitals) and the trial bands of a case."""
    make, a = LATTICES[case["lattice"]]
    lattice, n = make(a), (case["n"], case["n"], case["n3"])
    recip = S.reciprocal_rows(lattice)
    kfrac = S.mp_mesh(case["k1"], case["k2"], case["k3"])
    gcart0 = S.miller_of_index(n) @ recip
    gw = S.gw_rule(lattice, n)
    r = np.random.default_rng([11, seed])
    nocc, napp = _counts(case, case["occ"], 0), _counts(case, case["app"], 1)
    if case["op"].startswith("grad"):
        napp = nocc
    npw, gidx, phi, chi, app, fill = [], [], [], [], [], []
    for k, kf in enumerate(kfrac):
        kg2 = np.sum((gcart0 + kf @ recip) ** 2, axis=1)
        sel = np.nonzero(kg2 <= gw * gw + 1e-12)[0]
        sel = sel[np.lexsort((sel, np.round(kg2[sel], 10)))]
        env = np.exp(-kg2[sel] / 2.0)

        def block(m):
            c = (r.standard_normal((m, len(sel))) + 1j * r.standard_normal((m, len(sel)))) * env
            return np.linalg.qr(c.T)[0].T

        right = block(nocc[k])
        if case["method"] == "BITC":  # left orbitals near the right ones, <left_a|right_b> = delta_ab
            left = right + 0.3 * block(nocc[k])
            chi.append((np.conj(np.linalg.inv(np.conj(left) @ right.T)) @ left).reshape(-1))
        npw.append(len(sel))
        gidx.append(sel.astype(np.int32))
        phi.append(right.reshape(-1))
        app.append(block(napp[k]).reshape(-1))
        f = np.full(nocc[k], 2.0)
        f[-1] = 2.0 * r.uniform(0.2, 1.0)
        fill.append(f)
    A = np.zeros((2, 2)) if case["method"] == "HF" else np.full((2, 2), 0.5)
    F = np.array([[1.0, math.sqrt(0.5)], [math.sqrt(0.5), 1.0]]) if case["method"] != "HF" else np.ones((2, 2))
    sysm = S.System(lattice=lattice, recip=recip, volume=abs(float(np.linalg.det(lattice))), n=n, kfrac=kfrac,
                    npw=np.array(npw, np.int32), gindex=np.concatenate(gidx), nocc=nocc, filling=np.concatenate(fill),
                    phi_occ=np.concatenate(phi), chi_occ=np.concatenate(chi) if chi else None,
                    method=case["method"], A=A, F=F)
    return sysm, napp, np.concatenate(app)


def prepare(case, seed):
    sysm, napp, app = _make(case, seed)
    eng = tcx.Engine(0)
    eng.load_system(sysm)
    return {"case": case, "eng": eng, "sys": sysm, "nb": napp, "phi": app, "eig": np.zeros(int(napp.sum()), complex),
            "prec": tcx.PREC_FP32 if case["prec"] == "fp32" else tcx.PREC_FP64}


def run(state):
    eng, sysm, op, prec = state["eng"], state["sys"], state["case"]["op"], state["prec"]
    if op in ("apply_all", "davidson", "tc3a2a4b2b5"):  # an SCF iteration: new occupied orbitals first
        eng.set_states(sysm.nocc, sysm.filling, sysm.phi_occ, sysm.chi_occ)
    if op == "apply_all":
        h1, h2, h3 = eng.apply_all(state["nb"], state["phi"], precision=prec)
        return [h1, h2] if h3 is None else [h1, h2, h3]
    if op == "davidson":
        phi, _, eig, en = eng.davidson(state["nb"], state["phi"], state["eig"], precision=prec)
        return [eig, en, phi]
    if op == "grad_exchange":
        e, g = eng.grad_exchange(precision=prec)
        return [e.real, e.imag, g]
    if op == "grad_tc2":
        e, gl, gr, da = eng.grad_tc2(precision=prec)
        return [e.real, e.imag, gl, gr, da.real, da.imag]
    return getattr(eng, op)(state["nb"], state["phi"], precision=prec)


# ----------------------------------------------------------------------------- work and tolerance
def _pairs(case):
    """Expected (trial x occupied, occupied x occupied) band pairs of a case."""
    nk = case["k1"] * case["k2"] * case["k3"]

    def total(m):
        return nk * (m if not case["ragged"] else 0.5 * (max(1, m // 3) + m))

    return total(case["app"]) * total(case["occ"]), total(case["occ"]) ** 2


def work(case):
    make, a = LATTICES[case["lattice"]]
    n = (case["n"], case["n"], case["n3"])
    N = n[0] * n[1] * n[2]
    lattice = make(a)
    gw = S.gw_rule(lattice, n)
    npw = gw ** 3 / (6.0 * math.pi ** 2) * abs(float(np.linalg.det(lattice)))
    nk = case["k1"] * case["k2"] * case["k3"]
    app, occ = _pairs(case)
    left = 2 if case["method"] == "BITC" else 1
    # 3D FFTs of N points per band pair, as the operators are written
    tc3a = (app * 8 + occ * 7 * left)
    ffts = {"hf2x": 2 * app, "tc2x": 8 * app, "tc3a3b3b4b6": 21 * app, "tc3a2a4b2b5": tc3a,
            "davidson": 2 * 2 * app, "grad_exchange": 2 * occ, "grad_tc2": 3 * 8 * occ,
            "apply_all": 2 * app if case["method"] == "HF" else (8 + 21) * app + tc3a}[case["op"]]
    bands = math.sqrt(occ) * left + 2 * app / math.sqrt(occ)
    return {"bytes": 16.0 * npw * bands, "flops": ffts * 5.0 * N * math.log2(N)}


def tolerance(case):
    # measured against 64-bit sums in another order: FP64 1e-15 and FP32-split up to 1e-7 (2-norm);
    # a two-body term of 32-bit transforms in another order may differ by a few times that.  The
    # iterated call divides by level spacings, which magnifies both.
    if case["op"] == "davidson":
        return {"rel": 1e-9, "max": 1e-7} if case["prec"] == "fp64" else {"rel": 2e-5, "max": 1e-3}
    if case["prec"] == "fp64":
        return {"rel": 1e-13, "max": 1e-11}
    return {"rel": 1e-6, "max": 1e-4}


# ----------------------------------------------------------------------------- the same in 64 bits
class _Ref:
    """The operators as sums over band pairs with complex128 FFTs in plain torch."""

    def __init__(self, case, sysm):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.s, self.n = sysm, sysm.n
        n1, n2, n3 = sysm.n
        self.N, self.shape = n1 * n2 * n3, (n3, n2, n1)

        def centred(n):
            i = np.arange(n)
            return np.where(i <= n // 2, i, i - n)

        m3, m2, m1 = np.meshgrid(centred(n3), centred(n2), centred(n1), indexing="ij")
        G = np.stack([m1, m2, m3], -1) @ sysm.recip
        self.G = torch.as_tensor(np.moveaxis(G, -1, 0).copy(), device=self.dev)  # [3][n3][n2][n1]
        self.kc = torch.as_tensor(sysm.kfrac @ sysm.recip, device=self.dev)
        self.po = np.concatenate([[0], np.cumsum(sysm.npw)])
        self.NkV = sysm.nk * sysm.volume
        self.fill = np.split(sysm.filling, np.cumsum(sysm.nocc)[:-1])
        self.c_phi = self.blocks(sysm.nocc, sysm.phi_occ)
        self.c_chi = self.c_phi if sysm.chi_occ is None else self.blocks(sysm.nocc, sysm.chi_occ)
        self.phi = [self.real(k, c) for k, c in enumerate(self.c_phi)]
        self.chi = self.phi if sysm.chi_occ is None else [self.real(k, c) for k, c in enumerate(self.c_chi)]
        self.f = [torch.as_tensor(f, device=self.dev) for f in self.fill]
        self.rho = sum((f[:, None, None, None] * c.conj() * p).sum(0)
                       for f, c, p in zip(self.f, self.chi, self.phi)) / 2.0  # per spin
        self.div()

    def blocks(self, nb, c):
        out, o = [], 0
        for k in range(self.s.nk):
            m = int(nb[k]) * int(self.s.npw[k])
            out.append(torch.as_tensor(c[o:o + m].reshape(int(nb[k]), -1), device=self.dev))
            o += m
        return out

    def idx(self, k):
        return torch.as_tensor(self.s.gindex[self.po[k]:self.po[k + 1]].astype(np.int64), device=self.dev)

    def fwd(self, x):
        return torch.fft.fftn(x, dim=(-3, -2, -1)) / self.N

    def bwd(self, x):
        return torch.fft.ifftn(x, dim=(-3, -2, -1)) * self.N

    def real(self, k, c, d=None):
        """Orbitals c at k (or their (k+G)_d multiple) on the real-space grid."""
        g = torch.zeros((c.shape[0], self.N), dtype=torch.complex128, device=self.dev)
        g[:, self.idx(k)] = c
        g = g.reshape(-1, *self.shape)
        return self.bwd(g if d is None else g * (self.kc[k, d] + self.G[d]))

    def gather(self, k, w):
        return self.fwd(w).reshape(w.shape[0], -1)[:, self.idx(k)]

    def div(self):
        s = self.s
        self.alpha = (s.volume ** (1.0 / 3.0) / (2.0 * math.pi)) ** 2
        total = 0.0  # the same at every k of the mesh
        r = np.arange(-12, 13)
        shifts = np.stack(np.meshgrid(r, r, r, indexing="ij"), -1).reshape(-1, 3)
        for q in s.kfrac:
            g2 = np.sum(((s.kfrac[0] - q + shifts) @ s.recip) ** 2, axis=1)
            g2 = g2[g2 > 1e-8]
            total += float(np.sum(np.exp(-self.alpha * g2) / g2))
        self.vaux = FOURPI * total - FOURPI * self.alpha

    def u(self, x2, s):
        A, F2 = self.s.A[0, s], self.s.F[0, s] ** 2
        return torch.where(x2 < 1e-12, torch.full_like(x2, -FOURPI * A * F2),
                           FOURPI * A / (x2 * (x2 * F2 + 1.0)).clamp_min(1e-300))

    def tc2body(self, x2, s):
        A, F = self.s.A[0, s], self.s.F[0, s]
        p, f2 = math.pi * A * A / F ** 2, F * F * x2
        g = torch.sqrt(x2).clamp_min(1e-150)
        v = FOURPI / x2.clamp_min(1e-300) - FOURPI * A / (1.0 + f2) + (p / g) * (
            math.pi * f2 + (4.0 + 2.0 * f2) * torch.atan(F * g / 2.0) - (4.0 + 4.0 * f2) * torch.atan(F * g))
        return torch.where(x2 < 1e-12, torch.full_like(x2, -2.0 * p * F), v)

    def kq(self, k, q):
        K = self.G + (self.kc[k] - self.kc[q])[:, None, None, None]
        return K, (K * K).sum(0)

    # ------------------------------------------------------------------ exchange terms
    def projector(self, k, c, left):
        """Divergence correction: sum_b f dc |phi_b><left_b| on the bands c at k."""
        dc = -0.5 * (1.0 / math.sqrt(math.pi * self.alpha) - self.vaux / self.NkV)
        return (c @ left[k].conj().T * (dc * self.f[k])) @ self.c_phi[k]

    def hf2x(self, nb, app):
        out = []
        for k, c in enumerate(self.blocks(nb, app)):
            a = self.real(k, c)
            W = torch.zeros_like(a)
            for q in range(self.s.nk):
                x2 = self.kq(k, q)[1]
                v = torch.where(x2 < 1e-8, torch.zeros_like(x2), 1.0 / x2.clamp_min(1e-300))
                for j in range(len(a)):
                    V = self.bwd(self.fwd(self.phi[q].conj() * a[j]) * v)
                    W[j] += (self.f[q][:, None, None, None] * V * self.phi[q]).sum(0)
            out.append(-0.5 * FOURPI / self.NkV * self.gather(k, W) + self.projector(k, c, self.c_phi))
        return out

    def tc2x(self, nb, app):
        out = []
        grad = [[self.real(q, self.c_phi[q], d) for d in range(3)] for q in range(self.s.nk)]
        for k, c in enumerate(self.blocks(nb, app)):
            a, ga = self.real(k, c), [self.real(k, c, d) for d in range(3)]
            W = torch.zeros_like(a)
            for q in range(self.s.nk):
                K, x2 = self.kq(k, q)
                u, v2 = self.u(x2, 0), self.tc2body(x2, 0)
                for j in range(len(a)):
                    r = self.fwd(self.chi[q].conj() * a[j])
                    b = r * v2
                    t = 0.0
                    for d in range(3):
                        b += self.fwd(self.chi[q].conj() * ga[d][j]) * (K[d] * u)
                        t = t - self.bwd(r * (K[d] * u)) * grad[q][d]
                    W[j] += (self.f[q][:, None, None, None] * (self.bwd(b) * self.phi[q] + t)).sum(0)
            out.append(-0.5 / self.NkV * self.gather(k, W) + self.projector(k, c, self.c_chi))
        return out

    def dnu(self):
        x2 = (self.G ** 2).sum(0)
        n = self.fwd(self.rho)
        us = self.u(x2, 0) + self.u(x2, 1)
        return [self.bwd(us * self.G[d] * n) for d in range(3)]

    def tc3a3b3b4b6(self, nb, app):
        s, base = self.s, 1.0 / self.NkV ** 2
        fa3, fb3, fb4, fb6 = -base / 2, base / 2, -base / 4, base / 2
        dnu, n = self.dnu(), self.fwd(self.rho)
        x2g = (self.G ** 2).sum(0)
        dcp = self.NkV / math.sqrt(math.pi * self.alpha) - self.vaux
        t1, tG = 0.0, torch.zeros_like(n)
        for sp in range(2):
            A = s.A[0, sp]
            u = self.u(x2g, sp)
            t1 = t1 + FOURPI * A * (dcp * A + u[0, 0, 0]) * n[0, 0, 0]
            tG += FOURPI * A * u * n
        tG[0, 0, 0] = 0.0
        tR = self.bwd(tG)
        out = []
        for k, c in enumerate(self.blocks(nb, app)):
            a = self.real(k, c)
            W, Q = torch.zeros_like(a), torch.zeros((3, *a.shape), dtype=a.dtype, device=self.dev)
            o = torch.zeros_like(c)
            for q in range(s.nk):
                K, x2 = self.kq(k, q)
                us = [self.u(x2, 0), self.u(x2, 1)]
                fq = self.f[q][:, None, None, None]
                for j in range(len(a)):
                    r = self.fwd(self.chi[q].conj() * a[j]) * fq
                    y = 0.0
                    for d in range(3):
                        y = y + fb3 * fq * self.fwd(self.chi[q].conj() * (dnu[d] * a[j])) * (K[d] * us[0])
                        for sp in range(2):
                            p = self.bwd(r * (K[d] * us[sp]))
                            if sp == 0:
                                Q[d, j] += (p * self.phi[q]).sum(0)
                            y = y + fb6 * self.fwd(p * self.rho) * (K[d] * us[sp])
                    W[j] += (self.bwd(y) * self.phi[q]).sum(0)
            for j in range(len(a)):
                pp = self.chi[k].conj() * a[j]
                I = pp.mean((-3, -2, -1))
                dot = (pp * tR).mean((-3, -2, -1))
                cf = fb6 * self.f[k]
                o[j] += (cf * (t1 * I + dot)) @ self.c_phi[k]
                W[j] += ((cf * I)[:, None, None, None] * self.phi[k]).sum(0) * tR
                W[j] += fa3 * sum(Q[d, j] * dnu[d] for d in range(3))
            for q in range(s.nk):
                K, x2 = self.kq(k, q)
                u0 = self.u(x2, 0)
                for j in range(len(a)):
                    y = sum(self.fwd(self.chi[q].conj() * Q[d, j]) * (K[d] * u0) for d in range(3))
                    W[j] += fb4 * (self.f[q][:, None, None, None] * self.bwd(y) * self.phi[q]).sum(0)
            out.append(o + self.gather(k, W))
        return out

    def tc3a2a4b2b5(self, nb, app):
        s, base = self.s, 1.0 / self.NkV ** 2
        fa2, fa4, fb2, fb5 = -base / 8, base / 4, base / 4, -base / 4
        x2g = (self.G ** 2).sum(0)
        ug = [self.u(x2g, 0), self.u(x2g, 1)]
        a = [self.real(k, c) for k, c in enumerate(self.blocks(nb, app))]
        W = [torch.zeros_like(x) for x in a]
        V3, B2 = torch.zeros_like(self.rho), torch.zeros((3, *self.shape), dtype=torch.complex128, device=self.dev)
        dc2 = self.NkV / math.sqrt(math.pi * self.alpha) - self.vaux
        for q2 in range(s.nk):
            for i2 in range(len(self.phi[q2])):
                p2, c2, f2 = self.phi[q2][i2], self.chi[q2][i2], float(self.fill[q2][i2])
                Q2 = torch.zeros_like(p2)
                Q4, Q5 = torch.zeros_like(B2), torch.zeros_like(B2)
                for q1 in range(s.nk):
                    K, x2 = self.kq(q2, q1)
                    f1 = self.f[q1][:, None, None, None]
                    r = self.fwd(self.chi[q1].conj() * p2)
                    l = self.fwd(self.phi[q1].conj() * c2)
                    for sp in range(2):
                        u = self.u(x2, sp)
                        for d in range(3):
                            x = self.bwd(r * (K[d] * u))
                            y = x if self.chi is self.phi else self.bwd(l * (K[d] * u))
                            Q2 -= (f1 * x * y.conj()).sum(0)
                            if sp == 0:
                                Q4[d] += (f1 * x * self.phi[q1]).sum(0)
                                Q5[d] -= (f1 * y.conj() * self.chi[q1].conj()).sum(0)
                T = self.fwd(Q2)
                pa, pb = self.fwd(self.chi[q2].conj() * p2), self.fwd(c2.conj() * self.phi[q2])
                f1 = self.f[q2]
                pa0, pb0 = pa[:, 0, 0, 0], pb[:, 0, 0, 0]
                for sp in range(2):
                    A = s.A[0, sp]
                    t0 = FOURPI * A * (A * dc2 + ug[sp][0, 0, 0]) * (f1 * pa0 * pb0).sum()
                    tg = FOURPI * A * ug[sp] * ((f1 * pb0)[:, None, None, None] * pa
                                                + (f1 * pa0)[:, None, None, None] * pb).sum(0)
                    tg[0, 0, 0] = t0
                    T = T - tg
                V3 += f2 * T
                B2 += f2 * Q5 * p2
                for k in range(s.nk):
                    K, x2 = self.kq(k, q2)
                    u0 = self.u(x2, 0)
                    r = self.fwd(c2.conj() * a[k]) * (f2 * fa4)
                    b = 0.0
                    for d in range(3):
                        W[k] += Q4[d] * self.bwd(r * (K[d] * u0))
                        b = b + self.fwd(Q5[d] * a[k]) * (K[d] * u0)
                    W[k] += fb5 * f2 * self.bwd(b) * p2
        X = self.bwd(fb2 * sum(self.fwd(B2[d]) * self.G[d] for d in range(3)) * (ug[0] + ug[1]) + fa2 * V3)
        return [self.gather(k, W[k] + X * a[k]) for k in range(s.nk)]

    # ------------------------------------------------------------------ local terms
    def local(self, nb, app, V, vec=None):
        out = []
        for k, c in enumerate(self.blocks(nb, app)):
            w = V * self.real(k, c)
            if vec is not None:
                w = w - sum(vec[d] * self.real(k, c, d) for d in range(3))
            out.append(self.gather(k, w))
        return out

    def kinetic(self, nb, app):
        out = []
        for k, c in enumerate(self.blocks(nb, app)):
            kg = (self.G + self.kc[k][:, None, None, None]).reshape(3, -1)[:, self.idx(k)]
            out.append(0.5 * (kg * kg).sum(0) * c)
        return out

    def hartree(self, nb, app):
        x2 = (self.G ** 2).sum(0)
        n = self.fwd(self.rho)
        if self.s.method == "HF":
            v = torch.where(x2 < 1e-8, torch.zeros_like(x2), FOURPI / x2.clamp_min(1e-300))
            return self.local(nb, app, self.bwd(2.0 * v * n) / self.NkV)
        g = [0.0, 0.0, 0.0]
        for q in range(self.s.nk):
            fc = self.f[q][:, None, None, None] * self.chi[q].conj()
            for d in range(3):
                g[d] = g[d] + (fc * self.real(q, self.c_phi[q], d)).sum(0)
        v, vec = 0.0, [0.0, 0.0, 0.0]
        for sp in range(2):
            u = self.u(x2, sp)
            v = v + self.tc2body(x2, sp) * n
            for d in range(3):
                v = v + u * self.G[d] * self.fwd(g[d]) / 2.0
                vec[d] = vec[d] + u * self.G[d] * n
        return self.local(nb, app, self.bwd(v) / self.NkV, [self.bwd(x) / self.NkV for x in vec])

    def three_local(self, nb, app):
        dnu = self.dnu()
        x2 = (self.G ** 2).sum(0)
        us = self.u(x2, 0) + self.u(x2, 1)
        a1 = 0.5 / self.NkV ** 2 * sum(x * x for x in dnu)
        b1 = self.bwd(us * sum(self.G[d] * self.fwd(self.rho * dnu[d]) for d in range(3)))
        return self.local(nb, app, a1 - b1 / self.NkV ** 2)


def _flat(blocks):
    return torch.cat([b.reshape(-1) for b in blocks]).cpu().numpy()


def _dot(nb, a, fill, b):
    """(1/Nk) sum over bands of f <a|b>, per-band blocks."""
    return sum(complex((f[:, None] * x.conj() * y).sum()) for f, x, y in zip(fill, a, b)) / len(a)


def exact(case, seed):
    op = case["op"]
    if op == "davidson":  # what an iteration leaves depends on its algorithm, not on the operator alone
        return None
    rate = 1e10 if torch.cuda.is_available() else 2e8  # grid points transformed a second
    points = work(case)["flops"] / (5.0 * math.log2(case["n"] ** 2 * case["n3"]))
    if points / rate > 15.0 or op == "grad_tc2":  # grad_tc2: H^dagger and dE/dA as well, beyond a plain restatement
        return None
    sysm, nb, app = _make(case, seed)
    R = _Ref(case, sysm)
    if op == "apply_all":
        h1, h2 = R.kinetic(nb, app), R.hartree(nb, app)
        if case["method"] == "HF":
            return [_flat(h1), _flat(h2) + _flat(R.hf2x(nb, app))]
        h3 = _flat(R.three_local(nb, app)) + _flat(R.tc3a2a4b2b5(nb, app)) + _flat(R.tc3a3b3b4b6(nb, app))
        return [_flat(h1), _flat(h2) + _flat(R.tc2x(nb, app)), h3]
    if op == "grad_exchange":
        h = R.hf2x(sysm.nocc, sysm.phi_occ)
        grad = [f[:, None] * x / sysm.nk for f, x in zip(R.f, h)]
        e = 0.5 * _dot(sysm.nocc, R.c_phi, R.f, h)
        return [e.real, None, _flat(grad)]
    return _flat(getattr(R, op)(nb, app))
