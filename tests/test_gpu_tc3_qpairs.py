"""tc3a2a4b2b5's occupied-set pairs: half of them (bases that do not alias) or all, in blocks.

The record of an orbital pair serves both orders, in launches of one block of orbitals against
another; block sizes 1, 2, 3 and larger than the set put diagonal and off-diagonal blocks and their
remainders next to each other.  A basis with 2 (span of its Miller indices) >= n in some direction
aliases and forms every pair; the number of pairs that the passes count says which happened, on both
sides of that line (12x12x12 x1.0 has spans 5, 5, 4, x1.1 has 5, 5, 6).  Against the oracle: FP64 within
1e-10 relative, FP32-split within the rounding bound of its path (fp32_rounding).  Block sizes only change the
order of FP64 sums of the same products, except that a pair of a block with itself and of two
blocks swaps which of its two orders is transformed: 1e-12 in FP64.
"""
import numpy as np
import pytest

from oracle import oracle as O
from tc_amd import system as S
from tc_amd import tcx
from test_gpu_hf2x import fp32_rounding, per_band_rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("div", [True, False])  # the G = 0 terms are FP64 and outweigh the pairs
@pytest.mark.parametrize("method", ["TC", "BITC"])
@pytest.mark.parametrize("scale,n", [(1.0, (12, 12, 8)), (1.0, (8, 8, 30)), (1.0, (12, 12, 12)), (1.1, (12, 12, 12)),
                                     (1.9, (12, 12, 8))])
def test_blocks_against_oracle(engine, method, scale, n, div):
    lat = S.fcc_lattice(6.0)
    base = S.build_system(lat, n, (2, 2, 1), nbands=3, nocc=3, seed_stream=660, method=method,
                          A=np.array([[0.5, 0.4], [0.4, 0.5]]), gw=scale * S.gw_rule(lat, n), div_corr=div)
    sys_ = S.uneven_bands(base, [3, 1, 0, 2])
    engine.load_system(sys_)
    nb = np.array([1, 0, 2, 1], np.int32)
    _, phi = S.applied_bands(sys_, nb=nb, seed=661)
    ref = O.Oracle(sys_).tc3a2a4b2b5(nb, phi)
    mill = S.miller_of_index(n)[sys_.gindex]
    aliases = bool(np.any(2 * (mill.max(0) - mill.min(0)) >= np.array(n)))
    assert aliases == (scale > 1.0)
    n_occ = int(sys_.nocc.sum())
    pairs = (n_occ * n_occ if aliases else n_occ * (n_occ + 1) // 2) + int(nb.sum()) * n_occ  # q1-q2 + apply phase
    first = None
    for shape in ((0, 0), (1, 1), (2, 2), (3, 3), (5, 2), (64, 64)):
        engine.set_launch_shape("tc3", *shape)
        engine.set_states(sys_.nocc, sys_.filling, sys_.phi_occ, sys_.chi_occ)  # the sums are kept otherwise
        for prec, tol in ((tcx.PREC_FP64, 1e-10), (tcx.PREC_FP32, fp32_rounding(n, 4))):
            engine.enable_timing(True)
            got = engine.tc3a2a4b2b5(nb, phi, precision=prec)
            formed = engine.get_timing()[2]
            engine.enable_timing(False)
            assert list(formed[:3]) == [pairs] * 3
            rel = per_band_rel(sys_, nb, got, ref).max()
            print(method, n, scale, shape, "precision", prec, f"{rel:.3e}", flush=True)
            assert rel <= tol
            if prec == tcx.PREC_FP64:
                first = got if first is None else first
                assert np.abs(got - first).max() <= 1e-12 * np.abs(first).max()
    engine.set_launch_shape("tc3", 0, 0)
