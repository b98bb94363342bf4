"""tc2x in its two-channel form (bases that do not alias) and its four-channel form against the oracle.

Every compiled grid size, TC and BITC, both precisions, ragged bands with an empty k; then bases
around the limit of the form: a span of s Miller indices in a direction of n points takes two
channels when 2 s < n, and the four-channel form otherwise, so the cut-off radius is scaled across
that line.  FP64 within 1e-10 relative; FP32-split within the 3e-5 per-band bound of its
pipelines.
"""
import numpy as np
import pytest

from oracle import oracle as O
from tc_amd import system as S
from tc_amd import tcx
from test_gpu_hf2x import per_band_rel

pytestmark = pytest.mark.gpu


def check(engine, sys_, nb, seed):
    engine.load_system(sys_)
    _, phi = S.applied_bands(sys_, nb=nb, seed=seed)
    ref = O.Oracle(sys_).tc2x(nb, phi)
    for prec, tol in ((tcx.PREC_FP64, 1e-10), (tcx.PREC_FP32, 3e-5)):
        got = engine.tc2x(nb, phi, precision=prec)
        rel = per_band_rel(sys_, nb, got, ref).max()
        print(sys_.name, "precision", prec, f"per-band rel max {rel:.3e}", flush=True)
        assert rel <= tol


@pytest.mark.parametrize("grid", [6, 8, 10, 12, 16, 18, 20, 24, 30, 32, 36, 40, 48])
@pytest.mark.parametrize("method", ["TC", "BITC"])
def test_grid_sizes(engine, grid, method):
    sys_ = S.build_system(S.fcc_lattice(10.26 if grid > 20 else 6.0), (grid,) * 3, (2, 1, 1), nbands=3, nocc=2,
                          seed_stream=600 + grid, method=method, A=np.full((2, 2), 0.5), name=f"{method} {grid}^3")
    check(engine, sys_, np.array([3, 0] if grid % 4 else [1, 3], np.int32), 601)


@pytest.mark.parametrize("n", [(12, 12, 18), (20, 20, 12)])
@pytest.mark.parametrize("scale", [0.8, 1.0, 1.15, 1.4, 1.9])
def test_limit_of_the_form(engine, n, scale):
    lat = S.fcc_lattice(6.0)
    sys_ = S.build_system(lat, n, (4, 1, 2), nbands=2, nocc=2, seed_stream=640, method="BITC",
                          A=np.full((2, 2), 0.5), gw=scale * S.gw_rule(lat, n), name=f"BITC {n} x{scale}")
    check(engine, sys_, np.full(sys_.nk, 1, np.int32), 641)
