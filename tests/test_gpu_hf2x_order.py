"""The two pass orders of the FP32-split exchange pipeline against the oracle and each other.

Plane-first (xy planes, z pencils, xy planes; the automatic order) keeps only the (kx, ky) columns of
the pair records inside the pair density's G-space support; z-first (tcx_set_pipeline_order) keeps
them all.  Both are checked at every compiled grid size, and on mixed grids whose planes leave a
remainder in pass A's workgroups, against the FP64 oracle (per band, the rounding bound of the path)
and against each other (per band <= 1e-6: the same FP32 transforms in another order, FP64 sums), with
ragged band counts and several launch shapes; the plane-first records must hold fewer columns than the
grid.
"""
import numpy as np
import pytest

from oracle import oracle as O
from tc_amd import system as S
from tc_amd import tcx
from test_gpu_hf2x import fp32_rounding, per_band_rel

pytestmark = pytest.mark.gpu


def cell(grid, seed, nz=None):
    n = (grid, grid, nz or grid)
    if grid >= 32:  # the benchmark's fcc cell, reduced k-mesh and bands
        return S.build_system(S.fcc_lattice(10.26), n, (2, 1, 1), nbands=3, nocc=2, seed_stream=seed,
                              name=f"HF fcc a10.26 2x1x1k {n}")
    return S.tiny_system(method="HF", n=n, kmesh=(2, 2, 1), nbands=3, nocc=2, seed_stream=seed)


@pytest.mark.parametrize("grid,nz", [(n, n) for n in (6, 8, 10, 12, 16, 18, 20, 24, 30, 32, 36, 40, 48)]
                         + [(10, 8), (12, 8), (18, 20), (20, 10), (36, 40)])
def test_plane_first_and_z_first_vs_oracle(engine, grid, nz):
    sys_ = cell(grid, 500 + grid, nz)
    engine.load_system(sys_)
    nb = np.array([(i % 3) for i in range(sys_.nk)], np.int32)  # ragged, with an empty k
    _, phi = S.applied_bands(sys_, nb=nb, seed=501)
    ref = O.Oracle(sys_).hf2x(nb, phi)
    out = {}
    for order in (-1, 1, 0):
        engine.set_pipeline_order("hf2x", order)
        out[order] = engine.hf2x(nb, phi, precision=tcx.PREC_FP32)
        cols = engine.record_columns("hf2x")
        rel = per_band_rel(sys_, nb, out[order], ref)
        print(f"{sys_.n} order {order}: per-band rel max {rel.max():.3e}, record columns {cols:.1f} of {grid * grid}",
              flush=True)
        assert rel.max() <= fp32_rounding(sys_.n)
        if order == 0:
            assert cols == grid * grid
        else:
            assert cols < grid * grid
    engine.set_pipeline_order("hf2x", -1)
    assert np.array_equal(out[-1], out[1])  # automatic is plane-first
    rel = per_band_rel(sys_, nb, out[1], out[0])
    print(f"{sys_.n} plane-first vs z-first per-band rel max {rel.max():.3e}", flush=True)
    assert rel.max() <= 1e-6


@pytest.mark.parametrize("shape", [(1, 1), (3, 2), (7, 5), (0, 0)])
def test_plane_first_launch_shapes(engine, shape):
    """Results do not depend on how pairs are grouped into launches (FP64 sums in another
    order: 1e-12)."""
    sys_ = cell(16, 520)
    engine.load_system(sys_)
    nb = np.array([2, 0, 1, 2], np.int32)
    _, phi = S.applied_bands(sys_, nb=nb, seed=521)
    engine.set_pipeline_order("hf2x", 1)
    engine.set_launch_shape("hf2x", 0, 0)
    base = engine.hf2x(nb, phi, precision=tcx.PREC_FP32)
    engine.set_launch_shape("hf2x", *shape)
    got = engine.hf2x(nb, phi, precision=tcx.PREC_FP32)
    engine.set_launch_shape("hf2x", 0, 0)
    engine.set_pipeline_order("hf2x", -1)
    err = np.abs(got - base).max() / np.abs(base).max()
    print("shape", shape, err, flush=True)
    assert err <= 1e-12


def test_pipeline_order_errors(engine):
    for term, order in ((1, 0), (0, 2), (0, -2)):
        with pytest.raises(tcx.TcxError) as e:
            engine.set_pipeline_order(term, order)
        assert e.value.code == tcx.TCX_ERR_ARG


@pytest.mark.parametrize("gw,mesh", [(1.0, (4, 1, 1)), (1.35, (4, 3, 1)), (2.2, (2, 2, 1))])
def test_plane_first_wrapping_columns(engine, gw, mesh):
    """Bases whose differences reach past the grid (gw: multiple of the alias-free radius): the
    runs of the column set that wrap take every ky, and the two orders stay equal to FP32
    rounding and the oracle within the rounding bound."""
    lat = S.fcc_lattice(6.0)
    sys_ = S.build_system(lat, (18, 18, 12), mesh, nbands=3, nocc=2, seed_stream=530,
                          gw=gw * S.gw_rule(lat, (18, 18, 12)))
    engine.load_system(sys_)
    nb = np.full(sys_.nk, 2, np.int32)
    _, phi = S.applied_bands(sys_, nb=nb, seed=531)
    ref = O.Oracle(sys_).hf2x(nb, phi)
    out = {}
    for order in (1, 0):
        engine.set_pipeline_order("hf2x", order)
        out[order] = engine.hf2x(nb, phi, precision=tcx.PREC_FP32)
        assert per_band_rel(sys_, nb, out[order], ref).max() <= fp32_rounding(sys_.n)
    engine.set_pipeline_order("hf2x", -1)
    assert per_band_rel(sys_, nb, out[1], out[0]).max() <= 1e-6


def test_calls_that_return_rounding_keep_z_first(engine):
    """Phases of Davidson's eigenvectors and Im E_x are set by rounding, so with the automatic order
    they come from the z-first sums, bit for bit; an order that was asked for is taken."""
    sys_ = S.tiny_system(method="HF", n=(16, 16, 16), kmesh=(2, 2, 1), nbands=3, nocc=3, seed_stream=540)
    engine.load_system(sys_)
    nb, phi = S.applied_bands(sys_, nb=np.array([3, 3, 2, 3], np.int32), seed=541)
    eig = np.zeros(int(nb.sum()), complex)
    out = {}
    for order in (-1, 0, 1):
        engine.set_pipeline_order("hf2x", order)
        e, g = engine.grad_exchange(precision=tcx.PREC_FP32)
        out[order] = [np.array([e]), g, engine.davidson(nb, phi, eig, precision=tcx.PREC_FP32)[0]]
    engine.set_pipeline_order("hf2x", -1)
    for a, b, c in zip(out[-1], out[0], out[1]):
        assert np.array_equal(a, b)
        assert not np.array_equal(a, c)
    assert abs(out[1][0][0].real - out[0][0][0].real) <= 1e-6 * abs(out[0][0][0].real)
