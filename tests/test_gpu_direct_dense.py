"""The one-launch gridder of few records (k_direct, FP64 grids of one polarization)
at three and four grid rows, at its widest supports (27 x 27, 31 x 23: a tile and
its halo within 64 KB), and dense on few tiles, where its lanes take a record each.

Bars: 1e-12 of max|grid| (the oracle's FP32 products in another order of FP64
sums), with gradients 1e-6 (their FP32 screens may round differently); weights
(FP64 sums) 1e-12.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(hpg, oracle_mod, gsz, M, Mc, cf, rec, bar):
    n = len(rec)
    gs = hpg.GridderState.create(hpg.Device.Hip, 0, n, cf, gsz, (0.9, 1.1), M, Mc)
    gs.set_convolution_function(hpg.Device.Serial, cf)
    o = oracle_mod.Oracle(gsz, (0.9, 1.1), M, Mc)
    o.set_cf(cf.oversampling(),
             [(cf.extents(g), cf.values(g)) for g in range(cf.num_groups())])
    view = np.ascontiguousarray(rec).view(oracle_mod.visdata_dtype(1))
    for _ in range(2):  # a second call adds to the grid
        gs.grid_visibilities(hpg.Device.Serial, rec, True)
        o.grid_visibilities(view, True)
    exp = o.grid_values()
    assert np.abs(gs.grid_values() - exp).max() <= bar * np.abs(exp).max()
    np.testing.assert_allclose(gs.grid_weights(), o.grid_weights(), rtol=1e-12)


@pytest.mark.parametrize("gradient", [False, True])
@pytest.mark.parametrize("nr", [3, 4])
@pytest.mark.parametrize("radii", [[3], [13], [(15, 11), 2], [1, 4, (2, 12)]])
@pytest.mark.parametrize("n", [40, 900])
def test_rows_and_widest_supports(hpg, oracle_mod, n, radii, nr, gradient):
    from hpg_amd import workloads
    print(f"n {n} radii {radii} rows {nr} gradient {gradient}", flush=True)
    M, Mc = [[0], [-1], [2], [1]][:nr], [[1], [0], [-1], [2]][:nr]
    gsz = (97, 66, nr, 2)
    cf = workloads.random_cf(6, radii, nmueller=3, ncube=2, seed=25)
    rec = workloads.random_visibilities(n, 1, gsz, (0.9, 1.1), cf, seed=26, phase=True, margin=-3,
                                        gradient=gradient)
    if gradient:
        rec["cf_phase_gradient"][1::3] = 0.0
    _check(hpg, oracle_mod, gsz, M, Mc, cf, rec, 1e-6 if gradient else 1e-12)


@pytest.mark.parametrize("gradient", [False, True])
@pytest.mark.parametrize("sigma", [0.0, 1.5, 12.0])
@pytest.mark.parametrize("radii", [[0], [1], [3], [4], [7, 1], [12]])
@pytest.mark.parametrize("n", [33, 300, 2048])
def test_dense(hpg, oracle_mod, n, radii, sigma, gradient):
    """All records about one point at the corner of four tiles."""
    from hpg_amd import workloads
    print(f"n {n} radii {radii} sigma {sigma} gradient {gradient}", flush=True)
    gsz = (128, 128, 1, 1)
    cf = workloads.random_cf(6, radii, nmueller=2, ncube=2, seed=25)
    rec = workloads.random_visibilities(n, 1, gsz, (0.9, 1.1), cf, seed=26, phase=True,
                                        gradient=gradient)
    rec["uvw"][:, :2] = np.random.default_rng(4).normal(0, sigma, (n, 2)) + [0.3, 0.1]
    if gradient:
        rec["cf_phase_gradient"][1::3] = 0.0
    _check(hpg, oracle_mod, gsz, [[0]], [[1]], cf, rec, 1e-6 if gradient else 1e-12)
