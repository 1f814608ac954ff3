"""The one-launch gridder of few records (k_direct) against the oracle: supports
at the edges of its 8 x 8 blocks and of a tile, grids at and past tile edges,
batches up to and past its largest, one and two grid rows.

Bars: FP64 grids without phase gradients 1e-12 of max|grid| (the oracle's FP32
products in another order of FP64 sums), with gradients 1e-6 (their FP32 screens
may round differently); FP32 grids 1e-6; weights (FP64 sums) 1e-12.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gradient", [False, True])
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("gsz,radii,n", [
    ((64, 64, 1, 1), [3], 1),
    ((65, 95, 1, 2), [3], 600),
    ((97, 64, 1, 1), [0, 4, (8, 3), (2, 12)], 700),  # supports 1, 9, 17 x 7, 5 x 25
    ((130, 97, 2, 1), [3, 15], 513),                 # supports 7 and 31
    ((160, 160, 2, 2), [(1, 3)], 2048),              # the largest batch
    ((160, 160, 1, 1), [3], 2049),                   # and one more
])
def test_direct_vs_oracle(hpg, oracle_mod, gsz, radii, n, mode, gradient):
    from hpg_amd import workloads
    print(f"grid {gsz} radii {radii} n {n} mode {mode} gradient {gradient}", flush=True)
    M, Mc = ([[0]], [[1]]) if gsz[2] == 1 else ([[0], [1]], [[1], [-1]])
    cf = workloads.random_cf(6, radii, nmueller=2, ncube=2, seed=25)
    rec = workloads.random_visibilities(n, 1, gsz, (0.9, 1.1), cf, seed=26, phase=True, margin=-3,
                                        gradient=gradient)
    if gradient:
        rec["cf_phase_gradient"][1::3] = 0.0
    gs = hpg.GridderState.create(hpg.Device.Hip, 0, n, cf, gsz, (0.9, 1.1), M, Mc, grid_mode=mode)
    gs.set_convolution_function(hpg.Device.Serial, cf)
    o = oracle_mod.Oracle(gsz, (0.9, 1.1), M, Mc)
    o.set_cf(cf.oversampling(),
             [(cf.extents(g), cf.values(g)) for g in range(cf.num_groups())])
    view = np.ascontiguousarray(rec).view(oracle_mod.visdata_dtype(1))
    for _ in range(2):  # a second call adds to the grid
        gs.grid_visibilities(hpg.Device.Serial, rec, True)
        o.grid_visibilities(view, True)
    exp = o.grid_values()
    bar = 1e-6 if mode or gradient else 1e-12
    assert np.abs(gs.grid_values() - exp).max() <= bar * np.abs(exp).max()
    np.testing.assert_allclose(gs.grid_weights(), o.grid_weights(), rtol=1e-12)
