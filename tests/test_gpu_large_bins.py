"""Quadrant bins of large grids against the oracle, at the edges of a workgroup's
records and with all records in one bin."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gsz,n,one_tile", [
    ((2905, 2890, 1, 1), 1, False),      # 33,124 quadrants
    ((2905, 2890, 1, 1), 2049, False),
    ((2905, 2890, 1, 1), 5000, True),    # of one bin
    ((1500, 1490, 2, 2), 4100, False),   # two entries a record
    ((1500, 1490, 2, 2), 2048, True),
])
def test_large_grid_bins_vs_oracle(hpg, oracle_mod, gsz, n, one_tile):
    """Entries by quadrant on grids of more keys than the block-local bins take;
    FP32-compensated sums, 1e-6 of the largest value; weights (FP64) 1e-12."""
    from hpg_amd import workloads
    print(f"grid {gsz} n {n} one {one_tile}", flush=True)
    M = [[0]] if gsz[2] == 1 else [[0], [1]]
    cf = workloads.random_cf(5, [2, 1], nmueller=2, ncube=2, seed=15)
    rec = workloads.random_visibilities(n, 1, gsz, (0.9, 1.1), cf, seed=16, phase=True, margin=-2,
                                        gradient=True)
    rec["cf_phase_gradient"][1::3] = 0.0
    if one_tile:
        rec["uvw"][:, :2] = rec["uvw"][0, :2] + np.random.default_rng(3).uniform(0, 8, (n, 2))
    gs = hpg.GridderState.create(hpg.Device.Hip, 0, n, cf, gsz, (0.9, 1.1), M, M, grid_mode=1)
    gs.set_convolution_function(hpg.Device.Serial, cf)
    o = oracle_mod.Oracle(gsz, (0.9, 1.1), M, M)
    o.set_cf(cf.oversampling(),
             [(cf.extents(g), cf.values(g)) for g in range(cf.num_groups())])
    view = np.ascontiguousarray(rec).view(oracle_mod.visdata_dtype(1))
    for _ in range(2):
        gs.grid_visibilities(hpg.Device.Serial, rec, True)
        o.grid_visibilities(view, True)
    exp = o.grid_values()
    assert np.abs(gs.grid_values() - exp).max() <= 1e-6 * max(np.abs(exp).max(), 1e-30)
    np.testing.assert_allclose(gs.grid_weights(), o.grid_weights(), rtol=1e-12)
