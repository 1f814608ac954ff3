"""Register patches at the batch sizes where one workgroup, workgroups of 1024
records and of more prepare them, and at the most tiles that one workgroup counts,
against the oracle.

Bars: FP64 grids 1e-12 of max|grid| (the oracle's FP32 products in another order
of FP64 sums), weights (FP64 sums) 1e-12.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DIAG = [[0, -1, -1, -1], [-1, 1, -1, -1], [-1, -1, 2, -1], [-1, -1, -1, 3]]


@pytest.mark.parametrize("npol,gsz,M,n", [
    (2, (150, 170, 1, 2), [[0, 1]], 1),
    (2, (150, 170, 1, 2), [[0, 1]], 2048),
    (2, (150, 170, 1, 2), [[0, 1]], 2049),
    (2, (150, 170, 1, 2), [[0, 1]], 16_384),
    (2, (150, 170, 1, 2), [[0, 1]], 16_385),
    (4, (2048, 2048, 4, 1), DIAG, 2048),  # 16384 tiles of 16 x 16
    (4, (2048, 2048, 4, 1), DIAG, 2049),
    (4, (2049, 2048, 4, 1), DIAG, 2048),  # and more
])
def test_batches_vs_oracle(hpg, oracle_mod, npol, gsz, M, n):
    from hpg_amd import workloads
    print(f"grid {gsz} npol {npol} n {n}", flush=True)
    cf = workloads.random_cf(4, [2, 5], nmueller=4, ncube=2, seed=1)
    rec = workloads.random_visibilities(n, npol, gsz, (1.0, 1.0), cf, seed=2, phase=True, margin=-3)
    rec["uvw"][0] = 0.0
    if n > 2:
        rec["uvw"][-1, 0] = 1e4  # outside the grid
    gs = hpg.GridderState.create(hpg.Device.Hip, 0, n, cf, gsz, (1.0, 1.0), M, M)
    gs.set_convolution_function(hpg.Device.Serial, cf)
    o = oracle_mod.Oracle(gsz, (1.0, 1.0), M, M)
    o.set_cf(cf.oversampling(),
             [(cf.extents(g), cf.values(g)) for g in range(cf.num_groups())])
    view = np.ascontiguousarray(rec).view(oracle_mod.visdata_dtype(npol))
    for part in (slice(None), slice(n // 2 + 1)):  # the second call on the first's counts
        gs.grid_visibilities(hpg.Device.Serial, rec[part], True)
        o.grid_visibilities(view[part], True)
    exp = o.grid_values()
    assert np.abs(exp).max() > 0
    assert np.abs(gs.grid_values() - exp).max() <= 1e-12 * np.abs(exp).max()
    np.testing.assert_allclose(gs.grid_weights(), o.grid_weights(), rtol=1e-12)
