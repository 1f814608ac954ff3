"""The slice order of the degridder against the oracle: keys that are the bins
themselves, keys with lower bits sorted within a bin, and more keys than both
levels hold; batches at the edges of a workgroup's records, all records of one
slice, and records that are not degridded at both ends of the batch.

Bar: degridded values are FP64 sums rounded to FP32, 1e-6; a record that is
lost or taken twice is off by its whole value.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("one_slice", [False, True])
@pytest.mark.parametrize("ncube,nc,oversampling,n", [
    (2, 1, 4, 1),            # 162 slices: one bin each
    (2, 1, 4, 2047),
    (2, 1, 4, 2049),
    (30, 3, 8, 4097),        # 8670 slices x 3 cubes: bins of 32 keys
    (60, 70, 20, 6000),      # 100860 slices x 70 cubes: bins of 8192 keys
    (60, 3000, 20, 3000),    # 3e8 keys: their lowest bits left out
])
def test_order_vs_oracle(hpg, oracle_mod, monkeypatch, ncube, nc, oversampling, n, one_slice):
    from hpg_amd import workloads
    monkeypatch.setenv("HPGX_GRIDDER", "2")
    print(f"ncube {ncube} nc {nc} os {oversampling} n {n} one {one_slice}", flush=True)
    gsz, M = (24, 22, 1, nc), [[0, 1]]
    cf = workloads.random_cf(oversampling, [1], nmueller=2, ncube=ncube, seed=5)
    rec = workloads.random_visibilities(n, 2, gsz, (0.9, 1.1), cf, seed=6, phase=True, margin=-2)
    if one_slice:
        for name in ("uvw", "cf_index", "grid_cube"):
            rec[name] = rec[name][n // 2]
    if n > 1:
        rec["uvw"][0, 0] = rec["uvw"][-1, 0] = 1e4  # outside the grid
    gs = hpg.GridderState.create(hpg.Device.Hip, 0, n, cf, gsz, (0.9, 1.1), M, M)
    gs.set_convolution_function(hpg.Device.Serial, cf)
    o = oracle_mod.Oracle(gsz, (0.9, 1.1), M, M)
    o.set_cf(cf.oversampling(),
             [(cf.extents(g), cf.values(g)) for g in range(cf.num_groups())])
    rng = np.random.default_rng(7)
    model = rng.standard_normal(gsz[::-1]) + 1j * rng.standard_normal(gsz[::-1])
    gs.set_model(hpg.Device.Serial, model)
    o.set_model(model)
    exp = o.grid_visibilities(np.ascontiguousarray(rec).view(oracle_mod.visdata_dtype(2)), False,
                              do_degrid=True, do_grid=False)["vis"]
    for _ in range(2):  # the second call on the first one's counts and places
        pred = gs.degrid_get_predicted_visibilities(hpg.Device.Serial, rec)["visibilities"]
        np.testing.assert_allclose(pred, exp, rtol=1e-6, atol=1e-6 * max(np.abs(exp).max(), 1e-30))
