"""Register patches whose tiles' lists are split over several workgroups, against
the oracle: batches dense on a few tiles, evenly and about one point, on grids of
few tiles and of more than one workgroup scans.

Bars: FP64 grids 1e-12 of max|grid| (the oracle's FP32 products in another order
of FP64 sums), FP32-compensated grids 1e-6, weights (FP64 sums) 1e-12.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FULL = [[0, 1, 2, 3], [4, 5, 6, 7], [8, 9, 10, 11], [12, 13, 14, 15]]


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("npol,M,nm", [
    (2, [[0, 1]], 2), (2, [[0, -1], [-1, 1]], 2), (4, FULL[:3], 16), (4, FULL, 16)])
@pytest.mark.parametrize("gsz,radius,n,sigma", [
    ((40, 37), 1, 127, None),          # lists of up to a chunk, and up to two
    ((40, 37), 2, 700, None),
    ((130, 70), 3, 20_000, None),      # of many chunks, all tiles
    ((300, 280), 2, 30_000, 2.0),      # one tile's and its neighbours'
    ((300, 280), 20, 2500, 3.0),       # supports of several tiles
    ((2100, 2090), 4, 6000, 4.0),      # more than 16384 tiles of 16 x 16
])
def test_split_lists_vs_oracle(hpg, oracle_mod, gsz, radius, n, sigma, npol, M, nm, mode):
    from hpg_amd import workloads
    print(f"grid {gsz} radius {radius} n {n} sigma {sigma} npol {npol} mode {mode}", flush=True)
    gsz = gsz + (len(M), 1)
    cf = workloads.random_cf(4, [radius], nmueller=nm, seed=1)
    rec = workloads.random_visibilities(n, npol, gsz, (1.0, 1.0), cf, seed=2, phase=True)
    if sigma:
        rec["uvw"][:, :2] = np.random.default_rng(3).normal(0, sigma, (n, 2))
    gs = hpg.GridderState.create(hpg.Device.Hip, 0, n, cf, gsz, (1.0, 1.0), M, M, grid_mode=mode)
    gs.set_convolution_function(hpg.Device.Serial, cf)
    o = oracle_mod.Oracle(gsz, (1.0, 1.0), M, M)
    o.set_cf(cf.oversampling(), [(cf.extents(0), cf.values(0))])
    view = np.ascontiguousarray(rec).view(oracle_mod.visdata_dtype(npol))
    for part in (slice(None), slice(n // 3)):  # the second call on the first's counters
        gs.grid_visibilities(hpg.Device.Serial, rec[part], True)
        o.grid_visibilities(view[part], True)
    exp = o.grid_values()
    bar = 1e-6 if mode else 1e-12
    assert np.abs(gs.grid_values() - exp).max() <= bar * np.abs(exp).max()
    np.testing.assert_allclose(gs.grid_weights(), o.grid_weights(), rtol=1e-12)


@pytest.mark.parametrize("npol,M,nm,gsz", [
    (2, [[0, -1], [-1, 1]], 2, (512, 512)),  # 512 tiles of 32 x 16
    (2, [[0, -1], [-1, 1]], 2, (512, 496)),  # one row of tiles fewer
    (4, FULL, 16, (384, 370)),               # 576 of 16 x 16
])
@pytest.mark.parametrize("sigma", [None, 30.0])
def test_many_tiles_vs_oracle(hpg, oracle_mod, npol, M, nm, gsz, sigma):
    """Even lists, which stay whole where the tiles fill the chip, and a core's."""
    test_split_lists_vs_oracle(hpg, oracle_mod, gsz, 3, 50_000, sigma, npol, M, nm, 0)
