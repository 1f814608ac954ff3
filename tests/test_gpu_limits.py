"""Calls at the ends of what the entry points accept, against the oracle.

Bars: FP64 grids without phase gradients 1e-12 of max|grid| (the oracle's FP32
products in another order of FP64 sums), with gradients 1e-6 (their FP32 screens
may round differently); degridded values (FP64 sums rounded to FP32) 1e-6;
weights (FP64 sums) 1e-12.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FULL = [[0, 1, 2, 3], [4, 5, 6, 7], [8, 9, 10, 11], [12, 13, 14, 15]]
DIAG = [[0, -1, -1, -1], [-1, 1, -1, -1], [-1, -1, 2, -1], [-1, -1, -1, 3]]


def _pair(hpg, oracle_mod, gsz, M, Mc, cf, mode, n):
    gs = hpg.GridderState.create(hpg.Device.Hip, 0, n, cf, gsz, (0.9, 1.1), M, Mc,
                                 grid_mode=mode)
    gs.set_convolution_function(hpg.Device.Serial, cf)
    o = oracle_mod.Oracle(gsz, (0.9, 1.1), M, Mc)
    o.set_cf(cf.oversampling(),
             [(cf.extents(g), cf.values(g)) for g in range(cf.num_groups())])
    return gs, o


def _view(rec, oracle_mod):
    npol = rec.dtype["visibilities"].shape[0]
    return np.ascontiguousarray(rec).view(oracle_mod.visdata_dtype(npol))


def _set_model(hpg, gs, o, gsz):
    rng = np.random.default_rng(7)
    model = rng.standard_normal(gsz[::-1]) + 1j * rng.standard_normal(gsz[::-1])
    gs.set_model(hpg.Device.Serial, model)
    o.set_model(model)


def _check_grid(hpg, oracle_mod, gs, o, rec, bar):
    gs.grid_visibilities(hpg.Device.Serial, rec, True)
    o.grid_visibilities(_view(rec, oracle_mod), True)
    exp = o.grid_values()
    assert np.abs(exp).max() > 0
    assert np.abs(gs.grid_values() - exp).max() <= bar * np.abs(exp).max()
    np.testing.assert_allclose(gs.grid_weights(), o.grid_weights(), rtol=1e-12)


def _check_predictions(hpg, oracle_mod, gs, o, rec):
    pred = gs.degrid_get_predicted_visibilities(hpg.Device.Serial, rec)["visibilities"]
    exp = o.grid_visibilities(_view(rec, oracle_mod), False, do_degrid=True, do_grid=False)["vis"]
    assert np.abs(exp).max() > 0
    assert np.abs(pred - exp).max() <= 1e-6 * np.abs(exp).max()


@pytest.mark.parametrize("lo,hi", [(10, 14), (14, 18), (18, 25), (25, 300)])
@pytest.mark.parametrize("npol,M,nm", [(4, FULL, 16), (4, DIAG, 4), (2, [[0, 1], [1, 2]], 3)])
def test_large_phase_gradients(hpg, oracle_mod, npol, M, nm, lo, hi):
    """Phases on both sides of the change of their reduction (2^40) and far
    beyond what their rounding leaves of a turn: the same FP64 phases as the
    oracle's, so the same screens."""
    print(f"npol {npol} nm {nm} gradients 1e{lo} to 1e{hi}", flush=True)
    gsz, n = (60, 50, len(M), 1), 300
    from hpg_amd import workloads
    cf = workloads.random_cf(6, [3, (2, 9)], nmueller=nm, seed=1)
    rec = workloads.random_visibilities(n, npol, gsz, (0.9, 1.1), cf, seed=2, phase=True)
    rng = np.random.default_rng(3)
    rec["cf_phase_gradient"] = 10.0 ** rng.uniform(lo, hi, (n, 2)) * rng.choice([-1, 1], (n, 2))
    gs, o = _pair(hpg, oracle_mod, gsz, M, M, cf, 0, n)
    _set_model(hpg, gs, o, gsz)
    _check_predictions(hpg, oracle_mod, gs, o, rec)
    _check_grid(hpg, oracle_mod, gs, o, rec, 1e-6)
