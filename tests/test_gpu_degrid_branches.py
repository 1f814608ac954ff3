"""The slice-ordered degridder where its sort leaves out low key bits, and region
by region with supports of one pixel, against the oracle; and the roundings of its
sums.

Bar: degridded values are FP64 sums rounded to FP32, 1e-6; that of the roundings
stands with them.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(hpg, oracle_mod, gsz, M, cf, rec, npol):
    gs = hpg.GridderState.create(hpg.Device.Hip, 0, len(rec), cf, gsz, (0.9, 1.1), M, M)
    gs.set_convolution_function(hpg.Device.Serial, cf)
    o = oracle_mod.Oracle(gsz, (0.9, 1.1), M, M)
    o.set_cf(cf.oversampling(),
             [(cf.extents(g), cf.values(g)) for g in range(cf.num_groups())])
    rng = np.random.default_rng(7)
    model = rng.standard_normal(gsz[::-1]) + 1j * rng.standard_normal(gsz[::-1])
    gs.set_model(hpg.Device.Serial, model)
    o.set_model(model)
    view = np.ascontiguousarray(rec).view(oracle_mod.visdata_dtype(npol))
    exp = o.grid_visibilities(view, False, do_degrid=True, do_grid=False)["vis"]
    assert np.abs(exp).max() > 0
    for _ in range(2):  # the second call on the first one's counts and places
        pred = gs.degrid_get_predicted_visibilities(hpg.Device.Serial, rec)["visibilities"]
        np.testing.assert_allclose(pred, exp, rtol=1e-6, atol=1e-6 * np.abs(exp).max())


@pytest.mark.parametrize("n", [3000, 20_001])
def test_order_without_low_bits(hpg, oracle_mod, monkeypatch, n):
    from hpg_amd import workloads
    monkeypatch.setenv("HPGX_GRIDDER", "2")
    ncube, nc, oversampling = 220, 3000, 20
    nf = 2 * ((oversampling + 1) // 2) + 1  # fine offsets of an axis
    # 16384 bins of 2^14 keys are all that both levels of the sort hold
    assert 2**28 < ncube * nf * nf * nc < 2**32 - 1
    gsz = (24, 22, 1, nc)
    cf = workloads.random_cf(oversampling, [1], nmueller=2, ncube=ncube, seed=5)
    rec = workloads.random_visibilities(n, 2, gsz, (0.9, 1.1), cf, seed=6, phase=True, margin=-2)
    rec["uvw"][0, 0] = rec["uvw"][-1, 0] = 1e4  # outside the grid
    # runs of one slice and of its neighbours
    rec[1:200] = rec[1]
    rec["uvw"][100:200, 1] += np.arange(100) / oversampling / 1.1
    _check(hpg, oracle_mod, gsz, [[0, 1]], cf, rec, 2)


def test_regions_of_one_pixel_supports(hpg, oracle_mod):
    from hpg_amd import workloads
    gsz, n = (150, 140, 4, 1), 90_011
    # regions of 128 x 128: the batch reads each of their pixels over four times
    assert n / (gsz[0] * gsz[1]) * 128 * 128 >= 4 * 129 * 129
    cf = workloads.random_cf(3, [0], nmueller=4, seed=21)
    rec = workloads.random_visibilities(n, 4, gsz, (0.9, 1.1), cf, seed=22, phase=True)
    M = [[0, -1, -1, -1], [-1, 1, -1, -1], [-1, -1, 2, -1], [-1, -1, -1, 3]]
    _check(hpg, oracle_mod, gsz, M, cf, rec, 4)


@pytest.mark.parametrize("nr,npol", [(4, 4), (2, 2), (1, 2)])
def test_roundings_of_wide_supports(hpg, nr, npol):
    """FP64 predictions of 65 x 65 taps, one element a row, against sums in
    extended precision.  A sum of n random terms, each added with a rounding of
    0.4 x 2^-53 rms, is off by sqrt(n / 2) of them: in 16 lanes with two roundings
    a tap 528 in a row, 7e-16; in parts of 8 and 17 of them about 2e-16, with
    the norm, the division and the phasor 3e-16."""
    radius, size, n = 32, 96, 400
    side = 2 * radius + 1
    rng = np.random.default_rng(11)
    shape = (1, npol, side + 4, side + 4)  # oversampling 1, padding 2
    cfv = (0.5 + rng.random(shape) + 0.2j * rng.standard_normal(shape)).astype(np.complex64)
    cf = hpg.CFArray(1, [cfv])
    gsz = (size, size, nr, 1)
    M = [[v if v == r else -1 for v in range(npol)] for r in range(nr)]
    gs = hpg.GridderState.create(hpg.Device.Hip, 0, n, cf, gsz, (1.0, 1.0), M, M)
    gs.set_convolution_function(hpg.Device.Serial, cf)
    model = rng.standard_normal(gsz[::-1]) + 1j * rng.standard_normal(gsz[::-1])
    gs.set_model(hpg.Device.Serial, model)
    rec = np.zeros(n, hpg.visdata_dtype(npol))
    corner = rng.integers(0, size - side + 1, (n, 2))
    rec["frequency"] = 299792458.0
    rec["uvw"][:, :2] = corner + radius - size // 2
    rec["uvw"][:, 2] = 1.0
    got = gs.degrid_forward(rec)
    exp = np.empty((n, nr), np.clongdouble)
    for r in range(nr):
        c = cfv[0, r, 2:-2, 2:-2].astype(np.clongdouble)
        for i, (x, y) in enumerate(corner):
            exp[i, r] = (c * model[0, r, y:y + side, x:x + side]).sum() / c.sum()
    err = np.linalg.norm(got[:, :nr] - exp) / np.linalg.norm(exp)
    print(f"rows {nr}: error {float(err):.2e}", flush=True)
    assert err <= 5e-16
