"""The register-patch gridder (k_patch) and the slice-ordered degridder
(k_degrid) against the oracle at the edges of their tiles, patches and runs.

Bars: grids of FP64 mode without phase gradients hold the oracle's FP32
products summed in FP64 in another order, 1e-12 of max|grid| (with gradients
1e-6, whose FP32 screens may round differently); FP32-compensated grids 1e-6;
degridded values (FP64 sums rounded to FP32) 1e-6, gridded residuals 1e-5;
weights (FP64 sums) 1e-12.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FULL = [[0, 1, 2, 3], [4, 5, 6, 7], [8, 9, 10, 11], [12, 13, 14, 15]]
DIAG = [[0, -1, -1, -1], [-1, 1, -1, -1], [-1, -1, 2, -1], [-1, -1, -1, 3]]

# npol, grid size (edges before, at and past tiles of 16 and 32 pixels), M, Mc,
# Mueller elements: rows of four neighbouring elements, of one element each
# (equal and different for the two signs of w; two rows of one polarization),
# of any, and of fewer elements than the rows ask for
KINDS = [
    (4, (80, 79, 4, 2), FULL, FULL, 16),
    (4, (65, 81, 4, 1), DIAG, DIAG, 4),
    (4, (64, 96, 4, 1), DIAG, DIAG[::-1], 4),
    (4, (81, 64, 3, 1), FULL[:3], [FULL[2], FULL[0], FULL[1]], 13),
    (2, (97, 66, 2, 2), [[0, 1], [2, 3]], [[2, 3], [0, 1]], 4),
    (2, (96, 64, 2, 1), [[0, -1], [1, -1]], [[0, -1], [1, -1]], 2),
    (2, (70, 70, 1, 1), [[1, 0]], [[0, 1]], 2),
    (3, (70, 66, 2, 1), [[0, -1, 1], [2, 0, -1]], [[1, -1, 0], [-1, 2, 0]], 3),
    (1, (97, 65, 1, 1), [[0]], [[0]], 1),
    (1, (64, 70, 2, 1), [[0], [1]], [[1], [0]], 3),
]
# radii of a patch, of whole patches, past a tile
RADII = [[0, 1], [(1, 3), 4], [8, (16, 7)], [(18, 17), 3]]


def _inputs(hpg, kind, radii, n, seed, gradient):
    from hpg_amd import workloads
    npol, gsz, M, Mc, nm = KINDS[kind]
    cf = workloads.random_cf(6, radii, nmueller=nm, ncube=2, seed=seed)
    rec = workloads.random_visibilities(n, npol, gsz, (0.9, 1.1), cf, seed=seed + 1,
                                        phase=True, margin=-3, gradient=gradient)
    if gradient:
        rec["cf_phase_gradient"][1::3] = 0.0
    # records in runs of one CF slice, of 1 to 12 records and both signs of w
    rng = np.random.default_rng(seed + 2)
    at = 0
    while at < n // 2:
        k = int(rng.integers(1, 13))
        rec["uvw"][at:at + k, :2] = rec["uvw"][at, :2]
        rec["cf_index"][at:at + k] = rec["cf_index"][at]
        at += k
    # whole-pixel moves keep the slice
    move = rng.integers(-6, 7, (n, 2)) * (n // 2 > np.arange(n))[:, None]
    rec["uvw"][:, :2] += move / np.array([0.9, 1.1])
    return npol, gsz, M, Mc, cf, rec


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


def _planes_close(got, exp, bar):
    for g, e in zip(got.reshape(-1, *got.shape[2:]), exp.reshape(-1, *exp.shape[2:])):
        scale = np.abs(e).max()
        if scale == 0:
            assert np.abs(g).max() == 0
            continue
        assert np.abs(g - e).max() <= bar * scale


@pytest.mark.parametrize("gradient", [False, True])
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("radii", range(len(RADII)))
@pytest.mark.parametrize("kind", range(len(KINDS)))
def test_patches_vs_oracle(hpg, oracle_mod, monkeypatch, kind, radii, mode, gradient):
    monkeypatch.setenv("HPGX_GRIDDER", "2")  # register patches for every call
    print(f"kind {kind} radii {radii} mode {mode} gradient {gradient}", flush=True)
    npol, gsz, M, Mc, cf, rec = _inputs(hpg, kind, RADII[radii], 1100, 300 + kind, gradient)
    gs, o = _pair(hpg, oracle_mod, gsz, M, Mc, cf, mode, len(rec))
    # a second call adds to the grid
    for part in (rec[:1000], rec[1000:]):
        gs.grid_visibilities(hpg.Device.Serial, part, True)
        o.grid_visibilities(_view(part, oracle_mod), True)
    exp = o.grid_values()
    assert np.abs(exp).max() > 0
    _planes_close(gs.grid_values(), exp, 1e-6 if mode or gradient else 1e-12)
    np.testing.assert_allclose(gs.grid_weights(), o.grid_weights(), rtol=1e-12)


@pytest.mark.parametrize("gradient", [False, True])
@pytest.mark.parametrize("device", [False, True])
@pytest.mark.parametrize("kind,radii", [(k, k % len(RADII)) for k in range(len(KINDS))]
                         + [(0, 3), (1, 3), (8, 3), (9, 0)])
def test_slice_runs_vs_oracle(hpg, oracle_mod, monkeypatch, kind, radii, device, gradient):
    """Predictions and residuals of host and device records (read in place, the
    caller's batch unchanged)."""
    import torch
    monkeypatch.setenv("HPGX_GRIDDER", "2")
    print(f"kind {kind} radii {radii} device {device} gradient {gradient}", flush=True)
    npol, gsz, M, Mc, cf, rec = _inputs(hpg, kind, RADII[radii], 1103, 400 + kind, gradient)
    gs, o = _pair(hpg, oracle_mod, gsz, M, Mc, cf, 0, len(rec))
    rng = np.random.default_rng(9)
    shape = gsz[::-1]
    model = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    gs.set_model(hpg.Device.Serial, model)
    o.set_model(model)

    def call(name):
        f = getattr(gs, name)
        if not device:
            return f(hpg.Device.Serial, rec)
        dev = torch.from_numpy(rec.view(np.uint8).copy()).cuda()
        out = f(hpg.Device.Serial, dev).cpu().numpy().view(rec.dtype)
        assert np.array_equal(dev.cpu().numpy(), rec.view(np.uint8))
        return out

    pred = call("degrid_get_predicted_visibilities")
    pexp = o.grid_visibilities(_view(rec, oracle_mod), False, do_degrid=True, do_grid=False)
    assert np.abs(pexp["vis"]).max() > 0
    bar = 1e-6 * np.abs(pexp["vis"]).max()
    np.testing.assert_allclose(pred["visibilities"], pexp["vis"], rtol=1e-6, atol=bar)
    res = call("degrid_grid_get_residual_visibilities")
    rexp = o.grid_visibilities(_view(rec, oracle_mod), True, do_degrid=True, do_grid=True)
    np.testing.assert_allclose(res["visibilities"], rexp["vis"], rtol=1e-6, atol=bar)
    for name in rec.dtype.names:
        if name != "visibilities":
            assert np.array_equal(pred[name], rec[name]) and np.array_equal(res[name], rec[name])
    _planes_close(gs.grid_values(), o.grid_values(), 1e-5)


@pytest.mark.parametrize("M,nm,radius", [(DIAG, 4, 4), (FULL, 16, 3), (DIAG, 4, 0)])
def test_degrid_regions_vs_oracle(hpg, oracle_mod, M, nm, radius):
    """A batch dense enough to be degridded region by region (2^k pixels
    squares, several on this grid, edges between and at its ends)."""
    from hpg_amd import workloads
    gsz = (520, 300, 4, 2)
    n = 30_011
    cf = workloads.random_cf(3, [radius], nmueller=nm, seed=21)
    rec = workloads.random_visibilities(n, 4, gsz, (0.9, 1.1), cf, seed=22, phase=True,
                                        margin=-3)
    gs, o = _pair(hpg, oracle_mod, gsz, M, M, cf, 0, n)
    rng = np.random.default_rng(9)
    model = rng.standard_normal(gsz[::-1]) + 1j * rng.standard_normal(gsz[::-1])
    gs.set_model(hpg.Device.Serial, model)
    o.set_model(model)
    pred = gs.degrid_get_predicted_visibilities(hpg.Device.Serial, rec)
    pexp = o.grid_visibilities(_view(rec, oracle_mod), False, do_degrid=True, do_grid=False)
    np.testing.assert_allclose(pred["visibilities"], pexp["vis"], rtol=1e-6,
                               atol=1e-6 * np.abs(pexp["vis"]).max())


def test_patches_in_passes(hpg, monkeypatch):
    """Batches whose lists exceed the entry budget take several passes."""
    from hpg_amd import workloads
    gsz = (256, 200, 4, 1)
    cf = workloads.random_cf(4, [20], nmueller=16, seed=5)
    rec = workloads.random_visibilities(40_000, 4, gsz, (1.0, 1.0), cf, seed=6, phase=True)
    grids = []
    for budget in ("1", "64"):
        monkeypatch.setenv("HPGX_ENTRY_BUDGET_MB", budget)
        gs = hpg.GridderState.create(hpg.Device.Hip, 0, len(rec), cf, gsz, (1.0, 1.0), FULL)
        gs.set_convolution_function(hpg.Device.Serial, cf)
        gs.grid_visibilities(hpg.Device.Serial, rec)
        grids.append(gs.grid_values())
    _planes_close(grids[0], grids[1], 1e-12)


@pytest.mark.parametrize("nm,os_,radius", [(1, 20, 3), (3, 5, 2), (16, 20, 12), (16, 253, 1),
                                           (6, 1, 70), (70, 8, 1)])
def test_cf_layout_weights(hpg, oracle_mod, nm, os_, radius):
    """The CF slices' sums (the weights) and taps for element counts, supports
    and oversamplings at which the layout kernels change form."""
    from hpg_amd import workloads
    n = 400
    gsz = (160, 150, 1, 1)
    cf = workloads.random_cf(os_, [radius], nmueller=nm, seed=7)
    M = [[nm - 1]]
    rec = workloads.random_visibilities(n, 1, gsz, (0.9, 1.1), cf, seed=8)
    gs, o = _pair(hpg, oracle_mod, gsz, M, M, cf, 0, n)
    gs.grid_visibilities(hpg.Device.Serial, rec, True)
    o.grid_visibilities(_view(rec, oracle_mod), True)
    _planes_close(gs.grid_values(), o.grid_values(), 1e-12)
    np.testing.assert_allclose(gs.grid_weights(), o.grid_weights(), rtol=1e-12)


@pytest.mark.parametrize("mode", [0, 1])
def test_values_on_device(hpg, mode):
    """The grid and the model read back into device tensors equal the host
    copies bit for bit; an unset model reads as zero."""
    import torch
    from hpg_amd import workloads
    gsz = (37, 21, 2, 3)
    cf = workloads.random_cf(4, [2], nmueller=2, seed=1)
    rec = workloads.random_visibilities(500, 2, gsz, (1.0, 1.0), cf, seed=2)
    gs = hpg.GridderState.create(hpg.Device.Hip, 0, 500, cf, gsz, (1.0, 1.0),
                                 [[0, -1], [-1, 1]], grid_mode=mode)
    gs.set_convolution_function(hpg.Device.Serial, cf)
    assert not gs.model_values_device().any()
    gs.grid_visibilities(hpg.Device.Serial, rec)
    gs.normalize_by_weights(2.0)
    gs.apply_grid_fft(1.0, hpg.FFTSign.POSITIVE, True)
    on_device = gs.grid_values_device()
    assert on_device.dtype == torch.complex128 and tuple(on_device.shape) == gs.grid_shape
    assert np.array_equal(on_device.cpu().numpy(), gs.grid_values())
    model = torch.randn(gs.grid_shape, dtype=torch.complex128, device="cuda")
    gs.set_model(hpg.Device.Serial, model)
    assert torch.equal(gs.model_values_device(), model)
