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


def test_many_cf_cubes(hpg, oracle_mod):
    """A CF laid out by 65536 x 87 x 3 workgroups of 256 threads: more threads
    than 2^32."""
    from hpg_amd import workloads
    rng = np.random.default_rng(1)
    plane = rng.standard_normal((91, 5)) + 1j * rng.standard_normal((91, 5))
    values = plane.astype(np.complex64) * np.linspace(
        1, 2, 65536, dtype=np.float32)[:, None, None, None]
    cf = hpg.CFArray(1, [values])
    gsz, n = (20, 130, 1, 1), 200
    rec = workloads.random_visibilities(n, 1, gsz, (0.9, 1.1), cf, seed=2)
    gs, o = _pair(hpg, oracle_mod, gsz, [[0]], [[0]], cf, 0, n)
    _check_grid(hpg, oracle_mod, gs, o, rec, 1e-12)


def test_many_patches(hpg, oracle_mod):
    """2^31 pixels a plane: patches of 16 x 16 pixels by 512 threads each, 2^32.
    Against the middle of the same u, v on a small grid."""
    from hpg_amd import workloads
    gsz, small, n = (65536, 32768, 3, 1), (64, 64, 3, 1), 200
    M = [[0, 1], [1, -1], [-1, 0]]
    cf = workloads.random_cf(4, [3], nmueller=2, seed=1)
    # whole supports inside the small grid too
    rec = workloads.random_visibilities(n, 2, small, (0.9, 1.1), cf, seed=2, margin=5)
    gs = hpg.GridderState.create(hpg.Device.Hip, 0, n, cf, gsz, (0.9, 1.1), M, M, grid_mode=1)
    gs.set_convolution_function(hpg.Device.Serial, cf)
    gs.grid_visibilities(hpg.Device.Serial, rec, True)
    o = oracle_mod.Oracle(small, (0.9, 1.1), M, M)
    o.set_cf(cf.oversampling(), [(cf.extents(0), cf.values(0))])
    o.grid_visibilities(_view(rec, oracle_mod), True)
    for row, exp in enumerate(o.grid_values()[0]):
        got = gs.grid_window(32768 - 32, 16384 - 32, 64, 64, row, 0)
        assert np.abs(got - exp).max() <= 1e-6 * np.abs(exp).max()  # FP32 grid


def test_many_records_degridded(hpg):
    """2^28 + 300000 records, 16 by a workgroup of 256 threads: more threads
    than 2^32.  The batch repeats a small one, whose predictions it repeats."""
    import torch
    from hpg_amd import workloads
    gsz, part = (200, 180, 2, 1), 300_000
    M = [[0, -1], [-1, 1]]
    repeats = (1 << 28) // part + 2
    n = part * repeats
    cf = workloads.random_cf(4, [1], nmueller=2, seed=1)
    rec = workloads.random_visibilities(part, 2, gsz, (1.0, 1.0), cf, seed=2)
    gs = hpg.GridderState.create(hpg.Device.Hip, 0, n, cf, gsz, (1.0, 1.0), M, M)
    gs.set_convolution_function(hpg.Device.Serial, cf)
    model = torch.randn(gs.grid_shape, dtype=torch.complex128, device="cuda")
    gs.set_model(hpg.Device.Serial, model)
    one = torch.from_numpy(rec.view(np.uint8).reshape(part, -1)).cuda()
    exp = gs.degrid_get_predicted_visibilities(hpg.Device.Serial, one)
    got = gs.degrid_get_predicted_visibilities(hpg.Device.Serial, one.repeat(repeats, 1))
    vis = exp[:, :16].contiguous().view(torch.float32)
    bar = 1e-6 * vis.abs().max()
    for k, chunk in enumerate(got.split(part)):
        assert (chunk[:, :16].contiguous().view(torch.float32) - vis).abs().max() <= bar, k


@pytest.mark.parametrize("shift", [-7, -1, 1, 7])
@pytest.mark.parametrize("do_grid", [0, 1])
@pytest.mark.parametrize("npol,M", [(1, [[0]]), (2, [[0, 1]])])
def test_overlapping_device_records(hpg, npol, M, do_grid, shift):
    """Records returned some records before or behind their own place."""
    import ctypes
    import torch
    from hpg_amd import workloads
    print(f"npol {npol} do_grid {do_grid} shift {shift}", flush=True)
    gsz, n = (200, 180, 1, 1), 100_000
    cf = workloads.random_cf(4, [3], nmueller=2, seed=1)
    rec = workloads.random_visibilities(n, npol, gsz, (1.0, 1.0), cf, seed=2, margin=-3)
    gs = hpg.GridderState.create(hpg.Device.Hip, 0, n, cf, gsz, (1.0, 1.0), M, M)
    gs.set_convolution_function(hpg.Device.Serial, cf)
    rng = np.random.default_rng(3)
    gs.set_model(hpg.Device.Serial, rng.standard_normal(gsz[::-1]) + 0j)
    exp = (gs.degrid_grid_get_residual_visibilities if do_grid
           else gs.degrid_get_predicted_visibilities)(hpg.Device.Serial, rec)
    size = rec.dtype.itemsize
    src, dst = max(0, -shift) * size, max(0, shift) * size
    buf = torch.zeros((n + abs(shift)) * size, dtype=torch.uint8, device="cuda")
    buf[src:src + n * size] = torch.from_numpy(rec.view(np.uint8)).cuda()
    torch.cuda.synchronize()
    assert hpg._lib.lib().hpgx_grid_visibilities(
        gs._h, ctypes.c_void_p(buf.data_ptr() + src), n, npol, 0, 1, 1, do_grid,
        ctypes.c_void_p(buf.data_ptr() + dst), 1) == 0
    gs.fence()
    got = buf[dst:dst + n * size].cpu().numpy().view(rec.dtype)
    for name in rec.dtype.names:
        if name != "visibilities":
            assert np.array_equal(got[name], exp[name]), name
    bar = 1e-6 * np.abs(exp["visibilities"]).max()
    assert np.abs(got["visibilities"] - exp["visibilities"]).max() <= bar


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("npol,M,nm", [(1, [[0]], 1), (2, [[0, 1]], 2), (2, [[0, 1], [2, 1]], 3),
                                       (4, DIAG, 4), (4, FULL, 16)])
@pytest.mark.parametrize("sx,sy", [(65537, 3), (3, 65539), (65535, 1), (131075, 1)])
def test_wide_supports(hpg, oracle_mod, sx, sy, npol, M, nm, mode):
    """Supports of 2^16 pixels and more along one axis."""
    from hpg_amd import workloads
    print(f"support {sx} x {sy} npol {npol} nm {nm} mode {mode}", flush=True)
    gsz, n = (sx + 21, sy + 21, len(M), 1), 40
    cf = workloads.random_cf(1, [((sx - 1) // 2, (sy - 1) // 2), 1], nmueller=nm, seed=1)
    rec = workloads.random_visibilities(n, npol, gsz, (0.9, 1.1), cf, seed=2, phase=True)
    wide = rec["cf_index"][:, 1] == 0
    rng = np.random.default_rng(4)
    rec["uvw"][wide, :2] = rng.uniform(-9, 9, (wide.sum(), 2)) / np.array([0.9, 1.1])
    gs, o = _pair(hpg, oracle_mod, gsz, M, M, cf, mode, n)
    _set_model(hpg, gs, o, gsz)
    _check_predictions(hpg, oracle_mod, gs, o, rec)
    _check_grid(hpg, oracle_mod, gs, o, rec, 1e-6 if mode else 1e-12)


@pytest.mark.parametrize("gradient", [False, True])
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("rows,nm", [((0, 1, 2), 16), ((0, 1, 2), 12), ((3, 0, 2), 16)])
def test_three_rows_of_neighbouring_elements(hpg, oracle_mod, rows, nm, mode, gradient):
    """Rows of four neighbouring elements, whose patches' fourth lane has no row."""
    from hpg_amd import workloads
    gsz, n = (81, 64, 3, 2), 900
    M, Mc = [FULL[r] for r in rows], [FULL[r] for r in rows[::-1]]
    cf = workloads.random_cf(6, [(1, 3), 8], nmueller=nm, ncube=2, seed=1)
    rec = workloads.random_visibilities(n, 4, gsz, (0.9, 1.1), cf, seed=2, phase=True, margin=-3,
                                        gradient=gradient)
    gs, o = _pair(hpg, oracle_mod, gsz, M, Mc, cf, mode, n)
    _set_model(hpg, gs, o, gsz)
    _check_predictions(hpg, oracle_mod, gs, o, rec)
    _check_grid(hpg, oracle_mod, gs, o, rec, 1e-6 if mode or gradient else 1e-12)


# npol, M, Mc, Mueller elements of the two CF groups: elements that no row names
# before, between and behind those that rows do, rows of one polarization, rows
# that name elements which one group or both lack, or none at all
ELEMENTS = [
    (1, [[0]], [[0]], (16, 16)),
    (1, [[15]], [[3]], (16, 16)),
    (1, [[2]], [[5]], (6, 3)),
    (1, [[1], [7]], [[7], [-1]], (9, 2)),
    (1, [[4]], [[4]], (4, 6)),
    (2, [[0, -1], [-1, 15]], [[15, -1], [-1, 0]], (16, 16)),
    (2, [[1, 9]], [[9, 1]], (16, 10)),
    (2, [[6, 7], [12, 13]], [[12, 13], [6, 7]], (16, 14)),
    (3, [[0, 4, 8]], [[8, 4, 0]], (9, 5)),
    (4, [[0, -1, -1, -1], [-1, 5, -1, -1], [-1, -1, 10, -1], [-1, -1, -1, 15]],
     [[0, -1, -1, -1], [-1, 5, -1, -1], [-1, -1, 10, -1], [-1, -1, -1, 15]], (16, 11)),
    (4, [[20, 21, 22, 23]], [[4, 5, 6, 7]], (24, 24)),
    (4, [[20, 21, 22, 23]], [[4, 5, 6, 7]], (24, 2)),
    (2, [[-1, -1], [3, -1]], [[-1, -1], [-1, -1]], (4, 3)),
]


@pytest.mark.parametrize("gradient", [False, True])
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("radii", [[3, (1, 2)], [(6, 4), 9], [20, 2]])
@pytest.mark.parametrize("case", range(len(ELEMENTS)))
def test_few_of_a_cf_s_elements(hpg, oracle_mod, case, radii, mode, gradient):
    from hpg_amd import workloads
    print(f"case {case} radii {radii} mode {mode} gradient {gradient}", flush=True)
    npol, M, Mc, nms = ELEMENTS[case]
    gsz, n = (81, 70, len(M), 2), 2500
    groups = [workloads.random_cf(6, [r], nmueller=nm, ncube=2, seed=3 + k).values(0)
              for k, (r, nm) in enumerate(zip(radii, nms))]
    cf = hpg.CFArray(6, groups)
    rec = workloads.random_visibilities(n, npol, gsz, (0.9, 1.1), cf, seed=2, phase=True,
                                        margin=-3, gradient=gradient)
    gs, o = _pair(hpg, oracle_mod, gsz, M, Mc, cf, mode, n)
    _set_model(hpg, gs, o, gsz)
    o.grid_visibilities(_view(rec, oracle_mod), True)
    gs.grid_visibilities(hpg.Device.Serial, rec, True)
    copy = gs.copy()
    bar = 1e-6 if mode or gradient else 1e-12
    for s in (gs, copy):
        assert np.abs(s.grid_values() - o.grid_values()).max() <= bar * np.abs(
            o.grid_values()).max()
        np.testing.assert_allclose(s.grid_weights(), o.grid_weights(), rtol=1e-12)
        pred = s.degrid_get_predicted_visibilities(hpg.Device.Serial, rec)["visibilities"]
        exp = o.grid_visibilities(_view(rec, oracle_mod), False, do_degrid=True,
                                  do_grid=False)["vis"]
        assert np.abs(pred - exp).max() <= 1e-6 * np.abs(exp).max()
    # another CF in the same state, of other elements
    cf2 = workloads.random_cf(4, [2], nmueller=max(nms) + 1, ncube=2, seed=9)
    rec2 = workloads.random_visibilities(n, npol, gsz, (0.9, 1.1), cf2, seed=5, phase=True)
    gs.set_convolution_function(hpg.Device.Serial, cf2)
    o.set_cf(4, [(cf2.extents(0), cf2.values(0))])
    gs.grid_visibilities(hpg.Device.Serial, rec2, True)
    o.grid_visibilities(_view(rec2, oracle_mod), True)
    assert np.abs(gs.grid_values() - o.grid_values()).max() <= bar * np.abs(o.grid_values()).max()


def test_noalloc_register_patches(hpg):
    """Without allocations, calls by register patches need neither halos nor
    bins: they fit where the halo values alone (4096 keys of 1280 pixels, 84 MB)
    would not.  1e-12: the same products in another order of FP64 sums."""
    import ctypes
    import torch
    from hpg_amd import _lib, workloads
    gsz, n = (1024, 1024, 4, 1), 700
    cf = workloads.random_cf(4, [8], nmueller=4, seed=91)
    rec = workloads.random_visibilities(n, 4, gsz, (1.0, 1.0), cf, seed=92, phase=True)
    dev = torch.from_numpy(rec.view(np.uint8).copy()).cuda()
    torch.cuda.synchronize()
    states = []
    for noalloc in (False, True):
        gs = hpg.GridderState.create(hpg.Device.Hip, 0, n, cf, gsz, (1.0, 1.0), DIAG)
        gs.set_convolution_function(hpg.Device.Serial, cf)
        if noalloc:
            rc = _lib.lib().hpgx_grid_visibilities_noalloc(
                gs._h, ctypes.c_void_p(dev.data_ptr()), n, 4, 1)
            assert rc == 0, _lib.error_message(gs._h)
        else:
            gs.grid_visibilities(hpg.Device.Serial, dev)
        gs.fence()
        states.append(gs)
    exp = states[0].grid_values()
    assert np.abs(exp).max() > 0
    assert np.abs(states[1].grid_values() - exp).max() <= 1e-12 * np.abs(exp).max()
    np.testing.assert_allclose(states[1].grid_weights(), states[0].grid_weights(), rtol=1e-12)
