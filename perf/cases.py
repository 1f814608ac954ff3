"""Timing cases of the gridding path: one batch of visibilities through one public call each.

A case names the call (``op``) and the sizes it runs at:

  grid         grid_visibilities of a device-resident batch, into the state's grid
  predict      degrid_get_predicted_visibilities of a device-resident batch
  residual     degrid_grid_get_residual_visibilities of a device-resident batch
  degrid_grid  degrid_grid_visibilities of a device-resident batch
  forward      degrid_forward, the differentiable form's forward operator
  adjoint      degrid_adjoint, its adjoint
  fit          image -> model -> visibilities -> chi^2 -> image gradient (autograd)
  image        a whole dirty image of a host batch: reset, grid, normalize, FFT, shift, readback

``uv`` is "uniform" (u, v uniform within +-0.45 of the extent: the single-polarization
workload) or "gauss" (u, v ~ N(0, (sigma extent)^2), dense core and sparse edges: the
W- and A/W-projection workloads; records of the tail that fall off the grid are skipped).
CF group g has support smin .. smax pixels, linear in the group; a record's |w| picks it.

Gridding calls accumulate into the state's grid, as a program does that grids batch after
batch; the grid comes back as the state's own device buffer.  The weights come back where
the program waits for the call anyway (predictions returned, multi-polarization batches of
milliseconds, whole images); a single-polarization batch of microseconds is queued without
reading them.
"""
import math

import torch

import hpg_amd as hpg
from hpg_amd.autograd import degrid, image_to_model

C_LIGHT = 299792458.0
PAD = 2  # CF padding, in pixels per edge
DEV = "cuda"


# ---- the cases ---------------------------------------------------------------

def _case(name, op, mode, npol, mueller, nx, ny, cubes, records, groups, smin, smax, os, uv,
          sigma=0.2, screen=False, gradient=False):
    c = dict(op=op, mode=mode, npol=npol, mueller=mueller, nx=nx, ny=ny, cubes=cubes,
             records=records, groups=groups, smin=smin, smax=smax, os=os, uv=uv, sigma=sigma,
             screen=screen, gradient=gradient)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest calls: a short integration into a small grid, where launches count
        _case("small", "grid", "fp64", 1, "one", 512, 480, 1, 2000, 1, 7, 7, 20, "uniform"),
        # a quick look: host records to a finished dirty image in host memory (odd sizes)
        _case("quicklook", "image", "fp32", 1, "one", 301, 270, 1, 20_000, 1, 7, 7, 16,
              "uniform"),
        # the single-polarization workload, in both grid types
        _case("grid_1pol_fp32", "grid", "fp32", 1, "one", 1024, 1024, 1, 1_000_000, 1, 7, 7, 20,
              "uniform"),
        _case("grid_1pol_fp64", "grid", "fp64", 1, "one", 1024, 1024, 1, 1_000_000, 1, 7, 7, 20,
              "uniform"),
        # the same batch spread over a large grid of ragged sizes
        _case("grid_1pol_large", "grid", "fp32", 1, "one", 4001, 3750, 1, 1_000_000, 1, 7, 7, 20,
              "uniform"),
        # model prediction of that batch (calibration, subtraction)
        _case("predict_1pol", "predict", "fp32", 1, "one", 1024, 1024, 1, 1_000_000, 1, 7, 7, 20,
              "uniform"),
        # major-cycle residuals of the two parallel hands, small W kernels
        _case("residual_2pol", "residual", "fp64", 2, "diag", 1500, 1500, 2, 300_000, 8, 7, 17,
              16, "gauss"),
        # full-polarization gridding with supports below a tile
        _case("grid_fullpol", "grid", "fp32", 4, "full", 1024, 1024, 1, 200_000, 8, 9, 25, 16,
              "gauss"),
        # full-polarization W-projection: 64 w planes, supports 9-65
        _case("wproj", "degrid_grid", "fp64", 4, "full", 4096, 4096, 2, 500_000, 64, 9, 65, 20,
              "gauss"),
        # A/W-projection: supports 17-129, an aperture phase screen in every CF
        _case("awproj", "degrid_grid", "fp32", 4, "full", 4096, 4096, 2, 150_000, 32, 17, 129, 10,
              "gauss", sigma=0.25, screen=True),
        # the differentiable form: forward operator, and a whole image-domain fitting step
        _case("forward", "forward", "fp64", 4, "diag", 2048, 2048, 1, 1_000_000, 16, 9, 33, 16,
              "gauss", sigma=0.15),
        _case("fit_step", "fit", "fp64", 4, "diag", 1024, 1024, 1, 300_000, 16, 9, 33, 16,
              "gauss", sigma=0.15),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _odd(rng, lo, hi):
    return 2 * rng.randint(lo // 2, (hi - 1) // 2) + 1


def draw(rng):
    """A case of the listed ones' ranges: any kind of program above, at other sizes."""
    kind = rng.choice(["single", "single", "few", "fullpol", "wproj", "awproj", "diff", "image"])
    mode = rng.choice(["fp32", "fp64"])
    nx, ny = _log_int(rng, 128, 4096), 0
    ny = max(128, min(4096, int(nx * rng.uniform(0.7, 1.4))))
    if kind == "single":
        s = _odd(rng, 5, 9)
        return _case("", rng.choice(["grid", "grid", "predict"]), mode, 1, "one", nx, ny, 1,
                     _log_int(rng, 500, 1_000_000), 1, s, s, rng.choice([8, 10, 16, 20]),
                     "uniform", gradient=rng.random() < 0.15)
    if kind == "image":
        s = _odd(rng, 5, 9)
        npol = rng.choice([1, 2])
        return _case("", "image", mode, npol, "one" if npol == 1 else "diag",
                     _log_int(rng, 64, 1024), _log_int(rng, 64, 1024), 1,
                     _log_int(rng, 1000, 200_000), 1, s, s, rng.choice([8, 16]), "uniform")
    if kind in ("few", "fullpol"):
        nx, ny = max(256, min(nx, 2048)), max(256, min(ny, 2048))
        npol = 2 if kind == "few" else 4
        smin = _odd(rng, 7, 13)
        smax = _odd(rng, smin, 27)
        return _case("", rng.choice(["grid", "residual", "degrid_grid"]), mode, npol,
                     "diag" if kind == "few" else "full", nx, ny, rng.randint(1, 3),
                     _log_int(rng, 10_000, 200_000), rng.randint(2, 12), smin, smax,
                     rng.choice([8, 10, 16]), "gauss", gradient=rng.random() < 0.1)
    if kind == "wproj":
        nx, ny = max(1024, nx), max(1024, ny)
        smax = _odd(rng, 33, 65)
        return _case("", rng.choice(["grid", "residual", "degrid_grid"]), mode, 4, "full", nx, ny,
                     rng.randint(1, 2), _log_int(rng, 50_000, 400_000), rng.randint(8, 48), 9,
                     smax, rng.choice([10, 16]), "gauss")
    if kind == "awproj":
        nx, ny = max(2048, nx), max(2048, ny)
        return _case("", rng.choice(["grid", "degrid_grid"]), mode, 4, "full", nx, ny,
                     rng.randint(1, 2), _log_int(rng, 20_000, 100_000), rng.randint(8, 24), 17,
                     _odd(rng, 65, 129), rng.choice([8, 10]), "gauss", sigma=0.25, screen=True)
    nx = ny = min(2048, max(512, nx))
    smax = _odd(rng, 17, 33)
    op = rng.choice(["forward", "adjoint", "fit"])
    if op == "fit":
        nx = ny = min(1024, nx)
    return _case("", op, "fp64", 4, "diag", nx, ny, 1,
                 _log_int(rng, 50_000, 200_000 if op == "fit" else 1_000_000),
                 rng.randint(4, 16), 9, smax, rng.choice([8, 16]), "gauss", sigma=0.15)


# ---- inputs ------------------------------------------------------------------

def _radii(c):
    g = c["groups"]
    a, b = (c["smin"] - 1) // 2, (c["smax"] - 1) // 2
    return [a + int(round((b - a) * k / max(g - 1, 1))) for k in range(g)]


def _mueller(c):
    n = c["npol"]
    if c["mueller"] == "one":
        return [[0]]
    if c["mueller"] == "diag":
        return [[r if r == v else -1 for v in range(n)] for r in range(n)]
    return [[n * r + v for v in range(n)] for r in range(n)]


def _nelem(c):
    return 1 + max(m for row in _mueller(c) for m in row)


def _cf_groups(c, seed):
    """CF groups (1, element, y, x), complex64 on the GPU: a Gaussian taper; with several
    groups the w chirp exp(i pi k rho^2), one amplitude per Mueller element; with screen a
    phase per tap (an aperture illumination's)."""
    out = []
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed * 7919 + 17)
    nm, os_ = _nelem(c), c["os"]
    amp = 0.6 + 0.8 * torch.rand(nm, generator=gen, device=DEV, dtype=torch.float64)
    for k, r in enumerate(_radii(c)):
        ext = (2 * r + 1 + 2 * PAD) * os_
        t = (torch.arange(ext, device=DEV, dtype=torch.float64) - (r + PAD) * os_) / os_
        rho2 = t[None, :] ** 2 + t[:, None] ** 2
        sigma = max(r / 2.5, 1.0) if c["groups"] > 1 else r / 2.0
        base = torch.exp(-rho2 / (2 * sigma * sigma)).to(torch.complex64)
        if c["groups"] > 1:
            chirp = math.pi * 0.2 * (k + 0.5) / (c["groups"] * max(r, 1))
            base = base * torch.polar(torch.ones_like(rho2), chirp * rho2).to(torch.complex64)
        v = base[None, None] * amp[None, :, None, None].to(torch.float32)
        if c["screen"]:
            ph = torch.rand(v.shape, generator=gen, device=DEV) * (2 * math.pi)
            v = v * torch.polar(torch.ones_like(ph), ph)
        out.append(v.contiguous())
    return out


def _records(c, seed):
    """(n, itemsize) uint8 tensor of VisData records on the GPU."""
    n, npol = c["records"], c["npol"]
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed * 104729 + 5)
    dt = hpg.visdata_dtype(npol)
    rec = torch.zeros((n, dt.itemsize), dtype=torch.uint8, device=DEV)

    def put(name, value):
        off = dt.fields[name][1]
        b = value.contiguous().view(torch.uint8).reshape(n, -1)
        rec[:, off:off + b.shape[1]] = b

    def rand(*shape):
        return torch.rand(shape, generator=gen, device=DEV, dtype=torch.float64)

    put("visibilities", torch.randn((n, 2 * npol), generator=gen, device=DEV))
    put("weights", 0.5 + torch.rand((n, npol), generator=gen, device=DEV))
    cube = torch.randint(0, c["cubes"], (n,), generator=gen, device=DEV)
    freq = C_LIGHT * (1.0 + 0.01 * cube.to(torch.float64))
    put("frequency", freq)
    uvw = torch.empty((n, 3), dtype=torch.float64, device=DEV)
    for d, size in enumerate((c["nx"], c["ny"])):
        if c["uv"] == "uniform":
            # whole supports on the grid, also of the smallest grids
            edge = min(0.45 * size, size / 2.0 - (c["smax"] + 1) / 2.0 - 1.0)
            uvw[:, d] = (2 * rand(n) - 1) * edge
        else:
            uvw[:, d] = torch.randn(n, generator=gen, device=DEV, dtype=torch.float64) \
                * (c["sigma"] * size)
    uvw[:, :2] /= (freq / C_LIGHT)[:, None]
    w = rand(n) if c["groups"] > 1 else torch.zeros(n, dtype=torch.float64, device=DEV)
    grp = torch.clamp((w * c["groups"]).floor(), max=c["groups"] - 1).to(torch.int32)
    sign = torch.where(rand(n) < 0.5, -1.0, 1.0)
    uvw[:, 2] = w * sign
    put("uvw", uvw)
    put("grid_cube", cube.to(torch.int32))
    put("cf_index", torch.stack([torch.zeros_like(grp), grp], 1))
    if c["groups"] > 1:
        put("phase", 0.3 * (2 * rand(n) - 1))
    if c["gradient"]:
        put("cf_phase_gradient", 0.02 * (2 * rand(n, 2) - 1))
    return rec


def _complex(shape, gen):
    return torch.complex(
        torch.randn(shape, generator=gen, device=DEV, dtype=torch.float64),
        torch.randn(shape, generator=gen, device=DEV, dtype=torch.float64))


def _grid_size(c):
    return (c["nx"], c["ny"], len(_mueller(c)), c["cubes"])


class _DeviceArray:
    """The state's grid as __cuda_array_interface__ (no copy).  A tensor of it holds this
    object, and this object the state: the buffer lives as long as the tensor."""

    def __init__(self, gs, shape, kind):
        self.owner = gs
        ptr, _ = gs.grid_device_ptr()
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": kind,
                                         "strides": None, "version": 3}


def prepare(case, seed):
    c = case
    gsz = _grid_size(c)
    M = _mueller(c)
    mode = hpg.GridMode.FP64 if c["mode"] == "fp64" else hpg.GridMode.FP32_COMPENSATED
    cf = hpg.CFArray(c["os"], _cf_groups(c, seed))
    gs = hpg.GridderState.create(hpg.Device.Hip, 0, c["records"], cf, gsz, (1.0, 1.0), M, M,
                                 grid_mode=mode)
    gs.set_convolution_function(hpg.Device.Serial, cf)
    del cf
    shape = gs.grid_shape
    s = {"op": c["op"], "npol": c["npol"], "gs": gs, "rec": _records(c, seed)}
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed * 31 + 3)
    if c["op"] in ("predict", "residual", "degrid_grid", "forward"):
        gs.set_model(hpg.Device.Serial, _complex(shape, gen))
    if c["op"] == "adjoint":
        s["residuals"] = _complex((c["records"], c["npol"]), gen)
    if c["op"] == "fit":
        s["image"], s["data"], s["wts"] = _fit_inputs(c, gen)
    if c["op"] == "image":
        s["rec"] = s["rec"].cpu().numpy().view(hpg.visdata_dtype(c["npol"])).reshape(-1)
    s["grid"] = torch.as_tensor(
        _DeviceArray(gs, shape, "<c16" if c["mode"] == "fp64" else "<c8"), device=DEV)
    gs.fence()
    torch.cuda.empty_cache()
    return s


def _fit_inputs(c, gen):
    """A sky of point sources and noise, the data to fit, and their weights."""
    shape = (c["cubes"], c["npol"], c["ny"], c["nx"])
    image = 1e-4 * torch.randn(shape, generator=gen, device=DEV, dtype=torch.float64)
    y = torch.randint(0, c["ny"], (200,), generator=gen, device=DEV)
    x = torch.randint(0, c["nx"], (200,), generator=gen, device=DEV)
    flux = torch.exp(torch.rand(200, generator=gen, device=DEV, dtype=torch.float64)
                     * math.log(1e3)) * 1e-3
    image[:, :, y, x] += flux
    data = 3.0 * _complex((c["records"], c["npol"]), gen)
    wts = 0.5 + torch.rand((c["records"], c["npol"]), generator=gen, device=DEV,
                           dtype=torch.float64)
    return image.to(torch.float32), data, wts


# ---- one pass ----------------------------------------------------------------

def _split(records, npol):
    """The returned records: their visibilities as floats, and the rest as they are."""
    return {"visibilities": records[:, :8 * npol].view(torch.float32),
            "others": records[:, 8 * npol:]}


def run(state):
    op, gs, rec, npol = state["op"], state["gs"], state["rec"], state["npol"]
    host = hpg.Device.Serial
    if op == "grid":
        gs.grid_visibilities(host, rec)
        if npol == 1:
            return state["grid"]
        return {"grid": state["grid"], "weights": gs.grid_weights()}
    if op == "predict":
        return _split(gs.degrid_get_predicted_visibilities(host, rec), npol)
    if op == "residual":
        out = _split(gs.degrid_grid_get_residual_visibilities(host, rec), npol)
        return {**out, "grid": state["grid"], "weights": gs.grid_weights()}
    if op == "degrid_grid":
        gs.degrid_grid_visibilities(host, rec)
        return {"grid": state["grid"], "weights": gs.grid_weights()}
    if op == "forward":
        return gs.degrid_forward(rec)
    if op == "adjoint":
        gs.degrid_adjoint(rec, state["residuals"])
        return state["grid"]
    if op == "fit":
        image = state["image"].clone().requires_grad_(True)
        pred = degrid(image_to_model(image, gs), gs, rec)
        loss = (state["wts"] * (pred - state["data"]).abs() ** 2).sum()
        loss.backward()
        return {"loss": loss.detach(), "predicted": pred.detach(), "gradient": image.grad}
    # image
    gs.reset_grid()
    gs.grid_visibilities(host, rec)
    weights = gs.grid_weights()
    gs.normalize_by_weights(1.0)
    gs.apply_grid_fft(1.0, hpg.FFTSign.POSITIVE, True)
    gs.shift_grid(hpg.ShiftDirection.FORWARD)
    return {"image": gs.grid_values(), "weights": weights}


# ---- what a pass cannot do without -------------------------------------------

def work(case):
    """Bytes: the records, the CF as the caller holds it, grid and model once each way.
    Operations: 8 per tap, correlation and Mueller term gridded, the same degridded (all
    records taken as on the grid), 5 N log2 N a plane for an FFT."""
    c = case
    n, npol, op = c["records"], c["npol"], c["op"]
    radii = _radii(c)
    terms = sum(m >= 0 for row in _mueller(c) for m in row)
    s2 = sum((2 * r + 1) ** 2 for r in radii) / len(radii)
    cf = sum(((2 * r + 1 + 2 * PAD) * c["os"]) ** 2 for r in radii) * _nelem(c) * 8
    px = c["nx"] * c["ny"] * len(_mueller(c)) * c["cubes"]
    grid = px * (16 if c["mode"] == "fp64" else 8)
    rec = n * hpg.visdata_dtype(npol).itemsize
    one = 8.0 * n * s2 * terms
    fft = 5.0 * px * math.log2(c["nx"] * c["ny"])
    if op == "grid":
        b, f = rec + cf + 2 * grid, one
    elif op == "predict":
        b, f = 2 * rec + cf + 16 * px, one
    elif op == "residual":
        b, f = 2 * rec + cf + 16 * px + 2 * grid, 2 * one
    elif op == "degrid_grid":
        b, f = rec + cf + 16 * px + 2 * grid, 2 * one
    elif op == "forward":
        b, f = rec + cf + 16 * px + 16 * n * npol, one
    elif op == "adjoint":
        b, f = rec + cf + 16 * n * npol + 2 * grid, one
    elif op == "fit":
        # the image and its gradient, the model and its gradient, data, weights, predictions
        b = 2 * rec + 2 * cf + px * (4 + 4 + 2 * 16 + 2 * 16) + n * npol * (16 + 8 + 16)
        f = 2 * one + 2 * fft
    else:
        b, f = rec + cf + 2 * grid + 16 * px, one + fft
    return {"bytes": float(b), "flops": float(f)}


# ---- the same in 64 bits -----------------------------------------------------

class _Batch:
    """The records' fields, coordinates and CF positions in 64 bits."""

    def __init__(self, c, seed):
        self.c = c
        self.cf = _cf_groups(c, seed)
        self.rec = rec = _records(c, seed)
        npol = c["npol"]
        dt = hpg.visdata_dtype(npol)

        def get(name, nbytes, kind):
            off = dt.fields[name][1]
            return rec[:, off:off + nbytes].contiguous().view(kind)

        self.vis = torch.view_as_complex(
            get("visibilities", 8 * npol, torch.float32).reshape(-1, npol, 2).double())
        self.w = get("weights", 4 * npol, torch.float32).double()
        phase = get("phase", 8, torch.float64)[:, 0]
        self.phasor = torch.polar(torch.ones_like(phase), phase)
        uvw = get("uvw", 24, torch.float64).reshape(-1, 3)
        inv_lambda = get("frequency", 8, torch.float64)[:, 0] / C_LIGHT
        self.cube = get("grid_cube", 4, torch.int32)[:, 0].long()
        self.grp = get("cf_index", 8, torch.int32)[:, 1].long()
        self.grad = get("cf_phase_gradient", 16, torch.float64).reshape(-1, 2)
        self.pos_w = uvw[:, 2] > 0
        radii = torch.as_tensor(_radii(c), device=DEV)[self.grp]
        self.corner, self.fine = [], []
        self.inside = torch.ones_like(self.pos_w)
        for d, size in enumerate((c["nx"], c["ny"])):
            pos = uvw[:, d] * inv_lambda + size / 2.0
            near = torch.round(pos)
            self.fine.append(torch.round((near - pos) * c["os"]).long())
            corner = near.long() - radii
            self.corner.append(corner)
            self.inside &= (corner >= 0) & (corner + 2 * radii + 1 <= size)

    def chunks(self):
        """(records, their taps' flat positions in a plane (k, s, s), the elements' CF values
        by index, and the phase screen or None), some records of one group at a time."""
        c = self.c
        for g, cf in enumerate(self.cf):
            r = _radii(c)[g]
            s = 2 * r + 1
            every = torch.nonzero((self.grp == g) & self.inside)[:, 0]
            for i in torch.split(every, max(1, 24_000_000 // (s * s))):
                if not len(i):
                    continue
                t = torch.arange(s, device=DEV)
                ix = (t + PAD)[None] * c["os"] + self.fine[0][i][:, None]
                iy = (t + PAD)[None] * c["os"] + self.fine[1][i][:, None]
                px = (self.corner[1][i][:, None] + t)[:, :, None] * c["nx"] \
                    + (self.corner[0][i][:, None] + t)[:, None, :]
                screen = None
                if c["gradient"]:
                    ph = [-self.grad[i, d][:, None] * (r * c["os"] - self.fine[d][i])[:, None]
                          + self.grad[i, d][:, None] * c["os"] * t for d in (0, 1)]
                    ph = ph[1][:, :, None] + ph[0][:, None, :]
                    screen = torch.polar(torch.ones_like(ph), ph)
                at = iy[:, :, None] * cf.shape[-1] + ix[:, None, :]

                def element(m, cf=cf, at=at):
                    return torch.take(cf[0, m], at).to(torch.complex128)
                yield i, px, element, screen


def _exact_grid(b, gvis):
    """The grid and the weights' terms |sum c| w of gridding gvis (n, npol)."""
    c = b.c
    M = _mueller(c)
    nr, plane = len(M), c["nx"] * c["ny"]
    grid = torch.zeros((c["cubes"] * nr * plane, 2), dtype=torch.float64, device=DEV)
    weights = torch.zeros((c["cubes"], nr), dtype=torch.float64, device=DEV)
    for i, px, element, screen in b.chunks():
        neg = torch.where(b.pos_w[i], -1.0, 1.0)[:, None, None]
        for r, row in enumerate(M):
            total = torch.zeros(px.shape, dtype=torch.complex128, device=DEV)
            for v, m in enumerate(row):
                if m < 0:
                    continue
                e = element(m)
                e = torch.complex(e.real, e.imag * neg)
                weights[:, r].index_add_(0, b.cube[i], e.sum((1, 2)).abs() * b.w[i, v])
                total += (e if screen is None else e * screen) * gvis[i, v][:, None, None]
            at = (b.cube[i] * nr + r)[:, None, None] * plane + px
            grid.index_add_(0, at.reshape(-1), torch.view_as_real(total).reshape(-1, 2))
    shape = (c["cubes"], nr, c["ny"], c["nx"])
    return torch.view_as_complex(grid).reshape(shape), weights


def _exact_degrid(b, model):
    """(predictions, norms) of the model (cube, row, y, x)."""
    c = b.c
    M = _mueller(c)
    nr, plane = len(M), c["nx"] * c["ny"]
    flat = model.reshape(-1)
    a = torch.zeros((c["records"], c["npol"]), dtype=torch.complex128, device=DEV)
    W = torch.zeros_like(a)
    for i, px, element, screen in b.chunks():
        neg = torch.where(b.pos_w[i], 1.0, -1.0)[:, None, None]
        for r, row in enumerate(M):
            if all(m < 0 for m in row):
                continue
            mv = torch.take(flat, (b.cube[i] * nr + r)[:, None, None] * plane + px)
            if screen is not None:
                mv = mv * screen.conj()
            for v, m in enumerate(row):
                if m < 0:
                    continue
                e = element(m)
                e = torch.complex(e.real, e.imag * neg)
                a[i, v] += (e * mv).sum((1, 2))
                W[i, v] += e.sum((1, 2))
    W = torch.where(W == 0, torch.ones_like(W), W)
    return a / W * b.phasor.conj()[:, None], W


def exact(case, seed):
    """run()'s outputs of a new state by plain torch in 64 bits."""
    c = case
    op = c["op"]
    b = _Batch(c, seed)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed * 31 + 3)
    shape = (c["cubes"], len(_mueller(c)), c["ny"], c["nx"])
    if op == "fit":
        return _exact_fit(c, b, gen)
    vis = b.vis
    if op in ("predict", "residual", "degrid_grid", "forward"):
        pred, _ = _exact_degrid(b, _complex(shape, gen))
        if op == "forward":
            return pred
        keep = b.inside[:, None]
        vis = torch.where(keep, pred if op == "predict" else vis - pred, vis)
        out = {"visibilities": torch.view_as_real(vis).reshape(c["records"], -1), "others": None}
        if op == "predict":
            return out
    if op == "adjoint":
        r = _complex((c["records"], c["npol"]), gen)
        _, W = _exact_degrid(b, torch.zeros(shape, dtype=torch.complex128, device=DEV))
        gvis = r * b.phasor[:, None] / W.conj()
    else:
        gvis = vis * b.phasor[:, None] * b.w
    grid, weights = _exact_grid(b, gvis)
    if op == "residual":
        return {**out, "grid": grid, "weights": weights}
    if op == "image":
        z = grid / weights[:, :, None, None]
        z = torch.fft.ifft2(z, norm="forward")
        z = torch.fft.fftshift(z, dim=(-2, -1))
        return {"image": z.cpu().numpy(), "weights": weights.cpu().numpy()}
    if op == "adjoint" or c["npol"] == 1:
        return grid
    return {"grid": grid, "weights": weights}


def _exact_fit(c, b, gen):
    image, data, wts = _fit_inputs(c, gen)
    model = torch.fft.fftshift(torch.fft.fft2(image.to(torch.complex128)), dim=(-2, -1))
    pred, W = _exact_degrid(b, model)
    r = pred - data
    loss = (wts * (r.real ** 2 + r.imag ** 2)).sum()
    back, _ = _exact_grid(b, torch.where(b.inside[:, None], 2 * wts * r, torch.zeros_like(r))
                          * b.phasor[:, None] / W.conj())
    gradient = torch.fft.ifft2(torch.fft.ifftshift(back, dim=(-2, -1)), norm="forward").real
    return {"loss": loss, "predicted": pred, "gradient": gradient}
