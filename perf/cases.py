"""Timed cases of the fitting framework, through its public entry points.

Each case is one call a localization-microscopy program makes, with inputs
drawn the way the repository's own benchmark and tests draw them (photons,
backgrounds, widths, sensor maps), on the GPU, from a seed:

  fit       gaussmle_amd.device.fit_device on ROIs that are already in HBM:
            every PSF model, both cameras, both precisions, boxes 7..24 px
  batch     gaussmle_amd.batch.fit_batch_device: one call on ROIs of mixed box
            sizes and models
  host      gaussmle_amd.fit_arrays on host arrays, the call that replaces the
            reference's GPU branch
  boxes     gaussmle_amd.boxer.find_boxes_device: camera frames to ROIs
  simulate  gaussmle_amd.simulator.simulate_device: parameters to noisy ROIs
  epilogue  gaussmle_amd.device.epilogue_device: fit results to microns and
            p-values

`exact` restates each computed result in Float64 with plain torch.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parent.parent / "gaussmle.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import gaussmle_amd as g  # noqa: E402
from gaussmle_amd import batch as gb  # noqa: E402
from gaussmle_amd import boxer as gbx  # noqa: E402
from gaussmle_amd import device as gd  # noqa: E402
from gaussmle_amd import simulator as gs  # noqa: E402
from gaussmle_amd import synth  # noqa: E402

DEV = "cuda:0"
MODELS = ("xynb", "xynbs", "xynbsxsy", "astig")
N_PARAMS = {"xynb": 4, "xynbs": 5, "xynbsxsy": 6, "astig": 5}
SENSOR = 256                 # sCMOS calibration maps are SENSOR x SENSOR
BATCH_BOXES = (7, 9, 11, 13, 15)
BATCH_WEIGHTS = (0.1, 0.2, 0.4, 0.2, 0.1)
BATCH_STRIDE = 6
BOXER = {"overlap": 2.0, "sigma_small": 1.0, "sigma_large": 2.0, "minval": 5.0}
CELL = 64                    # one emitter per CELL x CELL pixels of a frame
PIXEL_UM = 0.1


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def _fit(name, model, box, n, camera="ideal", precision="fp32", iterations=20):
    return {"name": name, "kind": "fit", "model": model, "box": box, "n": n, "camera": camera,
            "precision": precision, "iterations": iterations}


def listed():
    return [
        # one camera frame's handful of emitters in an interactive or real-time loop: all latency
        _fit("fit_xynb7_100", "xynb", 7, 100),
        # the reference's default batch (10,000 ROIs of 11 px, fixed width)
        _fit("fit_xynb11_10k", "xynb", 11, 10_000),
        # the headline: a whole acquisition's ROIs in one launch
        _fit("fit_xynb11_1m", "xynb", 11, 1 << 20),
        # fitted width on an sCMOS sensor
        _fit("fit_xynbs13_scmos_1m", "xynbs", 13, 1_000_000, camera="scmos"),
        # the same with the Float64 final pass
        _fit("fit_xynbs13_scmos_mixed", "xynbs", 13, 250_000, camera="scmos", precision="mixed"),
        # astigmatic 3-D within +-d of focus, 30 iterations
        _fit("fit_astig15_1m", "astig", 15, 1_000_000, iterations=30),
        # wide boxes for wide spots
        _fit("fit_xynbs21_200k", "xynbs", 21, 200_000),
        # an uneven batch: five box sizes, three models, sCMOS
        {"name": "batch_scmos_1m", "kind": "batch", "n": 1_000_000},
        # host arrays in and out, as the drop-in call makes it (pageable memory, validation included)
        {"name": "host_xynb11_200k", "kind": "host", "model": "xynb", "box": 11, "n": 200_000},
        # camera frames of a full sensor to ROIs
        {"name": "boxes_2048_x32", "kind": "boxes", "ny": 2048, "nx": 2048, "frames": 32, "box": 11},
        # synthetic ROI stacks for tests and calibration
        {"name": "simulate_xynb11_1m", "kind": "simulate", "model": "xynb", "box": 11, "n": 1 << 20,
         "camera": "ideal"},
        # fit results of one acquisition to microns and p-values
        {"name": "epilogue_xynbs13_1m", "kind": "epilogue", "model": "xynbs", "box": 13, "n": 1 << 20},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("fit",) * 6 + ("batch", "host", "boxes", "simulate", "epilogue"))
    if kind == "fit":
        model = rng.choice(MODELS)
        # astigmatic spots are up to 2.9 px wide within +-d and need the larger boxes
        box = rng.randint(13, 24) if model == "astig" else rng.randint(7, 24)
        n = _log_int(rng, 50, min(600_000, 60_000_000 // (box * box)))
        return {"kind": "fit", "model": model, "box": box, "n": n, "camera": rng.choice(("ideal", "scmos")),
                "precision": rng.choice(("fp32", "fp32", "mixed")), "iterations": 30 if model == "astig" else 20}
    if kind == "batch":
        return {"kind": "batch", "n": _log_int(rng, 2_000, 600_000)}
    if kind == "host":
        return {"kind": "host", "model": rng.choice(MODELS[:3]), "box": rng.randint(7, 16),
                "n": _log_int(rng, 1_000, 150_000)}
    if kind == "boxes":
        return {"kind": "boxes", "ny": rng.randint(128, 2048), "nx": rng.randint(128, 2048),
                "frames": rng.randint(1, 24), "box": rng.randint(7, 16)}
    if kind == "simulate":
        return {"kind": "simulate", "model": rng.choice(MODELS[:3]), "box": rng.randint(7, 21),
                "n": _log_int(rng, 1_000, 200_000), "camera": rng.choice(("ideal", "scmos"))}
    return {"kind": "epilogue", "model": rng.choice(MODELS), "box": rng.randint(7, 24),
            "n": _log_int(rng, 1_000, 1 << 20)}


# ---------------------------------------------------------------------------
# Inputs, from the seed alone, on the GPU
# ---------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _uniform(gen, n, lo, hi):
    return torch.rand(n, generator=gen, device=DEV, dtype=torch.float64) * (hi - lo) + lo


def _psf(model):
    return {"xynb": g.GaussianXYNB(1.3), "xynbs": g.GaussianXYNBS(), "xynbsxsy": g.GaussianXYNBSXSY(),
            "astig": synth.ASTIG_CONFIG_PSF}[model]


def _constraints(model, box):
    """The reference's defaults for 11 px boxes, as its fitter passes them; those of the box's own size above 16 px."""
    if model == "astig":
        c = synth.astig_constraints()
        if box > 16:
            up = c.upper.copy()
            up[:2] = box + 2
            c = g.ParameterConstraints(c.lower, up, c.max_step)
        return c
    return g.default_constraints(_psf(model), 11 if box <= 16 else box)


def _theta(gen, model, box, n):
    """(n, P) Float64 true parameters: emitters within 1.5 px of the centre, 500-5000 photons (astigmatic:
    1000-10000), 1-20 background photons per pixel (2-30), widths 1-1.6 px (1.3-2 px above 16 px boxes), z within
    +-d of focus."""
    c = (box + 1) / 2
    x, y = _uniform(gen, n, c - 1.5, c + 1.5), _uniform(gen, n, c - 1.5, c + 1.5)
    if model == "astig":
        cols = [x, y, _uniform(gen, n, -100, 100), _uniform(gen, n, 1000, 10000), _uniform(gen, n, 2, 30)]
    else:
        cols = [x, y, _uniform(gen, n, 500, 5000), _uniform(gen, n, 1, 20)]
        widths = (1.0, 1.6) if box <= 16 else (1.3, 2.0)
        cols += [_uniform(gen, n, *widths) for _ in range(N_PARAMS[model] - 4)]
    return torch.stack(cols, 1)


def _widths(model, th):
    if model == "xynb":
        s = torch.full_like(th[:, 0], float(np.float32(1.3)))
        return s, s
    if model == "xynbs":
        return th[:, 4], th[:, 4]
    if model == "xynbsxsy":
        return th[:, 4], th[:, 5]
    p = [float(v) for v in _psf(model).psf_array()]
    ux, uy = (th[:, 2] - p[6]) / p[7], (th[:, 2] + p[6]) / p[7]
    return (p[0] * torch.sqrt(1 + ux**2 + p[2] * ux**3 + p[4] * ux**4),
            p[1] * torch.sqrt(1 + uy**2 + p[3] * uy**3 + p[5] * uy**4))


def _phi(box, mu, sigma):
    """Pixel-integrated Gaussian of pixels 1..box, (n, box)."""
    e = torch.arange(box + 1, device=DEV, dtype=torch.float64)[None, :] + 0.5
    s = torch.erf((e - mu[:, None]) / (math.sqrt(2.0) * sigma[:, None]))
    return 0.5 * (s[:, 1:] - s[:, :-1])


def _sensor_maps(gen):
    """(ny, nx) gain and read variance of an sCMOS sensor."""
    gain = torch.rand(SENSOR, SENSOR, generator=gen, device=DEV) * 0.2 + 0.4
    var = torch.exp(math.log(2.0) + 0.5 * torch.randn(SENSOR, SENSOR, generator=gen, device=DEV))
    return gain, var


def _corners(gen, n, box):
    return [torch.randint(1, SENSOR - box + 2, (n,), generator=gen, device=DEV, dtype=torch.int32) for _ in range(2)]


def _map_pixels(m, xc, yc, box):
    """A (ny, nx) map at each ROI's pixels, (n, column, row)."""
    k = torch.arange(box, device=DEV)
    return m[(yc.long() - 1)[:, None, None] + k[None, None, :], (xc.long() - 1)[:, None, None] + k[None, :, None]]


def _rois(gen, model, box, n, var=None):
    """(pixels, xc, yc): flat Float32 ROIs in the column-major layout; Poisson counts, with read noise of the sensor's
    variance for sCMOS."""
    th = _theta(gen, model, box, n)
    out = torch.empty(n, box, box, dtype=torch.float32, device=DEV)
    xc = yc = None
    if var is not None:
        xc, yc = _corners(gen, n, box)
    for a in range(0, n, 1 << 17):
        t = th[a:a + (1 << 17)]
        sx, sy = _widths(model, t)
        i_n, i_bg = (3, 4) if model == "astig" else (2, 3)
        mu = t[:, i_bg, None, None] + t[:, i_n, None, None] * _phi(box, t[:, 0], sx)[:, :, None] * _phi(
            box, t[:, 1], sy)[:, None, :]
        e = torch.poisson(mu.float(), generator=gen)
        if var is not None:
            sd = torch.sqrt(_map_pixels(var, xc[a:a + len(t)], yc[a:a + len(t)], box))
            e = e + sd * torch.randn(e.shape, generator=gen, device=DEV)
        out[a:a + len(t)] = e
    return out.reshape(-1), xc, yc


def _prepare_fit(case, gen):
    var = _sensor_maps(gen)[1] if case["camera"] == "scmos" else None
    data, xc, yc = _rois(gen, case["model"], case["box"], case["n"], var)
    P = N_PARAMS[case["model"]]
    # Float32 results, as the drop-in returns them; the buffers are a program's own and are used again
    out = {"params": torch.zeros(case["n"], P, device=DEV), "crlb": torch.zeros(case["n"], P, device=DEV),
           "llr": torch.zeros(case["n"], device=DEV)}
    return {"data": data, "xc": xc, "yc": yc, "out": out, "psf": _psf(case["model"]),
            "constraints": _constraints(case["model"], case["box"]),
            "var": None if var is None else var.t().contiguous().reshape(-1)}


def _batch_shapes(gen, n):
    boxes = torch.tensor(BATCH_BOXES, device=DEV)[torch.multinomial(
        torch.tensor(BATCH_WEIGHTS, device=DEV), n, replacement=True, generator=gen)]
    models = torch.randint(0, 3, (n,), generator=gen, device=DEV)
    return models, boxes


def _prepare_batch(case, gen):
    n = case["n"]
    models, boxes = _batch_shapes(gen, n)
    sizes = boxes * boxes
    offsets = torch.cumsum(sizes, 0) - sizes
    var = _sensor_maps(gen)[1]
    data = torch.empty(int(sizes.sum()), dtype=torch.float32, device=DEV)
    xc = torch.zeros(n, dtype=torch.int32, device=DEV)
    yc = torch.zeros(n, dtype=torch.int32, device=DEV)
    for m in range(3):
        for b in BATCH_BOXES:
            idx = torch.nonzero((models == m) & (boxes == b))[:, 0]
            if not len(idx):
                continue
            e, xs, ys = _rois(gen, MODELS[m], b, len(idx), var)
            xc[idx], yc[idx] = xs, ys
            data[(offsets[idx][:, None] + torch.arange(b * b, device=DEV)[None, :]).reshape(-1)] = e
    mb = gb.MixedBatch(models.cpu().numpy().astype(np.int8), boxes.cpu().numpy().astype(np.int8),
                       np.empty(0, np.float32), offsets.cpu().numpy(), {m: _psf(MODELS[m]) for m in range(3)},
                       {m: _constraints(MODELS[m], 11) for m in range(3)}, 20, var.cpu().numpy(), xc.cpu().numpy(),
                       yc.cpu().numpy())
    d = {"models": models.to(torch.int8), "boxes": boxes.to(torch.int8), "offsets": offsets, "data": data,
         "counts": mb.shape_counts(), "var": var.t().contiguous().reshape(-1), "xc": xc, "yc": yc,
         "workspace": torch.empty(int(g._lib.load().gmle_batch_workspace_bytes(n)), dtype=torch.uint8, device=DEV)}
    out = {"params": torch.zeros(n, BATCH_STRIDE, device=DEV), "crlb": torch.zeros(n, BATCH_STRIDE, device=DEV),
           "llr": torch.zeros(n, device=DEV)}
    return {"batch": mb, "d": d, "out": out}


def _prepare_host(case, gen):
    box, n = case["box"], case["n"]
    data = _rois(gen, case["model"], box, n)[0].cpu().numpy()
    fitter = g.GaussMLEFitter(_psf(case["model"]), device="gpu", constraints=_constraints(case["model"], box))
    return {"fitter": fitter, "psf": _psf(case["model"]),
            "data": data.reshape(n, box, box).transpose(2, 1, 0)}   # (row, column, roi), Fortran order


def _frames(gen, ny, nx, nf):
    """(nf, nx, ny) Float32 frames (column-major each): background 10, one emitter of 500-3000 photons per CELL x CELL
    cell, noise of variance equal to the mean."""
    mu = torch.full((nf, nx, ny), 10.0, device=DEV)
    cy, cx = max(1, ny // CELL), max(1, nx // CELL)
    k = nf * cx * cy
    half = 8
    jit = [_uniform(gen, k, half + 2.0, min(CELL, s) - half - 3.0) for s in (nx, ny)]
    at = torch.arange(k, device=DEV)
    f, col, row = at // (cx * cy), at // cy % cx, at % cy
    x, y = col * CELL + jit[0], row * CELL + jit[1]
    N = _uniform(gen, k, 500, 3000)
    ix, iy = torch.round(x).long(), torch.round(y).long()
    w = torch.arange(-half, half + 1, device=DEV)
    s = 1.0 / (math.sqrt(2.0) * 1.3)

    def integral(p, ip):
        e = (ip[:, None] + w[None, :] - p[:, None])
        return 0.5 * (torch.erf((e + 0.5) * s) - torch.erf((e - 0.5) * s))

    patch = N[:, None, None] * integral(x, ix)[:, :, None] * integral(y, iy)[:, None, :]
    # cells do not overlap, so no pixel is written twice
    mu[f[:, None, None], ix[:, None, None] + w[None, :, None], iy[:, None, None] + w[None, None, :]] += patch.float()
    return mu + torch.sqrt(mu) * torch.randn(mu.shape, generator=gen, device=DEV)


def _prepare_boxes(case, gen):
    ny, nx, nf, box = case["ny"], case["nx"], case["frames"], case["box"]
    cap = 2 * nf * max(1, ny // CELL) * max(1, nx // CELL) + 1024   # a program's bound on the detections
    ws = int(g._lib.load().gmle_boxer_workspace_bytes(ny, nx, nf))
    out = {"rois": torch.zeros(cap, box * box, device=DEV),
           "x_corners": torch.zeros(cap, dtype=torch.int32, device=DEV),
           "y_corners": torch.zeros(cap, dtype=torch.int32, device=DEV),
           "frames": torch.zeros(cap, dtype=torch.int32, device=DEV), "strength": torch.zeros(cap, device=DEV),
           "count": torch.zeros(1, dtype=torch.int64, device=DEV),
           "workspace": torch.empty(max(ws, 1), dtype=torch.uint8, device=DEV)}
    return {"frames": _frames(gen, ny, nx, nf).reshape(-1), "cap": cap, "out": out}


def _prepare_simulate(case, gen, seed):
    n, box = case["n"], case["box"]
    s = {"params": _theta(gen, case["model"], box, n).float().contiguous(), "psf": _psf(case["model"]),
         "seed": int(seed) + 1, "out": torch.zeros(n * box * box, device=DEV), "camera": None, "xc": None, "yc": None}
    if case["camera"] == "scmos":
        gain, var = (m.cpu().numpy() for m in _sensor_maps(gen))
        s["camera"] = g.SCMOSCamera.square(SENSOR, SENSOR, PIXEL_UM, readnoise=np.sqrt(var), offset=100.0, gain=gain,
                                           qe=0.82)
        s["xc"], s["yc"] = _corners(gen, n, box)
    return s


def _prepare_epilogue(case, gen):
    """Fit results: parameters near their truths, uncertainties of a few percent, chi^2 of good fits with one bad fit in
    fifty, and ROI corners on a 2048 x 2048 sensor."""
    n, box, model = case["n"], case["box"], case["model"]
    P = N_PARAMS[model]
    df = box * box - P
    chi2 = df + math.sqrt(2.0 * df) * torch.randn(n, generator=gen, device=DEV, dtype=torch.float64)
    bad = _uniform(gen, n, 0, 1) < 0.02
    chi2 = torch.where(bad, chi2 * _uniform(gen, n, 1.2, 3.0), chi2).clamp(min=0.1)
    xc, yc = [torch.randint(1, 2048 - box + 2, (n,), generator=gen, device=DEV, dtype=torch.int32) for _ in range(2)]
    return {"params": _theta(gen, model, box, n).float().contiguous(),
            "crlb": (_theta(gen, model, box, n).abs() * 0.03 + 0.01).float().contiguous(),
            "llr": (-0.5 * chi2).float(), "xc": xc, "yc": yc, "out": torch.zeros(n, 10, device=DEV)}


def prepare(case, seed):
    gen = _generator(seed)
    kind = case["kind"]
    if kind == "simulate":
        s = _prepare_simulate(case, gen, seed)
    else:
        s = {"fit": _prepare_fit, "batch": _prepare_batch, "host": _prepare_host, "boxes": _prepare_boxes,
             "epilogue": _prepare_epilogue}[kind](case, gen)
    s["case"] = case
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "fit":
        ny = nx = SENSOR if s["var"] is not None else 0
        r = gd.fit_device(s["psf"], c["box"], s["data"], s["constraints"], c["iterations"], c["precision"], 0, s["var"],
                          ny, nx, s["xc"], s["yc"], out=s["out"])
        return {k: r[k] for k in ("params", "crlb", "llr")}
    if kind == "batch":
        r = gb.fit_batch_device(s["batch"], s["d"], out=s["out"])
        return {k: r[k] for k in ("params", "crlb", "llr")}
    if kind == "host":
        r = g.fit_arrays(s["fitter"], s["data"], s["psf"])
        return {"params": r.params, "crlb": r.crlb, "llr": r.llr}
    if kind == "boxes":
        r = gbx.find_boxes_device(s["frames"], c["ny"], c["nx"], c["frames"], c["box"], max_boxes=s["cap"],
                                  out=s["out"], **BOXER)
        return {k: r[k] for k in ("rois", "x_corners", "y_corners", "frames", "strength", "count")}
    if kind == "simulate":
        return gs.simulate_device(s["psf"], c["box"], s["params"], s["seed"], s["camera"], s["xc"], s["yc"],
                                  out=s["out"])
    return gd.epilogue_device(s["params"], s["crlb"], s["llr"], PIXEL_UM, PIXEL_UM, MODELS.index(c["model"]), c["box"],
                              d_xc=s["xc"], d_yc=s["yc"], out=s["out"])


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _fit_flops(model, box, iterations):
    """FP32 operations of one separable fit: per iteration the pixels and both axes' edges, then the final pass and
    the initial estimates (an add or multiply is 1, an FMA 2; transcendentals are not counted)."""
    pix = {"xynb": 32, "xynbs": 45, "xynbsxsy": 50, "astig": 45}[model]
    axis = 13 if model == "xynb" else 23
    P = N_PARAMS[model]
    final = P * (P + 1) + 2 * P + 12
    return iterations * (box * box * pix + 2 * box * axis) + box * box * (final + 8)


def work(case):
    kind = case["kind"]
    if kind == "boxes":
        ny, nx, nf, box = case["ny"], case["nx"], case["frames"], case["box"]
        found = nf * max(1, ny // CELL) * max(1, nx // CELL)
        taps = 2 * (3 + 6)   # both radii (3 sigma) on each axis: a pair sum and an FMA per tap
        return {"bytes": 4.0 * ny * nx * nf + found * (4.0 * box * box + 16), "flops": ny * nx * nf * (3.0 * taps + 5)}
    n = case["n"]
    if kind == "batch":
        sizes = [(b, w / sum(BATCH_WEIGHTS)) for b, w in zip(BATCH_BOXES, BATCH_WEIGHTS)]
        return {"bytes": n * (sum(w * 4.0 * b * b for b, w in sizes) + 18 + 4 * (2 * BATCH_STRIDE + 1)),
                "flops": n * sum(w * _fit_flops(m, b, 20) / 3 for b, w in sizes for m in MODELS[:3])}
    box, P = case["box"], N_PARAMS[case["model"]]
    if kind == "epilogue":
        return {"bytes": n * (4.0 * (2 * P + 1) + 8 + 40), "flops": n * 100.0}
    if kind == "simulate":
        return {"bytes": n * (4.0 * P + 4.0 * box * box), "flops": n * box * box * 100.0}
    corners = 8.0 if case.get("camera") == "scmos" else 0.0
    return {"bytes": n * (4.0 * box * box + 4.0 * (2 * P + 1) + corners),
            "flops": n * float(_fit_flops(case["model"], box, case.get("iterations", 20)))}


# ---------------------------------------------------------------------------
# The same results in 64 bits, with plain torch
# ---------------------------------------------------------------------------
def _axis(box, mu, sigma, N):
    """Per-axis pixel integral and its derivatives (baselibrary's 1-D formulas), each (n, box)."""
    t = torch.arange(box + 1, device=DEV, dtype=torch.float64)[None, :] + 0.5 - mu[:, None]
    s = sigma[:, None]
    gss = torch.exp(-t * t / (2 * s * s))
    tg, t3g = t * gss, t * t * t * gss

    def diff(v):
        return v[:, 1:] - v[:, :-1]

    c = -N[:, None] / math.sqrt(2 * math.pi) / s
    S = c / s * diff(tg)
    return {"phi": 0.5 * diff(torch.erf(t / (math.sqrt(2.0) * s))), "D": c * diff(gss), "D2": c / s**2 * diff(tg),
            "S": S, "SS": -2 / s * S + c / s**4 * diff(t3g)}


def _width_terms(model, th):
    """(sx, sy) and, for the astigmatic model, their first and second z derivatives."""
    sx, sy = _widths(model, th)
    if model != "astig":
        return sx, sy, None
    p = [float(v) for v in _psf(model).psf_array()]
    out = []
    for s0, A, B, u in ((p[0], p[2], p[4], (th[:, 2] - p[6]) / p[7]), (p[1], p[3], p[5], (th[:, 2] + p[6]) / p[7])):
        a = 1 + u**2 + A * u**3 + B * u**4
        da = (2 * u + 3 * A * u**2 + 4 * B * u**3) / p[7]
        d2a = (2 + 6 * A * u + 12 * B * u**2) / p[7] ** 2
        r = torch.sqrt(a)
        out += [s0 / (2 * r) * da, -s0 / (4 * a * r) * da**2 + s0 / (2 * r) * d2a]
    return sx, sy, out


def _derivatives(model, box, th, second):
    """Model (n, box, box) [column, row], and per parameter its derivative and diagonal second derivative."""
    i_n, i_bg = (3, 4) if model == "astig" else (2, 3)
    N, bg = th[:, i_n], th[:, i_bg]
    sx, sy, dz = _width_terms(model, th)
    X, Y = _axis(box, th[:, 0], sx, N), _axis(box, th[:, 1], sy, N)

    def outer(a, b):
        return a[:, :, None] * b[:, None, :]

    pp = outer(X["phi"], Y["phi"])
    mu = bg[:, None, None] + N[:, None, None] * pp
    one = torch.ones_like(pp)
    du = {0: outer(X["D"], Y["phi"]), 1: outer(X["phi"], Y["D"]), i_n: pp, i_bg: one}
    d2 = {0: outer(X["D2"], Y["phi"]), 1: outer(X["phi"], Y["D2"])} if second else {}
    if model != "xynb":
        ax, ay = outer(X["S"], Y["phi"]), outer(X["phi"], Y["S"])
        aax, aay = (outer(X["SS"], Y["phi"]), outer(X["phi"], Y["SS"])) if second else (0.0, 0.0)
        if model == "xynbs":
            du[4], d2[4] = ax + ay, aax + aay
        elif model == "xynbsxsy":
            du[4], du[5], d2[4], d2[5] = ax, ay, aax, aay
        else:
            dx, ddx, dy, ddy = (v[:, None, None] for v in dz)
            du[2] = ax * dx + ay * dy
            d2[2] = aax * dx**2 + ax * ddx + aay * dy**2 + ay * ddy if second else 0.0
    return mu, du, d2


def _start(model, box, d):
    """Initial estimates from (n, column, row) pixels."""
    edge = torch.ones(box, box, dtype=torch.bool, device=DEV)
    edge[1:-1, 1:-1] = False
    bg = d[:, edge].mean(1)
    s = (d - bg[:, None, None]).clamp(min=0)
    k = torch.arange(1, box + 1, device=DEV, dtype=torch.float64)
    tot = s.sum((1, 2))
    mid = torch.full_like(tot, (box + 1) / 2)
    ok = tot > 10
    x = torch.where(ok, (s.sum(2) * k).sum(1) / tot, mid).clamp(1.5, box - 0.5)
    y = torch.where(ok, (s.sum(1) * k).sum(1) / tot, mid).clamp(1.5, box - 0.5)
    ph = tot.clamp(min=100)
    if model != "astig":
        return torch.stack([x, y, ph, bg] + [torch.full_like(x, 1.3)] * (N_PARAMS[model] - 4), 1)
    p = [float(v) for v in _psf(model).psf_array()]
    mxx = (s.sum(2) * (k[None, :] - x[:, None]) ** 2).sum(1)
    myy = (s.sum(1) * (k[None, :] - y[:, None]) ** 2).sum(1)
    rx, ry = ((m / tot).clamp(min=0.5) / q**2 for m, q in ((mxx, p[0]), (myy, p[1])))
    z = torch.where(ok, (-(rx - ry) * p[7] ** 2 / (4 * p[6])).clamp(-600, 600), torch.zeros_like(x))
    return torch.stack([x, y, z, ph, bg], 1)


def _crlb(F):
    """sqrt of the diagonal of the inverse of the (n, P, P) Fisher matrices with the reference's ridge."""
    P = F.shape[1]
    F = F + 1e-10 * F.abs().amax((1, 2))[:, None, None] * torch.eye(P, dtype=F.dtype, device=DEV)
    A = torch.cat([F, torch.eye(P, dtype=F.dtype, device=DEV).expand(len(F), P, P)], 2)
    for k in range(P):   # Gauss-Jordan without pivoting: the matrices are positive definite
        A[:, k] = A[:, k] / A[:, k, k, None]
        for i in range(P):
            if i != k:
                A[:, i] = A[:, i] - A[:, i, k, None] * A[:, k]
    return torch.sqrt(torch.diagonal(A[:, :, P:], dim1=1, dim2=2).clamp(min=0))


def _fit64(model, box, data, cons, iterations, var=None):
    """The fixed-iteration Newton fit of (n, column, row) Float32 pixels in Float64: (params, crlb, llr)."""
    lo, up, ms = (torch.from_numpy(np.asarray(a, dtype=np.float64)).to(DEV) for a in
                  (cons.lower, cons.upper, cons.max_step))
    d = data.double()
    th = _start(model, box, d)
    P = th.shape[1]
    for _ in range(iterations):
        mu, du, d2 = _derivatives(model, box, th, True)
        if var is None:
            ok = mu > 0.01
            cf = torch.where(ok, (d / mu - 1).clamp(max=1e4), 0.0)
            df = torch.where(ok, (d / mu**2).clamp(max=1e4), 0.0)
        else:
            v = mu + var
            cf, df = (d - mu) / v, 1 / v
        G = torch.stack([(du[k] * cf).sum((1, 2)) for k in range(P)], 1)
        H = torch.stack([((d2[k] * cf if k in d2 else 0.0) - du[k] ** 2 * df).sum((1, 2)) for k in range(P)], 1)
        step = torch.where(H.abs() > 1e-10, G / H, 0.0)
        th = torch.minimum(torch.maximum(th - torch.minimum(torch.maximum(step, -ms), ms), lo), up)
    mu, du, _ = _derivatives(model, box, th, False)
    if var is None:
        pos = mu > 0
        llr = torch.where(pos & (d > 0), d * torch.log(mu / d) + d - mu, torch.where(pos, -mu, 0.0)).sum((1, 2))
        w = torch.where(pos, 1 / mu, 0.0)
    else:
        v = mu + var
        llr = torch.where(v > 0, -0.5 * (d - mu) ** 2 / v, 0.0).sum((1, 2))
        w = torch.where(mu > 0, 1 / v, 0.0)
    F = torch.stack([torch.stack([(du[k] * w * du[m]).sum((1, 2)) for m in range(P)], 1) for k in range(P)], 1)
    return th, _crlb(F), llr


def _fit64_all(model, box, flat, cons, iterations, var=None, xc=None, yc=None):
    d = flat.view(-1, box, box)
    step = max(1, (1 << 23) // (box * box))
    parts = []
    for a in range(0, len(d), step):
        v = None if var is None else _map_pixels(var, xc[a:a + step], yc[a:a + step], box).double()
        parts.append(_fit64(model, box, d[a:a + step], cons, iterations, v))
    return [torch.cat(p) for p in zip(*parts)]


def _map_of(flat):
    return flat.view(SENSOR, SENSOR).t()


def _exact_batch(s):
    mb, d = s["batch"], s["d"]
    n = mb.n
    params = torch.full((n, BATCH_STRIDE), math.nan, dtype=torch.float64, device=DEV)
    crlb, llr = params.clone(), params[:, 0].clone()
    for m in range(3):
        for b in BATCH_BOXES:
            idx = torch.nonzero((d["models"] == m) & (d["boxes"] == b))[:, 0]
            if not len(idx):
                continue
            px = d["data"][(d["offsets"][idx][:, None] + torch.arange(b * b, device=DEV)[None, :]).reshape(-1)]
            p, c, v = _fit64_all(MODELS[m], b, px, mb.constraints[m], mb.iterations, _map_of(d["var"]), d["xc"][idx],
                                 d["yc"][idx])
            params[idx, :p.shape[1]], crlb[idx, :p.shape[1]], llr[idx] = p, c, v
    return {"params": params, "crlb": crlb, "llr": llr}


def _exact_epilogue(s):
    c = s["case"]
    P = N_PARAMS[c["model"]]
    p, u = s["params"].double(), s["crlb"].double()
    chi2 = -2.0 * s["llr"].double()
    out = torch.full((c["n"], 10), math.nan, dtype=torch.float64, device=DEV)
    px = float(PIXEL_UM)
    for a, q in ((0, s["xc"]), (1, s["yc"])):
        out[:, a] = (q.double() + p[:, a] - 2.0) * px
        out[:, 2 + a] = u[:, a] * px
    half = torch.full_like(chi2, 0.5 * (c["box"] ** 2 - P))
    out[:, 4] = torch.special.gammaincc(half, 0.5 * chi2)
    if P > 4 and c["model"] != "astig":
        for a in (0, 1):
            k = 4 if P == 5 else 4 + a
            out[:, 5 + a], out[:, 7 + a] = p[:, k] * px, u[:, k] * px
    out[:, 9] = chi2
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("simulate", "boxes"):
        # drawn counts, and copied pixels at whole-number places: no rounding to measure
        return None
    s = prepare(case, seed)
    if kind == "fit":
        var = None if s["var"] is None else _map_of(s["var"])
        r = _fit64_all(case["model"], case["box"], s["data"], s["constraints"], case["iterations"], var, s["xc"], s["yc"])
        return dict(zip(("params", "crlb", "llr"), r))
    if kind == "host":
        flat = torch.from_numpy(np.ascontiguousarray(s["data"].transpose(2, 1, 0))).to(DEV).reshape(-1)
        p, c, v = _fit64_all(case["model"], case["box"], flat, s["fitter"].constraints, s["fitter"].iterations)
        return {"params": p.t().cpu().numpy(), "crlb": c.t().cpu().numpy(), "llr": v.cpu().numpy()}
    if kind == "batch":
        return _exact_batch(s)
    return _exact_epilogue(s)
