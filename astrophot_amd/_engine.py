"""Host side of one component render: window geometry in float64, then the
gfx950 launches render -> psf_shift -> convolve through the C ABI.

This is Component_Model.sample (models/model_object.py:258-375) and the
per-component forward-mode Jacobian (models/_model_methods.py:260-347)
re-expressed as kernel launches:

* psf_mode "full": the working window is the sampling window padded by the
  PSF border (psf_image.py:71-93); the sub-pixel centre shift
  s = pc - round(pc) moves into a bilinearly shifted PSF and the grid is
  sampled at X = P (i - round(pc)) (model_object.py:320-325).  Centre
  derivatives come from d(shifted PSF)/ds, every other column from the render
  channels convolved with the shifted PSF.
* psf_mode "none": X = P (i - pc); every column, the centre included, comes
  from the render channels; a 1x1 unit kernel crops and accumulates.

The integration threshold reference is the Sersic total flux over the
working-grid pixel count (sersic_model.py:78-89) or the mean initial sample
(_model_methods.py:151-152).
"""

from __future__ import annotations

import ctypes
import functools
import math
from dataclasses import dataclass
from typing import Dict, List, Optional, Sequence, Tuple

import numpy as np
import torch

from . import AP_config
from . import _lib as L
from .errors import SpecificationConflict

PROFILE_CODE = {"sersic": L.APX_SERSIC, "exponential": L.APX_EXPONENTIAL, "gaussian": L.APX_GAUSSIAN,
                "moffat": L.APX_MOFFAT, "flat_sky": L.APX_FLAT_SKY}
# profile parameter name -> slot
PROFILE_SLOTS = {
    "sersic": {"n": L.APX_P_A, "Re": L.APX_P_B, "Ie": L.APX_P_C},
    "exponential": {"Re": L.APX_P_A, "Ie": L.APX_P_B},
    "gaussian": {"sigma": L.APX_P_A, "flux": L.APX_P_B},
    "moffat": {"n": L.APX_P_A, "Rd": L.APX_P_B, "I0": L.APX_P_C},
    "flat_sky": {"F": L.APX_P_A},
}
GEOM_SLOTS = {"q": L.APX_P_Q, "PA": L.APX_P_PA}
# parameters of an auxiliary PSF model (model_object.py:133-147) are keyed
# PSF_SLOT0 + their slot in the PSF model
PSF_SLOT0 = 16


def gauss_legendre(n: int):
    """Abscissae and weights on [-1, 1] (the table scipy.special.roots_legendre
    gives the reference, utils/operations.py:105-120)."""
    x, w = np.polynomial.legendre.leggauss(n)
    return x, w


def sersic_b(n):
    """utils/conversions/functions.py:7-22."""
    return (2 * n - 1 / 3 + 4 / (405 * n) + 46 / (25515 * n**2) + 131 / (1148175 * n**3)
            - 2194697 / (30690717750 * n**4))


def sersic_total_flux(Ie_lin, n, Re, q):
    """utils/conversions/functions.py:168-190."""
    b = sersic_b(n)
    return 2 * math.pi * Ie_lin * Re**2 * q * n * math.exp(b) * b ** (-2 * n) * math.exp(math.lgamma(2 * n))


@dataclass
class RenderRequest:
    """What one component render has to produce."""

    window: object                  # sampling (working) window before padding
    image: Optional[object] = None  # Model_Image to accumulate the value into
    jac: Optional[object] = None    # Jacobian_Image to accumulate columns into
    slot_cols: Optional[Dict[int, int]] = None  # slot -> Jacobian column
    dvdr: Optional[Dict[int, float]] = None     # slot -> d value / d rep
    region: Optional[object] = None  # window the result is clipped to (default: destination & window)


_UNIT_KERNEL = {}

# When a dict, every library launch below is bracketed by torch.cuda events on
# the launch stream: TIMING[name] collects (start, end, work) triples, with
# `work` the launch's algorithmic flops (convolve) or pixels (render).
TIMING = None


def _launch(name, work, fn):
    if TIMING is None:
        return fn()
    s = torch.cuda.Event(enable_timing=True)
    e = torch.cuda.Event(enable_timing=True)
    s.record()
    r = fn()
    e.record()
    TIMING.setdefault(name, []).append((s, e, work))
    return r


def _unit_kernel(device):
    k = _UNIT_KERNEL.get(device)
    if k is None:
        k = torch.ones((1, 1, 1), dtype=torch.float32, device=device)
        _UNIT_KERNEL[device] = k
    return k


@functools.lru_cache(maxsize=16)
def _gl(n):
    x, w = gauss_legendre(n)
    return tuple(float(v) for v in x), tuple(float(v) for v in w)


@functools.lru_cache(maxsize=8)
def _device(device):
    return torch.device(device)


@functools.lru_cache(maxsize=256)
def _render_bytes(npix):
    return int(L.load().apx_render_workspace_bytes(npix))


@functools.lru_cache(maxsize=256)
def _convolve_bytes(kh, kw):
    return int(L.load().apx_convolve_workspace_bytes(kh, kw))


def _buffer(owner, name, nbytes, device):
    """A device byte buffer of at least ``nbytes`` kept on ``owner`` between
    calls (work on one stream is ordered, so reuse is safe)."""
    cache = owner.__dict__.get("_apx_buffers")
    if cache is None:
        cache = owner.__dict__["_apx_buffers"] = {}
    b = cache.get(name)
    if b is None or b.numel() < nbytes or b.device != _device(device):
        b = torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device=device)
        cache[name] = b
    return b


def _box(dst_window, src_window, region):
    """Where ``region`` lands in ``dst`` and in ``src``, and its extent
    (image_object.py:450-457 via window_object.py:241-269)."""
    dr, dc = dst_window.get_self_indices(region)
    sr, sc = src_window.get_self_indices(region)
    h = min(dr.stop - dr.start, sr.stop - sr.start)
    w = min(dc.stop - dc.start, sc.stop - sc.start)
    return (dr.start, dc.start), (sr.start, sc.start), (max(h, 0), max(w, 0))


@dataclass
class Plan:
    """Launch descriptor and geometry of one component on one sampling window."""

    cp: object            # L.Component
    window: object        # padded working window
    bx: int
    by: int
    shift: Optional[Tuple[float, float]]
    psf_full: bool
    chan_slots: List[int]
    upscale: int = 1           # PSF upscale: working pixels per image pixel, per axis
    out_window: object = None  # where the convolved output lands (after the block sum)


@functools.lru_cache(maxsize=256)
def _template(kind, sm, im, quad_level, gridding, max_depth, radius, softening, tolerance) -> bytes:
    """The fields of an apx_component that the model's knobs alone decide."""
    cp = L.Component()
    cp.profile = PROFILE_CODE[kind]
    # sampling mode (_model_methods.py:82-148)
    if sm == "midpoint":
        cp.sampling = L.APX_SAMPLE_MIDPOINT
    elif sm == "simpsons":
        # _model_methods.py:97-109: corners, edge midpoints and centre of each
        # pixel weighted 1, 4, 16 / 36, the centre sample as the reference
        cp.sampling = L.APX_SAMPLE_QUAD
        cp.sample_quad = 3
        cp.sq_node[:3] = (-1.0, 0.0, 1.0)
        cp.sq_weight[:3] = (1.0 / 3.0, 4.0 / 3.0, 1.0 / 3.0)
    elif sm.startswith("quad"):
        cp.sampling = L.APX_SAMPLE_QUAD
        cp.sample_quad = int(sm[sm.find(":") + 1:])
        if not 1 <= cp.sample_quad <= L.APX_MAX_QUAD_LEVEL:
            raise SpecificationConflict(f"sampling quad level must be 1..{L.APX_MAX_QUAD_LEVEL}")
        x, w = _gl(cp.sample_quad)
        cp.sq_node[:cp.sample_quad], cp.sq_weight[:cp.sample_quad] = x, w
    elif sm == "trapezoid":
        # _model_methods.py:121-139: mean of the four pixel corners; the
        # reference is that mean plus its Laplacian
        cp.sampling = L.APX_SAMPLE_TRAPEZOID
        cp.sample_quad = 2
        cp.sq_node[:2] = (-1.0, 1.0)
        cp.sq_weight[:2] = (1.0, 1.0)
    else:
        raise SpecificationConflict(
            f"{{name}} has unknown sampling mode: {sm}. Should be one of: midpoint, simpsons, quad:level, trapezoid")
    if im not in ("none", "threshold", "radius"):
        raise SpecificationConflict(
            f"{{name}} has unknown integration mode: {im}. Should be one of: none, threshold, radius")
    cp.integrate = {"none": L.APX_INTEGRATE_NONE, "threshold": L.APX_INTEGRATE_THRESHOLD,
                    "radius": L.APX_INTEGRATE_RADIUS}[im]
    if cp.integrate:
        cp.quad_level, cp.gridding, cp.max_depth = quad_level, gridding, max_depth
        if im == "radius":
            cp.integrate_radius = radius
            cp.gridding, cp.max_depth = 1, 1
        if not 1 <= cp.quad_level <= L.APX_MAX_QUAD_LEVEL:
            raise SpecificationConflict(f"integrate_quad_level must be 1..{L.APX_MAX_QUAD_LEVEL}")
        x, w = _gl(cp.quad_level)
        cp.gl_node[:cp.quad_level], cp.gl_weight[:cp.quad_level] = x, w
    cp.softening, cp.tolerance = softening, tolerance
    return bytes(cp)


def plan(model, values, window, slot_cols=None, dvdr=None, channels=False, ref_npix=None) -> Plan:
    """Fill the apx_component of ``model`` for sampling ``window``.
    ``ref_npix`` (Sersic): the working-grid pixel count of the window the
    model is nominally sampled on, when only a part of it is rendered."""
    kind = model._profile
    psf_full = "full" in model.psf_mode and kind != "flat_sky"
    window = window.copy()
    cx, cy = values["center"].reshape(-1).tolist()
    P = window._P
    im = model.integrate_mode if kind != "flat_sky" else "none"
    # integrate_radius is in pixels of the model's own window
    radius = float(model.integrate_radius) * math.sqrt(abs(window._area)) if im == "radius" else 0.0
    quad = (int(model.integrate_quad_level), int(model.integrate_gridding), int(model.integrate_max_depth)) if im != "none" \
        else (0, 0, 0)
    try:
        cp = L.Component.from_buffer_copy(_template(kind, model.sampling_mode, im, *quad, radius, float(model.softening),
                                                    float(model.sampling_tolerance)))
    except SpecificationConflict as e:
        raise SpecificationConflict(str(e).replace("{name}", str(model.name))) from None

    shift = None
    upscale = 1
    out_window = window.copy()
    if psf_full:
        psf = model.psf
        if psf is None:
            raise SpecificationConflict(f"{model.name} has psf_mode 'full' but no PSF")
        upscale = psf_upscale(window, psf)
        if upscale != 1:
            # model_object.py:313-314: 1 / psf_upscale of an int32 tensor is a
            # float32 scalar, so the working pixelscale is P * float32(1/U) and
            # the working shape is the floor of the exact quotient n / float32(1/U)
            window = window.rescale_pixel(float(np.float32(1.0 / upscale)))
            # model_object.py:348-349: the block sum lands on that grid rescaled by U
            out_window = window.rescale_pixel(upscale)
            P = window._P
        bx, by = psf.psf_border_int
        window.pad_pixel((bx, by))
        pcx, pcy = window._x2p(cx, cy)
        ci, cj = round(pcx), round(pcy)  # ties to even, as torch.round
        if model.psf_subpixel_shift == "none":
            fx, fy = P[0] * (ci - pcx) + P[1] * (cj - pcy), P[2] * (ci - pcx) + P[3] * (cj - pcy)
        elif model.psf_subpixel_shift == "bilinear":
            shift = (pcx - ci, pcy - cj)
            fx = fy = 0.0
        else:
            raise SpecificationConflict(f"unrecognized subpixel shift method: {model.psf_subpixel_shift}")
    else:
        bx = by = 0
        pcx, pcy = window._x2p(cx, cy)
        ci, cj = round(pcx), round(pcy)
        fx, fy = P[0] * (ci - pcx) + P[1] * (cj - pcy), P[2] * (ci - pcx) + P[3] * (cj - pcy)
    nx, ny = window.nx, window.ny
    cp.nx, cp.ny = nx, ny
    cp.ci, cp.cj = int(ci), int(cj)
    cp.P[:] = P
    cp.frac[0], cp.frac[1] = fx, fy
    cp.pixel_area = window._area
    if kind == "flat_sky":
        cp.q, cp.pa = 1.0, 0.0
    elif getattr(model, "_is_psf", False):
        # PSF models evaluate on untransformed coordinates (psf_model_object.py:
        # 136-137): q = 1 and a position angle on the reference axis make the
        # kernel's rotation the identity
        cp.q, cp.pa = 1.0, math.pi / 2
    else:
        cp.q, cp.pa = float(values["q"]), float(values["PA"])
    for name, slot in PROFILE_SLOTS[kind].items():
        cp.prm[slot - L.APX_P_A] = float(values[name])
    if kind == "sersic":
        cp.mean_reference = 0
        cp.reference = sersic_total_flux(10 ** float(values["Ie"]), float(values["n"]),
                                         float(values["Re"]), float(values["q"])) / (ref_npix or nx * ny)
    else:
        cp.mean_reference = 1
    # Jacobian / adjoint channels: the centre acts through the shifted PSF when
    # psf_mode is "full" with a sub-pixel shift, through X, Y otherwise
    slot_cols = slot_cols or {}
    chan_slots = [s for s in sorted(slot_cols)
                  if not (psf_full and shift is not None and s in (L.APX_P_CX, L.APX_P_CY))]
    cp.nchan = 1 + (len(chan_slots) if channels else 0)
    if channels:
        for c, s in enumerate(chan_slots):
            cp.chan_slot[c + 1] = s
    for s, v in (dvdr or {}).items():
        if s < L.APX_NSLOT:  # an auxiliary PSF model's slots are not this render's
            cp.dvdr[s] = float(v)
    return Plan(cp, window, bx, by, shift, psf_full, chan_slots, upscale, out_window)


def psf_upscale(window, psf) -> int:
    """model_object.py:313: round(window pixel length / PSF pixel length)."""
    U = round(math.sqrt(window._area) / math.sqrt(psf.window._area))
    if U < 1:
        raise SpecificationConflict("PSF pixels must not be larger than the image pixels")
    return U


@dataclass
class Kernels:
    """Convolution kernels of one render: ``ptr`` -> [K] or [K, dK/dcx, dK/dcy]
    (kh x kw each, flipped); ``dk_ptr`` -> [K, dK_0 .. dK_(nd-1), 0] for the
    parameters ``dk_slots`` of an auxiliary PSF model."""

    ptr: int
    kh: int
    kw: int
    view: torch.Tensor
    dk_ptr: Optional[int] = None
    dk_slots: Tuple[int, ...] = ()


def psf_render(psf_model, dev, st, slots=(), dvdr=None):
    """Sample a PSF model on its window and normalise it (psf_model_object.py:
    180-264): (planes (1 + len(slots), ph, pw) float32 view, plane slots)."""
    lib = L.load()
    pl = plan(psf_model, psf_model._values(), psf_model.window, {s: 0 for s in slots}, dvdr or {},
              channels=bool(slots))
    cp = pl.cp
    n = cp.nx * cp.ny
    planes = _buffer(psf_model, "planes", 4 * cp.nchan * n, dev)
    wsb = _render_bytes(n)
    ws = _buffer(psf_model, "render_ws", wsb, dev)
    L.check(lib.apx_render_component(ctypes.byref(cp), L.ptr(planes), L.ptr(ws), wsb, st))
    if psf_model.normalize_psf:
        L.check(lib.apx_normalize_planes(L.ptr(planes), cp.nchan, n, st))
    return planes[:4 * cp.nchan * n].view(torch.float32).view(cp.nchan, cp.ny, cp.nx), pl.chan_slots


def _kernels(model, pl, dvdr, dev, st, psf_slots=()) -> Kernels:
    """Shifted, normalised, flipped PSF (+ centre derivatives, + derivatives
    in the parameters of an auxiliary PSF model) or a unit kernel."""
    lib = L.load()
    if not pl.psf_full:
        k = _unit_kernel(dev)
        return Kernels(L.ptr(k), 1, 1, k)
    aux = model._aux_psf()
    dplanes = None
    psf_slots = tuple(psf_slots) if aux is not None else ()
    if aux is not None:
        pdvdr = {s - PSF_SLOT0: d for s, d in dvdr.items() if s >= PSF_SLOT0}
        planes, chan = psf_render(aux, dev, st, psf_slots, pdvdr)
        psf_slots = tuple(chan)
        pdata = planes[0]
        dplanes = planes[1:] if psf_slots else None
    else:
        pdata = model.psf.data
        if pdata.dtype != torch.float32 or not pdata.is_contiguous():
            pdata = pdata.to(torch.float32).contiguous()
    ph, pw = int(pdata.shape[0]), int(pdata.shape[1])
    shifted = pl.shift is not None
    kh, kw = (ph + 2, pw + 2) if shifted else (ph, pw)
    sx, sy = pl.shift if shifted else (0.0, 0.0)
    dk_ptr = None
    if not shifted or psf_slots:
        nd = len(psf_slots)
        dbuf = _buffer(model, "dkernels", 4 * (nd + 2) * kh * kw, dev)
        L.check(lib.apx_psf_kernels_dparam(L.ptr(pdata), L.ptr(dplanes) if nd else 0, nd, ph, pw,
                                           1 if shifted else 0, sx, sy, L.ptr(dbuf), st))
        dk_ptr = L.ptr(dbuf)
    if shifted:
        kbuf = _buffer(model, "kernels", 4 * 3 * kh * kw, dev)
        pinv = (ctypes.c_double * 4)(*pl.window._Pi)
        L.check(lib.apx_psf_shift(L.ptr(pdata), ph, pw, sx, sy, pinv,
                                  float(dvdr.get(L.APX_P_CX, 1.0)), float(dvdr.get(L.APX_P_CY, 1.0)),
                                  L.ptr(kbuf), st))
        view = kbuf[:4 * 3 * kh * kw].view(torch.float32).view(3, kh, kw)
        return Kernels(L.ptr(kbuf), kh, kw, view, dk_ptr, psf_slots)
    view = dbuf[:4 * kh * kw].view(torch.float32).view(1, kh, kw)
    return Kernels(dk_ptr, kh, kw, view, dk_ptr, psf_slots)


def _dk_pairs(kern: Kernels, psf_cols):
    """(kernel pointer, (column, column)) per pair of auxiliary-PSF columns."""
    plane = 4 * kern.kh * kern.kw
    out = []
    for k in range(0, len(kern.dk_slots), 2):
        c0 = psf_cols[kern.dk_slots[k]]
        c1 = psf_cols[kern.dk_slots[k + 1]] if k + 1 < len(kern.dk_slots) else -1
        out.append((kern.dk_ptr + k * plane, (c0, c1)))
    return out


_NO_CHAN, _NO_DK = (-1,) * L.APX_MAX_CHAN, (-1, -1)


def _new_job(pl, kh, kw):
    job = L.ConvJob()
    job.nx, job.ny, job.nchan, job.kh, job.kw = pl.cp.nx, pl.cp.ny, pl.cp.nchan, kh, kw
    job.chan_col[:] = _NO_CHAN
    job.dk_col[:] = _NO_DK
    return job


def _sampled_part(model, req: RenderRequest):
    """The window actually rendered, and the Sersic threshold's pixel count.

    A component of a group is sampled on the whole group window and kept on
    its own (group_model_object.py:183-231, model_object.py:258-375).  On the
    kept pixels that equals sampling just the kept region plus what reaches
    it: the PSF border (psf_mode "full") or one pixel for the curvature
    stencil, clipped to the window, as long as the integration threshold
    still divides the Sersic flux by the whole window's working-grid pixel
    count (sersic_model.py:87-89).  Other profiles take the mean of the whole
    grid as the threshold reference and are rendered on the whole window."""
    region = req.region
    w = req.window
    if region is None or model._profile != "sersic" or getattr(model, "_is_psf", False) or req.jac is not None:
        return w, None
    if "full" in model.psf_mode and model.psf is not None and psf_upscale(w, model.psf) != 1:
        return w, None
    part = region & w
    if part.nx * part.ny >= w.nx * w.ny:
        return w, None
    if "full" in model.psf_mode:
        bx, by = model.psf.psf_border_int
    else:
        part = part.copy()
        part.pad_pixel((1, 1))
        part = part & w
        bx = by = 0
    if part.nx < 3 or part.ny < 3:
        return w, None
    return part, (w.nx + 2 * bx) * (w.ny + 2 * by)


def render(model, values: Dict[str, torch.Tensor], req: RenderRequest):
    """Render ``model`` with parameter ``values`` (host float64) on
    ``req.window``; accumulate into ``req.image`` / ``req.jac``."""
    lib = L.load()
    dvdr = req.dvdr or {}
    all_cols = req.slot_cols or {}
    slot_cols = {s: c for s, c in all_cols.items() if s < PSF_SLOT0}
    psf_cols = {s - PSF_SLOT0: c for s, c in all_cols.items() if s >= PSF_SLOT0}
    sample_window, ref_npix = _sampled_part(model, req)
    pl = plan(model, values, sample_window, slot_cols, dvdr, channels=req.jac is not None, ref_npix=ref_npix)
    cp, nx, ny = pl.cp, pl.cp.nx, pl.cp.ny
    dev = AP_config.ap_device
    planes = _buffer(model, "planes", 4 * cp.nchan * ny * nx, dev)
    wsb = _render_bytes(nx * ny)
    ws = _buffer(model, "render_ws", wsb, dev)
    st = L.stream()
    _launch("render", nx * ny, lambda: L.check(
        lib.apx_render_component(ctypes.byref(cp), L.ptr(planes), L.ptr(ws), wsb, st)))
    if getattr(model, "_is_psf", False) and model.normalize_psf:
        L.check(lib.apx_normalize_planes(L.ptr(planes), cp.nchan, nx * ny, st))
    kern = _kernels(model, pl, dvdr, dev, st, sorted(psf_cols) if req.jac is not None else ())
    kptr, kh, kw = kern.ptr, kern.kh, kern.kw
    # crop back to the sampling window, then window-aware accumulation
    cwsb = _convolve_bytes(kh, kw)
    cws = _buffer(model, "conv_ws", cwsb, dev)
    job = _new_job(pl, kh, kw)
    bx, by, U, out_w = pl.bx, pl.by, pl.upscale, pl.out_window
    if req.image is not None:
        # default: the part of the image the sampling window covers
        region = req.region if req.region is not None else (req.image.window & out_w)
        (dy, dx), (sy, sx), (h, w) = _box(req.image.window, out_w, region)
        img = req.image.data
        if img.dtype != torch.float32 or not img.is_contiguous():
            raise SpecificationConflict("model image must be contiguous float32")
        j1 = job if req.jac is None else _job_copy(job)
        j1.nchan = 1
        j1.x0, j1.y0, j1.ow, j1.oh = bx + U * sx, by + U * sy, U * w, U * h
        if U == 1:
            j1.img, j1.img_row, j1.img_x0, j1.img_y0 = L.ptr(img), img.shape[1], dx, dy
            j1.img_w, j1.img_h = img.shape[1], img.shape[0]
        elif h > 0 and w > 0:
            fine = _fine(model, "fine_img", (U * h, U * w, 1), dev)
            j1.img, j1.img_row, j1.img_x0, j1.img_y0, j1.img_w, j1.img_h = L.ptr(fine), U * w, 0, 0, U * w, U * h
        if h > 0 and w > 0:
            _launch("convolve", 2.0 * kh * kw * h * w * U * U, lambda: L.check(
                lib.apx_convolve(ctypes.byref(j1), L.ptr(planes), kptr, L.ptr(cws), cwsb, st)))
            if U != 1:
                _block_sum(lib, fine, U, (h, w), img, 1, (dx, dy), [0], st)
    if req.jac is not None and (slot_cols or psf_cols):
        # default: the part of the Jacobian the sampling window covers (a
        # component on a sub-window of a group's Jacobian lands at its own pixels)
        region = req.region if req.region is not None else (req.jac.window & out_w)
        (dy, dx), (sy, sx), (h, w) = _box(req.jac.window, out_w, region)
        jd = req.jac.data
        if not jd.is_contiguous() or jd.dtype != torch.float32:
            raise SpecificationConflict("Jacobian must be contiguous float32")
        npj = int(jd.shape[2])
        centre_dk = pl.psf_full and pl.shift is not None
        dest = [slot_cols[s] for s in pl.chan_slots]
        if centre_dk:
            dest += [slot_cols[s] for s in (L.APX_P_CX, L.APX_P_CY) if s in slot_cols]
        dest += [psf_cols[s] for s in sorted(psf_cols)]
        # the columns this render writes: in place, or through a fine-grid
        # buffer holding just them when the PSF is upscaled
        col = {c: c for c in dest} if U == 1 else {c: k for k, c in enumerate(dest)}
        col[-1] = -1
        j2 = _job_copy(job)
        j2.x0, j2.y0, j2.ow, j2.oh = bx + U * sx, by + U * sy, U * w, U * h
        if U == 1:
            j2.jac, j2.jac_row, j2.jac_np, j2.jac_x0, j2.jac_y0 = L.ptr(jd), jd.shape[1] * npj, npj, dx, dy
            j2.jac_w, j2.jac_h = jd.shape[1], jd.shape[0]
        elif h > 0 and w > 0:
            if len(dest) > L.APX_MAX_BLOCK_COLS:
                raise SpecificationConflict(f"an upscaled render writes at most {L.APX_MAX_BLOCK_COLS} columns")
            fine = _fine(model, "fine_jac", (U * h, U * w, len(dest)), dev)
            j2.jac, j2.jac_row, j2.jac_np, j2.jac_x0, j2.jac_y0 = L.ptr(fine), U * w * len(dest), len(dest), 0, 0
            j2.jac_w, j2.jac_h = U * w, U * h
        for c, s in enumerate(pl.chan_slots):
            j2.chan_col[c + 1] = col[slot_cols[s]]
        if centre_dk:
            j2.dk_col[0] = col[slot_cols.get(L.APX_P_CX, -1)]
            j2.dk_col[1] = col[slot_cols.get(L.APX_P_CY, -1)]
        nk = (cp.nchan - 1) + (2 if j2.dk_col[0] >= 0 or j2.dk_col[1] >= 0 else 0)
        if h > 0 and w > 0 and nk > 0:
            _launch("convolve_jac", 2.0 * kh * kw * h * w * nk * U * U, lambda: L.check(
                lib.apx_convolve(ctypes.byref(j2), L.ptr(planes), kptr, L.ptr(cws), cwsb, st)))
        # auxiliary PSF parameters: conv(value plane, dK/dtheta), two columns a launch
        for ptr, (c0, c1) in (_dk_pairs(kern, psf_cols) if h > 0 and w > 0 else ()):
            j3 = _job_copy(j2)
            j3.nchan = 1
            j3.chan_col[:] = [-1] * L.APX_MAX_CHAN
            j3.dk_col[0], j3.dk_col[1] = col[c0], col[c1]
            _launch("convolve_jac", 2.0 * kh * kw * h * w * 2 * U * U, lambda: L.check(
                lib.apx_convolve(ctypes.byref(j3), L.ptr(planes), ptr, L.ptr(cws), cwsb, st)))
        if U != 1 and h > 0 and w > 0:
            _block_sum(lib, fine, U, (h, w), jd, npj, (dx, dy), dest, st)
    return ws


def vjp(model, values, window, G, G_window, slot_cols, dvdr, region=None):
    """Hand-written adjoint of ``render`` (value image only): returns
    {column: sum over pixels of G * d image / d rep(column)} for the columns
    in ``slot_cols``, as float64 device scalars in one tensor indexed like
    ``sorted(slot_cols.values())``.

    G (float32, G_window's shape) is carried back through the convolution
    (correlation with the unflipped shifted PSF), then apx_render_vjp
    recomputes the render and reduces against it; the centre columns of a
    shifted-PSF model, and the parameters of an auxiliary PSF model, are
    sum(G * conv(deep, dK)) with dK the kernel's derivative."""
    lib = L.load()
    dev = AP_config.ap_device
    st = L.stream()
    all_cols = slot_cols
    slot_cols = {s: c for s, c in all_cols.items() if s < PSF_SLOT0}
    psf_cols = {s - PSF_SLOT0: c for s, c in all_cols.items() if s >= PSF_SLOT0}
    pl = plan(model, values, window, slot_cols, dvdr, channels=True)
    cp, nx, ny, bx, by, U = pl.cp, pl.cp.nx, pl.cp.ny, pl.bx, pl.by, pl.upscale
    region = G_window if region is None else region
    (dy, dx), (sy, sx), (h, w) = _box(G_window, pl.out_window, region)
    out = torch.zeros(len(all_cols), dtype=torch.float64, device=dev)
    col_index = {c: k for k, c in enumerate(sorted(all_cols.values()))}
    if h <= 0 or w <= 0:
        return out, col_index
    # the adjoint of the U x U block sum gives every fine pixel of a block its
    # coarse pixel's G
    Gc = G[dy:dy + h, dx:dx + w]
    if U != 1:
        Gc = Gc.repeat_interleave(U, dim=0).repeat_interleave(U, dim=1)
    sx, sy, h, w = U * sx, U * sy, U * h, U * w
    Gw = torch.zeros((ny, nx), dtype=torch.float32, device=dev)
    Gw[by + sy:by + sy + h, bx + sx:bx + sx + w] = Gc
    kern = _kernels(model, pl, dvdr, dev, st, sorted(psf_cols))
    kh, kw = kern.kh, kern.kw
    cwsb = _convolve_bytes(kh, kw)
    cws = _buffer(model, "conv_ws", cwsb, dev)
    if pl.psf_full:
        # B = adjoint of the convolution: correlation with the unflipped taps
        taps = torch.flip(kern.view[0], dims=(0, 1)).contiguous()
        B = torch.zeros((ny, nx), dtype=torch.float32, device=dev)
        jb = _new_job(pl, kh, kw)
        jb.nchan = 1
        jb.x0, jb.y0, jb.ow, jb.oh = 0, 0, nx, ny
        jb.img, jb.img_row, jb.img_w, jb.img_h, jb.img_x0, jb.img_y0 = L.ptr(B), nx, nx, ny, 0, 0
        jb.zero_outside = 1
        L.check(lib.apx_convolve(ctypes.byref(jb), L.ptr(Gw), L.ptr(taps), L.ptr(cws), cwsb, st))
    else:
        B = Gw
    value = _buffer(model, "planes", 4 * ny * nx, dev)
    wsb = _render_bytes(nx * ny)
    ws = _buffer(model, "render_ws", wsb, dev)
    centre_dk = pl.psf_full and pl.shift is not None and (L.APX_P_CX in slot_cols or L.APX_P_CY in slot_cols)
    psf_dk = pl.psf_full and bool(kern.dk_slots) and bool(psf_cols)
    if cp.nchan > 1:
        g = torch.empty(cp.nchan - 1, dtype=torch.float64, device=dev)
        L.check(lib.apx_render_vjp(ctypes.byref(cp), L.ptr(B), L.ptr(value), L.ptr(g), L.ptr(ws), wsb, st))
        for c, s in enumerate(pl.chan_slots):
            out[col_index[slot_cols[s]]] += g[c]
    elif centre_dk or psf_dk:
        L.check(lib.apx_render_component(ctypes.byref(cp), L.ptr(value), L.ptr(ws), wsb, st))
    pairs = []
    if centre_dk:
        pairs.append((kern.ptr, (slot_cols.get(L.APX_P_CX, -1), slot_cols.get(L.APX_P_CY, -1))))
    if psf_dk:
        pairs.extend(_dk_pairs(kern, psf_cols))
    if pairs:
        Gb = Gc.double()
        C = torch.empty((h, w, 2), dtype=torch.float32, device=dev)
        for ptr, cols in pairs:
            C.zero_()
            jc = _new_job(pl, kh, kw)
            jc.nchan = 1
            jc.x0, jc.y0, jc.ow, jc.oh = bx + sx, by + sy, w, h
            jc.jac, jc.jac_row, jc.jac_w, jc.jac_h, jc.jac_np, jc.jac_x0, jc.jac_y0 = L.ptr(C), 2 * w, w, h, 2, 0, 0
            jc.dk_col[0], jc.dk_col[1] = (0 if cols[0] >= 0 else -1), (1 if cols[1] >= 0 else -1)
            L.check(lib.apx_convolve(ctypes.byref(jc), L.ptr(value), ptr, L.ptr(cws), cwsb, st))
            for k in range(2):
                if cols[k] >= 0:
                    out[col_index[cols[k]]] += (Gb * C[..., k].double()).sum()
    return out, col_index


def _fine(model, name, shape, dev):
    """A zeroed float32 buffer of ``shape`` on the fine (PSF-upscaled) grid."""
    n = shape[0] * shape[1] * shape[2]
    buf = _buffer(model, name, 4 * n, dev)[:4 * n].view(torch.float32).view(*shape)
    buf.zero_()
    return buf


def _block_sum(lib, fine, U, hw, dst, dst_pix, dxy, cols, st):
    """Sum the U x U blocks of ``fine`` (fine rows x fine cols x len(cols))
    into ``dst`` (rows x cols x dst_pix, or rows x cols) at pixel ``dxy``,
    channel k into offset cols[k] (image_object.py:348-376, 450-457)."""
    job = L.BlockSum()
    job.scale, job.nc, job.h, job.w = U, len(cols), hw[0], hw[1]
    job.src_h, job.src_w = int(fine.shape[0]), int(fine.shape[1])
    job.dst, job.dst_pix = L.ptr(dst), dst_pix
    job.dst_h, job.dst_w = int(dst.shape[0]), int(dst.shape[1])
    job.dst_row = int(dst.shape[1]) * dst_pix
    job.dst_x0, job.dst_y0 = dxy
    job.col[:len(cols)] = list(cols)
    L.check(lib.apx_block_sum_add(ctypes.byref(job), L.ptr(fine), st))


def _job_copy(job):
    j = L.ConvJob()
    ctypes.pointer(j)[0] = job
    return j
