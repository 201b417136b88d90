"""Batched independent fits: many cutouts, one Sersic each, fitted together on
one GPU by the device-resident Levenberg-Marquardt of ``csrc/batch.hip``.

Each cutout is what a reference user would fit with

    tgt = ap.image.Target_Image(data=d, pixelscale=ps, variance=v, psf=psf, origin=o)
    m = ap.models.AstroPhot_Model(model_type="sersic galaxy model", target=tgt,
                                  psf_mode="full", parameters=p0)
    ap.fit.LM(m).fit()

and the batch gives every cutout that result (same render, same LM control
flow, fit/lm.py:248-493), all cutouts at once: one tick is one LM sub-step of
every unfinished fit; a tick is captured in a HIP graph and replayed.
"""

from __future__ import annotations

import ctypes
import math
from dataclasses import dataclass
from typing import Dict, List, Optional, Sequence

import numpy as np
import torch

from . import AP_config
from . import _lib as L
from .errors import SpecificationConflict

NP = 7
PARAM_NAMES = ("center_x", "center_y", "q", "PA", "n", "Re", "Ie")
STATUS = {0: "running", 1: "success", 2: "success by immobility. Convergence not guaranteed",
          3: "fail. Could not find step to improve Chi^2", 4: "fail. Maximum iterations", 5: "skipped"}


CONV_IMPL = {0: "default", 1: "valu", 2: "mfma", 3: "sep"}


def rank_one_factors(psfs, rtol: float = 1e-6):
    """(u, v) with psf = outer(u, v) to ``rtol`` of the PSF's largest value,
    or None, for each PSF: the skeleton through the largest element,
    u = P[:, c*], v = P[r*, :] / P[r*, c*], which reproduces a rank-one image
    exactly and is checked against the image itself."""
    out = [None] * len(psfs)
    groups: Dict[tuple, List[int]] = {}
    for k, p in enumerate(psfs):
        groups.setdefault(tuple(np.shape(p)), []).append(k)
    for (h, w), idx in groups.items():
        P = np.stack([np.asarray(psfs[k], dtype=np.float64) for k in idx])      # (m, h, w)
        flat = np.abs(P).reshape(len(idx), -1).argmax(axis=1)
        r, c = flat // w, flat % w
        m = np.arange(len(idx))
        piv = P[m, r, c]
        safe = np.where(piv == 0, 1.0, piv)
        u = P[m, :, c]                                                          # (m, h)
        v = P[m, r, :] / safe[:, None]                                          # (m, w)
        err = np.abs(u[:, :, None] * v[:, None, :] - P).reshape(len(idx), -1).max(axis=1)
        ok = (piv != 0) & (err <= rtol * np.abs(piv))
        for j, k in enumerate(idx):
            if ok[j]:
                out[k] = (u[j], v[j])
    return out


class Galaxy(ctypes.Structure):
    """apx_batch_galaxy."""

    _fields_ = [("nx", ctypes.c_int32), ("ny", ctypes.c_int32), ("ph", ctypes.c_int32), ("pw", ctypes.c_int32),
                ("pix_off", ctypes.c_int64), ("psf_off", ctypes.c_int64), ("work_off", ctypes.c_int64),
                ("tap_off", ctypes.c_int64), ("chunk_off", ctypes.c_int64), ("tile_off", ctypes.c_int64),
                ("origin", ctypes.c_double * 2), ("ref_npix", ctypes.c_int64), ("sep_off", ctypes.c_int64)]


class Batch(ctypes.Structure):
    """apx_batch."""

    _p = ctypes.c_void_p
    _fields_ = [("ngal", ctypes.c_int32), ("max_kernel", ctypes.c_int32),
                ("npix", ctypes.c_int64), ("nwork", ctypes.c_int64), ("nchunk", ctypes.c_int64),
                ("ntile", ctypes.c_int64), ("ntap", ctypes.c_int64),
                ("P", ctypes.c_double * 4), ("softening", ctypes.c_double), ("tolerance", ctypes.c_double),
                ("quad_level", ctypes.c_int32), ("gridding", ctypes.c_int32), ("max_depth", ctypes.c_int32),
                ("max_iter", ctypes.c_int32), ("relative_tolerance", ctypes.c_double), ("L0", ctypes.c_double),
                ("gal", _p), ("data", _p), ("weight", _p), ("psf", _p), ("psf_sep", _p), ("model0", _p),
                ("model1", _p),
                ("jac", _p), ("planes", _p), ("taps", _p), ("state", _p), ("scratch", _p),
                ("conv_impl", ctypes.c_int32), ("conv_blocks", ctypes.c_int32), ("quad_blocks", ctypes.c_int32),
                ("quad_group", ctypes.c_int32), ("chunk_blocks", ctypes.c_int32), ("sep_all", ctypes.c_int32),
                ("quad_group_value", ctypes.c_int32)]


SIGNATURES = {
    "apx_batch_plan": (ctypes.c_int, [ctypes.POINTER(Galaxy), ctypes.c_int32, ctypes.POINTER(Batch)]),
    "apx_batch_state_bytes": (ctypes.c_int64, []),
    "apx_batch_scratch_bytes": (ctypes.c_int64, [ctypes.POINTER(Batch)]),
    "apx_batch_render": (ctypes.c_int, [ctypes.POINTER(Batch), ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int32,
                                        ctypes.c_void_p]),
    "apx_batch_jacobian": (ctypes.c_int, [ctypes.POINTER(Batch), ctypes.c_void_p, ctypes.c_void_p,
                                          ctypes.c_int32, ctypes.c_void_p]),
    "apx_batch_moment_init": (ctypes.c_int, [ctypes.POINTER(Batch), ctypes.c_void_p, ctypes.c_void_p]),
    "apx_sersic_light_fraction": (ctypes.c_double, [ctypes.c_double, ctypes.c_double]),
    "apx_batch_start": (ctypes.c_int, [ctypes.POINTER(Batch), ctypes.c_void_p, ctypes.c_void_p]),
    "apx_batch_tick": (ctypes.c_int, [ctypes.POINTER(Batch), ctypes.c_void_p]),
    "apx_batch_results": (ctypes.c_int, [ctypes.POINTER(Batch)] + [ctypes.c_void_p] * 7),
    "apx_batch_start_fallback": (ctypes.c_int, [ctypes.POINTER(Batch), ctypes.c_void_p, ctypes.c_void_p,
                                                ctypes.c_void_p]),
    "apx_batch_counters": (ctypes.c_int, [ctypes.POINTER(Batch), ctypes.c_void_p, ctypes.c_void_p]),
}
L.register(SIGNATURES)


@dataclass
class Cutout:
    """One fit: data and variance (ny, nx), PSF (odd, unit sum) and the plane
    coordinates of the cutout's corner (pixel -0.5, -0.5)."""

    data: np.ndarray
    variance: np.ndarray
    psf: np.ndarray
    origin: Sequence[float] = (0.0, 0.0)


def values_to_rep(v: np.ndarray) -> np.ndarray:
    """[cx, cy, q, PA, n, Re, Ie] values -> representation
    (utils/conversions/optimization.py:6-14, 50-54)."""
    v = np.asarray(v, dtype=np.float64)
    r = v.copy()
    r[..., 2] = np.tan((v[..., 2] - 0.0) * np.pi / 1.0 - np.pi / 2)
    r[..., 3] = np.mod(v[..., 3], np.pi)
    r[..., 4] = np.tan((v[..., 4] - 0.36) * np.pi / (8.0 - 0.36) - np.pi / 2)
    r[..., 5] = v[..., 5] - 1.0 / (v[..., 5] - 0.0)
    return r


def values_to_rep_device(v: torch.Tensor) -> torch.Tensor:
    """``values_to_rep`` on a float64 device tensor."""
    r = v.clone()
    r[..., 2] = torch.tan((v[..., 2] - 0.0) * math.pi / 1.0 - math.pi / 2)
    r[..., 3] = torch.remainder(v[..., 3], math.pi)
    r[..., 4] = torch.tan((v[..., 4] - 0.36) * math.pi / (8.0 - 0.36) - math.pi / 2)
    r[..., 5] = v[..., 5] - 1.0 / (v[..., 5] - 0.0)
    return r


def rep_to_values(r: np.ndarray) -> np.ndarray:
    """Inverse of ``values_to_rep`` (optimization.py:17-25, 50-54)."""
    r = np.asarray(r, dtype=np.float64)
    v = r.copy()
    v[..., 2] = (np.arctan(r[..., 2]) + np.pi / 2) * 1.0 / np.pi
    v[..., 3] = np.mod(r[..., 3], np.pi)
    v[..., 4] = (np.arctan(r[..., 4]) + np.pi / 2) * (8.0 - 0.36) / np.pi + 0.36
    v[..., 5] = (r[..., 5] + np.sqrt(r[..., 5] ** 2 + 4)) * 0.5
    return v


def conv_grids(ntile: int, impl: int) -> List[int]:
    """Workgroup counts to time for a convolution: no more than it has work items, a
    tile each, or for the MFMA kernel (2) one of the 7 passes of a tile."""
    items = ntile * (7 if impl == 2 else 1)
    return sorted({min(c, items) for c in (1024, 2048, 4096, 8192, 16384)})


class BatchFit:
    """All cutouts resident on the GPU; ``fit(rep0)`` runs every LM to the end."""

    def __init__(self, cutouts: List[Cutout], pixelscale=1.0, max_iter=100, relative_tolerance=1e-5, L0=1.0,
                 sampling_tolerance=1e-2, softening=1e-3, integrate_quad_level=3, integrate_gridding=5,
                 integrate_max_depth=3, data=None, variance=None):
        self.lib = L.load()
        dev = AP_config.ap_device
        ng = len(cutouts)
        if ng == 0:
            raise SpecificationConflict("BatchFit needs at least one cutout")
        self.cutouts = cutouts
        gal = (Galaxy * ng)()
        for k, c in enumerate(cutouts):
            ny, nx = np.shape(c.data)
            ph, pw = np.shape(c.psf)
            gal[k].nx, gal[k].ny, gal[k].ph, gal[k].pw = nx, ny, ph, pw
            gal[k].origin[0], gal[k].origin[1] = float(c.origin[0]), float(c.origin[1])
        b = Batch()
        L.check(self.lib.apx_batch_plan(gal, ng, ctypes.byref(b)))
        P = torch.as_tensor(pixelscale, dtype=torch.float64).reshape(-1)
        if P.numel() == 1:
            P = torch.tensor([P.item(), 0.0, 0.0, P.item()], dtype=torch.float64)
        b.P[:] = [float(x) for x in P]
        b.softening, b.tolerance = softening, sampling_tolerance
        b.quad_level, b.gridding, b.max_depth = integrate_quad_level, integrate_gridding, integrate_max_depth
        b.max_iter, b.relative_tolerance, b.L0 = max_iter, relative_tolerance, L0
        # rank-one factors of every PSF that has them (the separable convolution)
        factors = rank_one_factors([c.psf for c in cutouts])
        self.sep_all = all(f is not None for f in factors)
        if self.sep_all:
            off = 0
            for k, (u, v) in enumerate(factors):
                gal[k].sep_off = off
                off += len(u) + len(v)
            self.psf_sep = torch.as_tensor(np.concatenate([np.concatenate(f) for f in factors]),
                                           dtype=torch.float32).to(dev)
            b.psf_sep, b.sep_all = self.psf_sep.data_ptr(), 1
        self.gal_host = gal
        # cutout origins (ngal x 2) as an array: reading them back from the
        # ctypes records costs about a microsecond per cutout
        self.origins = np.array([[float(c.origin[0]), float(c.origin[1])] for c in cutouts], dtype=np.float64)
        self.origins_dev = torch.as_tensor(self.origins, device=dev)
        f32 = dict(dtype=torch.float32, device=dev)
        self.gal_dev = torch.frombuffer(bytearray(gal), dtype=torch.uint8).to(dev)
        if data is not None:  # flat device arrays in cutout order
            self.data = torch.as_tensor(data, dtype=torch.float32, device=dev).reshape(-1).contiguous()
            self.weight = (1.0 / torch.as_tensor(variance, device=dev).double()).to(torch.float32).reshape(-1)
            if self.data.numel() != b.npix or self.weight.numel() != b.npix:
                raise SpecificationConflict("flat data / variance do not match the cutout sizes")
        else:
            self.data = torch.cat([torch.as_tensor(c.data, dtype=torch.float32).reshape(-1)
                                   for c in cutouts]).to(dev)
            self.weight = torch.cat([(1.0 / torch.as_tensor(c.variance, dtype=torch.float64)).to(torch.float32)
                                     .reshape(-1) for c in cutouts]).to(dev)
        self.psf = torch.cat([torch.as_tensor(c.psf, dtype=torch.float32).reshape(-1) for c in cutouts]).to(dev)

        self.model0 = torch.zeros(b.npix, **f32)
        self.model1 = torch.zeros(b.npix, **f32)
        self.jac = torch.zeros(b.npix * NP, **f32)
        self.planes = torch.zeros(6 * b.nwork, **f32)
        self.taps = torch.zeros(b.ntap, **f32)
        self.state = torch.zeros(ng * self.lib.apx_batch_state_bytes(), dtype=torch.uint8, device=dev)
        for name in ("gal", "data", "weight", "psf", "model0", "model1", "jac", "planes", "taps", "state"):
            src = self.gal_dev if name == "gal" else getattr(self, name)
            setattr(b, name, src.data_ptr())
        self.scratch = torch.zeros(self.lib.apx_batch_scratch_bytes(ctypes.byref(b)), dtype=torch.uint8, device=dev)
        b.scratch = self.scratch.data_ptr()
        self.b = b
        self.ngal = ng
        self.npix = b.npix
        self._rep = torch.zeros((ng, NP), dtype=torch.float64, device=dev)
        self._chi2 = torch.zeros(ng, dtype=torch.float64, device=dev)
        self._status = torch.zeros(ng, dtype=torch.int32, device=dev)
        self._iters = torch.zeros(ng, dtype=torch.int32, device=dev)
        self._fbran = torch.zeros(ng, dtype=torch.int32, device=dev)
        self._done = torch.zeros(1, dtype=torch.int32, device=dev)
        self.graph = None
        self.ticks = 0

    # -- rendering --------------------------------------------------------
    def render(self, rep, out=None, parts=3) -> torch.Tensor:
        """All cutouts rendered at ``rep`` (ngal x 7, representation) into one
        flat float32 tensor (cutouts concatenated row-major).  ``parts``: 1 =
        working planes only, 2 = convolution of the planes of a previous
        parts=1 call, 3 = both."""
        rep = torch.as_tensor(rep, dtype=torch.float64, device=self.data.device).contiguous()
        self._render_rep = rep
        if out is None:
            out = torch.zeros(self.npix, dtype=torch.float32, device=self.data.device)
        L.check(self.lib.apx_batch_render(ctypes.byref(self.b), rep.data_ptr(), out.data_ptr(), parts,
                                          L.stream()))
        return out

    def jacobian(self, rep, out=None, parts=3):
        """All cutouts rendered at ``rep`` into ``out`` (as render) and their
        Jacobians with respect to the 7 representation-space parameters,
        returned as an (npix, 7) view of the batch's J buffer (stored
        parameter-major, 7 x npix, cutouts concatenated).  ``parts`` as in render.  The LM state of the
        fits is left untouched."""
        rep = torch.as_tensor(rep, dtype=torch.float64, device=self.data.device).contiguous()
        self._render_rep = rep
        if out is None:
            out = torch.zeros(self.npix, dtype=torch.float32, device=self.data.device)
        L.check(self.lib.apx_batch_jacobian(ctypes.byref(self.b), rep.data_ptr(), out.data_ptr(), parts,
                                            L.stream()))
        return out, self.jac.view(NP, self.npix).t()

    def moment_init(self) -> torch.Tensor:
        """Moment-based starting parameters of every cutout from its data
        (ngal x 7, representation space, float64 on the device)."""
        rep = torch.empty((len(self.gal_host), NP), dtype=torch.float64, device=self.data.device)
        L.check(self.lib.apx_batch_moment_init(ctypes.byref(self.b), rep.data_ptr(), L.stream()))
        return rep

    # -- launch-shape autotuning ---------------------------------------------
    def _time(self, fn, n=4, skip=1) -> float:
        evs = []
        for _ in range(n):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            fn()
            b.record()
            evs.append((a, b))
        torch.cuda.synchronize()
        return float(np.mean([a.elapsed_time(b) for a, b in evs[skip:]]))

    def autotune(self, rep=None) -> Dict:
        """Pick the launch shape of this batch by timing candidates on it (HIP
        events on the launch stream), one stage at a time:
          convolution  VALU or MFMA kernel x workgroup count, on the Jacobian-
                       stage convolution of every cutout (the costliest launch);
          quadrature   lanes per refined pixel (32 or 64, or one lane per
                       level-2 sub-pixel with 10 pixels a workgroup: 25) x
                       workgroup count on the Jacobian stage, then the lane
                       grouping of the value-only renders on the first 16
                       LM ticks of every fit,
          chunks       workgroup count of the per-chunk render kernels,
                       both on the Jacobian-stage render planes.
        The winners stay in the batch descriptor for every later render, Jacobian
        and LM tick; returns them with the timings (ms)."""
        if rep is None:
            rep = getattr(self, "_render_rep", None)
        if rep is None:
            raise SpecificationConflict("autotune needs parameters to render at")
        rep = torch.as_tensor(rep, dtype=torch.float64, device=self.data.device).contiguous()
        out = torch.zeros(self.npix, dtype=torch.float32, device=self.data.device)
        b = self.b
        log = {"conv": {}, "quad": {}, "quad_value": {}, "chunk": {}}
        self.jacobian(rep, out=out, parts=1)
        impls = [1] + ([2] if b.max_kernel <= 67 else []) + ([3] if self.sep_all and b.max_kernel <= 61 else [])
        best = None
        for impl in impls:
            for blocks in conv_grids(int(b.ntile), impl):
                b.conv_impl, b.conv_blocks = impl, blocks
                ms = self._time(lambda: self.jacobian(rep, out=out, parts=2))
                log["conv"][f"{CONV_IMPL[impl]}:{blocks}"] = ms
                if best is None or ms < best[0]:
                    best = (ms, impl, blocks)
        b.conv_impl, b.conv_blocks = best[1], best[2]
        groups = [0] + ([64] if b.gridding * b.gridding <= 32 else []) + \
            ([25] if (b.quad_level, b.gridding) == (3, 5) else [])
        best = None
        for grp in groups:
            for blocks in (512, 1024, 2048, 4096):
                b.quad_group, b.quad_blocks = grp, blocks
                ms = self._time(lambda: self.jacobian(rep, out=out, parts=1))
                log["quad"][f"{grp or (32 if b.gridding * b.gridding <= 32 else 64)}:{blocks}"] = ms
                if best is None or ms < best[0]:
                    best = (ms, grp, blocks)
        b.quad_group, b.quad_blocks = best[1], best[2]
        # the value-only renders (LM probe and trial points) pick their own
        # grouping, timed on what they render in a fit: the first 16 LM ticks
        # of every fit from rep (each candidate from the same start)
        best = None
        for grp in groups:
            b.quad_group_value = grp if grp else (32 if b.gridding * b.gridding <= 32 else 64)

            def ticks():
                self.start(rep)
                for _ in range(16):
                    self.tick()

            ms = self._time(ticks, n=3, skip=1)
            log["quad_value"][str(b.quad_group_value)] = ms
            if best is None or ms < best[0]:
                best = (ms, b.quad_group_value)
        b.quad_group_value = best[1]
        best = None
        for blocks in sorted({min(c, int(b.nchunk)) for c in (2048, 4096, 8192, 16384)}):
            b.chunk_blocks = blocks
            ms = self._time(lambda: self.jacobian(rep, out=out, parts=1))
            log["chunk"][str(blocks)] = ms
            if best is None or ms < best[0]:
                best = (ms, blocks)
        b.chunk_blocks = best[1]
        self.graph = None  # a captured tick holds the old launch shape
        choice = {"conv_impl": CONV_IMPL[b.conv_impl], "conv_blocks": b.conv_blocks,
                  "quad_group": b.quad_group or (32 if b.gridding * b.gridding <= 32 else 64),
                  "quad_group_value": b.quad_group_value,
                  "quad_blocks": b.quad_blocks, "chunk_blocks": b.chunk_blocks}
        self.tuning = {"choice": choice, "timings_ms": log}
        return self.tuning

    def counters(self) -> Dict[str, int]:
        """Work counters of the last render / Jacobian stage (apx_batch_counters)."""
        out = torch.zeros(8, dtype=torch.int32, device=self.data.device)
        L.check(self.lib.apx_batch_counters(ctypes.byref(self.b), out.data_ptr(), L.stream()))
        c = out.cpu().tolist()
        return {"fits": c[0], "chunks": c[1], "tiles": c[2], "refined": c[3], "undecided_select": c[4],
                "redone": c[5], "level3_float": c[6], "level3_double": c[7]}

    def quad_evaluations(self, counts: Dict[str, int]) -> int:
        """Profile evaluations of the float32 level-2/3 quadrature pass."""
        per = (self.b.gridding ** 2) * (self.b.quad_level ** 2)
        return per * (counts["refined"] + counts["level3_float"])

    def conv_flops(self) -> float:
        """Algorithmic flops of one value convolution of every cutout:
        sum of 2 (ph+2)(pw+2) nx ny."""
        return float(sum(2.0 * (g.ph + 2) * (g.pw + 2) * g.nx * g.ny for g in self.gal_host))

    def split(self, flat: torch.Tensor) -> List[torch.Tensor]:
        out = []
        for g in self.gal_host:
            out.append(flat[g.pix_off:g.pix_off + g.nx * g.ny].view(g.ny, g.nx))
        return out

    # -- fitting ------------------------------------------------------------
    def start(self, rep0, fallback=None):
        """Start every fit from ``rep0``; with ``fallback`` (ngal x 7) a failed
        run restarts once from its fallback row within the same ticks."""
        rep0 = torch.as_tensor(rep0, dtype=torch.float64, device=self.data.device).contiguous()
        self._rep0 = rep0
        if fallback is None:
            L.check(self.lib.apx_batch_start(ctypes.byref(self.b), rep0.data_ptr(), L.stream()))
        else:
            fallback = torch.as_tensor(fallback, dtype=torch.float64, device=self.data.device).contiguous()
            self._fb = fallback
            L.check(self.lib.apx_batch_start_fallback(ctypes.byref(self.b), rep0.data_ptr(), fallback.data_ptr(),
                                                      L.stream()))
        self.ticks = 0

    def tick(self):
        L.check(self.lib.apx_batch_tick(ctypes.byref(self.b), L.stream()))
        self.ticks += 1

    def done_count(self) -> int:
        L.check(self.lib.apx_batch_results(ctypes.byref(self.b), self._rep.data_ptr(), self._chi2.data_ptr(),
                                           self._status.data_ptr(), self._iters.data_ptr(),
                                           self._fbran.data_ptr(), self._done.data_ptr(), L.stream()))
        return int(self._done.item())

    def capture(self, ticks_per_graph: int = 4):
        """Capture ``ticks_per_graph`` ticks in one HIP graph (after one eager
        tick has loaded every kernel)."""
        self.graph = torch.cuda.CUDAGraph()
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            with torch.cuda.graph(self.graph, stream=stream):
                for _ in range(ticks_per_graph):
                    L.check(self.lib.apx_batch_tick(ctypes.byref(self.b), L.stream()))
        torch.cuda.current_stream().wait_stream(stream)
        self.ticks_per_graph = ticks_per_graph

    def fit(self, rep0, max_ticks: int = 4000, check_every: int = 8, use_graph: bool = True, fallback=None):
        """Run every fit to completion (a failed run restarts once from its
        ``fallback`` row when given).  Returns a dict of host arrays: rep,
        values, chi2 (reduced), status, iterations (all runs), fallback."""
        self.start(rep0, fallback)
        self.tick()
        if use_graph:
            if self.graph is None:
                self.capture(check_every)
            while self.ticks < max_ticks:
                self.graph.replay()
                self.ticks += self.ticks_per_graph
                if self.done_count() == self.ngal:
                    break
        else:
            while self.ticks < max_ticks:
                for _ in range(check_every):
                    self.tick()
                if self.done_count() == self.ngal:
                    break
        self.done_count()
        rep = self._rep.cpu().numpy()
        return {"rep": rep, "values": rep_to_values(rep), "chi2": self._chi2.cpu().numpy(),
                "status": self._status.cpu().numpy(), "iterations": self._iters.cpu().numpy(),
                "fallback": self._fbran.cpu().numpy().astype(bool), "ticks": self.ticks}
