"""Parity of the gfx950 path with the float64 oracle on identical inputs.

Tolerances (max-norm relative to the oracle's max):
  model image  1e-5   (float32 render vs float64 oracle)
  Jacobian     2e-4 per column (float32 analytic partials vs float64 forward AD)
"""

import ctypes
import math

import numpy as np
import pytest
import torch

import astrophot_amd as ap
from oracle import hotpath as H
from tests.pairs import GAL, component, rel_err, single, target

pytestmark = pytest.mark.gpu

IMG_TOL = 1e-5
JAC_TOL = 2e-4

PSF11 = H.gaussian_psf(1.5, 11, 1.0)


@pytest.mark.parametrize("kind", ["sersic", "exponential", "gaussian", "moffat", "flat_sky"])
@pytest.mark.parametrize("integrate", ["none", "threshold"])
def test_render_psf_none(kind, integrate):
    om, m = single(kind, GAL[kind], integrate_mode=integrate)
    ref = om.forward(om.vector_representation())
    got = m().data
    assert got.is_cuda
    assert rel_err(got, ref) < IMG_TOL


@pytest.mark.parametrize("kind", ["sersic", "exponential", "gaussian", "moffat"])
@pytest.mark.parametrize("integrate", ["none", "threshold"])
def test_render_psf_full(kind, integrate):
    om, m = single(kind, GAL[kind], psf=PSF11, psf_mode="full", integrate_mode=integrate)
    ref = om.forward(om.vector_representation())
    got = m().data
    assert rel_err(got, ref) < IMG_TOL


@pytest.mark.parametrize("kind", ["sersic", "exponential", "gaussian", "moffat", "flat_sky"])
@pytest.mark.parametrize("psf_mode", ["none", "full"])
def test_jacobian(kind, psf_mode):
    if kind == "flat_sky" and psf_mode == "full":
        pytest.skip("sky models never convolve (sky_model_object.py:21-27)")
    kw = dict(psf=PSF11, psf_mode="full") if psf_mode == "full" else {}
    om, m = single(kind, GAL[kind], **kw)
    rep = om.vector_representation()
    Jref = om.jacobian(rep)
    J = m.jacobian(parameters=rep.clone(), as_representation=True).data
    assert J.shape == Jref.shape
    for k in range(J.shape[-1]):
        assert rel_err(J[..., k], Jref[..., k]) < JAC_TOL, k


def test_sersic_quad_sampling():
    """sampling_mode quad:5 (the reference fixtures' truth render, tests/utils.py:64)."""
    om, m = single("sersic", GAL["sersic"], psf=PSF11, psf_mode="full", sampling_mode="quad:5")
    ref = om.forward(om.vector_representation())
    assert rel_err(m().data, ref) < IMG_TOL


@pytest.mark.parametrize("kind", ["sersic", "exponential", "gaussian", "moffat"])
@pytest.mark.parametrize("integrate", ["none", "threshold"])
def test_trapezoid_sampling(kind, integrate):
    """sampling_mode "trapezoid" (_model_methods.py:121-139): the mean of the
    four pixel corners, selection by its Laplacian.  Image, Jacobian columns
    and the adjoint against the oracle, with the PSF convolved."""
    om, m = single(kind, GAL[kind], psf=PSF11, psf_mode="full", sampling_mode="trapezoid",
                   integrate_mode=integrate)
    rep = om.vector_representation()
    assert rel_err(m().data, om.forward(rep)) < IMG_TOL
    Jref = om.jacobian(rep)
    J = m.jacobian(parameters=rep.clone(), as_representation=True).data
    for k in range(J.shape[-1]):
        assert rel_err(J[..., k], Jref[..., k]) < JAC_TOL, k
    G = torch.tensor(np.random.default_rng(3).normal(size=(m.window.ny, m.window.nx)))
    r = rep.clone().requires_grad_(True)
    ref, = torch.autograd.grad((om.forward(r) * G).sum(), r)
    got = m.vjp(G.float(), parameters=rep.clone(), as_representation=True).cpu()
    assert ((got - ref).abs() / ref.abs().max()).max() < JAC_TOL, (got, ref)


def test_trapezoid_sampling_psf_none():
    om, m = single("sersic", GAL["sersic"], sampling_mode="trapezoid")
    assert rel_err(m().data, om.forward(om.vector_representation())) < IMG_TOL


def upscaled_pair(kind, U, nx=30, ny=26):
    """A model whose PSF is U times finer than the image (target_image.py:
    303-324), in the oracle and on the GPU."""
    psf = H.gaussian_psf(1.3, 13, 1.0 / U)
    params = dict(GAL[kind], center=[15.3, 12.6])
    oc = H.Component(kind, H.Grid(nx, ny), dict(params), psf=torch.tensor(psf), psf_mode="full", psf_upscale=U)
    tgt = ap.image.Target_Image(data=np.zeros((ny, nx)), pixelscale=1.0, psf=psf, psf_upscale=U)
    m = ap.models.AstroPhot_Model(name=f"up{kind}{U}", model_type=f"{kind} galaxy model", target=tgt,
                                  psf_mode="full", parameters=params)
    return H.Model([oc]), m


@pytest.mark.parametrize("U", [2, 3])
@pytest.mark.parametrize("kind", ["sersic", "moffat"])
def test_psf_upscale(kind, U):
    """model_object.py:313-349: sampled and convolved on the U-times finer
    grid, U x U blocks summed back (with U = 3 the reference's float32 1/U
    leaves the last row and column empty).  Image, Jacobian and adjoint
    against the oracle."""
    om, m = upscaled_pair(kind, U)
    rep = om.vector_representation()
    ref = om.forward(rep)
    got = m().data
    assert rel_err(got, ref) < IMG_TOL
    if U == 3:
        assert float(got[-1].abs().max()) == 0.0 and float(got[:, -1].abs().max()) == 0.0
    Jref = om.jacobian(rep)
    J = m.jacobian(parameters=rep.clone(), as_representation=True).data
    assert J.shape == Jref.shape
    for k in range(J.shape[-1]):
        assert rel_err(J[..., k], Jref[..., k]) < JAC_TOL, k
    G = torch.tensor(np.random.default_rng(5).normal(size=tuple(ref.shape)))
    r = rep.clone().requires_grad_(True)
    gref, = torch.autograd.grad((om.forward(r) * G).sum(), r)
    gv = m.vjp(G.float(), parameters=rep.clone(), as_representation=True).cpu()
    assert ((gv - gref).abs() / gref.abs().max()).max() < JAC_TOL, (gv, gref)


def test_lm_with_upscaled_psf_matches_oracle():
    """fit.LM through the upscaled render and Jacobian (PSF upscale 2) against
    the oracle's float64 LM on the same seeded data (variance = model/5 +
    0.01) from the same +-3 % start: parameters 1e-4, chi^2 1e-6.  (The
    bilinear PSF shift makes the model piecewise linear in the centre with a
    kink at every working-grid pixel; on the twice finer grid the kinks are
    twice as dense, and from +-10 % the reference LM's curvature test damps
    both fits into immobility.)"""
    om, m = upscaled_pair("sersic", 2)
    img = om.forward(om.vector_representation()).numpy()
    rng = np.random.default_rng(9)
    var = img / 5.0 + 0.01
    data = img + rng.normal(size=img.shape) * np.sqrt(var)
    oc = om.components[0]
    start_vals = om.vector_values().numpy() * (1 + rng.uniform(-0.03, 0.03, 7))
    o_start = oc.val_to_rep(torch.tensor(start_vals))
    lm_o = H.LM(om, torch.tensor(data), weight=torch.tensor(1 / var), initial_state=o_start).fit()
    psf = H.gaussian_psf(1.3, 13, 0.5)
    tgt = ap.image.Target_Image(data=data, pixelscale=1.0, variance=var, psf=psf, psf_upscale=2)
    fit_m = ap.models.AstroPhot_Model(name="upfit", model_type="sersic galaxy model", target=tgt,
                                      psf_mode="full", parameters=dict(GAL["sersic"], center=[15.3, 12.6]))
    fit_m.parameters.vector_set_values(torch.tensor(start_vals))
    start = fit_m.parameters.vector_representation()
    assert torch.allclose(start, o_start, rtol=1e-12, atol=1e-12)
    lm_g = ap.fit.LM(fit_m, initial_state=start).fit()
    assert lm_o.message.startswith("success"), lm_o.message
    assert lm_g.message.startswith("success"), lm_g.message
    vo = oc.rep_to_values(torch.as_tensor(lm_o.res()))
    v_o = torch.cat([vo[k].reshape(-1) for k in ("center", "q", "PA", "n", "Re", "Ie")])
    v_g = fit_m.parameters.vector_values()
    err = ((v_g - v_o).abs() / v_o.abs().clamp_min(1.0)).max().item()
    assert err < 1e-4, (err, v_g, v_o)
    chi_o, chi_g = min(lm_o.loss_history), min(lm_g.loss_history)
    assert abs(chi_g - chi_o) / chi_o < 1e-6, (chi_g, chi_o)


def test_group_c0_like():
    """Sersic + flat sky group with a 25x25 Gaussian PSF (the 100x100 C0 setup at 64x64)."""
    nx = ny = 64
    psf = H.gaussian_psf(1.5, 25, 1.0)
    tgt = target(nx, ny, psf=psf)
    p = {"center": [32.3, 31.7], "q": 0.7, "PA": 0.6, "n": 2.0, "Re": 8.0, "Ie": 1.0}
    oc, mc = component("sersic", p, tgt, nx, ny, psf=psf, psf_mode="full")
    os_, ms = component("flat_sky", {"F": math.log10(0.5)}, tgt, nx, ny)
    om = H.Model([oc, os_], window=H.Grid(nx, ny))
    g = ap.models.AstroPhot_Model(name="grp", model_type="group model", models=[mc, ms], target=tgt)
    rep = om.vector_representation()
    assert np.allclose(rep.numpy(), g.parameters.vector_representation().numpy())
    assert rel_err(g().data, om.forward(rep)) < IMG_TOL
    J = g.jacobian(parameters=rep.clone(), as_representation=True).data
    Jref = om.jacobian(rep)
    for k in range(J.shape[-1]):
        assert rel_err(J[..., k], Jref[..., k]) < JAC_TOL, k


def test_group_subwindows_union_and_jacobian_scatter():
    """Two Sersic components on overlapping sub-windows of a 72 x 64 image plus
    a sky on all of it: the group renders over the union of the windows with
    each component confined to its own window (group_model_object.py:92-129,
    183-231), and each component's Jacobian columns land in the group
    Jacobian at its own pixels, zero elsewhere (group_model_object.py:233-283,
    jacobian_image.py:79-118) -- against the oracle."""
    nx, ny = 72, 64
    psf = H.gaussian_psf(1.2, 11, 1.0)
    tgt = target(nx, ny, psf=psf)
    wins = [((4, 44), (6, 50)), ((30, 70), (14, 60))]  # [xmin, xmax), [ymin, ymax) in pixels
    pars = [{"center": [24.6, 27.2], "q": 0.6, "PA": 0.9, "n": 2.2, "Re": 5.0, "Ie": 1.1},
            {"center": [49.3, 37.8], "q": 0.8, "PA": 2.1, "n": 1.1, "Re": 7.0, "Ie": 0.6}]
    ocs, ms = [], []
    for k, (((x0, x1), (y0, y1)), p) in enumerate(zip(wins, pars)):
        g = H.Grid(x1 - x0, y1 - y0, ref_ij=(-0.5 - x0, -0.5 - y0))
        ocs.append(H.Component("sersic", g, dict(p), psf=torch.as_tensor(psf, dtype=torch.float64), psf_mode="full"))
        ms.append(ap.models.AstroPhot_Model(name=f"sub{k}", model_type="sersic galaxy model", target=tgt,
                                            parameters=dict(p), psf_mode="full", window=[[x0, x1], [y0, y1]]))
    osky, msky = component("flat_sky", {"F": math.log10(0.3)}, tgt, nx, ny)
    om = H.Model(ocs + [osky], window=H.Grid(nx, ny))
    grp = ap.models.AstroPhot_Model(name="subgrp", model_type="group model", models=ms + [msky], target=tgt)
    rep = om.vector_representation()
    assert np.allclose(rep.numpy(), grp.parameters.vector_representation().numpy())
    assert rel_err(grp().data, om.forward(rep)) < IMG_TOL
    J = grp.jacobian(parameters=rep.clone(), as_representation=True).data
    Jref = om.jacobian(rep)
    assert J.shape == Jref.shape
    for k in range(J.shape[-1]):
        assert rel_err(J[..., k], Jref[..., k]) < JAC_TOL, k
    # the first component's columns vanish outside its window
    (x0, x1), (y0, y1) = wins[0]
    outside = torch.ones(ny, nx, dtype=torch.bool)
    outside[y0:y1, x0:x1] = False
    assert float(J[..., :7].cpu()[outside].abs().max()) == 0.0


def test_saved_group_renders_the_same(tmp_path):
    """A group saved to YAML and loaded by filename (core_model.py:386-449,
    group_model_object.py:325-365) renders, and differentiates, bit for bit
    as the group it was saved from."""
    nx, ny = 60, 52
    tgt = target(nx, ny, psf=H.gaussian_psf(1.3, 11, 1.0))
    a = ap.models.AstroPhot_Model(name="a", model_type="sersic galaxy model", target=tgt, psf_mode="full",
                                  parameters={"center": [24.3, 22.8], "q": 0.7, "PA": 0.4, "n": 1.7,
                                              "Re": 6.0, "Ie": 0.9}, window=[[2, 50], [0, 48]])
    b = ap.models.AstroPhot_Model(name="b", model_type="moffat galaxy model", target=tgt,
                                  parameters={"center": [40.1, 30.6], "q": 0.8, "PA": 2.0, "n": 2.5,
                                              "Rd": 3.0, "I0": 0.5})
    grp = ap.models.AstroPhot_Model(name="g", model_type="group model", models=[a, b], target=tgt)
    fn = str(tmp_path / "g.yaml")
    grp.save(fn)
    new = ap.models.AstroPhot_Model(name="g", filename=fn, target=tgt)
    assert torch.equal(new().data, grp().data)
    assert torch.equal(new.jacobian().data, grp.jacobian().data)


def test_chi2_and_normal_equations():
    lib = ap._lib.load()
    torch.manual_seed(0)
    n, npar = 5000, 7
    dev = "cuda"
    J = torch.randn(n, npar, device=dev, dtype=torch.float32)
    m = torch.rand(n, device=dev)
    y = torch.rand(n, device=dev)
    w = torch.rand(n, device=dev) + 0.5
    mask = (torch.rand(n, device=dev) < 0.1).to(torch.uint8)
    wsb = lib.apx_reduce_workspace_bytes(n, npar)
    ws = torch.empty(wsb, dtype=torch.uint8, device=dev)
    out = torch.zeros(1, dtype=torch.float64, device=dev)
    st = ap._lib.stream()
    ap._lib.check(lib.apx_chi2(m.data_ptr(), y.data_ptr(), w.data_ptr(), mask.data_ptr(), n, out.data_ptr(),
                               ws.data_ptr(), wsb, st))
    keep = mask == 0
    ref = (w.double() * (y.double() - m.double()) ** 2)[keep].sum()
    assert abs(out.item() - ref.item()) <= 1e-9 * abs(ref.item())
    hess = torch.zeros(npar, npar, dtype=torch.float64, device=dev)
    grad = torch.zeros(npar, dtype=torch.float64, device=dev)
    ap._lib.check(lib.apx_normal_equations(J.data_ptr(), m.data_ptr(), y.data_ptr(), w.data_ptr(), mask.data_ptr(),
                                           n, npar, hess.data_ptr(), grad.data_ptr(), ws.data_ptr(), wsb, st))
    Jd, wd = J.double()[keep], w.double()[keep]
    Href = Jd.T @ (wd[:, None] * Jd)
    gref = Jd.T @ (wd * (y.double() - m.double())[keep])
    assert torch.allclose(hess, Href, rtol=1e-5, atol=1e-5 * Href.abs().max().item())
    assert torch.allclose(grad, gref, rtol=1e-5, atol=1e-5 * gref.abs().max().item())


def test_lm_solve_matches_reference_formula():
    lib = ap._lib.load()
    torch.manual_seed(1)
    npar = 8
    A = torch.randn(40, npar, dtype=torch.float64)
    hess = (A.T @ A).cuda()
    grad = torch.randn(npar, dtype=torch.float64).cuda()
    for Lval in (1e-9, 1e-3, 1.0, 1e4):
        h = torch.empty_like(grad)
        st = torch.zeros(1, dtype=torch.int32, device="cuda")
        ap._lib.check(lib.apx_lm_solve(hess.data_ptr(), grad.data_ptr(), npar, Lval, h.data_ptr(), st.data_ptr(),
                                       ap._lib.stream()))
        ref = H.lm_damped_solve(Lval, grad.cpu(), hess.cpu())
        assert st.item() == 0
        assert torch.allclose(h.cpu(), ref, rtol=1e-9, atol=1e-12)


@pytest.mark.parametrize("level,gridding,depth", [(3, 5, 3), (3, 5, 2), (3, 5, 1), (3, 4, 3), (5, 3, 3), (7, 8, 2), (1, 2, 3)])
def test_integration_settings(level, gridding, depth):
    """The level-1 and deep passes at other Gauss-Legendre orders, griddings
    and depths than the default's (a cuspy, well resolved Sersic refines at
    every level): image, Jacobian and adjoint against the oracle, at the
    repository's bars (1e-5 of the image's max; 2e-4 of a column's)."""
    p = dict(GAL["sersic"], n=4.5, Re=5.0)
    om, m = single("sersic", p, psf=PSF11, psf_mode="full", integrate_quad_level=level, integrate_gridding=gridding,
                   integrate_max_depth=depth, sampling_tolerance=1e-3)
    rep = om.vector_representation()
    assert rel_err(m().data, om.forward(rep).reshape(36, 40)) < 1e-5
    J = m.jacobian(parameters=rep.clone(), as_representation=True).data
    ref = om.jacobian(rep).reshape(36, 40, -1)
    for k in range(7):
        assert rel_err(J[..., k], ref[..., k]) < 2e-4, k
    G = torch.randn(36, 40, generator=torch.Generator().manual_seed(level), dtype=torch.float64)
    g = m.vjp(G, parameters=rep.clone())
    gref = (ref * G[..., None]).sum(dim=(0, 1))
    scale = (ref * G[..., None]).abs().sum(dim=(0, 1))
    assert bool(((g.cpu() - gref).abs() <= 2e-4 * scale).all())


@pytest.mark.parametrize("level,gridding,depth,tol,many", [
    (2, 5, 2, 1e-4, True), (4, 2, 3, 1e-4, True), (4, 5, 2, 1e-2, False), (6, 2, 3, 1e-2, False), (6, 3, 2, 1e-4, True),
    (5, 3, 3, 1e-4, True), (5, 1, 3, 1e-8, True), (7, 4, 2, 1e-8, True), (7, 8, 2, 1e-3, False)])
def test_integration_orders_and_list_lengths(level, gridding, depth, tol, many):
    """Every way the level-1 terms are added (by lane reads, over 16, 32 and 64
    lanes), and the deep pass with more listed pixels than its 1,024 workgroups
    (four pixels a workgroup) and with fewer (one), rules without a central node
    among them: image, Jacobian and adjoint at the bars of
    test_integration_settings."""
    p = dict(GAL["sersic"], n=4.5, Re=5.0)
    om, m = single("sersic", p, psf=PSF11, psf_mode="full", integrate_quad_level=level, integrate_gridding=gridding,
                   integrate_max_depth=depth, sampling_tolerance=tol)
    rep = om.vector_representation()
    assert rel_err(m().data, om.forward(rep).reshape(36, 40)) < 1e-5
    refined = int(m._apx_buffers["render_ws"].view(torch.int32)[1])
    assert refined > 0 and (refined > 1024) == many
    J = m.jacobian(parameters=rep.clone(), as_representation=True).data
    ref = om.jacobian(rep).reshape(36, 40, -1)
    for k in range(7):
        assert rel_err(J[..., k], ref[..., k]) < 2e-4, k
    G = torch.randn(36, 40, generator=torch.Generator().manual_seed(level), dtype=torch.float64)
    g = m.vjp(G, parameters=rep.clone())
    gref = (ref * G[..., None]).sum(dim=(0, 1))
    scale = (ref * G[..., None]).abs().sum(dim=(0, 1))
    assert bool(((g.cpu() - gref).abs() <= 2e-4 * scale).all())


@pytest.mark.parametrize("kh,kw,ow,oh,nchan,zero,shared", [
    (1, 1, 70, 33, 1, 0, False), (19, 19, 64, 16, 2, 0, False), (21, 21, 65, 17, 3, 0, False), (53, 21, 130, 31, 2, 0, False),
    (23, 67, 63, 48, 2, 1, False), (67, 67, 100, 40, 4, 1, False), (69, 69, 64, 24, 2, 0, False), (27, 27, 66, 20, 3, 0, True),
    (91, 91, 40, 20, 2, 0, False)])
def test_convolve_shapes(kh, kw, ow, oh, nchan, zero, shared):
    """apx_convolve at the edges of its three kernels and their tiles: value,
    centre and channel columns at an offset in the destinations, added to what
    is there; ``zero``: taps that reach outside the planes read 0; ``shared``:
    two channels added to one column.  float32 sums of kh kw products in a
    fixed order against float64: 1e-5 of the sum of their magnitudes."""
    lib = ap._lib.load()
    g = torch.Generator().manual_seed(kh + ow)
    rnd = lambda *s: torch.randn(s, generator=g).cuda()  # noqa: E731
    m = 0 if zero else 1
    nx, ny = ow + m * (kw - 1) + 3, oh + m * (kh - 1) + 2
    x0, y0 = (1, 1) if zero else ((kw - 1) // 2 + 2, (kh - 1) // 2 + 1)
    planes, kern = rnd(nchan, ny, nx), rnd(3, kh, kw)
    img, jac = rnd(oh + 3, ow + 5), rnd(oh + 3, ow + 5, nchan + 3)
    ref_i, ref_j = img.double(), jac.double()
    job = ap._lib.ConvJob()
    job.nx, job.ny, job.nchan, job.kh, job.kw, job.x0, job.y0, job.ow, job.oh = nx, ny, nchan, kh, kw, x0, y0, ow, oh
    job.img, job.img_row, job.img_w, job.img_h, job.img_x0, job.img_y0 = img.data_ptr(), ow + 5, ow + 5, oh + 3, 4, 2
    job.jac, job.jac_np, job.jac_row = jac.data_ptr(), nchan + 3, (ow + 5) * (nchan + 3)
    job.jac_w, job.jac_h, job.jac_x0, job.jac_y0 = ow + 5, oh + 3, 4, 2
    job.dk_col[0], job.dk_col[1] = nchan + 1, 0
    col = [0] + [1 if shared else c for c in range(1, nchan)]
    job.chan_col[:nchan] = col
    job.zero_outside = zero
    wsb = lib.apx_convolve_workspace_bytes(kh, kw)
    ws = torch.empty(wsb, dtype=torch.uint8, device="cuda")
    pad = torch.nn.functional.pad(planes.double().cpu(), (kw, kw, kh, kh))
    box = pad[:, kh + y0 - (kh - 1) // 2:kh + y0 + oh + (kh - 1) // 2, kw + x0 - (kw - 1) // 2:kw + x0 + ow + (kw - 1) // 2]
    conv = lambda p, k: torch.nn.functional.conv2d(p[None, None], k.double().cpu()[None, None])[0, 0].cuda()  # noqa: E731
    tol = 1e-5 * float(conv(box.abs().max(0).values, kern.abs().max(0).values).max())
    ref_i[2:2 + oh, 4:4 + ow] += conv(box[0], kern[0])
    for k, c in ((1, nchan + 1), (2, 0)):
        ref_j[2:2 + oh, 4:4 + ow, c] += conv(box[0], kern[k])
    for c in range(1, nchan):
        ref_j[2:2 + oh, 4:4 + ow, col[c]] += conv(box[c], kern[0])
    ap._lib.check(lib.apx_convolve(ctypes.byref(job), planes.data_ptr(), kern.data_ptr(), ws.data_ptr(), wsb, ap._lib.stream()))
    assert float((img.double() - ref_i).abs().max()) <= tol
    assert float((jac.double() - ref_j).abs().max()) <= tol


def conv_job(planes, kern, img=None, jac=None, x0=0, y0=0, ow=0, oh=0):
    """An apx_conv_job on every output pixel of img or jac, zero outside the planes."""
    job = ap._lib.ConvJob()
    job.nchan, job.ny, job.nx = planes.shape
    job.kh, job.kw = kern.shape[1:]
    job.x0, job.y0, job.ow, job.oh, job.zero_outside = x0, y0, ow, oh, 1
    job.chan_col[:], job.dk_col[:] = [-1] * 8, [-1] * 2
    if img is not None:
        job.img, job.img_row, job.img_w, job.img_h = img.data_ptr(), ow, ow, oh
    if jac is not None:
        job.jac, job.jac_np, job.jac_row, job.jac_w, job.jac_h = jac.data_ptr(), jac.shape[2], ow * jac.shape[2], ow, oh
    return job


def conv_float64(box, kern):
    """Full convolution of the rows and columns around a box that the kernel covers."""
    return torch.nn.functional.conv2d(box.double().cpu()[None, None], kern.double().cpu()[None, None])[0, 0].cuda()


@pytest.mark.parametrize("side,ow,cols,dk", [(21, 70, [2, 2, 2], [2, -1]), (27, 40, [0, 1, 0], [1, 1]), (67, 130, [1, 1, 0], [0, 1])])
def test_convolve_shared_columns_without_workspace(side, ow, cols, dk):
    """Passes that add to one Jacobian column, and kernels of 21 to 67 rows, need
    no workspace: the columns' sums against float64, 1e-5 of the sum of the
    magnitudes as test_convolve_shapes."""
    g = torch.Generator().manual_seed(side)
    planes, kern = torch.randn(4, ow, ow, generator=g).cuda(), torch.randn(3, side, side, generator=g).cuda()
    jac = torch.randn(ow, ow, 3, generator=g).cuda()
    ref, tol = jac.double(), 0.0
    pad = torch.nn.functional.pad(planes, (side // 2,) * 4)
    for p, k, c in [(0, 1, dk[0]), (0, 2, dk[1]), (1, 0, cols[0]), (2, 0, cols[1]), (3, 0, cols[2])]:
        if c >= 0:
            ref[..., c] += conv_float64(pad[p], kern[k])
            tol += 1e-5 * float(conv_float64(pad[p].abs(), kern[k].abs()).max())
    job = conv_job(planes, kern, jac=jac, ow=ow, oh=ow)
    job.chan_col[1], job.chan_col[2], job.chan_col[3] = cols
    job.dk_col[0], job.dk_col[1] = dk
    ap._lib.check(ap._lib.load().apx_convolve(ctypes.byref(job), planes.data_ptr(), kern.data_ptr(), None, 0, ap._lib.stream()))
    assert float((jac.double() - ref).abs().max()) <= tol


def test_convolve_rows_of_half_a_billion_pixels():
    """A plane row of more than 2^29 pixels, whose bytes exceed a buffer resource:
    the last columns and the first ones, zero beyond either end."""
    g = torch.Generator().manual_seed(1)
    nx, ow, side = 2 ** 29 + 77, 150, 21
    plane, kern = torch.zeros(1, 1, nx, device="cuda"), torch.randn(1, side, side, generator=g).cuda()
    plane[0, 0, :400], plane[0, 0, -400:] = torch.randn(400, generator=g).cuda(), torch.randn(400, generator=g).cuda()
    lib = ap._lib.load()
    for x0 in (0, nx - ow):
        img = torch.zeros(1, ow, device="cuda")
        job = conv_job(plane, kern, img=img, x0=x0, ow=ow, oh=1)
        ap._lib.check(lib.apx_convolve(ctypes.byref(job), plane.data_ptr(), kern.data_ptr(), None, 0, ap._lib.stream()))
        row = torch.nn.functional.pad(plane[0, 0, :ow + 10] if x0 == 0 else plane[0, 0, -(ow + 10):],
                                      (10, 0) if x0 == 0 else (0, 10))
        box = torch.nn.functional.pad(row[None], (0, 0, 10, 10))
        want = conv_float64(box, kern[0])
        assert float((img.double() - want).abs().max()) <= 1e-5 * float(conv_float64(box.abs(), kern[0].abs()).max())


def test_convolve_of_more_tiles_than_a_launch():
    """A one-column image of 4.2 million tiles, past the 2^31 threads a launch is
    kept below: the rows around the cut, the first and the last."""
    g = torch.Generator().manual_seed(2)
    side = 21
    cut = ((2 ** 31 - 1) // 512 // 8) * 8 * 32
    ny = cut + 100
    plane, kern = torch.zeros(1, ny, 1, device="cuda"), torch.randn(1, side, side, generator=g).cuda()
    where = [0, cut - 100, ny - 200]
    for y in where:
        plane[0, y:y + 200, 0] = torch.randn(200, generator=g).cuda()
    img = torch.zeros(ny, 1, device="cuda")
    job = conv_job(plane, kern, img=img, ow=1, oh=ny)
    ap._lib.check(ap._lib.load().apx_convolve(ctypes.byref(job), plane.data_ptr(), kern.data_ptr(), None, 0, ap._lib.stream()))
    for y in where:
        lo, hi = max(y - 50, 0), min(y + 250, ny)
        rows = plane[0, max(lo - 10, 0):min(hi + 10, ny)]
        box = torch.nn.functional.pad(rows, (10, 10, 10 if lo == 0 else 0, 10 if hi == ny else 0))
        want = conv_float64(box, kern[0])
        assert float((img[lo:hi].double() - want).abs().max()) <= 1e-5 * float(conv_float64(box.abs(), kern[0].abs()).max())


@pytest.mark.parametrize("npar", [1, 2, 13, 15, 16, 17, 64])
def test_lm_solve_sizes_and_bad_pivots(npar):
    """The one-wave solve (up to 16) and the workgroup one at the edges of
    their ranges; with an indefinite matrix both report the first bad pivot and
    solve by elimination.  1e-9 relative: condition below 1e5, float64."""
    lib = ap._lib.load()
    g = torch.Generator().manual_seed(npar)
    A = torch.randn(4 * npar + 8, npar, dtype=torch.float64, generator=g)
    grad = torch.randn(npar, dtype=torch.float64, generator=g)
    for bad in (None, npar // 2):
        hess = A.T @ A
        if bad is not None:
            hess[bad, bad] = -50.0
        h = torch.empty(npar, dtype=torch.float64, device="cuda")
        st = torch.full((1,), 7, dtype=torch.int32, device="cuda")
        hd, gd = hess.cuda(), grad.cuda()
        ap._lib.check(lib.apx_lm_solve(hd.data_ptr(), gd.data_ptr(), npar, 0.5, h.data_ptr(), st.data_ptr(), ap._lib.stream()))
        ref = H.lm_damped_solve(0.5, grad, hess)
        assert st.item() == (0 if bad is None else bad + 1)
        assert float((h.cpu() - ref).norm() / ref.norm()) < 1e-9


@pytest.mark.parametrize("npix,npar", [(1, 1), (3, 16), (255, 13), (1023, 7), (4097, 16), (70001, 5), (600000, 13)])
@pytest.mark.parametrize("masked", [False, True])
def test_lm_products_sizes(npix, npar, masked):
    """chi^2, the normal equations and rpp at ragged sizes, from one pixel to
    more than one step of every workgroup.  float64 sums of float64 products
    (chi^2, rpp): 1e-11; J^T W J sums at most 256 float32 products in a chain:
    1e-5 of the largest entry, as test_chi2_and_normal_equations."""
    lib = ap._lib.load()
    g = torch.Generator(device="cuda").manual_seed(npix + npar)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    J, m, y, m1 = rnd(npix, npar), rnd(npix), rnd(npix), rnd(npix)
    w = torch.rand(npix, generator=g, device="cuda") + 0.1
    mask = (rnd(npix) > 1).to(torch.uint8) if masked else None
    keep = torch.ones(npix, device="cuda", dtype=torch.float64) if mask is None else (mask == 0).double()
    wsb = lib.apx_reduce_workspace_bytes(npix, npar)
    ws = torch.empty(wsb, dtype=torch.uint8, device="cuda")
    chi2, hess, grad, rpp = (torch.empty(s, dtype=torch.float64, device="cuda") for s in ((1,), (npar, npar), (npar,), (npar,)))
    h = rnd(npar).double()
    p, st = ap._lib.ptr, ap._lib.stream()
    ap._lib.check(lib.apx_chi2(p(m), p(y), p(w), p(mask), npix, p(chi2), p(ws), wsb, st))
    ap._lib.check(lib.apx_normal_equations(p(J), p(m), p(y), p(w), p(mask), npix, npar, p(hess), p(grad), p(ws), wsb, st))
    ap._lib.check(lib.apx_rpp(p(J), p(m), p(m1), p(w), p(mask), npix, npar, p(h), 0.1, p(rpp), p(ws), wsb, st))
    Jd, wd = J.double(), w.double() * keep
    r = y.double() - m.double()
    ref = (wd * r * r).sum()
    assert abs(float(chi2 - ref)) <= 1e-11 * float(ref) + 1e-300
    Href, gref = Jd.T @ (wd[:, None] * Jd), Jd.T @ (wd * r)
    v = 20.0 * (wd * (m1 - m).double() / 0.1 - wd * (Jd @ h))
    assert float((hess - Href).abs().max()) <= 1e-5 * float(Href.abs().max())
    assert float((grad - gref).abs().max()) <= 1e-5 * float((Jd.abs().T @ (wd * r.abs())).max())
    assert float((rpp - Jd.T @ v).abs().max()) <= 1e-11 * float((Jd.abs().T @ v.abs()).max())


@pytest.mark.parametrize("kind", ["sersic", "exponential", "gaussian", "moffat", "flat_sky"])
@pytest.mark.parametrize("psf_mode", ["none", "full"])
def test_adjoint_vjp(kind, psf_mode):
    """Hand-written adjoint vs the oracle's reverse-mode autograd gradient and
    vs J^T G from the forward-mode Jacobian (tolerance 2e-4 of the max)."""
    if kind == "flat_sky" and psf_mode == "full":
        pytest.skip("sky models never convolve")
    kw = dict(psf=PSF11, psf_mode="full") if psf_mode == "full" else {}
    om, m = single(kind, GAL[kind], **kw)
    rep = om.vector_representation()
    rng = np.random.default_rng(11)
    G = torch.tensor(rng.normal(size=(m.window.ny, m.window.nx)))
    r = rep.clone().requires_grad_(True)
    ref, = torch.autograd.grad((om.forward(r) * G).sum(), r)
    got = m.vjp(G.float(), parameters=rep.clone(), as_representation=True).cpu()
    scale = ref.abs().max()
    assert ((got - ref).abs() / scale).max() < JAC_TOL, (got, ref)
    J = m.jacobian(parameters=rep.clone(), as_representation=True).data.double().cpu()
    jtg = (J * G[..., None]).sum(dim=(0, 1))
    assert ((got - jtg).abs() / scale).max() < JAC_TOL


def test_autograd_function_group():
    """torch.autograd through differentiable_sample on the C0-like group."""
    nx = ny = 48
    psf = H.gaussian_psf(1.5, 11, 1.0)
    tgt = target(nx, ny, psf=psf)
    p = {"center": [24.3, 23.6], "q": 0.7, "PA": 0.6, "n": 2.0, "Re": 6.0, "Ie": 1.0}
    oc, mc = component("sersic", p, tgt, nx, ny, psf=psf, psf_mode="full")
    os_, ms = component("flat_sky", {"F": math.log10(0.5)}, tgt, nx, ny)
    om = H.Model([oc, os_], window=H.Grid(nx, ny))
    g = ap.models.AstroPhot_Model(name="grp_ad", model_type="group model", models=[mc, ms], target=tgt)
    rep = om.vector_representation()
    W = torch.tensor(np.random.default_rng(3).uniform(0.5, 1.5, (ny, nx)))
    r = rep.clone().requires_grad_(True)
    ref, = torch.autograd.grad(((om.forward(r) - 1.0) ** 2 * W).sum(), r)
    r2 = rep.clone().cuda().requires_grad_(True)
    img = ap.models.differentiable_sample(g, r2)
    loss = ((img.double() - 1.0) ** 2 * W.cuda()).sum()
    loss.backward()
    assert ((r2.grad.cpu() - ref).abs() / ref.abs().max()).max() < JAC_TOL
    # central finite differences of the oracle (h = 1e-3 in representation space)
    h = 1e-3
    for k in range(len(rep)):
        a, b = rep.clone(), rep.clone()
        a[k] += h
        b[k] -= h
        fd = ((((om.forward(a) - 1.0) ** 2 * W).sum() - ((om.forward(b) - 1.0) ** 2 * W).sum()) / (2 * h)).item()
        assert abs(r2.grad[k].item() - fd) <= 2e-3 * max(abs(fd), ref.abs().max().item() * 1e-3), (k, fd)


def _masked_pair():
    nx, ny = 40, 36
    mask = torch.zeros((ny, nx))
    mask[10, 13] = 1
    mask[17:20, 19:23] = 1
    tgt = target(nx, ny, psf=PSF11)
    p = dict(GAL["sersic"])
    plain = ap.models.AstroPhot_Model(name="plain", model_type="sersic galaxy model", target=tgt, parameters=dict(p),
                                      psf_mode="full")
    masked = ap.models.AstroPhot_Model(name="masked", model_type="sersic galaxy model", target=tgt,
                                       parameters=dict(p), psf_mode="full", mask=mask)
    return tgt, mask, plain, masked


def test_model_mask():
    """model_object.py:370-371 (reference test_model.py:139-161): masked
    samples are zero, the others are the unmasked model's; the Jacobian is the
    derivative of the masked sample and the adjoint its transpose."""
    tgt, mask, plain, masked = _masked_pair()
    keep = torch.logical_not(mask).float().cuda()
    img = masked().data
    assert img[10, 13].item() == 0.0 and img[11, 12].item() != 0.0
    assert torch.equal(img, plain().data * keep)
    J = masked.jacobian().data
    Jp = plain.jacobian().data
    assert torch.equal(J, Jp * keep[..., None])
    G = torch.tensor(np.random.default_rng(4).normal(size=(36, 40)), dtype=torch.float32)
    rep = masked.parameters.vector_representation().clone()
    got = masked.vjp(G, parameters=rep.clone(), as_representation=True).cpu()
    Jr = masked.jacobian(parameters=rep.clone(), as_representation=True).data.double().cpu()
    jtg = (Jr * G.double()[..., None]).sum(dim=(0, 1))
    assert ((got - jtg).abs() / jtg.abs().max()).max() < JAC_TOL


def test_masked_member_keeps_other_light():
    """A group sampled into an image it is handed calls each member on the
    shared working image (group_model_object.py:217-229): a member's mask
    zeroes only its own samples (model_object.py:370-373), not the light the
    other members put there."""
    tgt, mask, plain, masked = _masked_pair()
    sky = ap.models.AstroPhot_Model(name="sky", model_type="flat sky model", target=tgt,
                                    parameters={"F": math.log10(0.5)})
    grp = ap.models.AstroPhot_Model(name="g", model_type="group model", models=[sky, masked], target=tgt)
    img = grp.make_model_image()
    grp.sample(image=img)
    keep = torch.logical_not(mask).float().cuda()
    want = sky().data + plain().data * keep
    assert float((img.data - want).abs().max()) <= 1e-6 * float(want.abs().max())
    assert img.data[10, 13].item() == pytest.approx(sky().data[10, 13].item(), rel=1e-6)
    own = grp()
    assert float((own.data - want).abs().max()) <= 1e-6 * float(want.abs().max())
    # group Jacobian: the masked member's columns vanish at its masked pixels
    J = grp.jacobian().data
    assert float(J[10, 13, 1:].abs().max()) == 0.0 and J[10, 13, 0].item() != 0.0


def test_group_with_upscaled_psf():
    """Sersic + flat sky group on a target whose PSF is 3 times finer
    (target_image.py:303-324): the group image and Jacobian against the
    oracle; the sky ignores the PSF."""
    nx, ny, U = 42, 38, 3
    psf = H.gaussian_psf(1.2, 15, 1.0 / U)
    tgt = ap.image.Target_Image(data=np.zeros((ny, nx)), pixelscale=1.0, psf=psf, psf_upscale=U)
    p = {"center": [21.3, 18.6], "q": 0.7, "PA": 0.6, "n": 2.0, "Re": 6.0, "Ie": 1.0}
    oc = H.Component("sersic", H.Grid(nx, ny), dict(p), psf=torch.tensor(psf), psf_mode="full", psf_upscale=U)
    osky = H.Component("flat_sky", H.Grid(nx, ny), {"F": math.log10(0.5)})
    om = H.Model([oc, osky], window=H.Grid(nx, ny))
    ms = ap.models.AstroPhot_Model(name="s_up", model_type="sersic galaxy model", target=tgt, parameters=dict(p),
                                   psf_mode="full")
    mk = ap.models.AstroPhot_Model(name="sky_up", model_type="flat sky model", target=tgt,
                                   parameters={"F": math.log10(0.5)})
    g = ap.models.AstroPhot_Model(name="g_up", model_type="group model", models=[ms, mk], target=tgt)
    rep = om.vector_representation()
    assert np.allclose(rep.numpy(), g.parameters.vector_representation().numpy())
    assert rel_err(g().data, om.forward(rep)) < IMG_TOL
    J = g.jacobian(parameters=rep.clone(), as_representation=True).data
    Jref = om.jacobian(rep)
    for k in range(J.shape[-1]):
        assert rel_err(J[..., k], Jref[..., k]) < JAC_TOL, k


@pytest.mark.parametrize("ph,pw,sx,sy", [(1, 1, 0.3, -0.4), (3, 5, -0.5, 0.5), (51, 51, 0.25, 0.0), (123, 125, 0.1, 0.45),
                                         (125, 123, -0.3, 0.2), (129, 129, 0.49, -0.49), (5, 129, 0.0, 0.0)])
def test_psf_shift_of_any_side(ph, pw, sx, sy):
    """The shifted, normalised PSF and its two shift derivatives against float64
    numpy: padded sides up to 126 x 126 values go through LDS, larger ones do not.
    Both take float64 steps and round once: 2^-24 of each plane's largest value,
    taken as 1.2e-7."""
    import ctypes
    from astrophot_amd import _lib as L
    rng = np.random.default_rng(ph * 131 + pw)
    psf = (0.1 + rng.random((ph, pw))).astype(np.float32)
    pad = np.zeros((ph + 2, pw + 2))
    pad[1:-1, 1:-1] = psf
    r, c = np.meshgrid(np.arange(ph + 2.0), np.arange(pw + 2.0), indexing="ij")
    x, y = c - sx, r - sy
    xf, yf = np.floor(x).astype(int), np.floor(y).astype(int)
    x0, x1 = np.clip(xf, 0, pw), np.clip(xf + 1, 1, pw + 1)
    y0, y1 = np.clip(yf, 0, ph), np.clip(yf + 1, 1, ph + 1)
    fa, fb, fc, fd = pad[y0, x0], pad[y1, x0], pad[y0, x1], pad[y1, x1]
    v = fa * (x1 - x) * (y1 - y) + fb * (x1 - x) * (y - y0) + fc * (x - x0) * (y1 - y) + fd * (x - x0) * (y - y0)
    dx = -(-fa * (y1 - y) - fb * (y - y0) + fc * (y1 - y) + fd * (y - y0))
    dy = -(-fa * (x1 - x) + fb * (x1 - x) - fc * (x - x0) + fd * (x - x0))
    S = v.sum()
    ref = [v / S, dx / S - v * dx.sum() / S ** 2, dy / S - v * dy.sum() / S ** 2]
    out = torch.empty((3, ph + 2, pw + 2), dtype=torch.float32, device="cuda")
    pinv = (ctypes.c_double * 4)(1.0, 0.0, 0.0, 1.0)
    src = torch.tensor(psf, device="cuda")
    L.check(L.load().apx_psf_shift(src.data_ptr(), ph, pw, sx, sy, ctypes.cast(pinv, ctypes.c_void_p), 1.0, 1.0,
                                   out.data_ptr(), L.stream()))
    for got, want in zip(out.cpu().numpy(), ref):
        assert np.abs(got[::-1, ::-1] - want).max() <= 1.2e-7 * max(np.abs(want).max(), 1e-30)


@pytest.mark.parametrize("kh,kw,ow,oh,nchan", [(21, 67, 513, 321, 4), (67, 21, 449, 352, 5), (67, 67, 640, 337, 3),
                                               (33, 35, 1985, 513, 1)])
def test_convolve_two_blocks_a_workgroup(kh, kw, ow, oh, nchan):
    """apx_convolve where its launch has 512 workgroups of two 16-row blocks or
    more: whole and half last blocks, one-column last tiles, zero outside."""
    test_convolve_shapes(kh, kw, ow, oh, nchan, 0, False)
    test_convolve_shapes(kh, kw, ow, oh, nchan, 1, False)


@pytest.mark.parametrize("mode", ["midpoint", "trapezoid"])
@pytest.mark.parametrize("px,py", [(22, 18), (16, 21), (0, 0)])
def test_selection_at_its_threshold(mode, px, py):
    """A pixel whose curvature sits at the selection threshold is decided in
    float64 whichever side it falls: the tolerance at which the oracle's pixel
    switches between its sample and its quadrature is found by bisection, and
    the image agrees with the oracle's a part in 1e8 to either side of it (the
    float32 test cannot tell), at the repository's bar of 1e-5 of the max.  Last,
    a Gaussian wide enough (sigma 300 px) that no pixel of a wave is decided in
    float32."""
    p = dict(GAL["sersic"], center=[20.0, 18.0], q=0.98, n=1.5, Re=3.0)
    knobs = dict(sampling_mode=mode, integrate_max_depth=1)

    def at(tol):
        om, m = single("sersic", p, sampling_tolerance=tol, **knobs)
        return om.forward(om.vector_representation()).reshape(36, 40), m

    lo, hi = 1e-9, 1e6  # selected, not selected
    v_lo, v_hi = float(at(lo)[0][py, px]), float(at(hi)[0][py, px])
    assert v_lo != v_hi
    for _ in range(60):
        mid = math.sqrt(lo * hi)
        if float(at(mid)[0][py, px]) == v_hi:
            hi = mid
        else:
            lo = mid
    for tol in (lo * (1 - 1e-8), hi * (1 + 1e-8)):
        ref, m = at(tol)
        assert rel_err(m().data, ref) < 1e-5
    om, m = single("gaussian", dict(GAL["gaussian"], sigma=300.0, flux=6.0), sampling_tolerance=1e-12, **knobs)
    assert rel_err(m().data, om.forward(om.vector_representation()).reshape(36, 40)) < 1e-5
