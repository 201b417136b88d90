"""Batched fits (csrc/batch.hip) against the single-model path and the oracle.

* render: every cutout of the batch equals the single-model render of the
  same Sersic (psf_mode "full") within 1e-6 of its max;
* fits: each batched LM ends where the single-model LM (astrophot_amd.fit.LM)
  ends: reduced chi^2 within 1e-6 relative and parameters within 1e-4
  relative, or (at most one fit, along a direction the data barely
  constrain) within 1 % of the parameter's statistical uncertainty;
  two small cutouts are also checked against the float64 oracle LM.
"""

import math

import numpy as np
import pytest
import torch

import astrophot_amd as ap
from astrophot_amd.batch import BatchFit, Cutout, rep_to_values, values_to_rep
from oracle import hotpath as H

pytestmark = pytest.mark.gpu

PARAM_RTOL = 1e-4
CHI2_RTOL = 1e-6


def make_cutouts(n, seed, sizes=(32, 80), snr=(30, 300)):
    rng = np.random.default_rng(seed)
    truths, cut_shapes = [], []
    for _ in range(n):
        s = int(round(math.exp(rng.uniform(math.log(sizes[0]), math.log(sizes[1])))))
        sig = rng.uniform(1.0, 2.0)
        side = 2 * math.ceil(4 * sig) + 1
        psf = H.gaussian_psf(sig, side, 1.0)
        v = np.array([s / 2 + rng.uniform(-1, 1), s / 2 + rng.uniform(-1, 1), rng.uniform(0.4, 0.95),
                      rng.uniform(0, math.pi), rng.uniform(0.8, 4.0), math.exp(rng.uniform(math.log(2), math.log(s / 6))),
                      rng.uniform(0.0, 1.0)])
        truths.append(v)
        cut_shapes.append((s, psf))
    return truths, cut_shapes, rng


def test_batch_render_matches_single_model():
    truths, shapes, rng = make_cutouts(6, seed=1)
    cuts = [Cutout(np.zeros((s, s)), np.ones((s, s)), psf) for s, psf in shapes]
    bf = BatchFit(cuts)
    rep = values_to_rep(np.stack(truths))
    imgs = bf.split(bf.render(rep))
    for k, ((s, psf), v) in enumerate(zip(shapes, truths)):
        tgt = ap.image.Target_Image(data=np.zeros((s, s)), pixelscale=1.0, psf=ap.image.PSF_Image(data=psf, pixelscale=1.0))
        p = {"center": [v[0], v[1]], "q": v[2], "PA": v[3], "n": v[4], "Re": v[5], "Ie": v[6]}
        m = ap.models.AstroPhot_Model(name=f"b{k}", model_type="sersic galaxy model", target=tgt, parameters=p,
                                      psf_mode="full")
        ref = m().data
        err = float((imgs[k] - ref).abs().max() / ref.abs().max())
        assert err < 1e-6, (k, err)


@pytest.mark.parametrize("quad_group", [0, 25])
def test_batch_render_matches_oracle(quad_group):
    """The batched render (float32 samples, float64 refinement decisions)
    against the float64 oracle: within 1e-5 of the image max, and within 1e-5
    of the pixel's own value wherever it is above 1 % of the max, including
    cusp-like (n = 6) and barely resolved (Re = 1.5 px) profiles where the
    adaptive quadrature refines most; with 32 lanes per refined pixel and with
    one lane per level-2 sub-pixel (quad_group 25)."""
    vals = [[20.3, 21.7, 0.6, 0.7, 2.5, 6.0, 1.0], [24.0, 23.5, 0.35, 2.2, 6.0, 4.0, 0.5],
            [15.6, 16.2, 0.9, 1.0, 0.6, 1.5, 1.2], [40.1, 38.8, 0.5, 0.3, 4.0, 20.0, -0.3]]
    sides = [41, 48, 32, 80]
    psfs = [H.gaussian_psf(s_, 2 * math.ceil(4 * s_) + 1, 1.0) for s_ in (1.5, 1.0, 2.2, 3.0)]
    bf = BatchFit([Cutout(np.zeros((s, s)), np.ones((s, s)), psf) for s, psf in zip(sides, psfs)])
    bf.b.quad_group = quad_group
    imgs = bf.split(bf.render(values_to_rep(np.array(vals))))
    for k, (s, psf, v) in enumerate(zip(sides, psfs, vals)):
        p = {"center": [v[0], v[1]], "q": v[2], "PA": v[3], "n": v[4], "Re": v[5], "Ie": v[6]}
        om = H.Model([H.Component("sersic", H.Grid(s, s), p, psf=torch.tensor(psf), psf_mode="full")])
        ref = om.forward(om.vector_representation()).reshape(s, s)
        got = imgs[k].double().cpu()
        assert float((got - ref).abs().max() / ref.abs().max()) < 1e-5, k
        bright = ref > 1e-2 * ref.max()
        assert float(((got - ref).abs() / ref)[bright].max()) < 1e-5, k


@pytest.mark.parametrize("quad_group", [32, 25])
@pytest.mark.parametrize("n", [2, 9, 513, 1100, 4099])
def test_refined_pixel_lists_of_any_fit_count(n, quad_group):
    """The lists of refined and undecided pixels are packed several fits a
    workgroup, by their number: below 1,024 fits one, from 4,096 eight.  A fit's
    render and Jacobian have the same bits whichever others share the lists, so
    the first, a middle and the last fit equal a batch of that fit alone."""
    truths, shapes, _ = make_cutouts(7, seed=11, sizes=(16, 33))
    which = np.arange(n) % 7
    cut = [Cutout(np.zeros((s, s)), np.ones((s, s)), psf) for s, psf in shapes]

    def images(idx):
        bf = BatchFit([cut[i] for i in idx])
        bf.b.quad_group = quad_group
        rep = values_to_rep(np.stack([truths[i] for i in idx]))
        img, J = bf.jacobian(rep)
        cols = [bf.split(J[:, c].contiguous()) for c in range(7)]
        return bf.split(bf.render(rep)), bf.split(img), cols

    many = images(which)
    for k in {0, n // 2, n - 1}:
        one = images(which[k:k + 1])
        assert torch.equal(many[0][k], one[0][0])
        assert torch.equal(many[1][k], one[1][0])
        for jm, jo in zip(many[2], one[2]):
            assert torch.equal(jm[k], jo[0])


@pytest.mark.parametrize("quad_group", [32, 25])
@pytest.mark.parametrize("n", [1, 40])
def test_short_and_long_refined_lists_agree(n, quad_group):
    """Few refined or undecided pixels get a workgroup or 16 lanes each, many a
    group or a lane each, by the list's length against the launch's size
    (quad_blocks): the same bits either way, with tolerances that leave many
    pixels near a threshold and at every level."""
    truths, shapes, _ = make_cutouts(n, seed=3, sizes=(24, 50))
    cuts = [Cutout(np.zeros((s, s)), np.ones((s, s)), psf) for s, psf in shapes]
    for tol in (1e-2, 1e-4):
        bf = BatchFit(cuts, sampling_tolerance=tol)
        bf.b.quad_group = quad_group
        rep = values_to_rep(np.stack(truths))
        out = []
        for blocks in (1, 4096):
            bf.b.quad_blocks = blocks
            img, J = bf.jacobian(rep)
            out.append((img.clone(), J.clone(), bf.render(rep).clone()))
        for a, b in zip(*out):
            assert torch.equal(a, b)


@pytest.mark.parametrize("quad_group", [32, 25])
def test_both_branches_of_the_list_passes_are_taken(quad_group):
    """Three copies of a nearly round, centred galaxy, whose pixels come to a
    threshold by eights: the lengths of the three lists (refined pixels, undecided
    selections, pixels redone in float64) are on the long side of every rule for a
    launch of one workgroup and on the short side for one of 4,096, and the bits
    are the same."""
    v = np.array([16.5, 16.5, 0.999999, 0.3, 3.0, 3.0, 0.5])
    bf = BatchFit([Cutout(np.zeros((33, 33)), np.ones((33, 33)), H.gaussian_psf(1.0, 9, 1.0))] * 3)
    bf.b.quad_group = quad_group
    rep = values_to_rep(np.stack([v] * 3))
    for tol in (8.36e-4, 6.52e-4, 6.03e-4):
        bf.b.tolerance = tol
        out = []
        for blocks in (1, 4096):
            bf.b.quad_blocks = blocks
            img, J = bf.jacobian(rep)
            counts = [bf.counters()]
            out.append((img.clone(), J.clone(), bf.render(rep).clone()))
            counts.append(bf.counters())
            for c in counts:
                assert 2 < c["refined"] <= 2048
                assert 16 < c["undecided_select"] <= 16 * 4096
                assert 2 < c["redone"] <= 2048
        for a, b in zip(*out):
            assert torch.equal(a, b)


def test_batch_jacobian_matches_single_model():
    """apx_batch_jacobian: every cutout's model and its 7 representation-space
    Jacobian columns equal the single-model jacobian(as_representation=True)
    within the Jacobian parity bar (2e-4 of each column's max)."""
    truths, shapes, rng = make_cutouts(4, seed=3)
    cuts = [Cutout(np.zeros((s, s)), np.ones((s, s)), psf) for s, psf in shapes]
    bf = BatchFit(cuts)
    rep = values_to_rep(np.stack(truths))
    model, J = bf.jacobian(rep)
    imgs = bf.split(model)
    for k, ((s, psf), v, g) in enumerate(zip(shapes, truths, bf.gal_host)):
        tgt = ap.image.Target_Image(data=np.zeros((s, s)), pixelscale=1.0, psf=ap.image.PSF_Image(data=psf, pixelscale=1.0))
        p = {"center": [v[0], v[1]], "q": v[2], "PA": v[3], "n": v[4], "Re": v[5], "Ie": v[6]}
        m = ap.models.AstroPhot_Model(name=f"j{k}", model_type="sersic galaxy model", target=tgt, parameters=p,
                                      psf_mode="full")
        ref = m().data
        assert float((imgs[k] - ref).abs().max() / ref.abs().max()) < 1e-6, k
        rj = m.jacobian(as_representation=True).flatten("data")
        got = J[g.pix_off:g.pix_off + s * s]
        for c in range(7):
            err = float((got[:, c].double() - rj[:, c].double()).abs().max() / rj[:, c].abs().max())
            assert err < 2e-4, (k, c, err)


def _problem(n, seed):
    truths, shapes, rng = make_cutouts(n, seed)
    cuts, starts = [], []
    bf0 = BatchFit([Cutout(np.zeros((s, s)), np.ones((s, s)), psf) for s, psf in shapes])
    imgs = bf0.split(bf0.render(values_to_rep(np.stack(truths))))
    for (s, psf), v, img in zip(shapes, truths, imgs):
        img = img.double().cpu().numpy()
        var = img / 5.0 + 0.01
        data = img + rng.normal(size=img.shape) * np.sqrt(var)
        cuts.append(Cutout(data, var, psf))
        start = v * (1 + rng.uniform(-0.05, 0.05, 7))
        start[3] = v[3] + rng.uniform(-0.1, 0.1)
        start[2] = min(start[2], 0.97)
        starts.append(start)
    return cuts, np.stack(starts)


@pytest.mark.parametrize("graph,impl", [(False, 0), (True, 0), (True, 3)])
def test_batch_fits_match_single_model_lm(graph, impl):
    """impl 0: the default (MFMA) convolution; impl 3: the separable one,
    whose probe and trial epilogues run inside the captured LM ticks."""
    cuts, starts = _problem(6, seed=2)
    bf = BatchFit(cuts)
    assert bf.sep_all
    bf.b.conv_impl = impl
    res = bf.fit(values_to_rep(starts), use_graph=graph)
    assert (res["status"] > 0).all(), res["status"]
    degenerate = []
    for k, c in enumerate(cuts):
        ny, nx = c.data.shape
        tgt = ap.image.Target_Image(data=c.data, pixelscale=1.0, variance=c.variance,
                                    psf=ap.image.PSF_Image(data=c.psf, pixelscale=1.0))
        v = starts[k]
        p = {"center": [v[0], v[1]], "q": v[2], "PA": v[3], "n": v[4], "Re": v[5], "Ie": v[6]}
        m = ap.models.AstroPhot_Model(name=f"f{k}", model_type="sersic galaxy model", target=tgt, parameters=p,
                                      psf_mode="full")
        lm = ap.fit.LM(m, initial_state=m.parameters.vector_representation()).fit()
        want = m.parameters.vector_values().numpy()
        got = res["values"][k]
        err = np.max(np.abs(got - want) / np.maximum(np.abs(want), 1.0))
        assert abs(res["chi2"][k] - min(lm.loss_history)) / min(lm.loss_history) < CHI2_RTOL
        if err >= PARAM_RTOL:
            # a direction the data barely constrain: the two paths' float32
            # sums (MFMA vs VALU convolution) differ by ~1e-7 of the model and
            # move the end point along it; it must stay far inside the
            # statistical uncertainty (1 % of sigma from the LM covariance)
            sigma = np.sqrt(np.abs(np.diag(lm.covariance_matrix.numpy())))
            assert np.all(np.abs(got - want) <= 0.01 * sigma), (k, got, want, sigma)
            degenerate.append(k)
        # both fits ended; at the optimum the last attempted step may or may not
        # find a float32-noise improvement, so the exit message can differ
        assert res["status"][k] > 0 and lm.message != ""
    assert len(degenerate) <= 1, degenerate


@pytest.mark.parametrize("impl", [0, 3])
def test_two_stream_ticks_are_deterministic(impl):
    """A tick renders each sub-step's probe point on the caller's stream and
    its trial point on a second stream; both read the fit states and write
    their own work lists, planes and taps.  Fits replayed from the captured
    graph twice and run from eager ticks must agree bit for bit: a race
    between the two branches would show here as a difference."""
    cuts, starts = _problem(12, seed=31)
    bf = BatchFit(cuts)
    bf.b.conv_impl = impl
    rep0 = values_to_rep(starts)
    runs = [bf.fit(rep0, use_graph=True), bf.fit(rep0, use_graph=True), bf.fit(rep0, use_graph=False)]
    assert (runs[0]["status"] > 0).all(), runs[0]["status"]
    for r in runs[1:]:
        for key in ("rep", "chi2", "status", "iterations"):
            np.testing.assert_array_equal(r[key], runs[0][key], err_msg=key)


def test_batch_fit_matches_oracle_lm():
    cuts, starts = _problem(2, seed=5)
    bf = BatchFit(cuts)
    res = bf.fit(values_to_rep(starts))
    for k, c in enumerate(cuts):
        ny, nx = c.data.shape
        v = starts[k]
        p = {"center": [v[0], v[1]], "q": v[2], "PA": v[3], "n": v[4], "Re": v[5], "Ie": v[6]}
        om = H.Model([H.Component("sersic", H.Grid(nx, ny), p, psf=torch.tensor(c.psf), psf_mode="full")])
        lm = H.LM(om, torch.tensor(c.data), weight=torch.tensor(1 / c.variance)).fit()
        rv = om.components[0].rep_to_values(torch.as_tensor(lm.res()))
        want = np.concatenate([rv["center"].numpy(), [rv[k2].item() for k2 in ("q", "PA", "n", "Re", "Ie")]])
        err = np.max(np.abs(res["values"][k] - want) / np.maximum(np.abs(want), 1.0))
        assert err < PARAM_RTOL, (k, res["values"][k], want)
        assert abs(res["chi2"][k] - min(lm.loss_history)) / min(lm.loss_history) < CHI2_RTOL


def test_fallback_restart_and_skipped_starts():
    """apx_batch_start_fallback: with max_iter = 1 no run can converge (success
    needs three history entries), so every fit ends its first run at max_iter,
    restarts once from its fallback row, and ends exactly where a plain run
    from that row ends.  A non-finite start is skipped (status 5) without
    touching the other fits."""
    cuts, starts = _problem(6, seed=21)
    bf = BatchFit(cuts, max_iter=1)
    rep_a = torch.tensor(values_to_rep(starts), dtype=torch.float64, device="cuda")
    rep_b = rep_a.clone()
    rep_b[:, 5] += 0.3
    both = bf.fit(rep_a, fallback=rep_b, use_graph=False)
    plain_b = bf.fit(rep_b, use_graph=False)
    assert both["fallback"].all() and (both["iterations"] == 2).all(), (both["fallback"], both["iterations"])
    assert (both["status"] == 4).all()
    np.testing.assert_array_equal(both["rep"], plain_b["rep"])
    np.testing.assert_array_equal(both["chi2"], plain_b["chi2"])
    bf2 = BatchFit(cuts)
    full = bf2.fit(rep_a, use_graph=False)
    rep_nan = rep_a.clone()
    rep_nan[2, 0] = float("nan")
    part = bf2.fit(rep_nan, use_graph=False)
    assert part["status"][2] == 5 and not part["fallback"].any()
    keep = np.arange(6) != 2
    np.testing.assert_array_equal(part["rep"][keep], full["rep"][keep])


def test_launch_shapes_agree_and_autotune():
    """Every launch shape the autotuner may pick (VALU or MFMA convolution,
    32 or 64 lanes per refined pixel or one lane per level-2 sub-pixel with
    10 pixels a workgroup, workgroup counts) renders the same model and
    Jacobian (float32 summation order only: 1e-6 of each column's max), and
    autotune() leaves one of them in the descriptor."""
    truths, shapes, rng = make_cutouts(5, seed=8)
    cuts = [Cutout(np.zeros((s, s)), np.ones((s, s)), psf) for s, psf in shapes]
    bf = BatchFit(cuts)
    rep = torch.tensor(values_to_rep(np.stack(truths)), dtype=torch.float64, device="cuda")
    ref_r = bf.render(rep).clone()
    ref_m, ref_j = [t.clone() for t in bf.jacobian(rep)]
    assert bf.counters()["level3_float"] > 0  # the level-3 branch runs
    for impl, grp, cb, qb, kb in ((1, 0, 0, 0, 0), (2, 64, 7, 3, 5), (1, 64, 1, 1, 1), (2, 0, 4096, 4096, 9),
                                  (3, 0, 0, 0, 0), (3, 64, 5, 2, 3), (1, 25, 0, 0, 0), (3, 25, 5, 1, 3),
                                  (2, 25, 7, 4096, 5)):
        b = bf.b
        b.conv_impl, b.quad_group, b.conv_blocks, b.quad_blocks, b.chunk_blocks = impl, grp, cb, qb, kb
        r = bf.render(rep)
        assert float((r - ref_r).abs().max() / ref_r.abs().max()) < 1e-6, (impl, grp)
        m, j = bf.jacobian(rep)
        assert float((m - ref_m).abs().max() / ref_m.abs().max()) < 1e-6, (impl, grp)
        scale = ref_j.abs().amax(dim=0)
        assert float(((j - ref_j).abs().amax(dim=0) / scale).max()) < 1e-6, (impl, grp)
    tuning = bf.autotune(rep)
    ch = tuning["choice"]
    assert ch["conv_impl"] in ("mfma", "valu", "sep") and ch["quad_group"] in (25, 32, 64)
    assert ch["conv_blocks"] > 0 and ch["quad_blocks"] > 0 and ch["chunk_blocks"] > 0
    m, j = bf.jacobian(rep)
    assert float((m - ref_m).abs().max() / ref_m.abs().max()) < 1e-6



def test_separable_convolution_sheared_pixels_and_refusal():
    """conv_impl 3 on a sheared pixelscale (the centre columns mix the two
    separable derivative convolutions through P^-1, as the MFMA taps do)
    agrees with the MFMA convolution to float32 summation order; a batch with
    a PSF that is not rank one refuses conv_impl 3."""
    truths, shapes, rng = make_cutouts(4, seed=13)
    P = [[0.9, 0.12], [-0.07, 1.1]]
    cuts = [Cutout(np.zeros((s, s)), np.ones((s, s)), psf) for s, psf in shapes]
    bf = BatchFit(cuts, pixelscale=P)
    rep = torch.tensor(values_to_rep(np.stack(truths)), dtype=torch.float64, device="cuda")
    bf.b.conv_impl = 2
    ref_m, ref_j = [t.clone() for t in bf.jacobian(rep)]
    bf.b.conv_impl = 3
    m, j = bf.jacobian(rep)
    assert float((m - ref_m).abs().max() / ref_m.abs().max()) < 1e-6
    scale = ref_j.abs().amax(dim=0)
    assert float(((j - ref_j).abs().amax(dim=0) / scale).max()) < 1e-6
    moffat = ap.utils.moffat_psf(3.0, 2.0, 11, 1.0)
    mixed = BatchFit(cuts[:2] + [Cutout(np.zeros((40, 40)), np.ones((40, 40)), moffat)])
    assert not mixed.sep_all
    mixed.b.conv_impl = 3
    rep3 = torch.tensor(values_to_rep(np.stack(truths[:2] + [truths[0]])), dtype=torch.float64, device="cuda")
    with pytest.raises(ap.errors.APXError, match="conv_impl 3"):
        mixed.render(rep3)


def test_quadrature_rerun_and_work_counters():
    """parts=4 re-runs the float32 level-2/3 quadrature pass on the previous
    render's lists: the planes, and so the convolved render, stay bit-equal;
    the work counters add that pass's level-3 sub-pixels once per run."""
    truths, shapes, rng = make_cutouts(5, seed=17)
    cuts = [Cutout(np.zeros((s, s)), np.ones((s, s)), psf) for s, psf in shapes]
    bf = BatchFit(cuts)
    rep = torch.tensor(values_to_rep(np.stack(truths)), dtype=torch.float64, device="cuda")
    ref = bf.render(rep).clone()
    c1 = bf.counters()
    assert c1["fits"] == 5 and c1["refined"] > 0 and c1["tiles"] == int(bf.b.ntile)
    assert bf.quad_evaluations(c1) == 225 * (c1["refined"] + c1["level3_float"])
    for _ in range(3):
        bf.render(rep, parts=4)
    c2 = bf.counters()
    assert c2["refined"] == c1["refined"] and c2["level3_float"] == 4 * c1["level3_float"]
    out = torch.zeros_like(ref)
    bf.render(rep, out=out, parts=2)
    assert torch.equal(out, ref)


def test_mfma_convolution_wide_psf():
    """A 65 x 65 Moffat PSF (67-px shifted kernel, 21 k-steps a column, 128 KiB
    of LDS a workgroup): the MFMA Jacobian-stage convolution agrees with the
    VALU one to float32 summation order -- 4489-term sums, so the bar is the
    image parity bar, 1e-5 of each column's max (about sqrt(4489) float32
    epsilons), rather than the 1e-6 of the short kernels above."""
    truths, shapes, rng = make_cutouts(3, seed=23, sizes=(70, 90))
    psf = ap.utils.moffat_psf(3.5, 2.9, 65, 1.0)
    cuts = [Cutout(np.zeros((s, s)), np.ones((s, s)), psf) for s, _ in shapes]
    bf = BatchFit(cuts)
    assert not bf.sep_all and bf.b.max_kernel == 67
    rep = torch.tensor(values_to_rep(np.stack(truths)), dtype=torch.float64, device="cuda")
    bf.b.conv_impl = 1
    ref_m, ref_j = [t.clone() for t in bf.jacobian(rep)]
    bf.b.conv_impl = 2
    m, j = bf.jacobian(rep)
    assert float((m - ref_m).abs().max() / ref_m.abs().max()) < 1e-5
    scale = ref_j.abs().amax(dim=0)
    assert float(((j - ref_j).abs().amax(dim=0) / scale).max()) < 1e-5


# double offsets in the per-fit LM state (csrc/batch.hip GalState): H (7 x 7),
# g (7) and chi2(m0) follow x, ev, L, init_chi2, hist, res_chi2, res_x,
# best_dx, best_chi2, best_L, scary_dx, scary_chi2, scary_L (57 doubles), and
# h, a, ha, rpp (32 doubles) sit between g and chi2(m0)
_H0, _G0, _C0 = 57, 57 + 49, 57 + 49 + 7 + 32


@pytest.mark.parametrize("impl", [0, 3])
def test_normal_equations_of_the_jacobian_stage(impl):
    """The first tick's Jacobian stage writes, per fit, H = J^T W J,
    g = J^T W (Y - m0) and chi2(m0) = sum W (Y - m0)^2 from per-tile partial
    sums (normal_kernel, tile_reduce_kernel).  Against float64 sums over the
    model and J that the same stage leaves in the batch buffers, on cutouts
    whose widths are not a multiple of 64 and heights not of 16 (partial
    tiles), with a masked-out pixel (zero weight) in each."""
    rng = np.random.default_rng(11)
    cuts, starts = [], []
    for ny, nx in ((37, 45), (19, 70), (33, 129)):
        sig = rng.uniform(1.0, 2.0)
        psf = H.gaussian_psf(sig, 2 * math.ceil(4 * sig) + 1, 1.0)
        data = rng.normal(size=(ny, nx)) + 2.0 * np.exp(-((np.arange(nx) - nx / 2) ** 2)[None, :] / 50.0
                                                      - ((np.arange(ny) - ny / 2) ** 2)[:, None] / 30.0)
        var = rng.uniform(0.5, 2.0, size=(ny, nx))
        var[ny // 3, nx // 4] = np.inf
        cuts.append(Cutout(data, var, psf))
        starts.append([nx / 2 + 0.3, ny / 2 - 0.2, 0.7, 0.8, 2.0, 4.0, 0.3])
    bf = BatchFit(cuts)
    bf.b.conv_impl = impl
    bf.start(values_to_rep(np.array(starts)))
    bf.tick()
    torch.cuda.synchronize()
    sb = bf.lib.apx_batch_state_bytes()
    st = bf.state.view(len(cuts), sb)[:, :8 * (_C0 + 1)].contiguous().view(torch.float64).cpu().numpy()
    m0 = bf.model0.double().cpu().numpy()
    J = bf.jac.view(7, bf.npix).double().cpu().numpy()
    Y = bf.data.double().cpu().numpy()
    Wt = bf.weight.double().cpu().numpy()
    for k, g in enumerate(bf.gal_host):
        sl = slice(g.pix_off, g.pix_off + g.nx * g.ny)
        Jk, w, r = J[:, sl], Wt[sl], Y[sl] - m0[sl]
        assert np.count_nonzero(w == 0) == 1
        Hw = (Jk * w) @ Jk.T
        gw = Jk @ (w * r)
        cw = float(np.sum(w * r * r))
        Hg = st[k, _H0:_H0 + 49].reshape(7, 7)
        gg = st[k, _G0:_G0 + 7]
        scale = np.sqrt(np.outer(np.diag(Hw), np.diag(Hw)))
        assert np.all(np.abs(Hg - Hw) <= 1e-5 * scale), (k, np.max(np.abs(Hg - Hw) / scale))
        gs = np.sqrt(np.diag(Hw) * cw)
        assert np.all(np.abs(gg - gw) <= 1e-5 * gs), (k, np.abs(gg - gw) / gs)
        assert abs(st[k, _C0] - cw) <= 1e-6 * cw, (k, st[k, _C0], cw)
