"""Host-side checks that need no GPU: the C-ABI library, window geometry,
parameter vectors and the launch descriptors the engine builds."""

import ctypes
import math
import os
import re

import numpy as np
import pytest
import torch
from scipy.special import roots_legendre

import astrophot_amd as ap
from astrophot_amd import _lib as L
from oracle import hotpath as H

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "astrophot_hip.h")


def header_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(apx_\w+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    assert L.LIB_PATH.exists(), "run python -m astrophot_amd._build"
    lib = ctypes.CDLL(str(L.LIB_PATH))
    syms = header_symbols()
    assert len(syms) >= 10
    for s in syms:
        assert hasattr(lib, s), s
    assert sorted(L.SIGNATURES) == syms


def test_struct_layouts_match_header():
    """ctypes mirrors of apx_component / apx_conv_job list every header field in order."""
    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    from astrophot_amd import batch as B
    for cname, cls in (("apx_component", L.Component), ("apx_conv_job", L.ConvJob),
                       ("apx_batch_galaxy", B.Galaxy), ("apx_batch", B.Batch), ("apx_group", L.Group),
                       ("apx_block_sum", L.BlockSum)):
        body = re.search(r"typedef struct %s \{(.*?)\} %s;" % (cname, cname), text, re.S).group(1)
        fields = []
        for decl in body.split(";"):
            decl = decl.strip()
            if not decl:
                continue
            decl = re.sub(r"^const\s+", "", decl)
            names = decl.split(None, 1)[1].replace("*", " ")
            for n in names.split(","):
                fields.append(re.sub(r"\[.*\]", "", n).strip())
        assert [f[0] for f in cls._fields_] == fields, cname


def test_library_workspace_queries_without_gpu():
    lib = ctypes.CDLL(str(L.LIB_PATH))
    lib.apx_render_workspace_bytes.restype = ctypes.c_int64
    lib.apx_render_workspace_bytes.argtypes = [ctypes.c_int64]
    assert lib.apx_render_workspace_bytes(1000) >= 8 * 1000


def test_sersic_light_fraction_matches_scipy():
    """The host growth curve the moment initialiser inverts, P(2n, b_n r^(1/n)),
    against scipy's regularised incomplete gamma; and the half-light property
    that defines b_n (exact up to the b_n polynomial's own accuracy)."""
    from scipy.special import gammainc
    lib = ctypes.CDLL(str(L.LIB_PATH))
    f = lib.apx_sersic_light_fraction
    f.restype = ctypes.c_double
    f.argtypes = [ctypes.c_double, ctypes.c_double]
    for n in (0.36, 0.5, 1.0, 2.5, 4.0, 8.0):
        b = H.sersic_n_to_b(torch.tensor(n, dtype=torch.float64)).item()
        for r in (0.05, 0.3, 1.0, 2.0, 7.5):
            assert abs(f(n, r) - gammainc(2 * n, b * r ** (1 / n))) < 1e-10, (n, r)
        assert abs(f(n, 1.0) - 0.5) < 2e-3, n


def test_product_fails_loudly_without_gpu():
    if torch.cuda.is_available():
        pytest.skip("GPU visible")
    with pytest.raises(ap.errors.APXError):
        L.load()


@pytest.mark.parametrize("P", [1.0, 0.8, [[0.9, 0.1], [-0.05, 1.1]]])
def test_window_geometry_matches_oracle(P):
    w = ap.image.Window(pixel_shape=(40, 30), pixelscale=P)
    g = H.Grid(40, 30, P)
    assert torch.allclose(w.origin, g.origin) and torch.allclose(w.end, g.end)
    xy = torch.tensor([3.3, -1.7], dtype=torch.float64)
    assert torch.allclose(w.plane_to_pixel(xy), g.plane_to_pixel(xy))
    assert torch.allclose(w.get_coordinate_meshgrid(), g.meshgrid())
    # pad / crop keep the plane position of pixels
    w2 = w.copy().pad_pixel((5, 4))
    g2 = g.copy().pad(5, 4)
    assert (w2.nx, w2.ny) == (g2.nx, g2.ny) and torch.allclose(w2.reference_imageij, g2.ref_ij)
    # intersection / union / indices (window_object.py:241-253, 483-523)
    o = ap.image.Window(pixel_shape=(12, 9), origin=w.pixel_to_plane(torch.tensor([30.5, 20.5])), pixelscale=P)
    og = H.Grid(12, 9, P, ref_xy=g.pixel_to_plane(torch.tensor([30.5, 20.5], dtype=torch.float64)))
    a, ag = w & o, g & og
    assert (a.nx, a.ny) == (ag.nx, ag.ny) and torch.allclose(a.origin, ag.origin)
    u, ug = w | o, g | og
    assert (u.nx, u.ny) == (ug.nx, ug.ny) and torch.allclose(u.origin, ug.origin)
    assert w.get_self_indices(o) == H.Grid.indices(g, og)


def test_window_slicing_kat():
    """test_window.py:87-103 style: a sub-window's indices into its parent."""
    w = ap.image.Window(pixel_shape=(100, 100), pixelscale=1.0)
    sub = w.copy().crop_to_pixel([[10, 30], [20, 45]])
    assert w.get_self_indices(sub) == (slice(20, 45), slice(10, 30))


def test_psf_border_and_odd_shape():
    """test_image.py:412-436: border of a 9x9 PSF is 5; even PSFs are rejected."""
    p = ap.image.PSF_Image(data=np.ones((9, 9)), pixelscale=1.0)
    assert p.psf_border_int == (5, 5)
    with pytest.raises(ap.errors.SpecificationConflict):
        ap.image.PSF_Image(data=np.ones((8, 9)), pixelscale=1.0)


def test_reduce_sums_blocks():
    """test_image.py:438-459."""
    img = ap.image.Target_Image(data=np.ones((30, 36)), pixelscale=1.0)
    small = img.reduce(3)
    assert tuple(small.data.shape) == (10, 12) and float(small.data[0, 0]) == 9.0


def test_parameter_kats():
    """test_parameter.py:117-161."""
    P = ap.param.Parameter_Node("low", limits=(1, None))
    P.value = 100.0
    with pytest.raises(ap.errors.InvalidParameter):
        P.value = -100.0
    P = ap.param.Parameter_Node("cyc", limits=(-1, 1), cyclic=True)
    P.value = 2.0
    assert P.value.item() == 0.0
    P.value = -2.0
    assert P.value.item() == 0.0


def test_parameter_vector_round_trip_masked():
    """test_parameter.py:379-418 (without the functional node)."""
    P1 = ap.param.Parameter_Node("t1", value=0.5, limits=(-1, 1))
    P2 = ap.param.Parameter_Node("t2", value=2.0)
    P3 = ap.param.Parameter_Node("t3", value=[4.0, 5.0], limits=(1.0, None))
    P6 = ap.param.Parameter_Node("t6", value=((5, 6), (7, 8)), limits=(None, 10.0))
    G = ap.param.Parameter_Node("g")
    for p in (P1, P2, P3, P6):
        G.link(p)
    assert len(G.vector_representation()) == 8
    mask = torch.tensor([1, 1, 0, 1, 0, 1, 0, 1], dtype=torch.bool)
    with ap.param.Param_Mask(G, mask):
        vec = G.vector_values().clone()
        G.vector_set_representation(G.vector_representation())
        assert torch.allclose(vec, G.vector_values(), rtol=1e-12)
        assert G.vector_values().numel() == 5


def test_model_parameter_order_and_reps_match_oracle():
    tgt = ap.image.Target_Image(data=np.zeros((36, 40)), pixelscale=1.0)
    p = {"center": [20.3, 17.6], "q": 0.6, "PA": 3.5, "n": 2.5, "Re": 6.0, "Ie": 1.0}
    m = ap.models.AstroPhot_Model(name="s", model_type="sersic galaxy model", target=tgt, parameters=p)
    oc = H.Component("sersic", H.Grid(40, 36), p)
    # PA wraps into [0, pi) on set (parameter.py:436-440)
    assert m["PA"].value.item() == pytest.approx(3.5 - math.pi)
    rep = m.parameters.vector_representation()
    assert torch.allclose(rep, oc.val_to_rep(oc.vector_values()).reshape(-1) if False else
                          H.Model([H.Component("sersic", H.Grid(40, 36), dict(p, PA=3.5 - math.pi))]).vector_representation())
    assert list(m.parameters.vector_names()) == ["center:0", "center:1", "q", "PA", "n", "Re", "Ie"]
    with pytest.raises(ap.errors.UnrecognizedModel):
        ap.models.AstroPhot_Model(name="x", model_type="nonexistent model", target=tgt)


class _FakeLib:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def f(*a):
            self.calls.append((name, a))
            return 1 << 12 if name.endswith("workspace_bytes") else 0
        return f


def test_engine_descriptors(monkeypatch):
    """Geometry handed to the render kernel equals the oracle's working grid."""
    fake = _FakeLib()
    monkeypatch.setattr(L, "load", lambda require_gpu=True: fake)
    monkeypatch.setattr(L, "stream", lambda: 0)
    psf = H.gaussian_psf(1.5, 11, 1.0)
    tgt = ap.image.Target_Image(data=np.zeros((36, 40)), pixelscale=0.8, psf=ap.image.PSF_Image(data=psf, pixelscale=0.8))
    p = {"center": [16.3, 14.1], "q": 0.6, "PA": 0.7, "n": 2.5, "Re": 6.0, "Ie": 1.0}
    m = ap.models.AstroPhot_Model(name="s", model_type="sersic galaxy model", target=tgt, parameters=p,
                                  psf_mode="full")
    m()
    comp = [a for n, a in fake.calls if n == "apx_render_component"][0][0]._obj
    g = H.Grid(40, 36, 0.8).pad(6, 6)  # 11x11 PSF: border ceil(12/2) = 6
    pc = g.plane_to_pixel(torch.tensor(p["center"], dtype=torch.float64))
    assert (comp.nx, comp.ny) == (g.nx, g.ny)
    assert (comp.ci, comp.cj) == tuple(int(v) for v in torch.round(pc))
    assert comp.frac[0] == 0.0 and comp.frac[1] == 0.0
    F = H.sersic_Ie_to_flux(torch.tensor(10.0, dtype=torch.float64), torch.tensor(2.5, dtype=torch.float64), 6.0, 0.6).item()
    assert comp.reference == pytest.approx(F / (g.nx * g.ny), rel=1e-12)
    assert comp.pixel_area == pytest.approx(0.64)
    shift = [a for n, a in fake.calls if n == "apx_psf_shift"][0]
    assert shift[3] == pytest.approx(float(pc[0] - torch.round(pc[0])))
    assert shift[4] == pytest.approx(float(pc[1] - torch.round(pc[1])))
    conv = [a for n, a in fake.calls if n == "apx_convolve"][0][0]._obj
    assert (conv.x0, conv.y0, conv.ow, conv.oh) == (6, 6, 40, 36)


@pytest.mark.parametrize("mode,code,n,nodes,weights", [
    ("midpoint", 0, None, None, None),
    ("simpsons", 1, 3, [-1.0, 0.0, 1.0], [1 / 3, 4 / 3, 1 / 3]),
    ("quad:4", 1, 4, list(roots_legendre(4)[0]), list(roots_legendre(4)[1])),
    ("trapezoid", 2, 2, [-1.0, 1.0], [1.0, 1.0]),
])
def test_sampling_mode_descriptors(monkeypatch, mode, code, n, nodes, weights):
    """_model_methods.py:82-148: each sampling mode's rule as the render
    kernel receives it; the weights w_u w_v / 4 sum to one on every pixel."""
    fake = _FakeLib()
    monkeypatch.setattr(L, "load", lambda require_gpu=True: fake)
    monkeypatch.setattr(L, "stream", lambda: 0)
    tgt = ap.image.Target_Image(data=np.zeros((20, 24)), pixelscale=1.0)
    m = ap.models.AstroPhot_Model(name="s", model_type="sersic galaxy model", target=tgt, sampling_mode=mode,
                                  parameters={"center": [12.3, 9.1], "q": 0.6, "PA": 0.7, "n": 2.5, "Re": 4.0,
                                              "Ie": 1.0})
    m()
    comp = [a for nm, a in fake.calls if nm == "apx_render_component"][0][0]._obj
    assert comp.sampling == code
    if n is not None:
        assert comp.sample_quad == n
        assert np.allclose(list(comp.sq_node)[:n], nodes, rtol=0, atol=1e-15)
        assert np.allclose(list(comp.sq_weight)[:n], weights, rtol=0, atol=1e-15)
        assert sum(weights) ** 2 / 4 == pytest.approx(1.0, abs=1e-14)


def test_unknown_sampling_mode_raises(monkeypatch):
    fake = _FakeLib()
    monkeypatch.setattr(L, "load", lambda require_gpu=True: fake)
    monkeypatch.setattr(L, "stream", lambda: 0)
    tgt = ap.image.Target_Image(data=np.zeros((20, 24)), pixelscale=1.0)
    m = ap.models.AstroPhot_Model(name="s", model_type="sersic galaxy model", target=tgt, sampling_mode="boole",
                                  parameters={"center": [12.3, 9.1], "q": 0.6, "PA": 0.7, "n": 2.5, "Re": 4.0,
                                              "Ie": 1.0})
    with pytest.raises(ap.errors.SpecificationConflict, match="trapezoid"):
        m()


@pytest.mark.parametrize("U", [2, 3])
def test_upscaled_render_geometry(monkeypatch, U):
    """model_object.py:313-349: the working grid of a PSF U times finer than
    the image is the window rescaled by float32(1/U) and padded by the PSF
    border in fine pixels; the convolved fine box is summed back in U x U
    blocks onto the image (one pixel short per axis for U = 3)."""
    fake = _FakeLib()
    monkeypatch.setattr(L, "load", lambda require_gpu=True: fake)
    monkeypatch.setattr(L, "stream", lambda: 0)
    psf = H.gaussian_psf(1.3, 13, 1.0 / U)
    tgt = ap.image.Target_Image(data=np.zeros((26, 30)), pixelscale=0.8, psf=psf, psf_upscale=U)
    assert float(tgt.psf.pixel_length) == pytest.approx(0.8 / U)
    m = ap.models.AstroPhot_Model(name="s", model_type="sersic galaxy model", target=tgt, psf_mode="full",
                                  parameters={"center": [12.3, 9.1], "q": 0.6, "PA": 0.7, "n": 2.5, "Re": 4.0,
                                              "Ie": 1.0})
    m()
    s = float(np.float32(1.0 / U))
    comp = [a for n, a in fake.calls if n == "apx_render_component"][0][0]._obj
    nfx, nfy = int(30 // s), int(26 // s)
    assert (comp.nx, comp.ny) == (nfx + 14, nfy + 14)  # 13 x 13 PSF: border 7 fine pixels
    assert comp.P[0] == pytest.approx(0.8 * s, rel=1e-15) and comp.pixel_area == pytest.approx((0.8 * s) ** 2)
    conv = [a for n, a in fake.calls if n == "apx_convolve"][0][0]._obj
    bs = [a for n, a in fake.calls if n == "apx_block_sum_add"][0][0]._obj
    assert (bs.scale, bs.nc, bs.w, bs.h) == (U, 1, nfx // U, nfy // U)
    assert (conv.x0, conv.y0, conv.ow, conv.oh) == (7, 7, U * bs.w, U * bs.h)
    assert (bs.dst_x0, bs.dst_y0, bs.dst_w, bs.dst_h) == (0, 0, 30, 26)


def test_rank_one_factors():
    """Separable-convolution eligibility: Gaussian PSFs (gaussian_psf, a
    block-averaged product of 1-D Gaussians) factor to rounding; a Moffat PSF,
    a zero PSF and a rank-two image do not."""
    from astrophot_amd.batch import rank_one_factors
    from astrophot_amd.utils import moffat_psf
    gs = [H.gaussian_psf(s, 2 * math.ceil(4 * s) + 1, 1.0) for s in (1.0, 1.7, 2.9)]
    rank2 = np.outer(np.arange(1.0, 8.0), np.ones(7)) + np.outer(np.ones(7), np.arange(7.0) ** 2)
    f = rank_one_factors(gs + [moffat_psf(3.0, 2.0, 11, 1.0), np.zeros((5, 5)), rank2])
    for p, uv in zip(gs, f[:3]):
        assert uv is not None and np.abs(np.outer(*uv) - p).max() <= 1e-15 * p.max()
    assert f[3:] == [None, None, None]


def test_device_decode_matches_the_host_decode():
    """The learned step decodes the network outputs and maps them to the LM
    representation with torch (on the GPU); on CPU tensors the torch versions
    must agree with the numpy ones (cnn.decode, batch.values_to_rep) to
    rounding, over outputs that reach every clamp."""
    from astrophot_amd.batch import values_to_rep, values_to_rep_device
    from astrophot_amd.cnn import decode, decode_device
    rng = np.random.default_rng(3)
    t = (rng.standard_normal((4096, 8)) * 3.0).astype(np.float32)
    sigma = rng.uniform(0.5, 20.0, 4096).astype(np.float32)
    v = decode(t, sigma)
    vd = decode_device(torch.as_tensor(t), torch.as_tensor(sigma)).numpy()
    assert vd.dtype == np.float64
    np.testing.assert_allclose(vd[:, :6], v[:, :6], rtol=1e-12, atol=1e-12)
    # log10(sigma) + 1.2 is float32 in both (numpy's promotion), and float32
    # log10 may round one ulp apart between the two libraries
    np.testing.assert_allclose(vd[:, 6], v[:, 6], rtol=0, atol=5e-7)
    # the clamps were reached
    assert (v[:, 2] == 0.98).any() and (v[:, 2] == 0.05).any() and (v[:, 4] == 7.5).any()
    r = values_to_rep(v)
    rd = values_to_rep_device(torch.as_tensor(v)).numpy()
    np.testing.assert_allclose(rd, r, rtol=1e-12, atol=1e-9)


LIMITS = [((None, None), False), ((0.0, None), False), ((None, 3.0), False), ((0.36, 8.0), False), ((0.0, math.pi), True)]


@pytest.mark.parametrize("limits,cyclic", LIMITS)
def test_float_parameter_maps_equal_the_tensor_maps(limits, cyclic):
    """The maps on Python floats against the tensor ones, at ordinary values,
    at the limits, at infinities and NaN: equal to the last bits of the two
    math libraries (4 ulp)."""
    from astrophot_amd import param as PM
    n = PM.Parameter_Node("p", limits=limits, cyclic=cyclic)
    for x in (0.5, 1.3, 2.7, -4.0, 1e300, math.inf, -math.inf, math.nan, 0.36, 0.0, 3.0, 8.0):
        t = torch.tensor(x, dtype=torch.float64)
        for tensor_map, float_map in ((n._leaf_rep_to_val, PM._rep_to_val1), (n._leaf_val_to_rep, PM._val_to_rep1),
                                      (n._leaf_dval_drep, PM._dval_drep1)):
            a, b = float(tensor_map(t)), float_map(x, *limits, cyclic)
            assert (math.isnan(a) and math.isnan(b)) or a == b or abs(a - b) <= 4 * 2.3e-16 * abs(a), (x, a, b)


def test_plain_vectors_equal_the_tensor_path():
    """Reading and setting the flat vector of a tree: a plain vector (Python
    floats) and one that carries a graph (tensor operations) leave the same
    values; a masked tree and a wrong length take the tensor path as before."""
    from astrophot_amd.errors import InvalidParameter
    from astrophot_amd.param import Param_Mask, Parameter_Node

    def tree():
        top = Parameter_Node("top")
        for k, (lim, cyc) in enumerate(LIMITS):
            top.link(Parameter_Node(f"p{k}", value=[1.1, 2.1] if k == 0 else 1.3 + 0.1 * k, limits=lim, cyclic=cyc))
        return top

    a, b = tree(), tree()
    rep = a.vector_representation() * 1.01 + 0.01
    a.vector_set_representation(rep)
    b.vector_set_representation(rep.clone().requires_grad_(True))
    assert not a["p0"].value.requires_grad and b["p0"].value.requires_grad
    assert torch.allclose(a.vector_values(), b.vector_values().detach(), rtol=1e-15, atol=0)
    assert [n.value.shape for n in a._leaves()] == [n.value.shape for n in b._leaves()]
    assert list(a.vector_identities()) == a._identities() and len(a._identities()) == 6
    a.vector_set_values(b.vector_values().detach())
    assert torch.equal(a.vector_values(), b.vector_values().detach())
    with Param_Mask(a, torch.tensor([True, False, True, True, False, True])):
        assert len(a.vector_values()) == len(a._identities()) == len(a.vector_identities()) == 4
        a.vector_set_values(a.vector_values() * 1.001)
    with pytest.raises((InvalidParameter, RuntimeError)):
        a.vector_set_values(torch.ones(9, dtype=torch.float64))


@pytest.mark.parametrize("limits,cyclic", [((2.0, 2.0), False), ((2.0, 2.0), True), ((3.0, 1.0), True), ((-0.0, 0.0), True)])
def test_float_parameter_maps_of_degenerate_limits(limits, cyclic):
    """Equal or crossed limits: the float maps give what the tensor maps do, NaN
    where those divide by zero, and raise nothing."""
    from astrophot_amd import param as PM
    n = PM.Parameter_Node("p", limits=limits, cyclic=cyclic)
    for x in (2.0, 0.5, -3.25, 0.0, math.inf, math.nan):
        t = torch.tensor(x, dtype=torch.float64)
        for tensor_map, float_map in ((n._leaf_rep_to_val, PM._rep_to_val1), (n._leaf_val_to_rep, PM._val_to_rep1),
                                      (n._leaf_dval_drep, PM._dval_drep1)):
            a, b = float(tensor_map(t)), float_map(x, *limits, cyclic)
            assert (math.isnan(a) and math.isnan(b)) or a == b or abs(a - b) <= 4 * 2.3e-16 * abs(a), (x, a, b)


def test_values_set_under_another_type_or_with_a_graph_are_kept():
    """Values of another type than the present one (set before it changed) are
    read as they are, not rounded to it, and a vector of the present type is not
    taken for them; a value that carries a graph keeps taking part in it."""
    from astrophot_amd import AP_config
    from astrophot_amd.param import Parameter_Node
    top = Parameter_Node("top")
    for k in range(2):
        top.link(Parameter_Node(f"p{k}", value=[1.1 + k, 1.6 + k]))
    old = AP_config.ap_dtype
    AP_config.ap_dtype = torch.float32
    try:
        assert torch.equal(top.vector_values(), torch.tensor([1.1, 1.6, 2.1, 2.6], dtype=torch.float64))
        with pytest.raises(RuntimeError):
            top.vector_set_values(torch.ones(4))
    finally:
        AP_config.ap_dtype = old
    top.vector_set_values(torch.ones(4, dtype=torch.float64, requires_grad=True))
    top.vector_set_values(torch.arange(4, dtype=torch.float64))
    assert top.vector_values().requires_grad and top.vector_values().tolist() == [0.0, 1.0, 2.0, 3.0]


def _pair():
    from astrophot_amd.param import Parameter_Node
    top = Parameter_Node("top")
    top.link(Parameter_Node("a", value=1.1, limits=(0.0, None)))
    top.link(Parameter_Node("b", value=2.1))
    return top


def test_vector_operations_are_followed_by_traces_and_transforms(monkeypatch):
    """A trace, a dispatch mode, a functorch transform and a tangent see the
    vector's operations, so the result follows the input; and where torch's
    private questions about them are gone, everything stays on the tensor path."""
    from torch.utils._python_dispatch import TorchDispatchMode
    from astrophot_amd import param as PM

    class Count(TorchDispatchMode):
        seen = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Count.seen += func is torch.ops.aten.sqrt.default
            return func(*args, **(kwargs or {}))

    top, v = _pair(), torch.tensor([0.7, 1.9], dtype=torch.float64)

    def run(x):
        top.vector_set_representation(x)
        return top.vector_values()

    want = run(v + 0.25)
    assert not want.requires_grad and PM._plain(v) and top._plain_leaves() is not None
    traced = torch.jit.trace(run, (v,), check_trace=False)
    assert torch.allclose(traced(v + 0.25), want, rtol=1e-15, atol=0)
    top.vector_set_values(v.clone())
    with Count():
        run(v)
    assert Count.seen == 1
    d = torch.func.jvp(run, (v,), (torch.ones_like(v),))[1]
    assert torch.allclose(d, top.vector_dval_drep(v).detach(), rtol=1e-15, atol=0)
    for owner, name in ((torch._C, "_are_functorch_transforms_active"), (torch._C, "_len_torch_dispatch_stack"),
                        (torch.autograd.forward_ad, "_current_level")):
        top = _pair()
        with monkeypatch.context() as m:
            m.delattr(owner, name)
            assert top._plain_leaves() is None
            if owner is torch._C:
                assert torch.allclose(run(v + 0.25), want, rtol=1e-15, atol=0)


def test_vectors_stay_on_the_host_under_a_default_device():
    """Values live on the host whatever torch's default device is."""
    top = _pair()
    with torch.device("meta"):
        assert top.vector_values().device.type == "cpu"
        top.vector_set_representation(torch.tensor([0.7, 1.9], dtype=torch.float64, device="cpu"))
        top.vector_set_values(top.vector_values())
    assert all(n.value.device.type == "cpu" for n in top._leaves())


@pytest.mark.parametrize("mask", [[True] * 5, [True, False, True, True, False], [False] * 5])
def test_masked_vectors_on_floats_equal_the_tensor_path(mask):
    """Under a mask, and after one, the vector is read and set by floats as
    without: the same values, masked ones untouched."""
    from astrophot_amd.param import Param_Mask, Parameter_Node
    made = []
    for graph in (False, True):
        top = Parameter_Node("top")
        for k, (lim, cyc) in enumerate(LIMITS[:4]):
            top.link(Parameter_Node(f"p{k}", value=[1.1, 2.1] if k == 1 else 1.3 + 0.1 * k, limits=lim, cyclic=cyc))
        with Param_Mask(top, torch.tensor(mask)):
            assert top._plain_leaves() is not None
            rep = top.vector_representation() * 1.01 + 0.01
            assert len(rep) == sum(mask)
            top.vector_set_representation(rep.requires_grad_(graph))
            made.append(top.vector_values().detach())
        assert top._plain_leaves() is not None or graph
        made.append(top.vector_values().detach())
    assert torch.allclose(made[0], made[2], rtol=1e-15, atol=0) and torch.allclose(made[1], made[3], rtol=1e-15, atol=0)


def test_stream_handle_without_the_private_interface(monkeypatch):
    """The current stream's handle comes from the public Stream object where torch
    has no raw one to give."""
    class Stream:
        cuda_stream = 77

    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: Stream() if device == 3 else None)
    monkeypatch.delattr(torch._C, "_cuda_getDevice", raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda device: 78 + device, raising=False)
    assert L.stream() == 81
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream")
    assert L.stream() == 77


def test_convolution_grids_reach_every_work_item():
    """The MFMA convolution's items are the 7 passes of a tile: a small batch's
    tuned launch can have a workgroup for each, and none has more."""
    from astrophot_amd.batch import conv_grids
    for ntile in (1, 4, 146, 147, 420, 5000):
        assert max(conv_grids(ntile, 2)) == min(7 * ntile, 16384)
        for impl in (1, 3):
            assert max(conv_grids(ntile, impl)) == min(ntile, 16384)
