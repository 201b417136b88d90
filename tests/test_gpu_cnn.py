"""The learned initialiser's kernels (csrc/cnn.hip) against torch float32 on
the CPU.

* apx_gemm_bf16: every operand orientation, split-K and the bias / ReLU
  epilogue, against a float32 matmul of the same bf16-rounded operands
  (tolerance: float32 accumulation order, 1e-5 of the scale);
* the network forward pass and every weight and bias gradient against torch
  autograd on the CPU through the same layers, with the same bf16 rounding
  points emulated (activations and back-propagated gradients rounded to bf16
  where the kernels store them);
* a short training run on renderer-generated cutouts lowers the loss.
"""

import ctypes

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from astrophot_amd import _lib as L
from astrophot_amd import cnn

pytestmark = pytest.mark.gpu

DEV = "cuda"


def bf(x):
    return x.to(torch.bfloat16).to(torch.float32)


@pytest.mark.parametrize("M,N,K,ta,tb,split", [(64, 64, 32, False, False, False), (100, 37, 75, False, False, False),
                                               (33, 130, 300, True, False, False), (70, 20, 96, False, True, False),
                                               (32, 32, 20000, True, False, True), (288, 32, 9000, True, False, True)])
def test_gemm_bf16_matches_float32(M, N, K, ta, tb, split):
    g = torch.Generator().manual_seed(M * 7 + N)
    A = torch.randn((K, M) if ta else (M, K), generator=g)
    B = torch.randn((N, K) if tb else (K, N), generator=g)
    bias = torch.randn(N, generator=g)
    Ab, Bb = A.to(torch.bfloat16).to(DEV), B.to(torch.bfloat16).to(DEV)
    sam, sak = (1, M) if ta else (K, 1)
    sbk, sbn = (1, K) if tb else (N, 1)
    C = torch.zeros((M, N), device=DEV)
    Cb = torch.zeros((M, N), dtype=torch.bfloat16, device=DEV)
    ws = torch.zeros(1 << 22, device=DEV) if split else None
    cnn.gemm(Ab, sam, sak, Bb, sbk, sbn, C, M, N, K, bias=bias.to(DEV), relu=True, Cb=Cb, ws=ws)
    Af, Bf = bf(A), bf(B)
    ref = torch.relu((Af.t() if ta else Af).double() @ (Bf.t() if tb else Bf).double() + bias.double())
    scale = float((Af.abs().double().t() if ta else Af.abs().double()).max() * (Bf.abs().max()) * K ** 0.5)
    assert float((C.cpu().double() - ref).abs().max()) < 1e-5 * scale
    assert torch.equal(Cb.cpu(), C.cpu().to(torch.bfloat16))


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [(8, 8, 8), (72, 40, 104), (64, 128, 32), (136, 64, 40), (65, 33, 31), (64, 64, 65)])
def test_gemm_wide_loads_equal_the_general_path(M, N, K, ta, tb):
    """Operands on 16 bytes (wide loads where the strides allow them) and the
    same operands 2 bytes off (the general path) give the same bits."""
    g = torch.Generator().manual_seed(M + N + K)
    out = []
    a = torch.randn(M * K, generator=g).to(torch.bfloat16).to(DEV)
    b = torch.randn(K * N, generator=g).to(torch.bfloat16).to(DEV)
    sam, sak = (1, M) if ta else (K, 1)
    sbk, sbn = (1, K) if tb else (N, 1)
    for off in (0, 1):
        A, B = (torch.cat([x.new_zeros(off), x])[off:] for x in (a, b))
        assert (A.data_ptr() % 16 == 0) == (off == 0)
        C = torch.zeros((M, N), device=DEV)
        cnn.gemm(A, sam, sak, B, sbk, sbn, C, M, N, K)
        out.append(C)
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("M,N,masked,off", [(1, 8, False, 0), (257, 8, True, 0), (1000, 32, True, 0), (4099, 64, False, 0),
                                            (2050, 128, True, 0), (1000, 32, True, 1), (77, 12, True, 0), (300, 37, False, 0),
                                            (5, 1028, True, 0)])
def test_gate_colsum(M, N, masked, off):
    """Gate, bf16 copy and column sums in one pass: 4-column and general
    paths (``off``: a source not on 16 bytes), remainders of the row steps.
    A sum adds at most 64 terms in a chain (rows of a thread, rows of a step,
    workgroups of a lane): 64 rounding errors of the column's sum of |v|."""
    g = torch.Generator().manual_seed(M + N)
    src = torch.randn(M * N + off, generator=g).to(DEV)[off:].view(M, N)
    mask = torch.randn(M, N, generator=g).to(DEV) if masked else None
    dst = torch.zeros((M, N), dtype=torch.bfloat16, device=DEV)
    out, ws = torch.zeros(N, device=DEV), torch.zeros(1 << 18, device=DEV)
    cnn.gate_colsum(src, M, N, dst, out, ws, mask=mask)
    ref = src if mask is None else torch.where(mask > 0, src, torch.zeros_like(src))
    assert torch.equal(dst, ref.to(torch.bfloat16))
    err = (out.double() - ref.double().sum(0)).abs()
    assert bool((err <= 64 * 2.0 ** -24 * ref.double().abs().sum(0)).all())


@pytest.mark.parametrize("M,N", [(1, 1), (7, 64), (130, 65), (1001, 8)])
def test_separate_gate_and_column_sums(M, N):
    """apx_cast_gate_bf16 with a gate and a float32 copy, and apx_colsum of that
    copy, the C entry points that gate_colsum does in one: a column is four chains
    of M / 4 additions."""
    g = torch.Generator().manual_seed(M)
    src, mask = torch.randn(M, N, generator=g).to(DEV), torch.randn(M, N, generator=g).to(DEV)
    dst, dstf, out = torch.zeros((M, N), dtype=torch.bfloat16, device=DEV), torch.zeros_like(src), torch.zeros(N, device=DEV)
    cnn.cast_bf16(src, dst, mask=mask, dstf=dstf)
    cnn.L.check(cnn.L.load().apx_colsum(dstf.data_ptr(), M, N, out.data_ptr(), cnn.L.stream()))
    ref = torch.where(mask > 0, src, torch.zeros_like(src))
    assert torch.equal(dst, ref.to(torch.bfloat16)) and torch.equal(dstf, ref)
    err = (out.double() - ref.double().sum(0)).abs()
    assert bool((err <= (M // 4 + 4) * 2.0 ** -24 * ref.double().abs().sum(0)).all())


def torch_reference(net, x, dout_seed=3):
    """The same network in torch on the CPU (float32), bf16 rounding where the kernels round."""
    params = []
    for lay in net.layers:
        w = bf(lay.w.cpu()).requires_grad_(True)
        b = lay.b.cpu().clone().requires_grad_(True)
        params.append((w, b))
    h = bf(x.cpu().float())
    acts = []
    for (cin, cout), (w, b) in zip(cnn.CONV, params[:4]):
        # w rows (ky, kx, ci) -> conv weight (cout, cin, 3, 3)
        W = w[:9 * cin].reshape(3, 3, cin, cout).permute(3, 2, 0, 1)
        z = F.conv2d(h, W, b, stride=2, padding=1)
        y = torch.relu(z)
        acts.append(y)
        h = RoundBF.apply(y)
    B = x.shape[0]
    flat = h.permute(0, 2, 3, 1).reshape(B, -1)  # NHWC flatten
    (w5, b5), (w6, b6) = params[4:]
    hid = torch.relu(flat @ w5 + b5)
    out = RoundBF.apply(hid) @ w6 + b6
    return out, params


class RoundBF(torch.autograd.Function):
    """bf16 rounding in the forward pass; the backward rounds the incoming
    gradient to bf16, as the kernels do before every gradient GEMM."""

    @staticmethod
    def forward(ctx, x):
        return bf(x)

    @staticmethod
    def backward(ctx, g):
        return bf(g)


def test_network_forward_and_gradients_match_torch():
    torch.manual_seed(0)
    net = cnn.InitNet(seed=1)
    B = 8
    img = torch.randn(B, 64, 64) * 3.0
    sigma = torch.full((B,), 1.5)
    x = net.input(img.to(DEV), sigma.to(DEV))
    out = net.forward(x, B).clone()
    xr = torch.asinh(img / 1.5).reshape(B, 1, 64, 64)
    ref, params = torch_reference(net, xr)
    scale = float(ref.abs().max())
    assert float((out.cpu() - ref.detach()).abs().max()) < 2e-2 * scale
    g = torch.Generator().manual_seed(5)
    dout = torch.randn((B, cnn.NOUT), generator=g)
    # the GPU backward takes dout rounded to bf16; give the CPU the same
    dout = bf(dout)
    net.backward(B, dout.to(DEV).contiguous())
    ref.backward(dout)
    for i, (lay, (w, b)) in enumerate(zip(net.layers, params)):
        gw_ref = w.grad
        gw = lay.gw.cpu()
        s = float(gw_ref.abs().max()) + 1e-12
        assert float((gw - gw_ref).abs().max()) < 3e-2 * s, (i, float((gw - gw_ref).abs().max()) / s)
        s = float(b.grad.abs().max()) + 1e-12
        assert float((lay.gb.cpu() - b.grad).abs().max()) < 3e-2 * s, i


def test_short_training_lowers_the_loss():
    from astrophot_amd.learned_init import Trainer
    net = cnn.InitNet(seed=2)
    tr = Trainer(net, pool=2048, seed=4)
    losses = tr.train(steps=240, batch=128, lr=2e-3)
    first, last = np.mean(losses[:20]), np.mean(losses[-20:])
    assert last < 0.5 * first, (first, last)


@pytest.mark.parametrize("B", [3, 70])
def test_implicit_convolution_equals_im2col_gemm(B):
    """apx_conv_s2_bf16 (the A operand read straight from the NHWC input)
    gives the bits of apx_im2col_s2 + apx_gemm_bf16 for every layer of the
    network (Cin 1: the gathered path; 32 and 64: 16-byte channel loads),
    including ragged batches that leave part of the last tile empty."""
    net = cnn.InitNet(seed=5)
    g = torch.Generator().manual_seed(B)
    x = (torch.randn(B * cnn.SIDE * cnn.SIDE, generator=g) * 0.5).to(torch.bfloat16).to(DEV)
    out_a = net.forward(x, B, keep_cols=True).clone()
    acts_a = [t.clone() for t in net._buffers(B)["yb"]]
    out_b = net.forward(x, B, keep_cols=False).clone()
    acts_b = net._buffers(B)["yb"]
    for a, b in zip(acts_a, acts_b):
        assert torch.equal(a, b)
    assert torch.equal(out_a, out_b)


@pytest.mark.parametrize("B,shift", [(1, 0), (3, 1), (511, 0), (513, 3), (1100, 0)])
def test_fused_convolutions_equal_the_layers(B, shift):
    """apx_init_features gives the bits of the input pass and the four
    convolutions run one after another, whatever the number of cutouts a
    workgroup takes (512 workgroups) and wherever the images start (shift floats
    past 16 bytes), and so does the whole prediction; NaN and infinite pixels and
    a zero sigma take the same way through."""
    net = cnn.InitNet(seed=2)
    for k, lay in enumerate(net.layers):
        lay.b.copy_(0.1 * torch.randn(lay.b.shape, generator=torch.Generator().manual_seed(k)))
    g = torch.Generator().manual_seed(B)
    base = (3 * torch.randn(B * 4096 + 4, generator=g)).to(DEV)
    images = base[shift:shift + B * 4096].view(B, 64, 64)
    sigma = (0.2 + torch.rand(B, generator=g)).to(DEV)
    images[0, 0, 0], images[-1, 63, 63], images[-1, 31, 32] = 1e30, float("inf"), -1e30
    if B > 2:
        images[1, 5, 7], sigma[2] = float("nan"), 0.0
    lib = L.load()
    wsb = lib.apx_init_features_workspace_bytes()
    ws, feat = torch.empty(wsb, dtype=torch.uint8, device=DEV), torch.empty(B * 1024, dtype=torch.bfloat16, device=DEV)
    w = (ctypes.c_void_p * 4)(*(lay.wb.data_ptr() for lay in net.layers[:4]))
    b = (ctypes.c_void_p * 4)(*(lay.b.data_ptr() for lay in net.layers[:4]))
    L.check(lib.apx_init_features(images.data_ptr(), sigma.data_ptr(), B, w, b, feat.data_ptr(), ws.data_ptr(), wsb,
                                  L.stream()))
    ref = net.forward(net.input(images, sigma), B, keep_cols=False).clone()
    same = lambda a, b: torch.equal(torch.nan_to_num(a), torch.nan_to_num(b)) and torch.equal(a.isnan(), b.isnan())  # noqa: E731
    assert same(feat.float(), net._buffers(B)["yb"][3].reshape(-1).float())
    assert same(net._infer(images, sigma), ref)


@pytest.mark.parametrize("B,H,W,C,Kp", [(2, 64, 64, 1, 32), (3, 7, 5, 8, 72), (2, 9, 16, 32, 288), (1, 1, 1, 4, 36),
                                        (2, 6, 7, 12, 112), (2, 5, 5, 3, 27), (3, 4, 4, 64, 584), (2, 8, 3, 8, 76)])
def test_im2col_and_its_adjoint_any_shape(B, H, W, C, Kp):
    """Both widths of im2col and col2im (8 columns and 4 channels a thread where
    rows stay on 16 bytes, one otherwise, and with operands 2 or 4 bytes past it)
    against the definition: im2col moves bits, col2im adds at most 4 float32
    values in a fixed order (4 x 2^-24 of their magnitudes)."""
    lib = L.load()
    g = torch.Generator().manual_seed(B * 100 + H)
    Ho, Wo = (H + 1) // 2, (W + 1) // 2
    M = B * Ho * Wo
    x = torch.randn(B, H, W, C, generator=g).to(torch.bfloat16)
    d = torch.randn(M, Kp, generator=g)
    pad = torch.nn.functional.pad(x.float(), (0, 0, 1, 2, 1, 2))
    ref = torch.zeros(B, Ho, Wo, Kp)
    back, mag = torch.zeros(B, H + 3, W + 3, C, dtype=torch.float64), torch.zeros(B, H + 3, W + 3, C, dtype=torch.float64)
    for t in range(9):
        ky, kx = divmod(t, 3)
        ref[..., t * C:(t + 1) * C] = pad[:, ky:ky + 2 * Ho:2, kx:kx + 2 * Wo:2]
        part = d.view(B, Ho, Wo, Kp)[..., t * C:(t + 1) * C].double()
        back[:, ky:ky + 2 * Ho:2, kx:kx + 2 * Wo:2] += part
        mag[:, ky:ky + 2 * Ho:2, kx:kx + 2 * Wo:2] += part.abs()
    for shift in (0, 1):
        xd = torch.zeros(x.numel() + 8, dtype=torch.bfloat16, device=DEV)
        xd[shift:shift + x.numel()] = x.reshape(-1).to(DEV)
        col = torch.full((M * Kp + 8,), 7.0, dtype=torch.bfloat16, device=DEV)
        L.check(lib.apx_im2col_s2(xd[shift:].data_ptr(), B, H, W, C, Kp, col[shift:].data_ptr(), L.stream()))
        assert torch.equal(col[shift:shift + M * Kp].float().cpu(), ref.reshape(-1))
        assert (col[shift + M * Kp:].float() == 7.0).all()
        dd = torch.zeros(M * Kp + 8, device=DEV)
        dd[shift:shift + M * Kp] = d.reshape(-1).to(DEV)
        dx = torch.full((x.numel() + 8,), 7.0, device=DEV)
        L.check(lib.apx_col2im_s2(dd[shift:].data_ptr(), B, H, W, C, Kp, dx[shift:].data_ptr(), L.stream()))
        got = dx[shift:shift + x.numel()].view(B, H, W, C).double().cpu()
        assert ((got - back[:, 1:H + 1, 1:W + 1]).abs() <= 4 * 2.0 ** -24 * mag[:, 1:H + 1, 1:W + 1]).all()
        assert (dx[shift + x.numel():] == 7.0).all()
