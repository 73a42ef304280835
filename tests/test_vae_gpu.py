"""The Wan2.2 VAE38 first-frame encoder on the library (fam.vae.FusedWanVAEEncoder) against the
oracle's restatement of VideoVAE38_.encode, which the reference module pins
(tests/golden/wan_vae_tiny.safetensors): fp32 oracle on bf16-valued weights and image, normwise
relative error <= 3e-2 on the latent (about 25 bf16 layers deep).  Plus the non-GEMM kernels
(im2col, channel RMS_norm, AvgDown3D, row softmax, latent normalisation) against torch."""
import math

import pytest
import torch
import torch.nn.functional as F

from oracle import fam_oracle as O

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _rel(y, ref):
    y, ref = y.float().cpu(), ref.float().cpu()
    return ((y - ref).abs().max() / ref.abs().max()).item()


def _lib():
    from fam import _capi
    return _capi.load()


def _s():
    return torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("H,W,C,stride", [(6, 10, 16, 1), (8, 12, 24, 2), (5, 7, 8, 1)])
def test_im2col3x3(H, W, C, stride):
    x = torch.randn(H * W, C, generator=torch.Generator().manual_seed(1)).to(BF)
    kp = (9 * C + 63) // 64 * 64
    ho, wo = (H, W) if stride == 1 else (H // 2, W // 2)
    out = torch.full((ho * wo, kp), 7.0, dtype=BF, device="cuda")
    xd = x.cuda()
    assert _lib().fam_im2col3x3(xd.data_ptr(), C, H, W, C, stride, out.data_ptr(), kp, kp, _s()) == 0
    img = x.reshape(1, H, W, C).permute(0, 3, 1, 2).float()
    pad = (1, 1, 1, 1) if stride == 1 else (0, 1, 0, 1)
    cols = F.unfold(F.pad(img, pad), 3, stride=stride)                # [1, C*9, L], (c, kh, kw)
    ref = cols.reshape(C, 9, ho * wo).permute(2, 1, 0).reshape(ho * wo, 9 * C)
    got = out.float().cpu()
    assert torch.equal(got[:, :9 * C], ref)
    assert torch.equal(got[:, 9 * C:], torch.zeros_like(got[:, 9 * C:]))


# Edges of the image on every side of a tile, C below, off and above the 64-wide K block, both
# strides, padded rows (every tile of the product: test_conv3x3_on_every_tile).
@pytest.mark.parametrize("H,W,C,N,stride,ldx", [
    (9, 17, 8, 12, 1, 8), (1, 130, 24, 64, 1, 32), (130, 1, 64, 20, 1, 64), (28, 56, 40, 100, 2, 48),
    (16, 20, 160, 96, 1, 160), (14, 28, 640, 640, 1, 640), (56, 112, 320, 640, 2, 320), (96, 96, 80, 256, 1, 80),
    (112, 224, 160, 160, 1, 160), (224, 256, 16, 512, 1, 16), (100, 125, 32, 1024, 1, 32), (128, 128, 56, 128, 1, 56)])
def test_conv3x3_equals_im2col_gemm(H, W, C, N, stride, ldx):
    """The same plan reads the same operands in the same order: the bits are the same."""
    from fam import _capi
    import ctypes
    lib = _lib()
    g = torch.Generator().manual_seed(H * 131 + W)
    x = torch.full((H * W, ldx), float("nan"), dtype=BF)   # the padding columns are never used
    x[:, :C] = torch.randn(H * W, C, generator=g).to(BF)
    kp = (9 * C + 63) // 64 * 64
    P = (H // stride) * (W // stride)
    w = torch.zeros(N, kp, dtype=BF)
    w[:, :9 * C] = (torch.randn(N, 9 * C, generator=g) / math.sqrt(9 * C)).to(BF)
    x, w = x.cuda(), w.cuda()
    bias, res = (torch.randn(*s, generator=g).to(BF).cuda() for s in ((N,), (P, N)))
    rows = torch.empty(P, kp, dtype=BF, device="cuda")
    assert lib.fam_im2col3x3(x.data_ptr(), ldx, H, W, C, stride, rows.data_ptr(), kp, kp, _s()) == 0
    wsf = lib.fam_gemm_ws_floats(P, N, kp)
    ws = torch.empty(max(wsf, 4), device="cuda")
    outs = []
    for conv in (False, True):
        y = torch.empty(P, N, dtype=BF, device="cuda")
        a = x if conv else rows
        d = _capi.GemmDesc()
        d.a, d.lda, d.w, d.ldw, d.bias = a.data_ptr(), a.stride(0), w.data_ptr(), kp, bias.data_ptr()
        d.out, d.ldo, d.M, d.N, d.K, d.act = y.data_ptr(), N, P, N, kp, _capi.FAM_ACT_NONE
        d.res, d.ldr, d.rows_per_batch = res.data_ptr(), N, P
        if conv:
            assert lib.fam_conv3x3(ctypes.byref(d), H, W, C, stride, ws.data_ptr(), wsf, _s()) == 0
        else:
            assert lib.fam_gemm_ws(ctypes.byref(d), ws.data_ptr(), wsf, _s()) == 0
        outs.append(y)
    assert torch.equal(outs[0], outs[1])
    img = x[:, :C].float().t().reshape(1, C, H, W).cpu()
    k = w[:, :9 * C].float().reshape(N, 3, 3, C).permute(0, 3, 1, 2).cpu()
    img = F.pad(img, (1, 1, 1, 1)) if stride == 1 else F.pad(img, (0, 1, 0, 1))
    ref = F.conv2d(img, k, bias.float().cpu(), stride=stride).reshape(N, P).t() + res.float().cpu()
    assert _rel(outs[1], ref) <= 1e-2


def _conv_and_gemm(H, W, C, N, act=0, gate=False, f32=False):
    """fam_conv3x3 of an H x W image and fam_gemm_ws of its neighbourhoods: (conv, gemm, rows, w, bias, res, gate)."""
    from fam import _capi
    import ctypes
    lib, P, kp = _lib(), H * W, (9 * C + 63) // 64 * 64
    g = torch.Generator().manual_seed(H * 131 + C)
    rn = lambda *s: torch.randn(*s, generator=g).to(BF)
    x, w = rn(P, C).cuda(), torch.zeros(N, kp, dtype=BF)
    w[:, :9 * C] = rn(N, 9 * C) / math.sqrt(9 * C)
    w, bias, res, gt = w.cuda(), rn(N).cuda(), rn(P, N).cuda(), rn(2, N).cuda()
    res = res.float() if f32 else res
    rows = torch.empty(P, kp, dtype=BF, device="cuda")
    assert lib.fam_im2col3x3(x.data_ptr(), C, H, W, C, 1, rows.data_ptr(), kp, kp, _s()) == 0
    wsf = lib.fam_gemm_ws_floats(P, N, kp)
    ws = torch.empty(max(wsf, 4), device="cuda")
    outs = []
    for conv in (True, False):
        y = torch.empty(P, N, dtype=torch.float32 if f32 else BF, device="cuda")
        a = x if conv else rows
        d = _capi.GemmDesc(a.data_ptr(), a.stride(0), w.data_ptr(), kp, bias.data_ptr(), y.data_ptr(), N, P, N, kp)
        d.act, d.res, d.ldr, d.rows_per_batch, d.gate_ns, d.out_f32 = act, res.data_ptr(), N, (P + 1) // 2, 1, int(f32)
        if gate:
            d.gate, d.gate_bs = gt.data_ptr(), N
        if conv:
            assert lib.fam_conv3x3(ctypes.byref(d), H, W, C, 1, ws.data_ptr(), wsf, _s()) == 0, lib.fam_last_error()
        else:
            assert lib.fam_gemm_ws(ctypes.byref(d), ws.data_ptr(), wsf, _s()) == 0, lib.fam_last_error()
        outs.append(y)
    return (*outs, rows, w, bias, res, gt)


# A shape for every tile the library's plan can choose on 256 CUs, for channels that are (second
# half) and are not (first) whole K blocks: 64 x 64 with four and two K slots, 128 x 96, 128 x 128
# with one and two K groups, 224 x 256, 256 x 256, and K splits of the 64, 128, 224 and 256 tiles.
@pytest.mark.parametrize("H,W,C,N", [
    (10, 16, 88, 20), (56, 56, 88, 768), (75, 100, 88, 640), (56, 56, 200, 768), (56, 56, 264, 768), (75, 100, 88, 1280),
    (75, 100, 88, 2048), (10, 16, 296, 20), (28, 28, 600, 1280), (64, 64, 720, 768), (64, 64, 1000, 1280),
    (16, 16, 64, 64), (56, 56, 64, 768), (190, 200, 64, 64), (190, 200, 64, 128), (56, 56, 256, 768), (112, 224, 64, 320),
    (75, 100, 64, 2048), (16, 16, 320, 64), (28, 28, 640, 1280), (100, 125, 640, 192), (64, 64, 1024, 1280)])
def test_conv3x3_on_every_tile(H, W, C, N):
    """The bits of the product on the laid-out neighbourhoods, and its value: fp32 accumulation, half a bf16
    ulp (2^-8 of the value at most) of the product with its bias and of the sum with the residual."""
    y, ref, rows, w, bias, res, _ = _conv_and_gemm(H, W, C, N)
    assert torch.equal(y, ref)
    v = rows.float() @ w.float().t() + bias.float()
    exact = v + res.float()
    assert ((y.float() - exact).abs() <= 2.0 ** -8 * (v.abs() + exact.abs()) + 1e-4).all()


@pytest.mark.parametrize("H,W,C,N", [(20, 24, 24, 100), (14, 28, 640, 640), (56, 56, 264, 768)])
@pytest.mark.parametrize("act,gate,f32", [("FAM_ACT_GELU_TANH", False, False), ("FAM_ACT_SILU", True, False),
                                          ("FAM_ACT_NONE", True, True), ("FAM_ACT_RELU", False, True)])
def test_conv3x3_epilogues(H, W, C, N, act, gate, f32):
    """Activation, a gate row per half of the pixels, and fp32 residual and output, whole and split K.  The
    product with its bias is rounded to bf16 (2^-8 of it at most) before the activation, whose slope is at
    most 1.13, and the gate; then the sum."""
    from fam import _capi
    y, ref, rows, w, bias, res, gt = _conv_and_gemm(H, W, C, N, getattr(_capi, act), gate, f32)
    assert torch.equal(y, ref)
    v = rows.float() @ w.float().t() + bias.float()
    f = {"FAM_ACT_GELU_TANH": lambda t: F.gelu(t, approximate="tanh"), "FAM_ACT_SILU": F.silu, "FAM_ACT_RELU": F.relu,
         "FAM_ACT_NONE": lambda t: t}[act]
    gated = gt.float()[torch.arange(H * W, device="cuda") // ((H * W + 1) // 2)] if gate else torch.ones_like(v)
    exact = res.float() + gated * f(v)
    assert ((y.float() - exact).abs() <= 2.0 ** -8 * (1.13 * (gated * v).abs() + exact.abs()) + 1e-4).all()


def test_vae_patch_im2col():
    H, W = 12, 20
    img = torch.randn(1, 3, H, W, generator=torch.Generator().manual_seed(2)).to(BF)
    out = torch.empty((H // 2) * (W // 2), 128, dtype=BF, device="cuda")
    imgd = img.cuda()
    assert _lib().fam_vae_patch_im2col(imgd.data_ptr(), H, W, out.data_ptr(), 128, _s()) == 0
    pt = O.vae_patchify(img.float(), 2)                                 # [1, 12, 6, 10]
    cols = F.unfold(F.pad(pt, (1, 1, 1, 1)), 3)
    ref = cols.reshape(12, 9, -1).permute(2, 1, 0).reshape(-1, 108)
    got = out.float().cpu()
    assert torch.equal(got[:, :108], ref)
    assert torch.equal(got[:, 108:], torch.zeros_like(got[:, 108:]))


@pytest.mark.parametrize("C,act", [(160, True), (640, False), (8, True)])
def test_chan_rmsnorm(C, act):
    from fam import _capi
    g = torch.Generator().manual_seed(3)
    x = (torch.randn(37, C, generator=g) * 3).to(BF)
    gamma = (1 + 0.2 * torch.randn(C, generator=g)).to(BF)
    y = torch.empty(37, C, dtype=BF, device="cuda")
    xd, gd = x.cuda(), gamma.cuda()   # (device copies held for the launch)
    rc = _lib().fam_chan_rmsnorm(xd.data_ptr(), C, 37, C, gd.data_ptr(),
                                 _capi.FAM_ACT_SILU if act else _capi.FAM_ACT_NONE, y.data_ptr(), C, _s())
    assert rc == 0
    ref = O.vae_rms_norm(x.float().t().reshape(1, C, 37, 1), gamma.float()).reshape(C, 37).t()
    if act:
        ref = F.silu(ref)
    assert _rel(y, ref) <= 1e-2


@pytest.mark.parametrize("Cin,Cout,ft,fs", [(16, 16, 1, 2), (16, 32, 2, 2), (24, 24, 1, 1)])
def test_vae_avgdown(Cin, Cout, ft, fs):
    H, W = 6, 8
    g = torch.Generator().manual_seed(4)
    x = torch.randn(H * W, Cin, generator=g).to(BF)
    add = torch.randn((H // fs) * (W // fs), Cout, generator=g).to(BF)
    out = torch.empty((H // fs) * (W // fs), Cout, dtype=BF, device="cuda")
    xd = x.cuda()
    for a in (None, add.cuda()):
        assert _lib().fam_vae_avgdown(xd.data_ptr(), Cin, H, W, Cin, Cout, ft, fs,
                                      a.data_ptr() if a is not None else None, Cout, out.data_ptr(), Cout, _s()) == 0
        ref = O.vae_avg_down(x.float().t().reshape(1, Cin, H, W), Cout, ft, fs).reshape(Cout, -1).t()
        if a is not None:
            ref = ref + add.float()
        assert _rel(out, ref) <= 1e-2


@pytest.mark.parametrize("rows", [1, 7, 33])
@pytest.mark.parametrize("C", [8, 120, 128, 136, 160, 256, 264, 512, 520, 1024, 1032])
def test_chan_rmsnorm_lane_groups(rows, C):
    """Every lane group and both register forms, at the widths where they change; a row of zeros."""
    from fam import _capi
    g = torch.Generator().manual_seed(rows * 7 + C)
    x = torch.randn(rows, C + 8, generator=g).to(BF)
    x[rows // 2] = 0
    gamma = (1 + 0.2 * torch.randn(C, generator=g)).to(BF)
    y = torch.full((rows + 1, C + 16), 7.0, dtype=BF, device="cuda")
    xd, gd = x.cuda(), gamma.cuda()
    assert _lib().fam_chan_rmsnorm(xd.data_ptr(), C + 8, rows, C, gd.data_ptr(), _capi.FAM_ACT_SILU, y.data_ptr(),
                                   C + 16, _s()) == 0
    ref = F.silu(F.normalize(x[:, :C].double(), dim=1) * math.sqrt(C) * gamma.double())
    # one bf16 rounding of a value whose fp32 error is far smaller
    assert ((y[:rows, :C].cpu().double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-6).all()
    assert (y[rows] == 7).all() and (y[:, C:] == 7).all()


@pytest.mark.parametrize("Cin,Cout,ft,fs,pad", [
    (8, 8, 1, 1, 0), (8, 16, 2, 1, 8), (160, 160, 1, 2, 0), (24, 48, 2, 2, 8),   # 8 outputs a thread
    (16, 16, 1, 2, 1), (12, 12, 1, 2, 0), (16, 8, 1, 2, 0), (16, 32, 1, 2, 0)])   # one output a thread
def test_vae_avgdown_forms(Cin, Cout, ft, fs, pad):
    """Both forms against exact group means of the folded layout, rows padded by `pad`."""
    H, W = 10, 6
    P = (H // fs) * (W // fs)
    g = torch.Generator().manual_seed(Cin + Cout)
    x, add = torch.randn(H * W, Cin + pad, generator=g).to(BF), torch.randn(P, Cout + pad, generator=g).to(BF)
    xd, ad = x.cuda(), add.cuda()
    ref = O.vae_avg_down(x[:, :Cin].double().t().reshape(1, Cin, H, W), Cout, ft, fs).reshape(Cout, -1).t()
    for a in (None, ad):
        out = torch.full((P + 1, Cout + pad), 7.0, dtype=BF, device="cuda")
        assert _lib().fam_vae_avgdown(xd.data_ptr(), Cin + pad, H, W, Cin, Cout, ft, fs,
                                      a.data_ptr() if a is not None else None, Cout + pad, out.data_ptr(), Cout + pad,
                                      _s()) == 0
        want = ref if a is None else ref + add[:, :Cout].double()
        # one bf16 rounding; the fp32 sums of at most 8 values of magnitude < 8 are exact to 2^-18
        assert ((out[:P, :Cout].cpu().double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -18).all()
        assert (out[P] == 7).all() and (out[:, Cout:] == 7).all()


@pytest.mark.parametrize("ldo", [128, 131])
def test_vae_patch_im2col_rows(ldo):
    H, W = 10, 14
    img = torch.randn(3, H, W, generator=torch.Generator().manual_seed(5)).to(BF)
    imgd = img.cuda()
    out = torch.full((35, ldo), 7.0, dtype=BF, device="cuda")
    assert _lib().fam_vae_patch_im2col(imgd.data_ptr(), H, W, out.data_ptr(), ldo, _s()) == 0
    t = img.float().reshape(3, H // 2, 2, W // 2, 2).permute(0, 4, 2, 1, 3).reshape(1, 12, H // 2, W // 2)
    ref = F.unfold(t, 3, padding=1).reshape(12, 9, 35).permute(2, 1, 0).reshape(35, 108)
    assert torch.equal(out[:, :108].float().cpu(), ref)
    assert (out[:, 108:128] == 0).all() and (out[:, 128:] == 7).all()


def test_softmax_rows_and_affine():
    g = torch.Generator().manual_seed(5)
    s = torch.randn(9, 70, generator=g) * 4
    p = torch.zeros(9, 128, dtype=BF, device="cuda")
    sd = s.cuda()
    assert _lib().fam_softmax_rows(sd.data_ptr(), 70, 9, 70, 0.3, p.data_ptr(), 128, _s()) == 0
    assert _rel(p[:, :70], torch.softmax(s * 0.3, -1)) <= 1e-2
    assert torch.count_nonzero(p[:, 70:]).item() == 0
    x = torch.randn(12, 5, generator=g).to(BF)
    mean, std = torch.randn(5, generator=g), 0.5 + torch.rand(5, generator=g)
    out = torch.empty(5, 12, dtype=BF, device="cuda")
    inv = (1 / std).float().cuda()
    xd, md = x.cuda(), mean.cuda()
    assert _lib().fam_chan_affine_nchw(xd.data_ptr(), 5, 12, 5, md.data_ptr(), inv.data_ptr(), out.data_ptr(),
                                       _s()) == 0
    assert _rel(out, ((x.float() - mean) / std).t()) <= 1e-2


def _encoder_case(cfg, H, W, seed):
    from fam.vae import FusedWanVAEEncoder
    p = {k: v.to(BF) for k, v in O.init_wan_vae_params(cfg, seed).items()}
    g = torch.Generator().manual_seed(seed + 1)
    img = torch.randn(1, 3, H, W, generator=g).clamp(-1, 1).to(BF)
    mean = 0.3 * torch.randn(cfg.z_dim, generator=g)
    std = 0.5 + torch.rand(cfg.z_dim, generator=g)
    enc = FusedWanVAEEncoder(cfg, p, height=H, width=W, mean=mean, std=std)
    y = enc.encode(img.cuda())
    ref = O.wan_vae_encode_first_frame({k: v.float() for k, v in p.items()}, cfg, img.float(), mean, std)
    return enc, img, y, ref


@pytest.mark.parametrize("H,W", [(64, 128), (48, 80)])
def test_vae_encoder_tiny_matches_oracle(H, W):
    """The golden config (dim 16, z 8) at both golden image sizes."""
    cfg = O.WanVaeConfig(dim=16, z_dim=8)
    enc, img, y, ref = _encoder_case(cfg, H, W, 2468)
    err = _rel(y, ref)
    print(f"vae tiny {H}x{W}: {enc.num_launches} launches, relerr {err:.3e}")
    assert y.shape == ref.shape == (1, 8, 1, H // 16, W // 16)
    assert err <= 3e-2
    enc.capture()
    assert torch.equal(enc.encode(img.cuda()), y)


def test_vae_encoder_wan22_shape():
    """The Wan2.2 VAE38 encoder (dim 160, z 48, widths 160-160-320-640-640) on FastWAM's first
    frame, 224 x 448 (latent 14 x 28 -> 7 x 14 video patches)."""
    cfg = O.WanVaeConfig()
    enc, img, y, ref = _encoder_case(cfg, 224, 448, 97)
    err = _rel(y, ref)
    print(f"vae wan2.2 224x448: {enc.num_launches} launches, relerr {err:.3e}")
    assert y.shape == (1, 48, 1, 14, 28)
    assert err <= 3e-2
