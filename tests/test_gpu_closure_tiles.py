"""LDS-tiled convolution kernels against float64 products: 32-column tiles
(W % 32 == 0, H % 8 == 0), where the layer calls of the training test run the
same kernels on both sides, and the bf16-only form on either side of the
number of tiles that changes its code (512).

Tolerances of the other layer tests: fp32 sums over at most 288 products (or
the pixels of a chunk), relative L2 below 1e-5; bf16 outputs are roundings of
the fp32 ones, so the forms of one call agree bit for bit."""

import pytest
import torch

import closure_ref as R
from test_gpu_closure import C, case, dev, random_conv, rl2, taps

pytestmark = pytest.mark.gpu

TILES = [(1, 8, 32, 32, 32), (2, 24, 96, 16, 32), (2, 16, 32, 32, 16), (3, 40, 32, 32, 32), (2, 8, 160, 16, 16)]


@pytest.mark.parametrize("B,H,W,Ci,Co", TILES + [(32, 64, 64, 32, 16), (129, 16, 64, 32, 16), (1, 4, 64, 32, 16)],
                         ids=str)
def test_forward_forms(B, H, W, Ci, Co):
    d, net = dev(), C()
    from dedalus import _hip
    case("tiles forward", B, H, W, Ci, Co)
    x, w, b = random_conv(B, H, W, Ci, Co, 41)
    xd, wd, bd = x.reshape(-1, Ci).to(d), taps(w).to(d), b.to(d)
    z = R.nchw_to_nhwc(R.conv_periodic(R.nhwc_to_nchw(x.double()), w.double()) + b.double().view(1, -1, 1, 1))
    f, _ = net.conv3x3(xd, wd, B, H, W, bias=bd)
    assert rl2(f, z.reshape(-1, Co)) < 1e-5
    for mode in (_hip.CONV_LINEAR, _hip.CONV_GELU):
        fb, both = net.conv3x3(xd, wd, B, H, W, bias=bd, mode=mode, out_bf16=True)
        _, one = net.conv3x3(xd, wd, B, H, W, bias=bd, mode=mode, out_f32=False, out_bf16=True)
        assert torch.equal(fb, f) and torch.equal(one, both)
        if mode == _hip.CONV_LINEAR:
            assert torch.equal(one, f.to(torch.bfloat16))


@pytest.mark.parametrize("B,H,W,Ci,Co", TILES, ids=str)
def test_gradients(B, H, W, Ci, Co):
    d, net = dev(), C()
    from dedalus import _hip
    case("tiles gradients", B, H, W, Ci, Co)
    x, w, _ = random_conv(B, H, W, Ci, Co, 42)
    g = torch.Generator().manual_seed(43)
    dz = torch.randn(B, H, W, Co, generator=g).to(torch.bfloat16)
    zp = torch.randn(B, H, W, Ci, generator=g)
    xd, dzd, zd = x.reshape(-1, Ci).to(d), dz.reshape(-1, Co).to(d), zp.reshape(-1, Ci).to(d)
    dx, dw = R.conv_grads(R.nhwc_to_nchw(x.double()), w.double(), R.nhwc_to_nchw(dz.double()))
    ref = R.nchw_to_nhwc(dx * R.gelu_grad(R.nhwc_to_nchw(zp.double()))).reshape(-1, Ci)
    _, wt = net.wprep(w.float().to(d), Co, Ci)
    f, both = net.conv3x3(dzd, wt, B, H, W, aux=zd, mode=_hip.CONV_GELU_GRAD, out_bf16=True)
    _, one = net.conv3x3(dzd, wt, B, H, W, aux=zd, mode=_hip.CONV_GELU_GRAD, out_f32=False, out_bf16=True)
    assert rl2(f, ref) < 1e-5
    assert torch.equal(both, f.to(torch.bfloat16)) and torch.equal(one, both)
    # one chunk for all tiles, fewer chunks than tiles, one per tile, more
    for nchunk in (1, 2, B * H * W // 256, 100):
        dwp = net.wgrad(xd, dzd, B, H, W, nchunk=nchunk)
        assert rl2(net.wunpack(dwp, Co, Ci), dw) < 1e-5, nchunk
        assert torch.equal(dwp, net.wgrad(xd, dzd, B, H, W, nchunk=nchunk))


@pytest.mark.parametrize("B,H,W,Ci,Co", [(1, 8, 32, 32, 32), (1, 4, 64, 16, 32)], ids=str)
@pytest.mark.parametrize("odd", ["x", "dz"])
def test_weight_gradient_alignment(B, H, W, Ci, Co, odd):
    """The tile kernel reads x and dz 8 bytes at a time; arrays that start on
    another 2-byte boundary go to the per-fragment kernel.  Which one ran shows
    in the partial sums: a single tile fills one chunk, 64-pixel chunks all four."""
    import ctypes
    from dedalus import _hip
    d, net = dev(), C()
    case("wgrad alignment", B, H, W, Ci, Co, odd)
    x, w, _ = random_conv(B, H, W, Ci, Co, 44)
    dz = torch.randn(B, H, W, Co, generator=torch.Generator().manual_seed(45)).to(torch.bfloat16)
    _, ref = R.conv_grads(R.nhwc_to_nchw(x.double()), w.double(), R.nhwc_to_nchw(dz.double()))

    def at(t, off):
        buf = torch.zeros(t.numel() + 8, dtype=torch.bfloat16, device=d)
        buf[off:off + t.numel()] = t.reshape(-1).to(d)
        return buf, ctypes.c_void_p(buf.data_ptr() + 2 * off)

    used = {}
    for off in (0, 4, 1):
        xb, xp = at(x, off if odd == "x" else 0)
        db, dp = at(dz, off if odd == "dz" else 0)
        part = torch.full((4, Co, 9, Ci), float("nan"), device=d)
        dw = torch.empty((Co, 9, Ci), device=d)
        _hip._check(_hip._lib.ddx_conv3x3_wgrad(net._stream(), B, H, W, Ci, Co, xp, dp, net._ptr(part), 4, net._ptr(dw)))
        torch.cuda.synchronize()
        assert rl2(net.wunpack(dw, Co, Ci), ref) < 1e-5, off
        used[off] = int((~part.isnan().flatten(1).any(1)).sum())
    assert used == {0: 1, 4: 1, 1: 4}
