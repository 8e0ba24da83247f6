"""The fused network on many images (row-by-row kernel) against the layer calls."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# one strip per image and several; a last strip that is shorter; strips in
# more than one round; both widths; 16-row images (fewer rows than the
# pipeline is deep)
@pytest.mark.parametrize("B,H,W", [(128, 64, 64), (256, 64, 64), (300, 32, 64), (130, 48, 64), (100, 96, 64),
                                   (1100, 16, 64), (256, 32, 32), (600, 64, 32), (77, 128, 32)])
def test_rows_match_layers(B, H, W):
    from dedalus import _hip
    from dedalus.closure.net import ClosureNet, Inference, pack, unpack
    _hip.init()
    print("case: network rows", B, H, W, flush=True)
    torch.manual_seed(B + H + W)
    net = ClosureNet(cin=3, cout=2, width=32, depth=5, seed=2, out_scale=1.0).cuda()
    with torch.no_grad():
        for b in net.biases:
            b.normal_(0, 0.1)
    n = B * H * W
    one = Inference(net, B, H, W)
    ref = Inference(net, B, H, W, fused=False)
    assert one.fused
    one.x[:, :3] = torch.randn(n, 3, device="cuda").bfloat16()
    ref.x.copy_(one.x)
    # the same products summed in the same order: equal bit for bit
    assert torch.equal(one.run(), ref.run())
    src = [torch.randn(n, dtype=torch.float64, device="cuda") for _ in range(3)]
    add = [torch.randn(n, dtype=torch.float64, device="cuda") for _ in range(2)]
    got, want = ([torch.empty_like(add[0]) for _ in range(2)] for _ in range(2))
    p = lambda ts: [t.data_ptr() for t in ts]
    one.run_fields(p(src), [0.7, 0.8, 0.25], p(got), [0.3, 0.4], add=p(add))
    pack([(t.data_ptr(), True) for t in src], n, 16, scale=[0.7, 0.8, 0.25], bf16=ref.x)
    unpack(ref.run(), 2, p(want), True, scale=[0.3, 0.4], add=p(add))
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def same(a, b):
    """Bit for bit, NaN for NaN."""
    return bool(((a == b) | (a.isnan() & b.isnan())).all())


# as the rule has it (asserted): one strip per image, several, a shorter last
# strip, 16-row images in one round and in two, 32-wide images alone on a CU
# and two to a CU; values that overflow, NaN, and products below the normal range
@pytest.mark.parametrize("values", ["normal", "tiny", "nonfinite"])
@pytest.mark.parametrize("B,H,W,S", [(256, 64, 64, 64), (128, 64, 64, 32), (67, 48, 64, 16), (40, 80, 64, 14),
                                     (400, 16, 64, 16), (200, 16, 64, 16), (25, 512, 32, 64), (19, 256, 32, 32),
                                     (300, 16, 32, 16), (600, 64, 32, 32), (1024, 32, 32, 32)])
def test_row_kernel(B, H, W, S, values):
    import ctypes
    from dedalus import _hip
    from dedalus.closure.net import ClosureNet, Inference
    _hip.init()
    chans = (3, 32, 32, 32, 32, 2)
    assert _hip._lib.ddx_conv_net_rows(B, H, W, 5, (ctypes.c_int * 6)(*chans)) == S
    print("case: row kernel", B, H, W, values, flush=True)
    torch.manual_seed(B + H + W)
    net = ClosureNet(cin=3, cout=2, width=32, depth=5, seed=2, out_scale=1.0).cuda()
    with torch.no_grad():
        for b in net.biases:
            b.normal_(0, 1e-38 if values == "tiny" else 0.1)
    one, ref = Inference(net, B, H, W), Inference(net, B, H, W, fused=False)
    x = torch.randn(B * H * W, 3, device="cuda")
    if values == "tiny":
        x *= 1e-37
    elif values == "nonfinite":
        x[W // 2] = float("inf")                   # first row of the first image
        x[(B - 1) * H * W + H * W // 2] = float("nan")
        x[(B // 2) * H * W + 3] = 3e38
    one.x[:, :3] = x.bfloat16()
    ref.x.copy_(one.x)
    got, want = one.run(), ref.run()
    assert same(got, want)
    if values == "nonfinite" and B > 4:
        assert got.view(B, -1)[1].isfinite().all()
