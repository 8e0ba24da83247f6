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
