"""The training passes in one native call each way (ddx_net_forward,
ddx_net_backward) against the layer calls they are made of: tile kernels 64
and 32 columns wide at their smallest images, shapes and widths on the
per-fragment kernels, more layers than one preparing or summing launch takes,
and partial gradients that need more than one summing launch.

The output and the weight gradients add in the same order, so they are equal;
a bias gradient sums the same fp32 values in double in another order, so the
two differ by their own roundings to fp32 (2 x 2^-24) and npix 2^-53 of the
sum of magnitudes."""

import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [((1, 4, 64), (2, 32, 32, 32, 32, 2)), ((3, 12, 64), (3, 16, 32, 16, 1)),
         ((1, 8, 32), (2, 32, 32, 2)), ((2, 24, 96), (16, 16, 32, 16)),
         ((2, 12, 32), (2, 32, 32, 2)), ((1, 5, 16), (3, 20, 48, 64, 4)),
         ((1, 4, 4), (1, 1)), ((2, 8, 64), (2,) + (16,) * 9 + (2,)),
         ((32, 64, 64), (2, 64, 64, 32, 2))]


def layer_calls(N, x, g, chans, ws, bs):
    B, H, W, cin = x.shape
    nl, npix = len(chans) - 1, B * H * W
    p16 = N.pad16
    a, _ = N.pack([(x.data_ptr() + 4 * c, False) for c in range(cin)], npix, p16(cin), pstride=cin)
    acts, zs, wts = [a], [], []
    for l in range(nl):
        wf, wt = N.wprep(ws[l], p16(chans[l + 1]), p16(chans[l]))
        wts.append(wt)
        bp = torch.zeros(p16(chans[l + 1]), device=x.device)
        bp[:chans[l + 1]] = bs[l]
        last = l == nl - 1
        z, a = N.conv3x3(acts[-1], wf, B, H, W, bias=bp, mode=0 if last else 1, out_f32=True, out_bf16=not last)
        if not last:
            zs.append(z)
            acts.append(a)
    cout = chans[-1]
    out = z[:, :cout].reshape(B, H, W, cout)
    dzb, dzf = N.pack([(g.data_ptr() + 4 * c, False) for c in range(cout)], npix, p16(cout), pstride=cout, f32=True)
    gw, gb, mag = [None] * nl, [None] * nl, [None] * nl
    for l in range(nl - 1, -1, -1):
        gw[l] = N.wunpack(N.wgrad(acts[l], dzb, B, H, W), chans[l + 1], chans[l])
        gb[l] = N.colsum(dzf)[:chans[l + 1]]
        mag[l] = dzf.double().abs().sum(0)[:chans[l + 1]]
        if l:
            dzf, dzb = N.conv3x3(dzb, wts[l], B, H, W, aux=zs[l - 1], mode=2, out_f32=True, out_bf16=True)
    return out, gw, gb, mag


@pytest.mark.parametrize("shape,chans", CASES, ids=str)
def test_network_calls_match_layers(shape, chans):
    from dedalus.closure import ClosureNet
    from dedalus.closure import net as N
    print("net calls", shape, chans, flush=True)
    d = torch.device("cuda")
    gen = torch.Generator().manual_seed(21)
    net = ClosureNet(cin=chans[0], cout=chans[-1], width=chans[1], depth=len(chans) - 1, seed=3, out_scale=1.0)
    net.chans = tuple(chans)
    for l in range(len(chans) - 1):
        net.weights[l] = torch.nn.Parameter(torch.randn(chans[l + 1], chans[l], 3, 3, generator=gen) * 0.2)
        net.biases[l] = torch.nn.Parameter(torch.randn(chans[l + 1], generator=gen) * 0.1)
    net = net.to(d)
    x = torch.randn(*shape, chans[0], generator=gen).to(d)
    g = torch.randn(*shape, chans[-1], generator=gen).to(d)
    out = net(x)
    out.backward(g)
    ref, gw, gb, mag = layer_calls(N, x, g, chans, [w.detach() for w in net.weights], [b.detach() for b in net.biases])
    torch.cuda.synchronize()
    assert torch.equal(out, ref)
    npix = shape[0] * shape[1] * shape[2]
    for l in range(len(chans) - 1):
        assert torch.equal(net.weights[l].grad, gw[l]), l
        bound = 2.0 ** -23 * gb[l].double().abs() + npix * 2.0 ** -53 * mag[l] + 1e-40
        assert ((net.biases[l].grad.double() - gb[l].double()).abs() <= bound).all(), l


def test_weights_larger_than_their_layers():
    """Weights within a layer's padding of 16 but beyond its channels compute
    the extra channels, which the next layer's weights may read; beyond the
    padding they are refused.  Smaller ones count as zeros there."""
    from dedalus import _hip
    from dedalus.closure import ClosureNet
    from dedalus.closure import net as N
    print("net calls, other weight shapes", flush=True)
    d = torch.device("cuda")
    gen = torch.Generator().manual_seed(22)
    chans = (3, 20, 20, 2)
    net = ClosureNet(cin=3, cout=2, width=20, depth=3, seed=3, out_scale=1.0).to(d)

    def put(shapes):
        for l, (co, ci) in enumerate(shapes):
            net.weights[l] = torch.nn.Parameter((torch.randn(co, ci, 3, 3, generator=gen) * 0.2).to(d))
            net.biases[l] = torch.nn.Parameter((torch.randn(chans[l + 1], generator=gen) * 0.1).to(d))

    x = torch.randn(2, 8, 64, 3, generator=gen).to(d)
    g = torch.randn(2, 8, 64, 2, generator=gen).to(d)
    for shapes in ([(24, 5), (20, 26), (3, 20)], [(18, 3), (20, 16), (1, 20)]):
        put(shapes)
        with torch.no_grad():
            out = net(x)
        ref = layer_calls(N, x, g, chans, [w.detach() for w in net.weights], [b.detach() for b in net.biases])[0]
        assert torch.equal(out, ref), shapes
        with pytest.raises(RuntimeError):       # their gradient has the layer's shape
            net(x).backward(g)
    put([(20, 3), (33, 20), (2, 20)])
    with pytest.raises(_hip.DDXError):
        net(x)
