"""fp32 products on the bf16 matrix cores (three-part operands, six products): the MACE
layer's weights GEMM at channel counts that fill its quads and launch rounds unevenly,
its error against float64, and infinities in W2."""
import numpy as np
import pytest
import torch

from oracle import mace as om

from helpers import gen, periodic_box

pytestmark = pytest.mark.gpu


def _layer(dev, n, c, seed, scale=1.0):
    import batmobile
    pos, cell = periodic_box(n, seed)
    graph = batmobile.Graph(pos.to(dev), cell, 5.0, c)
    layer = batmobile.MACEInteraction(c, 5.0, device=dev, generator=gen(seed + 1))
    layer.W2.mul_(scale)
    x = torch.randn(n, c, 16, generator=gen(seed + 2))
    go = torch.randn(n, c, 16, generator=gen(seed + 3))
    return pos, cell, graph, layer, x, go


# C: one quad and part of it, 20 quads (three ranges per XCD), 33 quads (more than one
# round); scale: weights whose lower parts reach down to 2^-100 and up to 2^100
@pytest.mark.parametrize("n,c,scale", [(60, 1, 1.0), (60, 7, 1.0), (150, 80, 1.0), (40, 130, 1.0),
                                       (60, 8, 2.0 ** -80), (60, 8, 2.0 ** 100)])
def test_layer_error_against_float64(bm, dev, n, c, scale):
    pos, cell, graph, layer, x, go = _layer(dev, n, c, 31, scale)
    p = pos.to(dev).requires_grad_(True)
    out = layer(graph, p, x.to(dev))
    (gp,) = torch.autograd.grad(out, p, go.to(dev))
    box = torch.diagonal(cell).numpy().astype(np.float64)
    want, gwant = om.layer_and_position_grad(
        pos.numpy(), box, x.numpy(), graph.src.cpu().numpy(), graph.dst.cpu().numpy(),
        layer.W1.cpu().numpy(), layer.b1.cpu().numpy(), layer.W2.cpu().numpy(), 5.0, go.numpy())
    # fp32: the radial basis and 64-term sums, a few 2^-24 each (measured about 1e-6)
    for got, ref in ((out.detach(), want), (gp, gwant)):
        d = got.cpu().double().numpy() - ref
        assert np.linalg.norm(d) <= 4e-6 * np.linalg.norm(ref)


def test_infinite_weight_stays_infinite(bm, dev):
    """An infinite W2 entry makes the same outputs infinite (not NaN) as the fp32 product
    R = h W2 does: path 0 (l1 = l2 = l_out = 0) of channel 1, hidden unit 5."""
    pos, cell, graph, layer, x, _ = _layer(dev, 80, 4, 41)
    layer.W2[5, 0 * 4 + 1] = float("inf")
    out = layer(graph, pos.to(dev), x.to(dev)).cpu()
    assert torch.isfinite(out[:, [0, 2, 3]]).all()
    assert torch.isfinite(out[:, 1, 1:]).all()   # path 0 writes component 0 only
    deg = torch.bincount(graph.dst.cpu(), minlength=80)
    assert not torch.isfinite(out[deg > 0, 1, 0]).any()
    # destinations with one edge: +-inf, the sign of h[5] x
    one = deg == 1
    assert torch.isinf(out[one, 1, 0]).all()
