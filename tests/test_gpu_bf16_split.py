"""fp32 products on the bf16 matrix cores (three-part operands, six products): the mixing
kernel of the weighted tensor product at the edges of its tiles, passes and chunks, the MACE
layer's weights GEMM at channel counts that fill its quads and launch rounds unevenly,
its error against float64, and infinities in W2."""
import numpy as np
import pytest
import torch

from oracle import mace as om
from oracle import tp as otp

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


# C: one quad and part of it, 20 quads (one range per XCD for few edges, three for many), 33
# quads (more than one round); scale: weights whose lower parts reach down to 2^-100 and up to
# 2^100
@pytest.mark.parametrize("n,c,scale", [(60, 1, 1.0), (60, 7, 1.0), (150, 80, 1.0), (400, 80, 1.0),
                                       (40, 130, 1.0), (60, 8, 2.0 ** -80), (60, 8, 2.0 ** 100)])
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
    """An infinite W2 entry of path 0 (l1 = l2 = l_out = 0, which no rotation mixes with other
    components) makes the same outputs infinite (not NaN) as the fp32 product R = h W2 does:
    channel 1, hidden unit 5."""
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


def _product_inputs(n, ci, co, seed):
    x = torch.randn(n, ci, 16, generator=gen(seed))
    y = torch.randn(n, 16, generator=gen(seed + 1))
    w = torch.randn(34, ci, co, generator=gen(seed + 2)) / ci ** 0.5
    g = torch.randn(n, co, 16, generator=gen(seed + 3))
    return x, y, w, g


# rows: one below and at the forward's line, a last tile of 15 rows, single rows; channels:
# parts of a tile, 1 to 4 tiles of a pass and past it, contracted channels of one 32-step, two,
# a partial second, and past one chunk of 64; the lines that the rounds of workgroups draw
@pytest.mark.parametrize("n,ci,co", [(3071, 8, 8), (3072, 1, 3), (3087, 33, 17), (3073, 64, 65),
                                     (3072, 20, 130), (3088, 130, 20), (3072, 72, 48), (1, 40, 96),
                                     (17, 48, 150), (8200, 4, 40), (3072, 8, 64), (3073, 8, 64),
                                     (4097, 12, 33), (5121, 16, 96), (2561, 16, 64)])
def test_mixing_kernel(bm, dev, n, ci, co):
    x, y, w, g = _product_inputs(n, ci, co, 51)
    out = bm.tensor_product(x.to(dev), y.to(dev), w.to(dev)).cpu().double().numpy()
    gx, gy, gw = bm.tensor_product_backward(x.to(dev), y.to(dev), w.to(dev), g.to(dev))
    only = bm.tensor_product_backward(x.to(dev), y.to(dev), w.to(dev), g.to(dev), False, True, False)
    assert torch.equal(only[1], gy)
    rows = np.unique(np.r_[:20, max(0, n // 2 - 8):n // 2, max(0, n - 20):n])
    rows = rows[rows < n]
    xs, ys, gs = (t[rows].double().numpy() for t in (x, y, g))
    want = otp.tensor_product(xs, ys, w.double().numpy())
    wx, wy, _ = otp.tensor_product_backward(xs, ys, w.double().numpy(), gs)
    # sums of up to 34 * 130 fp32 terms: a few 2^-24 times the square root of their number
    for got, ref in ((out[rows], want), (gx.cpu().double().numpy()[rows], wx),
                     (gy.cpu().double().numpy()[rows], wy)):
        assert np.linalg.norm(got - ref) <= 1e-6 * np.linalg.norm(ref)


# Sums of few products, where the parts' own error shows: y = (1, 0, ...) leaves one path per
# degree, so out and grad_input1 are sums of k products.  The dropped products are at most
# 2^-24 of each and fp32 rounds a few times by at most 2^-24 (6e-8), by 2.5e-8 (rms); grad_input2
# sums over channels and components besides.  same: one sign, and the leading bits at which
# truncated parts would drop most.
@pytest.mark.parametrize("same", [False, True])
@pytest.mark.parametrize("k", [1, 4, 8])
def test_short_sums_against_float64(bm, dev, k, same):
    x, _, w, g = _product_inputs(3072, k, k, 47)
    y = torch.zeros(3072, 16)
    y[:, 0] = 1.0
    if same:
        v = 1.0 + 2.0 ** -7 - 2.0 ** -23
        x, w, g = (torch.full_like(t, v) for t in (x, w, g))
    out = bm.tensor_product(x.to(dev), y.to(dev), w.to(dev))
    gx, gy, _ = bm.tensor_product_backward(x.to(dev), y.to(dev), w.to(dev), g.to(dev))
    d = [t.double().numpy() for t in (x, y, w, g)]
    wx, wy, _ = otp.tensor_product_backward(*d)
    for got, ref, tol in ((out, otp.tensor_product(*d[:3]), 1e-7), (gx, wx, 1e-7), (gy, wy, 2e-7)):
        assert np.linalg.norm(got.cpu().double().numpy() - ref) <= tol * np.linalg.norm(ref)


def test_values_that_bf16_rounds_to_infinity(bm, dev):
    """Up to the largest finite fp32 value: its products are those of fp32."""
    n, c = 3072, 20
    x, _, w, _ = _product_inputs(n, c, c, 48)
    y = torch.zeros(n, 16)
    y[:, 0] = 1.0
    big = torch.tensor([3.4028234e38, -3.4e38, 3.3961775e38])  # (the last: the least such value)
    x[5] = 0.0
    x[5, :3, 0] = big
    w[0, :3] = 0.25 * torch.eye(3, c)
    w[0, 3:] = 0.0
    out = bm.tensor_product(x.to(dev), y.to(dev), w.to(dev)).cpu()
    assert torch.equal(out[5, :3, 0], 0.25 * big)
    keep = [i for i in range(16) if i != 5]  # rows of the same wave
    d = [t[keep].double().numpy() for t in (x, y)]
    ref = otp.tensor_product(*d, w.double().numpy())
    assert np.linalg.norm(out[keep].double().numpy() - ref) <= 1e-6 * np.linalg.norm(ref)


def test_backward_past_the_grid_limit(bm, dev):
    """More rows than one launch's work-items (2^32) hold: the last rows equal their own call's.
    The inputs share one buffer (52 GB with the two gradients)."""
    n, m = 2 ** 28 + 100, 1000
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("not enough free device memory")
    y = torch.randn(n, 16, device=dev)
    w = torch.randn(34, 1, 1, generator=gen(45)).to(dev)
    x = y.view(n, 1, 16)
    gx, gy, _ = bm.tensor_product_backward(x, y, w, x, True, True, False)
    t = y[-m:].clone()
    wx, wy, _ = bm.tensor_product_backward(t.view(m, 1, 16), t, w, t.view(m, 1, 16), True, True, False)
    assert torch.equal(gx[-m:], wx) and torch.equal(gy[-m:], wy)
    del x, y, gx, gy
    torch.cuda.empty_cache()


def test_mixing_kernel_infinities(bm, dev):
    """inf in component 0 of one row's channel reaches that row's outputs through the paths
    (0, l, l) only, as sign(W y) inf, and no other row; the same for an infinite weight."""
    n, ci, co = 3072, 40, 24
    x, y, w, _ = _product_inputs(n, ci, co, 61)
    x[5, 3, 0] = float("inf")
    out = bm.tensor_product(x.to(dev), y.to(dev), w.to(dev)).cpu()
    l = torch.tensor([0] + [1] * 3 + [2] * 5 + [3] * 7)
    sign = torch.sign(w[l, 3, :].T * y[5])          # path l is (0, l, l)
    assert torch.equal(out[5], sign * float("inf"))
    keep = torch.arange(n) != 5
    assert torch.isfinite(out[keep]).all()
    x[5, 3, 0] = 1.0
    w[0, 7, 11] = float("-inf")
    out = bm.tensor_product(x.to(dev), y.to(dev), w.to(dev)).cpu()
    assert torch.equal(out[:, 11, 0], -torch.sign(x[:, 7, 0] * y[:, 0]) * float("inf"))
    out[:, 11, 0] = 0.0
    assert torch.isfinite(out).all()


@pytest.mark.parametrize("nk", [65, 72, 96, 130])
def test_mixing_kernel_infinite_weight_of_an_odd_step(bm, dev, nk):
    """A last chunk of 1 to 32 contracted channels has no second step: an infinite weight in
    its first one reaches one output channel, as sign(x y) inf or sign(g y) inf."""
    n, i = 3072, 20
    k = nk - 1
    x, y, w, _ = _product_inputs(n, nk, i, 63)
    w[0, k, 11] = float("inf")
    out = bm.tensor_product(x.to(dev), y.to(dev), w.to(dev)).cpu()
    assert torch.equal(out[:, 11, 0], torch.sign(x[:, k, 0] * y[:, 0]) * float("inf"))
    out[:, 11, 0] = 0.0
    assert torch.isfinite(out).all()
    x, y, w, g = _product_inputs(100, i, nk, 64)
    w[0, 11, k] = float("inf")
    gx, gy, _ = bm.tensor_product_backward(x.to(dev), y.to(dev), w.to(dev), g.to(dev), True, True,
                                           False)
    gx, gy = gx.cpu(), gy.cpu()
    assert torch.equal(gx[:, 11, 0], torch.sign(g[:, k, 0] * y[:, 0]) * float("inf"))
    gx[:, 11, 0] = 0.0
    assert torch.isfinite(gx).all()
    assert torch.equal(gy[:, 0], torch.sign(x[:, 11, 0] * g[:, k, 0]) * float("inf"))
    assert torch.isfinite(gy[:, 1:]).all()


def _cubic(n_side, spacing, tilt):
    """A cubic lattice: edges along the axes (y is the harmonics' pole) and the diagonals.
    tilt displaces every second plane along y in x and (by 0.7 of it) in z, so that the y edges
    of the atoms at x = 0 or z = 0, where a tilt of any size is kept, lie that far off the pole."""
    k = torch.arange(n_side, dtype=torch.float32) * spacing
    pos = torch.stack(torch.meshgrid(k, k, k, indexing="ij"), -1)
    pos[:, 1::2, :, 0] += tilt
    pos[:, 1::2, :, 2] += 0.7 * tilt
    return pos.reshape(-1, 3).contiguous(), torch.diag(torch.full((3,), n_side * spacing))


# 1e-22 to 1e-20: the square of the off-axis part of u is subnormal or 0; below, in reach of
# rounding and not
@pytest.mark.parametrize("tilt", [0.0, 4e-23, 1e-22, 1e-21, 1e-20, 1e-19, 1e-7, 1e-4, 1e-3])
def test_layer_edges_along_the_pole(bm, dev, tilt):
    import batmobile
    pos, cell = _cubic(4, 3.0, tilt)
    c = 6
    graph = batmobile.Graph(pos.to(dev), cell, 5.0, c)
    if tilt > 0.0:  # edges of the plane x = 0 keep the tilt
        dx = (pos[graph.dst.cpu()] - pos[graph.src.cpu()])[:, 0].abs()
        assert (dx == torch.tensor(tilt)).sum().item() >= 32
    layer = batmobile.MACEInteraction(c, 5.0, device=dev, generator=gen(72))
    x = torch.randn(pos.shape[0], c, 16, generator=gen(73))
    go = torch.randn(pos.shape[0], c, 16, generator=gen(74))
    p = pos.to(dev).requires_grad_(True)
    out = layer(graph, p, x.to(dev))
    (gp,) = torch.autograd.grad(out, p, go.to(dev))
    want, gwant = om.layer_and_position_grad(
        pos.numpy(), torch.diagonal(cell).numpy().astype(np.float64), x.numpy(),
        graph.src.cpu().numpy(), graph.dst.cpu().numpy(), layer.W1.cpu().numpy(),
        layer.b1.cpu().numpy(), layer.W2.cpu().numpy(), 5.0, go.numpy())
    for got, ref in ((out.detach(), want), (gp, gwant)):
        d = got.cpu().double().numpy() - ref
        assert np.linalg.norm(d) <= 4e-6 * np.linalg.norm(ref)


def _layer_against_oracle(dev, pos, cell, c, seed, **kw):
    """(out, gpos, want, gwant) of a layer on the graph of pos."""
    import batmobile
    graph = batmobile.Graph(pos.to(dev), cell, 5.0, c, **kw)
    layer = batmobile.MACEInteraction(c, 5.0, device=dev, generator=gen(seed))
    n = pos.shape[0]
    x = torch.randn(n, c, 16, generator=gen(seed + 1))
    go = torch.randn(n, c, 16, generator=gen(seed + 2))
    p = pos.to(dev).requires_grad_(True)
    out = layer(graph, p, x.to(dev))
    (gp,) = torch.autograd.grad(out, p, go.to(dev))
    want, gwant = om.layer_and_position_grad(
        pos.numpy(), torch.diagonal(cell).numpy().astype(np.float64), x.numpy(),
        graph.src.cpu().numpy(), graph.dst.cpu().numpy(), layer.W1.cpu().numpy(),
        layer.b1.cpu().numpy(), layer.W2.cpu().numpy(), 5.0, go.numpy())
    return out.detach().cpu().double().numpy(), gp.cpu().double().numpy(), want, gwant


def test_layer_self_loops(bm, dev):
    """An edge of no length: Y = (1, 0, ...), so only the paths with l2 = 0 act.  The basis is
    taken at r = 1e-10.  Its position gradient cancels against that of its reverse, itself."""
    pos, cell = periodic_box(60, 81)
    for got, ref in zip(*[iter(_layer_against_oracle(dev, pos, cell, 5, 82, self_loops=True)[i]
                               for i in (0, 2, 1, 3))] * 2):
        assert np.linalg.norm(got - ref) <= 4e-6 * np.linalg.norm(ref)


# two atoms at one place, below the length's lower bound 1e-10 along the pole, across and
# askew, below where squares are subnormal, and just above the bound
@pytest.mark.parametrize("d", [(0.0, 0.0, 0.0), (0.0, 5e-11, 0.0), (5e-11, 0.0, 0.0),
                               (3e-11, -4e-11, 6e-11), (2e-30, 1e-30, 0.0), (1e-10, 0.0, 1e-11)])
def test_layer_short_edges(bm, dev, d):
    """u = v / 1e-10 below the bound, the length a constant: the gradient of the two atoms is
    of the order of 1e10, those of the others are as ever."""
    pos = torch.tensor([[0.0, 0.0, 0.0], d, [1.0, 1.5, 2.0], [1.5, -1.0, 0.5]])
    out, gp, want, gwant = _layer_against_oracle(dev, pos, torch.diag(torch.full((3,), 20.0)), 5, 72)
    for got, ref in ((out, want), (gp[:2], gwant[:2]), (gp[2:], gwant[2:])):
        assert np.linalg.norm(got - ref) <= 4e-6 * np.linalg.norm(ref)


def test_layer_frame_error(bm, dev):
    """The edge's frame alone: W1 = 0 and b1 = 20 make h = 20 on every edge, so that the radial
    basis adds nothing.  Means over eight graphs, out / gradient: 1.9 / 2.9e-7; the product by CG
    entries, without a frame, had 2.3 / 3.1e-7, a frame off unit length by fp32 rounding
    2.6 / 3.7e-7."""
    import batmobile
    err = []
    for seed in range(8):
        n, c = 250, 8
        pos, cell = periodic_box(n, 100 + seed)
        graph = batmobile.Graph(pos.to(dev), cell, 5.0, c)
        layer = batmobile.MACEInteraction(c, 5.0, device=dev, generator=gen(72 + seed))
        layer.W1.zero_()
        layer.b1.fill_(20.0)
        x = torch.randn(n, c, 16, generator=gen(300 + seed))
        go = torch.randn(n, c, 16, generator=gen(400 + seed))
        p = pos.to(dev).requires_grad_(True)
        out = layer(graph, p, x.to(dev))
        (gp,) = torch.autograd.grad(out, p, go.to(dev))
        want = om.layer_and_position_grad(
            pos.numpy(), torch.diagonal(cell).numpy().astype(np.float64), x.numpy(),
            graph.src.cpu().numpy(), graph.dst.cpu().numpy(), layer.W1.cpu().numpy(),
            layer.b1.cpu().numpy(), layer.W2.cpu().numpy(), 5.0, go.numpy())
        err.append([np.linalg.norm(got.detach().cpu().double().numpy() - ref) / np.linalg.norm(ref)
                    for got, ref in zip((out, gp), want)])
    out_err, grad_err = np.mean(err, axis=0)
    print(f"frame error {out_err:.3g} {grad_err:.3g}")
    assert out_err <= 2.2e-7 and grad_err <= 3.1e-7


def test_layer_nan_position(bm, dev):
    """A NaN coordinate reaches every component of the atom's neighbours."""
    import batmobile
    pos, cell = periodic_box(80, 91)
    graph = batmobile.Graph(pos.to(dev), cell, 5.0, 4)
    layer = batmobile.MACEInteraction(4, 5.0, device=dev, generator=gen(92))
    x = torch.randn(80, 4, 16, generator=gen(93))
    src, dst = graph.src.cpu(), graph.dst.cpu()
    hit = torch.zeros(80, dtype=torch.bool)
    hit[dst[src == 7]] = True
    hit[7] = (dst == 7).any()
    for k in range(3):
        bad = pos.clone()
        bad[7, k] = float("nan")
        out = layer(graph, bad.to(dev), x.to(dev)).cpu()
        assert torch.isnan(out[hit]).all() and torch.isfinite(out[~hit]).all()


# the kernels that calls without a workspace take: two row tiles a workgroup, one, 128
# output channels, and past 128 with the rows staged and not
@pytest.mark.parametrize("n,ci,co", [(50, 32, 64), (17, 40, 24), (33, 24, 100), (9, 16, 130),
                                     (5, 8, 600)])
def test_backward_without_workspace(bm, dev, n, ci, co):
    import ctypes
    import os
    repo = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    lib = ctypes.CDLL(os.path.join(repo, "batmobile-evo_amd", "lib", "libbatmobile_hip.so"))
    P = ctypes.c_void_p
    fn = lib.batteries_tensor_product_backward_l3
    fn.restype = ctypes.c_int
    fn.argtypes = [P] * 7 + [ctypes.c_int64, ctypes.c_int, ctypes.c_int, P, ctypes.c_size_t, P]
    x, y, w, g = (t.to(dev) for t in _product_inputs(n, ci, co, 91))
    gx = torch.full_like(x, float("nan"))
    gy = torch.full_like(y, float("nan"))
    p = [P(t.data_ptr()) for t in (x, y, w, g, gx, gy)]
    stream = P(torch.cuda.current_stream().cuda_stream)
    assert fn(*p, None, n, ci, co, None, 0, stream) == 0
    torch.cuda.synchronize()
    wx, wy, _ = otp.tensor_product_backward(*(t.cpu().double().numpy() for t in (x, y, w, g)))
    for got, ref in ((gx, wx), (gy, wy)):
        d = got.cpu().double().numpy() - ref
        assert np.linalg.norm(d) <= 1e-6 * np.linalg.norm(ref)
