"""GPU kernels of the learned warm start against the FP64 U-Net oracle.

Operands are rounded to BF16 in both (the oracle rounds exactly where the
GEMM stages them), so single layers agree at FP32-accumulation precision
(1e-4); the whole network, where a 1-ulp BF16 flip of an activation
propagates, within 2e-2."""
import numpy as np
import pytest
import torch

from oracle.unet import OracleUNet, bf16, col2im3, im2col3, maxpool2, upsample2

pytestmark = pytest.mark.gpu


def rel(a, b):
    a = np.asarray(a, np.float64); b = np.asarray(b, np.float64)
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


@pytest.mark.parametrize('M,N,K', [(16, 16, 16), (37, 129, 70), (128, 4096, 1152), (200, 64, 33),
                                   (16, 72, 20000), (40, 300, 8200)])   # the last two split K
@pytest.mark.parametrize('ta,tb', [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_gemm_bf16(ctx, M, N, K, ta, tb):
    import ctypes as C
    from fhs._lib import lib
    from fhs.core import _ptr
    rng = np.random.default_rng(M + N + K + 2 * ta + tb)
    A = rng.normal(size=(K, M) if ta else (M, K)).astype(np.float32)
    B = rng.normal(size=(N, K) if tb else (K, N)).astype(np.float32)
    bias = rng.normal(size=M).astype(np.float32)
    Cd = torch.zeros((M, N), dtype=torch.float32, device='cuda')
    Ad, Bd, bd = dev(A), dev(B), dev(bias)     # held until the kernel has run
    ctx.check(lib().fhs_nn_gemm(ctx.h, M, N, K, _ptr(Ad), M if ta else K, ta, _ptr(Bd), K if tb else N, tb,
                                _ptr(Cd), N, 1.0, 0.0, _ptr(bd), 0), 'gemm')
    torch.cuda.synchronize()
    opA = bf16(A).T if ta else bf16(A)
    opB = bf16(B).T if tb else bf16(B)
    ref = opA @ opB + bias[:, None]
    assert rel(Cd.cpu().numpy(), ref) < 1e-5
    # beta = 1 accumulates into C (the weight-gradient use)
    ctx.check(lib().fhs_nn_gemm(ctx.h, M, N, K, _ptr(Ad), M if ta else K, ta, _ptr(Bd), K if tb else N, tb,
                                _ptr(Cd), N, 1.0, 1.0, None, 0), 'gemm beta')
    assert rel(Cd.cpu().numpy(), 2 * (opA @ opB) + bias[:, None]) < 1e-5


def test_layer_primitives(ctx):
    import ctypes as C
    from fhs._lib import lib
    from fhs.core import _ptr
    rng = np.random.default_rng(1)
    Cc, NB, H, W = 5, 2, 12, 10
    x = rng.normal(size=(Cc, NB * H * W)).astype(np.float32)
    xd = dev(x)
    col = torch.empty((Cc * 9, NB * H * W), dtype=torch.float32, device='cuda')
    ctx.check(lib().fhs_nn_im2col3(ctx.h, _ptr(xd), Cc, NB, H, W, _ptr(col)), 'im2col')
    assert rel(col.cpu().numpy(), im2col3(x.astype(np.float64), NB, H, W)) < 1e-7
    dcol = rng.normal(size=(Cc * 9, NB * H * W)).astype(np.float32)
    dcold = dev(dcol)
    din = torch.empty((Cc, NB * H * W), dtype=torch.float32, device='cuda')
    ctx.check(lib().fhs_nn_col2im3(ctx.h, _ptr(dcold), Cc, NB, H, W, _ptr(din)), 'col2im')
    assert rel(din.cpu().numpy(), col2im3(dcol.astype(np.float64), Cc, NB, H, W)) < 1e-6
    p = torch.empty((Cc, NB * H * W // 4), dtype=torch.float32, device='cuda')
    ctx.check(lib().fhs_nn_maxpool2(ctx.h, _ptr(xd), Cc * NB, H, W, _ptr(p)), 'pool')
    assert rel(p.cpu().numpy(), maxpool2(x.astype(np.float64), NB, H, W)[0]) == 0
    u = torch.empty((Cc, NB * H * W * 4), dtype=torch.float32, device='cuda')
    ctx.check(lib().fhs_nn_upsample2(ctx.h, _ptr(xd), Cc * NB, H, W, _ptr(u)), 'up')
    assert rel(u.cpu().numpy(), upsample2(x.astype(np.float64), Cc, NB, H, W)) == 0


def _oracle_of(net, bf):
    layers = [(l.W.cpu().numpy(), l.b.cpu().numpy(), l.relu) for l in net.layers()]
    return OracleUNet(layers, net.widths, bf=bf)


@pytest.mark.parametrize('widths,NB,H,W', [((4, 6, 8, 10), 2, 16, 16), ((16, 32, 64, 128), 1, 32, 48)])
def test_unet_forward_backward(ctx, widths, NB, H, W):
    from fhs.unet import UNet
    rng = np.random.default_rng(len(widths) + H)
    net = UNet(ctx, cin=8, cout=8, widths=widths, seed=3)
    x = rng.normal(size=(8, NB * H * W)).astype(np.float32)
    t = rng.normal(size=(8, NB * H * W)).astype(np.float32)
    y = net.forward(dev(x), NB, H, W)
    loss, g = net.mse(y, dev(t))
    net.zero_grad()
    gx = net.backward(g, NB, H, W)
    orc = _oracle_of(net, bf=True)
    yo = orc.forward(x.astype(np.float64), NB, H, W)
    assert rel(y.cpu().numpy(), yo) < 2e-2
    go = orc.backward(2.0 / y.numel() * (yo - t), NB, H, W)
    assert rel(gx.cpu().numpy(), go) < 2e-2
    for lg, lo in zip(net.layers(), orc.layers):
        assert rel(lg.dW.cpu().numpy(), lo['dW']) < 2e-2
        assert rel(lg.db.cpu().numpy(), lo['db']) < 2e-2


def test_unet_training_reduces_loss(ctx):
    from fhs.unet import UNet
    rng = np.random.default_rng(5)
    net = UNet(ctx, cin=8, cout=8, widths=(8, 16, 32, 64), seed=1)
    NB, H, W = 2, 32, 32
    x = rng.random((8, NB * H * W)).astype(np.float32)
    t = (0.5 * x + 0.1).astype(np.float32)
    xd, td = dev(x), dev(t)
    first = None
    for step in range(60):
        net.zero_grad()
        y = net.forward(xd, NB, H, W)
        loss, g = net.mse(y, td)
        first = loss if first is None else first
        net.backward(g, NB, H, W)
        net.adam(lr=2e-3)
    assert loss < 0.1 * first


@pytest.mark.parametrize('cin,cout,NB,H,W', [(8, 16, 1, 8, 32), (5, 3, 2, 9, 33), (16, 16, 1, 3, 7), (17, 40, 1, 20, 45),
                                             (64, 32, 2, 16, 64), (128, 128, 1, 8, 8), (24, 20, 3, 70, 38)])
@pytest.mark.parametrize('relu', [True, False])
def test_conv3x3(ctx, cin, cout, NB, H, W, relu):
    """The convolution and its gradients at the edges of their pixel tiles and
    channel groups, against the FP64 products of the BF16-rounded operands
    (1e-5: FP32 sums), and the bits of im2col, GEMM and col2im."""
    from fhs._lib import lib
    from fhs.core import _ptr
    rng = np.random.default_rng(cin + cout + W)
    Q = NB * H * W
    x, w, b, gy = (rng.normal(size=s).astype(np.float32) for s in ((cin, Q), (cout, cin * 9), (cout,), (cout, Q)))
    xd, wd, bd, gd = dev(x), dev(w), dev(b), dev(gy)
    y = torch.full((cout, Q), float('nan'), device='cuda')
    ctx.check(lib().fhs_nn_conv3x3(ctx.h, _ptr(xd), cin, NB, H, W, _ptr(wd), cout, _ptr(bd), int(relu), _ptr(y)), 'conv')
    col = im2col3(bf16(x), NB, H, W)
    ref = bf16(w) @ col + b[:, None].astype(np.float64)
    ref = np.maximum(ref, 0) if relu else ref
    assert rel(y.cpu().numpy(), ref) < 1e-5
    cd, yg = torch.empty((cin * 9, Q), device='cuda'), torch.empty_like(y)
    ctx.check(lib().fhs_nn_im2col3(ctx.h, _ptr(xd), cin, NB, H, W, _ptr(cd)), 'im2col')
    ctx.check(lib().fhs_nn_gemm(ctx.h, cout, Q, cin * 9, _ptr(wd), cin * 9, 0, _ptr(cd), Q, 0, _ptr(yg), Q, 1.0, 0.0,
                                _ptr(bd), int(relu)), 'gemm')
    assert torch.equal(y, yg)
    dw, db = dev(np.ones_like(w)), dev(np.ones_like(b))
    dx = torch.full((cin, Q), float('nan'), device='cuda')
    ctx.check(lib().fhs_nn_conv3x3_backward(ctx.h, _ptr(xd), cin, NB, H, W, _ptr(wd), cout, _ptr(y) if relu else None,
                                            _ptr(gd), _ptr(dw), _ptr(db), _ptr(dx)), 'conv backward')
    g = np.where(y.cpu().numpy() > 0, gy, 0) if relu else gy
    assert rel(dw.cpu().numpy() - 1.0, bf16(g) @ col.T) < 1e-5
    assert rel(db.cpu().numpy() - 1.0, g.astype(np.float64).sum(1)) < 1e-5
    assert rel(dx.cpu().numpy(), col2im3(bf16(w).T @ bf16(g), cin, NB, H, W)) < 1e-5
    gm, xg = dev(g.astype(np.float32)), torch.empty_like(dx)
    wg = dev(np.ones_like(w))
    ctx.check(lib().fhs_nn_gemm(ctx.h, cout, cin * 9, Q, _ptr(gm), Q, 0, _ptr(cd), Q, 1, _ptr(wg), cin * 9, 1.0, 1.0,
                                None, 0), 'gemm')
    assert torch.equal(dw, wg)
    ctx.check(lib().fhs_nn_gemm(ctx.h, cin * 9, Q, cout, _ptr(wd), cin * 9, 1, _ptr(gm), Q, 0, _ptr(cd), Q, 1.0, 0.0,
                                None, 0), 'gemm')
    ctx.check(lib().fhs_nn_col2im3(ctx.h, _ptr(cd), cin, NB, H, W, _ptr(xg)), 'col2im')
    assert torch.equal(dx, xg)


@pytest.mark.parametrize('net', [False, True])
def test_backward_after_the_input_was_reused(ctx, net):
    """A layer's, and the network's, gradients are those of the input that forward
    saw: writing to that tensor before backward changes none of them."""
    from fhs.unet import Conv3x3, UNet
    NB, H, W = 1, 8, 16
    rng = np.random.default_rng(11)
    x, gy = (dev(rng.normal(size=(8, NB * H * W))) for _ in range(2))
    grads = []
    for reuse in (False, True):
        m = UNet(ctx, 8, 8, widths=(8, 8), seed=2) if net else Conv3x3(ctx, 8, 8, True, np.random.default_rng(2))
        xin = x.clone()
        m.forward(xin, NB, H, W)
        if reuse:
            xin.zero_()
        dx = m.backward(gy.clone(), NB, H, W) if net else m.backward(gy.clone())
        layers = m.layers() if net else [m]
        grads.append([dx] + [t.clone() for p in layers for t in (p.dW, p.db)])
    assert all(torch.equal(a, b) for a, b in zip(*grads))
    assert all(float(g.abs().max()) > 0 for g in grads[0])
