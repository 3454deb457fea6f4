"""Every use of the analysis (set, accumulate, l21 step, weights, prior) and the
synthesis at the edges of their tiles (56 x 4 coefficients, 112 x 8 pixels),
for channel counts that fill a workgroup, do not, and exceed it; against the
FP64 oracle at the 1e-5 of the FP32 transforms."""
import numpy as np
import pytest
import torch

from oracle.wavelets import SaraDictionary as SaraRef

pytestmark = pytest.mark.gpu
TOL = 1e-5


def rel(a, b):
    return np.linalg.norm(np.asarray(a, dtype=np.float64) - b) / np.linalg.norm(b)


@pytest.mark.parametrize('Ny,Nx,L,nlevel', [(5, 3, 1, 2), (112, 8, 2, 1), (113, 9, 5, 4), (30, 250, 4, 4),
                                            (98, 64, 16, 4), (40, 33, 17, 3), (24, 20, 35, 2)])
def test_modes(ctx, Ny, Nx, L, nlevel):
    import fhs
    rng = np.random.default_rng(Ny + Nx + L)
    S = fhs.SaraDictionary(ctx, Ny, Nx, nlevel=nlevel)
    ref = SaraRef(Ny, Nx, nlevel=nlevel)
    x = rng.random((L, Nx, Ny)).astype(np.float32)
    xd = torch.from_numpy(x).cuda()
    c = np.stack([ref.psit(x[l].T.astype(np.float64)) for l in range(L)])
    out = torch.full((L, S.s), float('nan'), device='cuda')
    S.psit(xd, out=out)
    assert rel(out.cpu().numpy(), c) < TOL
    v1 = rng.standard_normal((L, S.s)).astype(np.float32)
    w = rng.random(S.s).astype(np.float32)
    acc = torch.from_numpy(v1).cuda()
    S.psit(xd, out=acc, accumulate=True)
    assert rel(acc.cpu().numpy(), v1 + c) < TOL
    for weights in (w, None):
        vd = torch.from_numpy(v1).cuda()
        vd, g1 = fhs.hs_update_dual_sparsity_distributed(
            vd, S, S, xd, None if weights is None else torch.from_numpy(weights).cuda(), 0.8, 0.3)
        r = v1.astype(np.float64) + c
        n = np.linalg.norm(r, axis=0)
        thr = 0.8 * (1.0 if weights is None else weights.astype(np.float64))
        vr = r - np.maximum(n - thr, 0) / (n + np.finfo(float).eps) * r
        assert rel(vd.cpu().numpy(), vr) < TOL
        gr = np.stack([0.3 * ref.psi(vr[l]).T for l in range(L)])
        assert rel(g1.cpu().numpy(), gr) < TOL
    wd = torch.full((S.s,), float('nan'), device='cuda')
    ctx.check(fhs.lib().fhs_sara_update_weights(ctx.h, S.h, xd.data_ptr(), L, 0.1, wd.data_ptr()), 'weights')
    n = np.linalg.norm(c, axis=0)
    assert rel(wd.cpu().numpy(), 0.1 / (0.1 + n)) < TOL
    assert abs(fhs.compute_sara_prior(xd, S) / n.sum() - 1) < TOL


@pytest.mark.parametrize('Ny,Nx', [(16, 12), (7, 5)])       # four pixels a thread, one
def test_dirac_block_keeps_infinities(ctx, Ny, Nx):
    """Without a threshold the Dirac coefficients are the scaled pixels, infinite
    ones too: no product with a zero factor turns them into NaN."""
    import fhs
    for bases in (('db2', 'db8', 'self'), ('self',)):
        S = fhs.SaraDictionary(ctx, Ny, Nx, bases=bases, nlevel=1)
        x = torch.ones((2, Nx, Ny), device='cuda')
        x[0, 1, 2], x[1, 3, 4] = float('inf'), -float('inf')
        want = x.reshape(2, -1) * np.float32(1 / np.sqrt(len(bases)))
        c = S.psit(x)[:, -Nx * Ny:]
        assert torch.equal(c, want)
        out = torch.full((2, S.s), 0.5, device='cuda')
        S.psit(x, out=out, accumulate=True)
        assert torch.allclose(out[:, -Nx * Ny:], want + 0.5)


@pytest.mark.parametrize('L', [3, 17])
def test_captured_step_outlives_its_dictionary(L):
    """A captured dual step needs its dictionary no more, which may also be created
    and dropped while the capture runs: replays give the eager step."""
    import gc
    import fhs
    ctx = fhs.Context(0)
    Ny, Nx = 60, 41
    rng = np.random.default_rng(L)
    x = torch.from_numpy(rng.random((L, Nx, Ny)).astype(np.float32)).cuda()
    S = fhs.SaraDictionary(ctx, Ny, Nx, nlevel=2)
    v0 = torch.from_numpy(rng.standard_normal((L, S.s)).astype(np.float32)).cuda()

    def step(S, v):
        return fhs.hs_update_dual_sparsity_distributed(v, S, S, x, None, 0.8, 0.3)

    want = [t.clone() for t in step(S, v0.clone())]      # also sizes the context's workspace
    v = v0.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ctx.bind_stream()
        D = fhs.SaraDictionary(ctx, Ny, Nx, nlevel=2)
        got = step(D, v)
        del D
        gc.collect()
    ctx.bind_stream()
    for seed in range(4):
        v.copy_(v0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
        again = step(S, v0.clone())                        # eager work between the replays
        assert torch.equal(again[0], want[0]) and torch.equal(again[1], want[1])


def _captured_nodes(ctx, f):
    """Nodes of the graph that a call captures."""
    import ctypes as C
    import fhs
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        ctx.bind_stream()
        f()
    ctx.bind_stream()
    n = C.c_size_t()
    assert fhs.lib().hipGraphGetNodes(C.c_void_p(graph.raw_cuda_graph()), None, C.byref(n)) == 0
    return n.value


def test_many_channels_take_no_more_launches():
    """The channels beyond a workgroup's 16 run in the same launches, not in a chain
    of launches of their own."""
    import fhs
    ctx = fhs.Context(0)
    S = fhs.SaraDictionary(ctx, 32, 24, nlevel=3)
    nodes = []
    for L in (16, 17, 64):
        x, c = torch.rand((L, 24, 32), device='cuda'), torch.empty((L, S.s), device='cuda')
        S.psit(x, out=c)                       # sizes the context's workspace
        torch.cuda.synchronize()
        nodes.append(_captured_nodes(ctx, lambda: S.psit(x, out=c)))
    assert nodes == [4, 4, 4], nodes           # three levels and the Dirac block


@pytest.mark.parametrize('Ny,Nx,L', [(1, 1, 1), (33, 17, 3), (600, 900, 2)])
def test_dirac_basis_alone(ctx, Ny, Nx, L):
    """Without wavelets the transforms are the identity, the dual step the threshold."""
    import fhs
    S = fhs.SaraDictionary(ctx, Ny, Nx, bases=('self',), nlevel=1)
    x = torch.randn((L, Nx, Ny), device='cuda')
    assert torch.equal(S.psit(x).reshape(x.shape), x)
    assert torch.equal(S.psi(x.reshape(L, -1), scale=0.5), 0.5 * x)
