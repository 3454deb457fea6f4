"""The tiled gridding adjoint (matrix cores, one wave per 16 x 16 quadrant) at
the sizes where it can go wrong: windows of one tap, of the slot count and one
less, anchors on every side of a tile and across the grid's wrap, fewer rows
than a group, more rows than a work item; against the FP64 sparse product
(1e-5: FP32 sums of at most a few thousand terms).  A non-finite visibility
reaches exactly the grid points of its window."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

pytestmark = pytest.mark.gpu
Kty, Ktx = 96, 64


def _problem(Ky, Kx, M, seed):
    rng = np.random.default_rng(seed)
    ky, kx = rng.integers(0, Kty, M), rng.integers(0, Ktx, M)
    ky[M // 2:], kx[M // 2:] = rng.integers(28, 36, M - M // 2), rng.integers(60, 64, M - M // 2)   # a dense, wrapping spot
    cy = (rng.standard_normal((M, Ky)) + 1j * rng.standard_normal((M, Ky))).astype(np.complex64)
    cx = (rng.standard_normal((M, Kx)) + 1j * rng.standard_normal((M, Kx))).astype(np.complex64)
    iy, ix = (ky[:, None] + np.arange(Ky)) % Kty, (kx[:, None] + np.arange(Kx)) % Ktx
    cols = (iy[:, :, None] + Kty * ix[:, None, :]).reshape(M, -1)
    vals = (cy.astype(complex)[:, :, None] * cx.astype(complex)[:, None, :]).reshape(M, -1)
    G = sp.csr_matrix((vals.ravel(), (np.repeat(np.arange(M), Ky * Kx), cols.ravel())), shape=(M, Kty * Ktx))
    y = (rng.standard_normal(M) + 1j * rng.standard_normal(M)).astype(np.complex64)
    return (ky + Kty * kx).astype(np.int32), cy, cx, G, y, rng.uniform(0.5, 1.5, M).astype(np.float32)


@pytest.mark.parametrize('M', [1, 3, 67, 6000])
@pytest.mark.parametrize('Ky,Kx', [(7, 7), (8, 8), (1, 8), (5, 1), (15, 15), (16, 16), (9, 3)])
def test_adjoint_tiles(ctx, Ky, Kx, M):
    import fhs
    a, cy, cx, G, y, lam = _problem(Ky, Kx, M, 10 * M + Ky)
    g = fhs.GMatrix.from_separable(ctx, a, cy, cx, Kty, Ktx)
    yd = torch.from_numpy(y).cuda()
    for l in (None, lam):
        out = fhs.apply_adjoint_operator(yd, g, None if l is None else torch.from_numpy(l).cuda()).cpu().numpy()
        ref = G.conj().T @ (y.astype(complex) if l is None else l.astype(float) * y)
        assert np.linalg.norm(out - ref) <= 1e-5 * np.linalg.norm(ref)


@pytest.mark.parametrize('K', [7, 15])
def test_non_finite_visibility_stays_in_its_window(ctx, K):
    import fhs
    a, cy, cx, G, y, _ = _problem(K, K, 500, K)
    bad = [3, 400]
    g = fhs.GMatrix.from_separable(ctx, a, cy, cx, Kty, Ktx)
    yd = torch.from_numpy(y).cuda()
    yd[bad[0]], yd[bad[1]] = float('nan'), complex(float('inf'), 0.0)
    out = fhs.apply_adjoint_operator(yd, g).cpu().numpy()
    hit = np.asarray(abs(G[bad]).sum(axis=0)).ravel() > 0
    assert np.array_equal(~np.isfinite(out), hit)
    y[bad] = 0
    ref = G.conj().T @ y.astype(complex)
    assert np.linalg.norm((out - ref)[~hit]) <= 1e-5 * np.linalg.norm(ref)
