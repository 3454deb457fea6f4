"""Scaled FFT of a real image: column pairs, mirrored and shared rows, and the
lengths whose workgroups hold 4, 8 or 16 values a thread."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('Ny,Nx,Kty,Ktx', [
    (1, 1, 16, 16), (7, 9, 16, 32), (33, 31, 64, 64), (100, 37, 256, 512), (512, 513, 1024, 1024), (9, 700, 32, 2048),
    (6, 2047, 16, 4096), (6, 3001, 16, 4096), (15, 21, 45, 45), (20, 41, 45, 128), (44, 13, 90, 32),
    (17, 500, 50, 1000), (500, 33, 1000, 72), (5, 2501, 18, 5120), (5, 11, 8192, 16), (5, 4000, 16, 8192),
    (5, 4097, 18, 8100)])
def test_scaled_fft(Ny, Nx, Kty, Ktx):
    """FP32 transforms of up to 2^26 points against FP64: log2(points) roundings of
    6e-8 add to 2e-6 at most."""
    import torch
    import fhs
    rng = np.random.default_rng(Ny + Nx + Kty)
    ctx = fhs.default_context(0)
    sy, sx = rng.uniform(0.5, 2, Ny).astype(np.float32), rng.uniform(0.5, 2, Nx).astype(np.float32)
    plan = fhs.NufftPlan(ctx, Ny, Nx, Kty, Ktx, sy.astype(np.float64), sx.astype(np.float64))
    L, sn = 2, sx[:, None].astype(np.float64) * sy
    x = rng.normal(size=(L, Nx, Ny)).astype(np.float32)
    F = plan.A(torch.from_numpy(x).cuda()).cpu().numpy().reshape(L, Ktx, Kty)
    ref = np.fft.fft2(x * sn, s=(Ktx, Kty))
    assert np.linalg.norm(F - ref) < 2e-6 * np.linalg.norm(ref)
    g = (rng.normal(size=(L, Ktx * Kty)) + 1j * rng.normal(size=(L, Ktx * Kty))).astype(np.complex64)
    scale = [1.0, 0.25]
    out = plan.At_real(torch.from_numpy(g).cuda(), scale).cpu().numpy().reshape(L, Nx, Ny)
    ref = np.fft.ifft2(g.reshape(L, Ktx, Kty).astype(np.complex128), norm='forward').real[:, :Nx, :Ny] * sn
    ref *= np.array(scale)[:, None, None]
    assert np.linalg.norm(out - ref) < 2e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize('Ny,Nx,Kty,Ktx,L', [
    (1, 1, 16, 16, 256), (33, 31, 64, 64, 128), (100, 37, 256, 512, 32), (100, 37, 256, 512, 31), (77, 128, 256, 256, 33),
    (512, 513, 1024, 1024, 4), (512, 513, 1024, 1024, 1), (9, 700, 32, 2048, 64), (6, 2047, 16, 4096, 1),
    (6, 2047, 1024, 4096, 8), (6, 3001, 1024, 4096, 8), (300, 700, 1024, 2048, 16)])
def test_adjoint_on_both_sides_of_its_rule(Ny, Nx, Kty, Ktx, L):
    """Launches that fill the chip transform half of the rows, smaller ones all of them
    with fewer rows a workgroup: both against FP64, with the bound of test_scaled_fft."""
    import torch
    import fhs
    rng = np.random.default_rng(Ny + Nx + L)
    ctx = fhs.default_context(0)
    sy, sx = rng.uniform(0.5, 2, Ny).astype(np.float32), rng.uniform(0.5, 2, Nx).astype(np.float32)
    plan = fhs.NufftPlan(ctx, Ny, Nx, Kty, Ktx, sy.astype(np.float64), sx.astype(np.float64))
    sn = torch.from_numpy(sx[:, None].astype(np.float64) * sy).cuda()
    x = torch.from_numpy(rng.normal(size=(L, Nx, Ny)).astype(np.float32)).cuda()
    ref = torch.fft.fft2(x.double() * sn, s=(Ktx, Kty))
    F = plan.A(x).reshape(L, Ktx, Kty)
    assert torch.linalg.vector_norm(F - ref) < 2e-6 * torch.linalg.vector_norm(ref)
    del F, ref
    g = torch.view_as_complex(torch.from_numpy(rng.normal(size=(L, Ktx * Kty, 2)).astype(np.float32)).cuda())
    out = plan.At_real(g).reshape(L, Nx, Ny)
    ref = torch.fft.ifft2(g.reshape(L, Ktx, Kty).to(torch.complex128), norm='forward').real[:, :Nx, :Ny] * sn
    assert torch.linalg.vector_norm(out - ref) < 2e-6 * torch.linalg.vector_norm(ref)
