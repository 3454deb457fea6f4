"""The data operator for every kind of channel count (one channel per XCD,
channels split over several, odd counts): each channel's rows and image equal
the single-channel operator's, so no unit of a launch is lost or done twice."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('N', [64, 20])          # tile-gridded rows, and the column gather
@pytest.mark.parametrize('L', [1, 2, 3, 4, 8, 12, 17])
def test_channels_match_single_channel(ctx, L, N):
    import fhs
    from fhs import solvers
    from fhs.nufft import Nufft2D
    lib = solvers.lib()
    rng = np.random.default_rng(100 * N + L)
    nf = Nufft2D(N, N)
    plan = nf.plan(ctx)
    Gs = []
    for l in range(L):
        u, v = rng.normal(0, np.pi / 4, (2, 500 + 300 * l)).clip(-3.1, 3.1)
        Gs.append(fhs.GMatrix.from_separable(ctx, *nf.separable_gpu(ctx, u, v), nf.Kty, nf.Ktx))
    D = fhs.DataOperator(ctx, plan, Gs, [[g.M] for g in Gs])
    x = torch.rand((L, N, N), device='cuda')
    y = torch.randn(D.Mtot, dtype=torch.complex64, device='cuda')
    out = torch.full_like(y, float('nan'))
    back = torch.full_like(x, float('nan'))
    ctx.check(lib.fhs_data_forward(ctx.h, D.h, x.data_ptr(), None, out.data_ptr()), 'data_forward')
    ctx.check(lib.fhs_data_adjoint(ctx.h, D.h, y.data_ptr(), None, None, back.data_ptr()), 'data_adjoint')
    for l, g in enumerate(Gs):
        rows = slice(D.row_offset[l], D.row_offset[l + 1])
        # the same kernels on the same rows, up to the order of FP32 sums
        ref = fhs.apply_direct_operator(plan.A(x[l]), g)
        img = plan.At_real(fhs.apply_adjoint_operator(y[rows].contiguous(), g))
        assert torch.linalg.vector_norm(out[rows] - ref) <= 1e-5 * torch.linalg.vector_norm(ref)
        assert torch.linalg.vector_norm(back[l] - img) <= 1e-5 * torch.linalg.vector_norm(img)
