"""Edges of the register FFTs and of the one-launch product: grids that leave
a remainder in every embedding (N < M/2), both precisions, batches.  The
product formed by torch.fft in complex128 is the reference."""
import numpy as np
import pytest

from conftest import rel
from test_rocfft_crosscheck import _torch_matvec

pytestmark = pytest.mark.gpu


# N = 5 ... 48: one launch (M = 16 ... 96); FP64 up to M = 64; above, three
# passes with 8, 12 and 16 elements per thread, up to the 4096-point FP64
# transform (72 KB of LDS)
@pytest.mark.parametrize("N", [5, 12, 13, 24, 31, 33, 47, 48, 49, 97, 130, 333, 513, 700, 1025, 2047])
def test_products_on_ragged_grids(N):
    """complex64 to 2e-6 and complex128 to 1e-12 (FP32 and FP64 rounding of a
    transform of at most 4096 points, measured 2e-7 and 1e-14), three vectors,
    one shared map and own maps, all modes; a single product equals the
    batched one bit for bit."""
    import torch
    from cugmres_amd import problems, solver
    print(f"ragged grid N={N}", flush=True)
    ctx = solver.Context(N, 0)
    g, g64 = ctx.spectrum_helmholtz(problems.KH, fp64=True)
    blk = ctx.block_helmholtz(problems.KH)
    rng = np.random.default_rng(N)
    B = 3 if N < 1024 else 1
    chi = torch.as_tensor(rng.uniform(0.0, 11.1, (B, N * N))).to(ctx.device)
    x = torch.as_tensor(rng.standard_normal((B, N * N)) + 1j * rng.standard_normal((B, N * N))).to(ctx.device)
    c32, x32 = chi.to(torch.float32), x.to(torch.complex64)
    ctx.set_radix_plan(0)   # one form of the N = 512 passes, whatever the batch
    for mode in (0, 1, 2):
        own = ctx.matvec_batched(g, c32, x32, mode)
        shared = ctx.matvec_batched(g, c32[0].contiguous(), x32, mode)
        for k in range(B):
            ref = _torch_matvec(torch, blk, c32[k].to(torch.float64), x32[k].to(torch.complex128), N, ctx.M, mode)
            assert rel(own[k].cpu().numpy(), ref.cpu().numpy()) < 2e-6, (mode, k)
            assert torch.equal(own[k], ctx.matvec(g, c32[k].contiguous(), x32[k].contiguous(), mode)), (mode, k)
            assert torch.equal(shared[k], ctx.matvec(g, c32[0].contiguous(), x32[k].contiguous(), mode)), (mode, k)
        y64 = ctx.matvec_c128(g64, chi[0].contiguous(), x[0].contiguous(), mode)
        ref = _torch_matvec(torch, blk, chi[0], x[0], N, ctx.M, mode)
        assert rel(y64.cpu().numpy(), ref.cpu().numpy()) < 1e-12, mode
    ctx.close()


# one N with a remainder for each embedding that the grids above leave out: M =
# 192, 512, 1024 (two-wave and one-wave form, radices 8 8 4 4 and 16 8 8) and 2048
# (16 elements per thread in complex64)
@pytest.mark.parametrize("N,plan", [(67, 0), (200, 0), (401, 0), (401, 1), (511, 0), (511, 1), (901, 0)])
def test_products_on_the_other_embeddings(N, plan):
    """Bounds as above: complex64 to 2e-6, complex128 to 1e-12 of the product by
    torch.fft, single and batched products equal bit for bit, all modes."""
    import torch
    from cugmres_amd import problems, solver
    print(f"ragged grid N={N} plan={plan}", flush=True)
    ctx = solver.Context(N, 0)
    g, g64 = ctx.spectrum_helmholtz(problems.KH, fp64=True)
    blk = ctx.block_helmholtz(problems.KH)
    rng = np.random.default_rng(N)
    B = 3
    chi = torch.as_tensor(rng.uniform(0.0, 11.1, (B, N * N))).to(ctx.device)
    x = torch.as_tensor(rng.standard_normal((B, N * N)) + 1j * rng.standard_normal((B, N * N))).to(ctx.device)
    c32, x32 = chi.to(torch.float32), x.to(torch.complex64)
    ctx.set_radix_plan(plan)
    for mode in (0, 1, 2):
        own = ctx.matvec_batched(g, c32, x32, mode)
        for k in range(B):
            ref = _torch_matvec(torch, blk, c32[k].to(torch.float64), x32[k].to(torch.complex128), N, ctx.M, mode)
            assert rel(own[k].cpu().numpy(), ref.cpu().numpy()) < 2e-6, (mode, k)
            assert torch.equal(own[k], ctx.matvec(g, c32[k].contiguous(), x32[k].contiguous(), mode)), (mode, k)
        y64 = ctx.matvec_c128(g64, chi[0].contiguous(), x[0].contiguous(), mode)
        ref = _torch_matvec(torch, blk, chi[0], x[0], N, ctx.M, mode)
        assert rel(y64.cpu().numpy(), ref.cpu().numpy()) < 1e-12, mode
    ctx.close()
