"""The fused weight gradient Re sum_b conj(g) . F x: against FP64 at the edges of
its launch rule (batch split 1, 4 and 16 ways, odd and single batches, one
point, inputs off a 16-byte boundary), and through autograd for gradients that
arrive lazily conjugated, strided or with a graph being recorded."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,batch,offset", [
    ([1], 5, 0), ([2], 1, 0), ([8], 3, 0), ([8], 4, 0), ([16, 16], 17, 0), ([1024], 1000, 0), ([64, 64], 15, 0),
    ([1 << 17], 7, 0), ([1 << 18], 5, 0), ([1 << 19], 3, 0), ([1 << 20], 9, 0), ([16, 64], 33, 1), ([32, 32, 32], 2, 0)])
def test_weight_gradient_vs_fp64(gpu_lib, dims, batch, offset):
    import torch
    from fftfpga_amd.autograd import weight_gradient
    n = int(np.prod(dims))
    gen = torch.Generator(device="cuda").manual_seed(n + batch)
    g, f = (torch.randn(n * batch + offset, dtype=torch.complex64, device="cuda", generator=gen)[offset:].view(batch, *dims)
            for _ in range(2))
    got = weight_gradient(g, f, len(dims))
    ref = (g.to(torch.complex128).conj() * f.to(torch.complex128)).real.sum(0)
    # exact products summed in FP64, then one rounding to FP32
    scale = (g.abs().double() * f.abs().double()).sum(0)
    assert got.shape == ref.shape and got.dtype == torch.float32
    assert bool(((got.double() - ref).abs() <= 2.0 ** -24 * ref.abs() + 1e-15 * scale).all())


@pytest.mark.parametrize("how", ["conj", "strided", "graph"])
def test_weight_gradient_through_autograd(gpu_lib, how):
    import torch
    from fftfpga_amd.autograd import fftn
    gen = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(3, 8, 16, 32, dtype=torch.complex64, device="cuda", generator=gen)
    w = torch.rand(8, 16, 32, device="cuda", generator=gen).requires_grad_(True)
    g = torch.randn(3, 8, 16, 32, dtype=torch.complex64, device="cuda", generator=gen)
    up = {"conj": g.conj(), "strided": g.transpose(2, 3).contiguous().transpose(2, 3), "graph": g}[how]
    (gw,) = torch.autograd.grad(fftn(x, 3, w), w, up, create_graph=how == "graph")
    f = torch.fft.fftn(x.to(torch.complex128), dim=(-3, -2, -1))
    ref = (up.to(torch.complex128).conj() * f).real.sum(0)
    assert (torch.linalg.vector_norm(gw.detach().double() - ref) / torch.linalg.vector_norm(ref)).item() <= 2e-6


def test_weight_gradient_refuses_mismatch(gpu_lib):
    import torch
    from fftfpga_amd.autograd import weight_gradient
    f = torch.zeros(2, 8, dtype=torch.complex64, device="cuda")
    with pytest.raises(ValueError):
        weight_gradient(f[:1], f, 1)
    with pytest.raises(ValueError):
        weight_gradient(f.to(torch.complex128), f, 1)
    assert weight_gradient(f[:0], f[:0], 1).tolist() == [0.0] * 8
