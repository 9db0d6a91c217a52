"""Contiguous rows of 16 points, as lines and as the rows of planes: tile edges,
directions, bit-reversed output, double and split precision, weights, in place."""
import pytest

pytestmark = pytest.mark.gpu
TOL = {"complex64": 2e-6, "complex128": 1e-14}
BREV = [int(f"{k:04b}"[::-1], 2) for k in range(16)]


def _input(shape, dtype, seed=1):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, dtype=getattr(torch, dtype), device="cuda", generator=g)


def _exact(x, rank, inverse):
    import torch
    dim = tuple(range(-rank, 0))
    x = x.to(torch.complex128)
    return torch.fft.ifftn(x, dim=dim, norm="forward") if inverse else torch.fft.fftn(x, dim=dim)


def _rel(y, e):
    return float((y - e).abs().pow(2).sum().sqrt() / e.abs().pow(2).sum().sqrt())


@pytest.mark.parametrize("batch", [1, 63, 64, 65, 255, 257, 32768, 32769, 100003])
@pytest.mark.parametrize("dtype", ["complex64", "complex128"])
@pytest.mark.parametrize("inverse", [False, True])
def test_lines(gpu_lib, batch, dtype, inverse):
    import torch
    print(batch, dtype, inverse, flush=True)
    x = _input((batch, 16), dtype, batch)
    e = _exact(x, 1, inverse)
    y = gpu_lib.c2c_dev(x, 1, inverse=inverse)
    assert _rel(y, e) <= TOL[dtype]
    if dtype == "complex64":
        assert torch.equal(gpu_lib.c2c_dev(x, 1, inverse=inverse, bitrev_1d=True), y[:, BREV])
        assert _rel(gpu_lib.c2c_dev(x, 1, inverse=inverse, split=True), e) <= TOL[dtype]
    gpu_lib.c2c_dev(x, 1, inverse=inverse, out=x)
    assert torch.equal(x, y)


@pytest.mark.parametrize("shape", [(3, 64, 16), (1, 128, 16), (40, 256, 16), (33, 512, 16), (2, 64, 64, 16), (5, 128, 32, 16),
                                   (3, 128, 16, 16)])
@pytest.mark.parametrize("inverse", [False, True])
def test_planes_and_boxes(gpu_lib, shape, inverse):
    import torch
    from fftfpga_amd.autograd import weighted_transform
    print(shape, inverse, flush=True)
    rank = len(shape) - 1
    for dtype in TOL:
        x = _input(shape, dtype, 3)
        e = _exact(x, rank, inverse)
        assert _rel(gpu_lib.c2c_dev(x, rank, inverse=inverse), e) <= TOL[dtype]
    x = _input(shape, "complex64", 3)
    assert _rel(gpu_lib.c2c_dev(x, rank, inverse=inverse, split=True), _exact(x, rank, inverse)) <= 2e-6
    wi, wo = (torch.rand(*shape[1:], device="cuda") for _ in range(2))
    y = weighted_transform(x, rank, w_in=wi, w_out=wo, inverse=inverse)
    assert _rel(y, wo * _exact(wi * x, rank, inverse)) <= 2e-6
