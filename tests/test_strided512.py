"""Strided lines of 512 points: 16 columns per workgroup up to 131072 lines, 32
past it, and every launch's result against FP64 on both sides of the line."""
import pytest

from test_plan_sim import describe


def test_columns(fl):
    cols = [[q["C"] for q in describe(fl, d, b)[0] if q["mode"] == 1 and q["lg"] == 9]
            for d, b in (([512, 64, 64], 1), ([512, 512], 256), ([512, 512], 257), ([512, 16, 32], 4), ([512, 512, 512], 1),
                         ([1 << 18], 60))]
    assert cols == [[16], [16], [32], [16], [], [16, 16]]
    # double and split precision keep theirs
    assert [q["C"] for q in describe(fl, [512, 512], 100, prec=1)[0] if q["mode"] == 1] == [8]
    assert [q["C"] for q in describe(fl, [512, 512], 100, flags=2)[0] if q["mode"] == 1] == [16]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(256, 512, 512), (257, 512, 512), (5, 512, 2), (3, 512, 16), (1, 512, 4096)])
@pytest.mark.parametrize("inverse", [False, True])
def test_against_fp64(gpu_lib, shape, inverse):
    import torch
    print(shape, inverse, flush=True)
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(*shape, dtype=torch.complex64, device="cuda", generator=g)
    e = torch.fft.ifft2(x.to(torch.complex128), norm="forward") if inverse else torch.fft.fft2(x.to(torch.complex128))
    y = gpu_lib.c2c_dev(x, 2, inverse=inverse)
    assert float((y - e).abs().pow(2).sum().sqrt() / e.abs().pow(2).sum().sqrt()) <= 2e-6
    gpu_lib.c2c_dev(x, 2, inverse=inverse, out=x)
    assert torch.equal(x, y)
