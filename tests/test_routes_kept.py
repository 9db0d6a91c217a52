"""Calls that keep an earlier route because the newer one is slower there: split
precision's long natural axes of up to 2^20 points, in place 2048-row arrays of
few columns."""
import pytest

from test_plan_sim import describe, run_plan


@pytest.mark.parametrize("n,batch,modes", [(1 << 15, 1, [1, 0]), (1 << 16, 3, [1, 0]), (1 << 16, 17, [1, 1])])
@pytest.mark.parametrize("inverse", [False, True])
def test_split_long_axes(fl, orc, n, batch, modes, inverse):
    import numpy as np
    p, copied = describe(fl, [n], batch, flags=2)
    assert [q["mode"] for q in p] == modes
    x = orc.uniform(n * batch, 3).astype(np.complex128)
    ref = np.fft.ifft(x.reshape(batch, n)) * n if inverse else np.fft.fft(x.reshape(batch, n))
    got = run_plan(p, copied, x, inverse)
    assert np.linalg.norm(got - ref.reshape(-1)) <= 1e-12 * np.linalg.norm(ref)
    assert [q["mode"] for q in describe(fl, [n], batch)[0]] == [1, 1]


def test_columns(fl):
    assert [q["mode"] for q in describe(fl, [2048, 1024], 1)[0]] == [3, 0]
    assert [q["mode"] for q in describe(fl, [2048, 1024], 1, aliased=True)[0]] == [0, 1, 1]
    assert [q["mode"] for q in describe(fl, [2048, 512], 3, aliased=True)[0]] == [3, 0]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 1 << 15), (3, 1 << 16), (2, 1 << 14), (17, 1 << 16)])
@pytest.mark.parametrize("inverse", [False, True])
def test_split_against_fp64(gpu_lib, shape, inverse):
    import torch
    print(shape, inverse, flush=True)
    g = torch.Generator(device="cuda").manual_seed(2)
    x = torch.randn(*shape, dtype=torch.complex64, device="cuda", generator=g)
    dim = tuple(range(1, len(shape)))
    f = torch.fft.ifftn if inverse else torch.fft.fftn
    e = f(x.to(torch.complex128), dim=dim, norm="forward" if inverse else "backward")
    y = gpu_lib.c2c_dev(x, len(dim), inverse=inverse, split=True)
    assert float((y - e).abs().pow(2).sum().sqrt() / e.abs().pow(2).sum().sqrt()) <= 2e-6
    gpu_lib.c2c_dev(x, len(dim), inverse=inverse, split=True, out=x)
    assert torch.equal(x, y)
