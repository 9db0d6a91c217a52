"""Boxes with planes of 65536 points and more in two passes, the y axis split
between them: the factorisation and the plans on the CPU, and on the GPU the
result against FP64 at every depth and split, both directions, weights, batches."""
import numpy as np
import pytest

from test_plan_sim import describe

# (nz, ny, nx): every r (4, 8, 16), the shortest and longest z of each, every first-pass shape
SHAPES = [(16, 128, 512), (256, 128, 512), (32, 512, 128), (64, 512, 128), (16, 256, 512), (128, 256, 512),
          (16, 512, 256), (128, 512, 256), (16, 512, 512), (64, 512, 512)]


def test_split_formula():
    """X[k + LY d] = sum_a W_R^{a d} W_{R LY}^{a k} T_a[k], T_a[k] = sum_b x[a + R b] W_LY^{b k}."""
    rng = np.random.default_rng(5)
    for R, LY in ((4, 32), (8, 64), (16, 32)):
        n = R * LY
        x = rng.standard_normal(n) + 1j * rng.standard_normal(n)
        T = np.stack([np.fft.fft(x[a::R]) for a in range(R)])
        a, k = np.arange(R)[:, None], np.arange(LY)[None, :]
        X = np.fft.fft(T * np.exp(-2j * np.pi * a * k / n), axis=0)
        assert np.allclose(X.reshape(-1), np.fft.fft(x))


def test_tile_maps():
    """The second pass's loads, LDS slots and stores: each point of a tile once."""
    for nz, R in ((16, 4), (256, 4), (128, 8), (64, 16), (16, 16)):
        J, ZT, CC, TPL = 16 // R, nz * R // 16, 16 * R, nz // 16
        tid = np.arange(nz * R)
        loads = np.stack([(tid // 16 + ZT * j) * CC + 16 * r + tid % 16 for j in range(J) for r in range(R)])
        assert np.array_equal(np.sort(loads.reshape(-1)), np.arange(nz * CC))
        stores = np.stack([((tid // CC) + TPL * p) * CC + tid % CC for p in range(16)])
        assert np.array_equal(np.sort(stores.reshape(-1)), np.arange(nz * CC))


@pytest.mark.parametrize("shape", SHAPES)
def test_plans(fl, shape):
    nz, ny, nx = shape
    p, copied = describe(fl, list(shape), 2)
    assert [(q["mode"], q["src"], q["dst"]) for q in p] == [(7, 0, 1), (8, 1, 1)] and not copied
    A, B = p
    r = A["M"]
    assert r == B["M"] and A["K"] * r == ny and A["K"] * nx == 16384 and A["NT"] == 512
    assert A["nouter"] == 2 * nz * r and B["NT"] == nz * r <= 1024 and B["K"] == A["K"] and B["ncol"] == nx
    # in place, double precision, split precision and the flags keep their passes
    for kw in ({"aliased": True}, {"prec": 1}, {"flags": 2}, {"flags": 4}, {"flags": 8}):
        assert not {7, 8} & {q["mode"] for q in describe(fl, list(shape), 2, **kw)[0]}


@pytest.mark.parametrize("shape,inverse", [((16, 128, 512), False), ((16, 512, 256), True), ((16, 512, 512), False)])
def test_replay(fl, shape, inverse):
    """Both passes as the plan places them, against the oracle transform."""
    nz, ny, nx = shape
    A, B = describe(fl, list(shape), 1)[0]
    R, LY = A["M"], A["K"]
    assert A["in_o"] == A["out_o"] == LY * nx and B["in_o"] == nz * ny * nx and B["in_p"] == B["out_p"] == ny * nx
    rng = np.random.default_rng(1)
    x = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)

    def dft(v, ax):
        return np.fft.ifft(v, axis=ax) * v.shape[ax] if inverse else np.fft.fft(v, axis=ax)
    t = np.empty(nz * ny * nx, complex)
    for p in range(A["nouter"]):  # plane p: rows a + R b of plane p / R, written as a plane of its own
        a, z = p % R, p // R
        first = (p - a) * LY * nx + a * nx
        rows = first + R * nx * np.arange(LY)[:, None] + np.arange(nx)[None, :]
        assert rows.max() < (z + 1) * ny * nx
        t[p * LY * nx:(p + 1) * LY * nx] = dft(dft(x.reshape(-1)[rows], 1), 0).reshape(-1)
    t = t.reshape(nz, R, LY, nx)
    ak = np.arange(R)[:, None] * np.arange(LY)[None, :] * (512 // ny)
    assert ak.max() < 512
    w = np.exp((2j if inverse else -2j) * np.pi * ak / 512)
    y = dft(dft(t * w[None, :, :, None], 1), 0).reshape(shape)
    ref = np.fft.ifftn(x) * x.size if inverse else np.fft.fftn(x)
    assert np.linalg.norm(y - ref) <= 1e-12 * np.linalg.norm(ref)


def test_plans_left_alone(fl):
    for shape, batch in (((8, 512, 512), 2), ((512, 128, 512), 1), ((128, 512, 512), 1), ((256, 512, 256), 1), ((64, 256, 256), 1),
                         ((64, 1024, 128), 1), ((64, 64, 1024), 1), ((64, 128, 256), 4), ((128, 128, 128), 2)):
        assert not {7, 8} & {q["mode"] for q in describe(fl, list(shape), batch)[0]}, shape


def _exact(x, inverse):
    import torch
    x = x.to(torch.complex128)
    return torch.fft.ifftn(x, dim=(-3, -2, -1), norm="forward") if inverse else torch.fft.fftn(x, dim=(-3, -2, -1))


def _rel(y, e):
    return float((y - e).abs().pow(2).sum().sqrt() / e.abs().pow(2).sum().sqrt())


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("inverse", [False, True])
def test_against_fp64(gpu_lib, shape, inverse):
    import torch
    print(shape, inverse, flush=True)
    batch = 3 if shape[0] * shape[1] * shape[2] <= 1 << 22 else 1
    g = torch.Generator(device="cuda").manual_seed(sum(shape))
    x = torch.randn(batch, *shape, dtype=torch.complex64, device="cuda", generator=g)
    kept = x.clone()
    y = gpu_lib.c2c_dev(x, 3, inverse=inverse)
    assert torch.equal(x, kept)
    e = _exact(x, inverse)
    assert _rel(y, e) <= 2e-6
    gpu_lib.c2c_dev(x, 3, inverse=inverse, out=x)  # in place: the line passes
    assert _rel(x, e) <= 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(16, 128, 512), (32, 512, 256), (16, 512, 512)])
def test_weights(gpu_lib, shape):
    import torch
    from fftfpga_amd.autograd import weighted_transform
    g = torch.Generator(device="cuda").manual_seed(7)
    x = torch.randn(2, *shape, dtype=torch.complex64, device="cuda", generator=g)
    wi, wo = (torch.rand(*shape, device="cuda", generator=g) for _ in range(2))
    for inverse in (False, True):
        y = weighted_transform(x, 3, w_in=wi, w_out=wo, inverse=inverse)
        assert _rel(y, wo * _exact(wi * x, inverse)) <= 2e-6
