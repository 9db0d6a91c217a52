"""Small boxes in one pass (sides 16 to 64, up to 16384 FP32 or 8192 FP64
points), and strided passes whose arrays have fewer columns than a tile (tiles
over several arrays).  The box kernel's column, row and LDS maps are replayed
on the CPU; the rule that picks it is checked; on the GPU both run against the
oracle per box, odd counts, weights, in place, every kind."""
import itertools

import numpy as np
import pytest
from test_plan_sim import describe, emulate_line

SHAPES = [s for s in itertools.product((16, 32, 64), repeat=3) if np.prod(s) <= 16384]


def emulate_box(x):
    """k_fft_box's exchanges for one box: z columns, rows along x, y columns per plane."""
    LZ, LY, LX = x.shape
    S = LY * LX
    lpx, n = LX + LX // 16, LZ * LY * LX
    lds = np.full(max(LZ * (S + 1), LZ * LY * lpx, LZ * LY * (LX + 1)), np.nan + 0j)
    rows = lambda row, p: row * lpx + p + (p >> 4)  # noqa: E731
    cols = lambda z, c, p: z * LY * (LX + 1) + p * (LX + 1) + c  # noqa: E731
    flat = x.reshape(-1)
    for c in range(S):  # z, written as rows (z, y)
        y = emulate_line(flat[np.arange(LZ) * S + c])
        idx = rows(np.arange(LZ) * LY + c // LX, c % LX)
        assert np.isnan(lds[idx]).all()
        lds[idx] = y
    new = np.full_like(lds, np.nan)
    for r in range(LZ * LY):  # x, written as columns of plane z
        y = emulate_line(lds[rows(r, np.arange(LX))])
        idx = cols(r // LY, np.arange(LX), r % LY)
        assert np.isnan(new[idx]).all()
        new[idx] = y
    out = np.full(n, np.nan + 0j)
    for z in range(LZ):
        for c in range(LX):
            e = z * S + np.arange(LY) * LX + c
            assert np.isnan(out[e]).all()
            out[e] = emulate_line(new[cols(z, c, np.arange(LY))])
    assert not np.isnan(out).any()
    return out.reshape(x.shape)


@pytest.mark.parametrize("shape", [(16, 16, 16), (16, 16, 32), (32, 16, 16), (16, 32, 16), (16, 16, 64), (64, 16, 16)])
def test_box_maps(shape):
    r = np.random.default_rng(1)
    x = r.standard_normal(shape) + 1j * r.standard_normal(shape)
    assert np.allclose(emulate_box(x), np.fft.fftn(x), atol=1e-9)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("shape", SHAPES)
def test_rule(fl, shape, prec):
    points = int(np.prod(shape))
    least = 1 if points <= 8192 or shape[1] * shape[2] < 1024 else 64
    for count in {max(1, least - 1), least, least + 1}:
        for aliased in (False, True):
            p, final_copy = describe(fl, list(shape), count, prec=prec, aliased=aliased)
            box = count >= least and (prec == 0 or points <= 8192)
            assert (p[0]["mode"] == 6) == box and not final_copy
            if box:
                assert len(p) == 1 and p[0]["NT"] == points // 16 and p[0]["nouter"] == count
                assert (p[0]["src"], p[0]["dst"]) == ((1, 1) if aliased else (0, 1))
    # separate passes where asked for, in split precision, and for boxes inside more dimensions' worth of planes
    assert all(q["mode"] != 6 for q in describe(fl, list(shape), least, 4, prec=prec)[0])
    if prec == 0:
        assert all(q["mode"] != 6 for q in describe(fl, list(shape), least, 2)[0])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["complex64", "complex128"])
@pytest.mark.parametrize("shape", SHAPES)
def test_boxes_vs_oracle(gpu_lib, orc, shape, dtype):
    import torch
    points = int(np.prod(shape))
    count = 3 if points <= 8192 or shape[1] * shape[2] < 1024 else 65
    x = orc.gauss(points * count, points).astype(dtype)
    tol = 2e-6 if dtype == "complex64" else 1e-14
    for inv in (False, True):
        ref = orc.fftnd(x, list(shape), batch=count, inverse=inv).reshape(count, -1)
        xt = torch.from_numpy(x.reshape(count, *shape)).cuda()
        y = gpu_lib.c2c_dev(xt, 3, inverse=inv)
        assert np.array_equal(xt.cpu().numpy().reshape(-1), x)
        gpu_lib.c2c_dev(xt, 3, inverse=inv, out=xt)
        assert torch.equal(xt, y)
        d = np.linalg.norm(y.cpu().numpy().reshape(count, -1) - ref, axis=1) / np.linalg.norm(ref, axis=1)
        print(f"{shape} {dtype} inv={inv} worst box {d.max():.3e}", flush=True)
        assert d.max() <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("shape,count", [((16, 16, 16), 5), ((32, 16, 16), 1), ((16, 64, 16), 65)])
def test_box_weights(gpu_lib, orc, shape, count):
    import torch
    from fftfpga_amd.autograd import weighted_transform
    n = int(np.prod(shape))
    x = orc.gauss(n * count, 3).reshape(count, *shape)
    w = np.abs(orc.uniform(n, 4).real).reshape(shape).astype(np.float32)
    xt, wt = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda()
    for inv in (False, True):
        out = weighted_transform(xt, 3, inverse=inv, w_in=wt, w_out=wt).cpu().numpy()
        ref = orc.fftnd((x * w).reshape(-1), list(shape), batch=count, inverse=inv) * w
        assert orc.rel_l2(out, ref) <= 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("shape,rank,dtype,split,fusion", [
    ((5, 128, 16, 16), 3, "complex64", False, True), ((3, 16, 16, 16), 3, "complex64", True, True),
    ((7, 16, 16, 16), 3, "complex64", False, False), ((1, 512, 16, 16), 3, "complex64", True, True),
    ((3, 32, 2), 2, "complex64", False, True), ((129, 64, 4), 2, "complex64", False, True), ((3, 256, 8), 2, "complex64", False, True),
    ((33, 4, 8, 8), 3, "complex64", False, True), ((5, 2, 2, 2), 3, "complex64", False, True), ((3, 512, 4), 2, "complex128", False, True),
    ((17, 8, 16, 4), 3, "complex128", False, True), ((3, 2048, 4), 2, "complex64", False, True)])
def test_few_columns_vs_oracle(gpu_lib, orc, shape, rank, dtype, split, fusion):
    import torch
    dims, n = list(shape[len(shape) - rank:]), int(np.prod(shape))
    batch = n // int(np.prod(dims))
    x = orc.gauss(n, 5).astype(dtype)
    tol = 2e-6 if dtype == "complex64" else 1e-14
    for inv in (False, True):
        ref = orc.fftnd(x, dims, batch=batch, inverse=inv).reshape(batch, -1)
        xt = torch.from_numpy(x.reshape(batch, *dims)).cuda()
        y = gpu_lib.c2c_dev(xt, rank, inverse=inv, split=split, plane_fusion=fusion)
        gpu_lib.c2c_dev(xt, rank, inverse=inv, split=split, plane_fusion=fusion, out=xt)
        assert torch.equal(xt, y)
        d = np.linalg.norm(y.cpu().numpy().reshape(batch, -1) - ref, axis=1) / np.linalg.norm(ref, axis=1)
        assert d.max() <= tol
