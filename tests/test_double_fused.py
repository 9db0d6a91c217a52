"""Double precision through the fused passes: plane passes up to 8192 points
and the y-split pair of 128^3 blocks.  Plans replayed on the CPU against the
oracle; the kernels against it on the GPU at the smallest and largest planes,
odd batches, both directions, in place, and against the separate line passes."""
import numpy as np
import pytest
from test_plan_sim import describe, run_plan

# 1e-14: the line passes measure 4e-16 to 6e-16 at these sizes
TOL = 1e-14


@pytest.mark.parametrize("dims,batch,modes", [
    ([16, 64], 1, [2]), ([64, 16], 3, [2]), ([32, 32, 32], 2, [2, 1]), ([8, 64, 64], 1, [2, 1]), ([4, 64, 128], 1, [2, 1]),
    ([4, 128, 64], 3, [2, 1]), ([2, 128, 128], 1, [0, 1, 1]), ([128, 128, 128], 1, [4, 5]), ([2, 16, 32], 1, [0, 1, 1])])
@pytest.mark.parametrize("inverse", [False, True])
def test_double_plans(fl, orc, dims, batch, modes, inverse):
    passes, final_copy = describe(fl, dims, batch, prec=1)
    assert [p["mode"] for p in passes] == modes and not final_copy
    x = orc.uniform(int(np.prod(dims)) * batch, 41)
    got = run_plan(passes, final_copy, x, inverse)
    ref = orc.fftnd(x, dims, batch=batch, inverse=inverse).reshape(-1)
    assert np.linalg.norm(got - ref) <= 1e-12 * np.linalg.norm(ref)


def test_double_in_place_needs_no_buffer(fl):
    """In place these shapes ran without a temporary buffer and still do."""
    for dims in ([128, 128, 128], [64, 64, 64], [16, 64], [4, 128, 64]):
        passes, final_copy = describe(fl, dims, 1, prec=1, aliased=True)
        assert not final_copy and all(p["src"] == p["dst"] == 1 for p in passes)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,rank", [
    ((16, 64), 2), ((3, 64, 16), 2), ((32, 32), 2), ((5, 32, 32, 32), 3), ((64, 64, 64), 3), ((7, 64, 128), 2),
    ((3, 4, 128, 64), 3), ((16, 16, 128), 3), ((128, 128, 128), 3), ((3, 128, 128, 128), 3)])
@pytest.mark.parametrize("inv", [False, True])
def test_double_vs_oracle(gpu_lib, orc, shape, rank, inv):
    import torch
    n, dims = int(np.prod(shape)), list(shape[len(shape) - rank:])
    batch = n // int(np.prod(dims))
    r = np.random.default_rng(n)
    x = r.standard_normal(n) + 1j * r.standard_normal(n)
    xt = torch.from_numpy(x.reshape(batch, *dims)).cuda()
    y = gpu_lib.c2c_dev(xt, rank, inverse=inv)
    assert np.array_equal(xt.cpu().numpy().reshape(-1), x)
    ref = orc.fftnd(x, dims, batch=batch, inverse=inv).reshape(-1)
    err = np.linalg.norm(y.cpu().numpy().reshape(-1) - ref) / np.linalg.norm(ref)
    lines = gpu_lib.c2c_dev(xt, rank, inverse=inv, plane_fusion=False)
    base = np.linalg.norm(lines.cpu().numpy().reshape(-1) - ref) / np.linalg.norm(ref)
    gpu_lib.c2c_dev(xt, rank, inverse=inv, out=xt)
    place = np.linalg.norm(xt.cpu().numpy().reshape(-1) - ref) / np.linalg.norm(ref)
    print(f"{shape} inv={inv} fused={err:.3e} lines={base:.3e} in place={place:.3e}", flush=True)
    assert max(err, base, place) <= TOL
