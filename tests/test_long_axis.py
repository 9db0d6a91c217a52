"""Long contiguous axes in natural order: a strided pass that leaves its lines
contiguous, then the second half of the axis as a strided axis.  The plans are
replayed on the CPU against the oracle (both directions, in and out of place,
several buffers and strides), the kernels run against it on the GPU at the
smallest and largest lengths and at each change of the split."""
import numpy as np
import pytest
from test_plan_sim import describe, run_plan

TOL32, TOL64 = 2e-6, 1e-14


@pytest.mark.parametrize("dims,batch,flags,prec", [
    ([1 << 14], 3, 0, 0), ([1 << 15], 2, 0, 0), ([1 << 17], 1, 0, 0), ([1 << 19], 1, 0, 0), ([1 << 21], 1, 0, 0),
    ([1 << 21], 1, 4, 0), ([1 << 21], 1, 2, 0), ([4, 1 << 14], 2, 0, 0), ([2, 2, 1 << 14], 1, 0, 0),
    ([32, 1 << 15], 1, 4, 0),
    ([1 << 13], 3, 0, 1), ([1 << 16], 1, 0, 1), ([1 << 18], 1, 0, 1), ([1 << 19], 1, 0, 1), ([8, 1 << 13], 1, 0, 1)])
@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("aliased", [False, True])
def test_natural_order_plans(fl, orc, dims, batch, flags, prec, inverse, aliased):
    passes, final_copy = describe(fl, dims, batch, flags, prec=prec, aliased=aliased)
    assert not final_copy
    # no pass scatters single points: adjacent columns or adjacent points in every store
    assert all(p["out_c"] == 1 or p["out_p"] == 1 for p in passes)
    x = orc.uniform(int(np.prod(dims)) * batch, 31)
    got = run_plan(passes, final_copy, x, inverse, aliased=aliased)
    ref = orc.fftnd(x, dims, batch=batch, inverse=inverse).reshape(-1)
    assert np.linalg.norm(got - ref) <= 1e-12 * np.linalg.norm(ref)


@pytest.mark.parametrize("lg", range(14, 24))
def test_natural_order_needs_no_buffer_out_of_place(fl, lg):
    """One more pass than two only past 2^22 points; a two-pass plan with both
    halves in single strided passes runs without a temporary buffer."""
    p, _ = describe(fl, [1 << lg], 1)
    assert len(p) == (3 if lg == 23 else 2)
    if lg <= 20:
        assert [(q["src"], q["dst"]) for q in p] == [(0, 1), (1, 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("n,batch,dtype,split,inv,inplace", [
    (1 << 14, 1, "complex64", False, False, False), (1 << 14, 5, "complex64", False, True, True),
    (1 << 15, 3, "complex64", False, False, False), (1 << 17, 3, "complex64", False, True, False),
    (1 << 18, 1, "complex64", False, False, True), (1 << 20, 3, "complex64", False, True, False),
    (1 << 21, 1, "complex64", False, False, False), (1 << 22, 1, "complex64", False, True, True),
    (1 << 23, 1, "complex64", False, False, False), (1 << 16, 3, "complex64", True, False, False),
    (1 << 20, 1, "complex64", True, True, False), (1 << 21, 1, "complex64", True, False, False),
    (1 << 13, 5, "complex128", False, True, False), (1 << 15, 1, "complex128", False, False, True),
    (1 << 18, 3, "complex128", False, False, False), (1 << 20, 1, "complex128", False, True, False)])
def test_natural_order_vs_oracle(gpu_lib, orc, n, batch, dtype, split, inv, inplace):
    import torch
    x = orc.uniform(n * batch, n % 1009).astype(dtype)
    xt = torch.from_numpy(x.reshape(batch, n)).cuda()
    y = gpu_lib.c2c_dev(xt, 1, inverse=inv, split=split, out=xt if inplace else None)
    if not inplace:
        assert np.array_equal(xt.cpu().numpy().reshape(-1), x)
    ref = orc.fftnd(x, [n], batch=batch, inverse=inv).reshape(-1)
    err = np.linalg.norm(y.cpu().numpy().reshape(-1) - ref) / np.linalg.norm(ref)
    print(f"n={n} batch={batch} {dtype} split={split} rel_l2={err:.3e}", flush=True)
    assert err <= (TOL32 if dtype == "complex64" else TOL64)
