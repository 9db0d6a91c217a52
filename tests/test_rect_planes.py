"""Plane passes of rectangular planes with a side of 256 or 512: the rule that
picks them (by points and number of planes), plans replayed on the CPU, and the
kernels on the GPU against the oracle and against the separate line passes, per
kind (FP32, split precision, FP64), with weights, in place, odd plane counts."""
import numpy as np
import pytest
from test_plan_sim import describe, run_plan

SHAPES = [(16, 256), (256, 16), (16, 512), (512, 16), (32, 256), (256, 32), (64, 256), (256, 64), (32, 512), (512, 32),
          (128, 256), (256, 128), (64, 512), (512, 64)]
MOST = {"f32": 32768, "split": 16384, "f64": 8192}


def _least(ly, lx):
    return {4096: 1, 8192: 16, 16384: 128, 32768: 256}[ly * lx]


@pytest.mark.parametrize("kind", ["f32", "split", "f64"])
@pytest.mark.parametrize("ly,lx", SHAPES)
def test_rule(fl, ly, lx, kind):
    flags, prec = (2 if kind == "split" else 0), int(kind == "f64")
    n = _least(ly, lx)
    for count in {max(1, n - 1), n, n + 1}:
        p, final_copy = describe(fl, [ly, lx], count, flags, prec=prec)
        assert (p[0]["mode"] == 2) == (count >= n and ly * lx <= MOST[kind]) and not final_copy
        if p[0]["mode"] == 2:  # in place without a temporary buffer, one workgroup per plane
            assert len(p) == 1 and not p[0]["transposing"] and p[0]["NT"] <= 1024
            q, _ = describe(fl, [ly, lx], count, flags, prec=prec, aliased=True)
            assert [(v["mode"], v["src"], v["dst"]) for v in q] == [(2, 1, 1)]
    assert describe(fl, [ly, lx], 300, flags | 4, prec=prec)[0][0]["mode"] != 2


@pytest.mark.parametrize("dims,batch,flags,prec", [
    ([4, 16, 512], 4, 0, 0), ([2, 256, 16], 2, 2, 0), ([8, 32, 256], 2, 0, 1), ([64, 512], 256, 0, 0), ([2, 64, 256], 64, 2, 0)])
@pytest.mark.parametrize("inverse", [False, True])
def test_plans(fl, orc, dims, batch, flags, prec, inverse):
    passes, final_copy = describe(fl, dims, batch, flags, prec=prec)
    assert passes[0]["mode"] == 2
    x = orc.uniform(int(np.prod(dims)) * batch, 51)
    got = run_plan(passes, final_copy, x, inverse)
    ref = orc.fftnd(x, dims, batch=batch, inverse=inverse).reshape(-1)
    assert np.linalg.norm(got - ref) <= 1e-12 * np.linalg.norm(ref)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["f32", "split", "f64"])
@pytest.mark.parametrize("ly,lx", SHAPES)
def test_vs_oracle(gpu_lib, orc, ly, lx, kind):
    import torch
    if ly * lx > MOST[kind]:
        pytest.skip("line passes")
    count = _least(ly, lx) + (2 if ly * lx <= 8192 else 1)
    x = orc.gauss(count * ly * lx, ly + lx).astype(np.complex128 if kind == "f64" else np.complex64)
    tol = 1e-14 if kind == "f64" else 2e-6  # the repository's bar; FP64 line passes measure 4e-16
    for inv in (False, True):
        ref = orc.fftnd(x, [ly, lx], batch=count, inverse=inv)
        xt = torch.from_numpy(x.reshape(count, ly, lx)).cuda()
        y = gpu_lib.c2c_dev(xt, 2, inverse=inv, split=kind == "split")
        assert np.array_equal(xt.cpu().numpy().reshape(-1), x)
        gpu_lib.c2c_dev(xt, 2, inverse=inv, split=kind == "split", out=xt)
        assert torch.equal(xt, y)
        # every plane by itself, so that one wrong plane is not lost in the sum
        d = np.linalg.norm((y.cpu().numpy() - ref).reshape(count, -1), axis=1) / np.linalg.norm(ref.reshape(count, -1), axis=1)
        print(f"{ly}x{lx} {kind} inv={inv} worst plane {d.max():.3e}", flush=True)
        assert d.max() <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("ly,lx", [(16, 512), (256, 32), (64, 256), (512, 32), (128, 256), (512, 64)])
def test_weights(gpu_lib, orc, ly, lx):
    import torch
    from fftfpga_amd.autograd import weighted_transform
    count = _least(ly, lx) + 1
    x = orc.gauss(count * ly * lx, 3).reshape(count, ly, lx)
    w = np.abs(orc.uniform(ly * lx, 4).real).reshape(ly, lx).astype(np.float32)
    xt, wt = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda()
    for inv in (False, True):
        out = weighted_transform(xt, 2, inverse=inv, w_out=wt).cpu().numpy()
        ref = orc.fftnd(x.reshape(-1), [ly, lx], batch=count, inverse=inv) * w
        assert orc.rel_l2(out, ref) <= 2e-6
        both = weighted_transform(xt, 2, inverse=inv, w_in=wt, w_out=wt).cpu().numpy()
        ref = orc.fftnd((x * w).reshape(-1), [ly, lx], batch=count, inverse=inv) * w
        assert orc.rel_l2(both, ref) <= 2e-6


@pytest.mark.gpu
def test_uneven_batch_of_long_planes(gpu_lib, orc):
    """Uneven batches keep the schedules they had for planes with a side over 128."""
    import torch
    from fftfpga_amd.multi import MultiPlan
    shapes = [(16, 16, 256), (32, 32, 32)]
    n = [int(np.prod(s)) for s in shapes]
    x = orc.uniform(sum(n), 9)
    xt = torch.from_numpy(x).cuda()
    out = torch.empty_like(xt)
    plan = MultiPlan(shapes, xt, out)
    assert plan.schedule()["mode"] == 1
    plan()
    plan.check()
    y = out.cpu().numpy()
    for s, a, b in zip(shapes, (0, n[0]), (n[0], n[0] + n[1])):
        assert orc.rel_l2(y[a:b], orc.fftnd(x[a:b], list(s)).reshape(-1)) <= 2e-6
