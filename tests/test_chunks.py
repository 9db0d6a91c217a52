"""Batches of 128^3 blocks run the y-split pair in chunks of blocks: every block
equals the same block alone, bit for bit, at the batch sizes around the first
chunked one and with an uneven last chunk; directions, in place, weights, and
the grouped launches of an uneven batch."""
import pytest

pytestmark = pytest.mark.gpu
N = 128


def _input(batch, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(batch, N, N, N, dtype=torch.complex64, device="cuda", generator=g)


@pytest.mark.parametrize("batch", [11, 12, 13, 17, 25])
@pytest.mark.parametrize("inverse", [False, True])
def test_blocks_equal_single_blocks(gpu_lib, batch, inverse):
    import torch
    x = _input(batch, batch)
    kept = x.clone()
    y = gpu_lib.c2c_dev(x, 3, inverse=inverse)
    assert torch.equal(x, kept)
    for b in range(batch):
        assert torch.equal(y[b], gpu_lib.c2c_dev(x[b], 3, inverse=inverse)), b
    gpu_lib.c2c_dev(x, 3, inverse=inverse, out=x)
    assert torch.equal(x, y)


def test_weighted_blocks_equal_single_blocks(gpu_lib):
    import torch
    from fftfpga_amd.autograd import weighted_transform
    x, w = _input(13, 3), torch.rand(N, N, N, device="cuda")
    for kw in ({"w_in": w}, {"w_out": w}, {"w_in": w, "w_out": w, "inverse": True}):
        y = weighted_transform(x, 3, **kw)
        for b in range(13):
            assert torch.equal(y[b], weighted_transform(x[b], 3, **kw)), (b, list(kw))


@pytest.mark.parametrize("inverse", [False, True])
def test_grouped_blocks_equal_single_blocks(gpu_lib, inverse):
    import torch
    from fftfpga_amd.multi import MultiPlan
    shapes = [(N, N, N)] * 7 + [(32, 32, 32)] * 3 + [(N, N, N)] * 6 + [(64, 64, 64)]
    sizes = [s[0] ** 3 for s in shapes]
    x = _input(-(-sum(sizes) // N ** 3), 9).view(-1)[:sum(sizes)].contiguous()
    out = torch.empty_like(x)
    plan = MultiPlan(shapes, x, out, inverse=inverse)
    assert plan.schedule()["mode"] == 2
    plan()
    plan.check()
    at = 0
    for s, n in zip(shapes, sizes):
        assert torch.equal(out[at:at + n].view(s), gpu_lib.c2c_dev(x[at:at + n].view(s), 3, inverse=inverse))
        at += n


@pytest.mark.parametrize("n64", [128, 129, 161])
def test_grouped_planes_equal_single_transforms(gpu_lib, n64):
    """64^3 groups up to and past 256 MiB (one launch pair, then chunks), between
    members of other shapes."""
    import torch
    from fftfpga_amd.multi import MultiPlan
    shapes = [(32, 32, 32)] * 5 + [(64, 64, 64)] * (n64 - 1) + [(32, 64, 64), (64, 64, 64)]
    sizes = [s[0] * s[1] * s[2] for s in shapes]
    x = _input(-(-sum(sizes) // N ** 3), n64).view(-1)[:sum(sizes)].contiguous()
    out = torch.empty_like(x)
    plan = MultiPlan(shapes, x, out)
    assert plan.schedule()["mode"] == 2
    plan()
    plan.check()
    at = 0
    for s, n in zip(shapes, sizes):
        assert torch.equal(out[at:at + n].view(s), gpu_lib.c2c_dev(x[at:at + n].view(s), 3)), (at, s)
        at += n
