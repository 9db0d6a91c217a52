"""What the library's users have it do, as measurable cases.

A case is a plain dict: `kind` says which public entry point carries it and
the rest are that call's sizes and options.  Each listed case says what it
stands for; draw() gives other members of the same ranges.

kind      entry point                                       options
c2c       fftfpga_amd.c2c_dev on a GPU tensor               rank, dims, batch, dtype, inverse, bitrev, split
pair      c2c_dev forward, then the unnormalised inverse    rank, dims, batch
multi     multi.MultiPlan over cubes of mixed sizes         c32, c64, c128 (how many of each side)
fixed     autograd.fft3/fftn with a fixed real weight       rank, dims, batch   (forward + input gradient)
learned   autograd.fftn with a weight that has a gradient   rank, dims, batch   (forward + both gradients)
host      fftfpgaf_c2c_3d_ddr(_batch) on host arrays        n, batch, inverse
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fft3d-fpga_amd"))

import fftfpga_amd as fl  # noqa: E402
from fftfpga_amd import autograd, multi  # noqa: E402

_started = False


def _start():
    """The library as a program starts it, once per process."""
    global _started
    if not _started:
        if fl.fpga_initialize("AMD HIP", fl.LIB_PATH, False) != 0:
            raise RuntimeError(f"fpga_initialize failed: {fl.last_error()}")
        _started = True


# ---- cases -------------------------------------------------------------------------

def _c2c(dims, batch=1, dtype="complex64", inverse=False, bitrev=False, split=False):
    d = list(dims) + [0] * (3 - len(dims))
    return {"kind": "c2c", "rank": len(dims), "n0": d[0], "n1": d[1], "n2": d[2], "batch": batch, "dtype": dtype,
            "inverse": inverse, "bitrev": bitrev, "split": split}


def _sized(kind, dims, batch=1):
    d = list(dims) + [0] * (3 - len(dims))
    return {"kind": kind, "rank": len(dims), "n0": d[0], "n1": d[1], "n2": d[2], "batch": batch}


def _multi(c32, c64, c128):
    return {"kind": "multi", "c32": c32, "c64": c64, "c128": c128}


def _host(n, batch, inverse):
    return {"kind": "host", "n": n, "batch": batch, "inverse": inverse}


def listed():
    return [
        # one small box of a solver or a particle-mesh step: launch latency counts
        dict(_c2c((64, 64, 64)), name="3d_64"),
        # the benchmark's default: forward and unnormalised inverse of one 256^3 field
        dict(_sized("pair", (256, 256, 256)), name="3d_256_pair"),
        # the largest field, in the split-precision mode
        dict(_c2c((512, 512, 512), split=True), name="3d_512_split"),
        # one large image or aperture
        dict(_c2c((4096, 4096)), name="2d_4096"),
        # one long signal, output order of the reference's 1D engine
        dict(_c2c((1 << 22,), bitrev=True), name="1d_4m_bitrev"),
        # a few long signals in natural order (spectra that are read by frequency)
        dict(_c2c((1 << 20,), batch=3), name="1d_1m_natural"),
        # many short signals (range lines, audio frames), an odd number of them, inverse
        dict(_c2c((1024,), batch=10007, inverse=True), name="1d_1k_lines"),
        # double precision, inverse, two fields
        dict(_c2c((128, 128, 128), batch=2, dtype="complex128", inverse=True), name="3d_128_double"),
        # batches of boxes of uneven sizes through one plan
        dict(_multi(256, 160, 32), name="uneven_448"),
        # the differentiable batch: y = W . FFT3(x), gradient of x for a given upstream gradient
        dict(_sized("fixed", (128, 128, 128), 16), name="grad_16x128"),
        # a learned spectral filter on a non-cubic grid, odd batch: gradients of x and of W
        dict(_sized("learned", (32, 64, 128), 9), name="learned_filter"),
        # the drop-in C entry point on host arrays: copy in, transform, copy out
        dict(_host(256, 1, False), name="host_3d_256"),
    ]


def _lg(rng, lo, hi):
    return 1 << rng.randint(lo, hi)


def _batch(rng, points, most):
    """A batch of any number, spread over the logarithm, that keeps batch x points within `most`."""
    top = max(1, most // points)
    return max(1, min(top, int(round(math.exp(rng.uniform(0.0, math.log(top)))))))


def _dims(rng, rank, lo, hi, least, most):
    """`rank` powers of two 2^lo..2^hi, cubic half the time, with least <= product <= most."""
    while True:
        if rng.random() < 0.5:
            d = [_lg(rng, lo, hi)] * rank
        else:
            d = [_lg(rng, lo, hi) for _ in range(rank)]
        if least <= math.prod(d) <= most:
            return d


def draw(rng: random.Random):
    kind = rng.choice(["c2c3", "c2c3", "c2c2", "lines", "long", "double", "split", "pair", "multi", "fixed", "learned", "host"])
    if kind in ("c2c3", "pair", "split"):
        d = _dims(rng, 3, 4, 9, 1 << 12, 1 << 25)
        b = _batch(rng, math.prod(d), 1 << 25)
        if kind == "pair":
            return _sized("pair", d, b)
        return _c2c(d, b, inverse=rng.random() < 0.5, split=kind == "split")
    if kind == "c2c2":
        d = _dims(rng, 2, 5, 12, 1 << 12, 1 << 24)
        return _c2c(d, _batch(rng, math.prod(d), 1 << 25), inverse=rng.random() < 0.5)
    if kind == "lines":
        n = _lg(rng, 6, 13)
        return _c2c((n,), _batch(rng, n, 1 << 25), inverse=rng.random() < 0.5, bitrev=rng.random() < 0.5)
    if kind == "long":
        n = _lg(rng, 14, 22)
        return _c2c((n,), _batch(rng, n, 1 << 24), inverse=rng.random() < 0.5, bitrev=rng.random() < 0.5)
    if kind == "double":
        rank = rng.randint(1, 3)
        d = (_lg(rng, 6, 16),) if rank == 1 else _dims(rng, rank, 4, 9 if rank == 3 else 11, 1 << 12, 1 << 23)
        return _c2c(d, _batch(rng, math.prod(d), 1 << 23), dtype="complex128", inverse=rng.random() < 0.5)
    if kind == "multi":
        return _multi(rng.randint(1, 300), rng.randint(0, 200), rng.randint(0, 32))
    if kind in ("fixed", "learned"):
        rank = rng.choice([2, 3, 3])
        d = _dims(rng, rank, 4, 8, 1 << 12, 1 << 24)
        return _sized(kind, d, _batch(rng, math.prod(d), 1 << 25))
    n = _lg(rng, 4, 8)
    return _host(n, rng.randint(1, max(1, (1 << 24) // n ** 3)) if n >= 128 else rng.randint(1, 9), rng.random() < 0.5)


# ---- inputs --------------------------------------------------------------------------

def _dims_of(case):
    return [case["n0"], case["n1"], case["n2"]][: case["rank"]]


def _sides(case):
    """Cube sides of an uneven batch, shuffled as the benchmark's batch is (the order is part of the case)."""
    s = [32] * case["c32"] + [64] * case["c64"] + [128] * case["c128"]
    random.Random(2).shuffle(s)
    return s


def _complex(n, seed, dtype=torch.complex64, normal=False):
    """n complex values on the GPU from `seed` alone: U[-1, 1) or N(0, 1) per component."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    real = torch.float64 if dtype == torch.complex128 else torch.float32
    v = torch.empty(2 * n, dtype=real, device="cuda")
    v = v.normal_(generator=g) if normal else v.uniform_(-1.0, 1.0, generator=g)
    return torch.view_as_complex(v.view(n, 2))


def _inputs(case, seed):
    kind = case["kind"]
    if kind == "multi":
        return {"x": _complex(sum(s ** 3 for s in _sides(case)), seed, normal=True)}
    if kind == "host":
        r = np.random.default_rng(seed)
        shape = (case["batch"],) + (case["n"],) * 3
        x = r.random(shape + (2,), dtype=np.float32) * np.float32(2) - np.float32(1)
        return {"x": np.ascontiguousarray(x.view(np.complex64).reshape(shape))}
    d, b = _dims_of(case), case["batch"]
    if kind in ("fixed", "learned"):
        g = torch.Generator(device="cuda").manual_seed(seed + 1000003)
        return {"x": _complex(b * math.prod(d), seed, normal=True).view(b, *d),
                "g": _complex(b * math.prod(d), seed + 2000003, normal=True).view(b, *d),
                "w": torch.rand(d, generator=g, device="cuda")}
    dtype = torch.complex128 if case.get("dtype") == "complex128" else torch.complex64
    x = _complex(b * math.prod(d), seed, dtype)
    if case.get("split"):
        # sparse small spikes, the mode's reason: a wide range within one field
        n = x.numel() // 1000
        g = torch.Generator(device="cuda").manual_seed(seed + 1000003)
        at = 1000 * torch.arange(n, device="cuda") + torch.randint(0, 1000, (n,), generator=g, device="cuda")
        x[at] += 1e-3 * torch.view_as_complex(torch.randint(0, 2, (n, 2), generator=g, device="cuda").float() * 2 - 1)
    return {"x": x.view(b, *d)}


def prepare(case, seed):
    _start()
    state = dict(case=case, **_inputs(case, seed))
    kind = case["kind"]
    if kind == "multi":
        shapes = [(s, s, s) for s in _sides(case)]
        state["out"] = torch.empty_like(state["x"])
        state["plan"] = multi.MultiPlan(shapes, state["x"], state["out"])
    elif kind in ("fixed", "learned"):
        state["x"].requires_grad_(True)
        state["w"].requires_grad_(kind == "learned")
    elif kind == "host":
        state["out"] = np.empty_like(state["x"])
    return state


# ---- one pass --------------------------------------------------------------------------

def run(state):
    case, x = state["case"], state["x"]
    kind = case["kind"]
    if kind == "c2c":
        return fl.c2c_dev(x, case["rank"], inverse=case["inverse"], bitrev_1d=case["bitrev"], split=case["split"])
    if kind == "pair":
        spectrum = fl.c2c_dev(x, case["rank"])
        return [spectrum, fl.c2c_dev(spectrum, case["rank"], inverse=True)]
    if kind == "multi":
        state["plan"]()
        return state["out"]
    if kind in ("fixed", "learned"):
        y = autograd.fftn(x, case["rank"], state["w"])
        wrt = (x, state["w"]) if kind == "learned" else (x,)
        return [y.detach(), *torch.autograd.grad(y, wrt, state["g"])]
    n, b, out = case["n"], case["batch"], state["out"]
    if b == 1:
        t = fl.fftfpgaf_c2c_3d_ddr(n, x, out, case["inverse"])
    else:
        t = fl.fftfpgaf_c2c_3d_ddr_batch(n, x, out, case["inverse"], how_many=b)
    if not t.valid:
        raise RuntimeError(f"transform failed: {fl.last_error()}")
    return out


# ---- what one pass cannot do without ------------------------------------------------------

def _flops(dims, count):
    n = math.prod(dims)
    return 5.0 * n * math.log2(n) * count


def work(case):
    kind = case["kind"]
    if kind == "multi":
        s = _sides(case)
        return {"bytes": 16.0 * sum(v ** 3 for v in s), "flops": sum(_flops((v, v, v), 1) for v in s)}
    if kind == "host":
        n, b = case["n"], case["batch"]
        return {"bytes": 16.0 * n ** 3 * b, "flops": _flops((n, n, n), b)}
    d, b = _dims_of(case), case["batch"]
    n = math.prod(d)
    if kind == "c2c":
        return {"bytes": (32.0 if case["dtype"] == "complex128" else 16.0) * n * b, "flops": _flops(d, b)}
    if kind == "pair":  # the input in, the spectrum and the inverse out
        return {"bytes": 24.0 * n * b, "flops": 2 * _flops(d, b)}
    # x, g and W in; y and the gradients out
    learned = kind == "learned"
    return {"bytes": 32.0 * n * b + (8.0 if learned else 4.0) * n,
            "flops": 2 * _flops(d, b) + (6.0 if learned else 4.0) * n * b}


# ---- the same values in 64 bits --------------------------------------------------------------

def _dft64(x, rank, inverse):
    """Unnormalised DFT over the last `rank` dims in complex128, batch by batch."""
    dim = tuple(range(-rank, 0))
    f = torch.fft.ifftn if inverse else torch.fft.fftn
    return f(x.to(torch.complex128), dim=dim, norm="forward" if inverse else "backward")


def _bitrev(n):
    bits = n.bit_length() - 1
    i, r = np.arange(n), np.zeros(n, np.int64)
    for _ in range(bits):
        r, i = (r << 1) | (i & 1), i >> 1
    return torch.from_numpy(r)


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "multi":
        out, at = torch.empty(s["x"].numel(), dtype=torch.complex128, device="cuda"), 0
        for v in _sides(case):
            n = v ** 3
            out[at:at + n] = _dft64(s["x"][at:at + n].view(v, v, v), 3, False).reshape(-1)
            at += n
        return out
    if kind == "host":
        return _dft64(torch.from_numpy(s["x"]).cuda(), 3, case["inverse"]).cpu().numpy()
    rank = case["rank"]
    if kind == "c2c":
        y = _dft64(s["x"], rank, case["inverse"])
        return y[:, _bitrev(case["n0"]).to(y.device)] if case["bitrev"] else y
    if kind == "pair":
        y = _dft64(s["x"], rank, False)
        return [y, _dft64(y, rank, True)]
    f, w, g = _dft64(s["x"], rank, False), s["w"].double(), s["g"].to(torch.complex128)
    out = [w * f, _dft64(w * g, rank, True)]
    if kind == "learned":
        out.append((g.conj() * f).real.sum(0))
    return out
