"""Performance cases of the FFT engine: what a program that links it asks of it.

Every case goes through the public plan surface (``FftPlan``, ``FftBatch``) as
such a program does: the plan and the device buffers are made once, a pass
executes them.  Plans use the planner's own kernel choices (no tuning table is
loaded).  Axis 0 of an FFT shape is the contiguous one, so the torch views of
the buffers list the axes in reverse.

Families (the listed cases, and what ``draw`` varies):

* ``c2c``   a batch of complex transforms, one direction, out of place or in
            place (orthonormal there, so that a buffer can be transformed
            again and again);
* ``pair``  a forward transform and the inverse of its spectrum, the two ends
            of a filter or a spectral solver (complex, or real with the packed
            half spectrum);
* ``r2c``   real lines to packed half spectra;
* ``batch`` many 1D transforms of uneven lengths in one ``FftBatch`` launch.
"""
import math
import random

import torch

from wgpufft_amd import (FftBatch, FftConfig, FftDirection, FftPlan, FftPrecision, Normalization)

PRECISION = {"f32": FftPrecision.F32, "f64": FftPrecision.F64, "df64": FftPrecision.Df64}
ELEMENT = {"f32": 8, "f64": 16, "df64": 16}

# Line lengths and line counts of the uneven batch (bench.py's batched workload).
UNEVEN_LENGTHS = (120, 343, 1001, 127, 1009, 4096, 65536)
# Points of the largest drawn case per family: no more work than the listed ones.
MAX_POINTS = 1 << 23


def listed():
    return [
        # one short line, the smallest request of a serving mix: call and launch cost
        dict(name="line_1000", family="c2c", precision="f32", shape="1000", batch=1, inverse=False, in_place=False),
        # a small image of the serving mix, to the spectrum and back: a few launches, little data
        dict(name="image_192x128_pair", family="pair", precision="f32", shape="192x128", batch=1, real=False),
        # speech frames: 25 ms windows at 16 kHz, eight minutes of them at a 10 ms hop
        dict(name="frames_400_r2c", family="r2c", precision="f32", shape="400", batch=48000),
        # the plain 1D batch: 4096 lines of 1024 points
        dict(name="lines_1024", family="c2c", precision="f32", shape="1024", batch=4096, inverse=False, in_place=True),
        # prime lines (no mixed-radix split): 1009 points
        dict(name="lines_1009", family="c2c", precision="f32", shape="1009", batch=8192, inverse=True, in_place=False),
        # the headline 2D transform: forward and inverse
        dict(name="image_4096x2048_pair", family="pair", precision="f32", shape="4096x2048", batch=1, real=False),
        # filtering three full-HD planes: ragged real image, packed spectrum and back
        dict(name="image_1920x1080_real", family="pair", precision="f32", shape="1920x1080", batch=3, real=True),
        # a particle-mesh grid step: real volume, packed spectrum and back
        dict(name="volume_144x120x108_real", family="pair", precision="f32", shape="144x120x108", batch=1, real=True),
        # a spectral solver's volume in double precision: forward and inverse
        dict(name="volume_256_f64_pair", family="pair", precision="f64", shape="256x256x256", batch=1, real=False),
        # long smooth lines that no power of two fits: four channels of a million points
        dict(name="long_1000000", family="c2c", precision="f32", shape="1000000", batch=4, inverse=False, in_place=False),
        # one very long double-precision line
        dict(name="long_2p24_f64", family="c2c", precision="f64", shape="16777216", batch=1, inverse=False,
             in_place=False),
        # many queued transforms of uneven lengths served by one persistent launch
        dict(name="uneven_batch_128", family="batch", precision="f32", count=128, mix_seed=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth(n):
    for p in (2, 3, 5, 7, 11, 13):
        while n % p == 0:
            n //= p
    return n == 1


def _next_smooth(n, even=False):
    while not _smooth(n) or (even and n % 2):
        n += 1
    return n


def _length(rng, lo, hi):
    """A power of two, a smooth length or any length, log-uniform in [lo, hi]."""
    n = _log_int(rng, lo, hi)
    c = rng.random()
    if c < 0.35:
        return 1 << max(1, round(math.log2(n)))
    return _next_smooth(n) if c < 0.75 else n


def draw(rng):
    c = rng.random()
    if c < 0.15:  # single short lines and few of them
        return dict(family="c2c", precision="f32", shape=str(_length(rng, 64, 8192)), batch=_log_int(rng, 1, 8),
                    inverse=rng.random() < 0.5, in_place=False)
    if c < 0.40:  # batches of lines
        n = _length(rng, 64, 8192)
        prec = rng.choice(["f32", "f32", "f32", "f64"])
        points = _log_int(rng, 1 << 18, MAX_POINTS if prec == "f32" else MAX_POINTS // 4)
        return dict(family="c2c", precision=prec, shape=str(n), batch=max(1, points // n), inverse=rng.random() < 0.5,
                    in_place=rng.random() < 0.5)
    if c < 0.50:  # real lines
        n = _next_smooth(_log_int(rng, 64, 8192), even=True)
        return dict(family="r2c", precision="f32", shape=str(n), batch=max(1, _log_int(rng, 1 << 18, 2 * MAX_POINTS) // n))
    if c < 0.72:  # images, complex and real
        n0, n1 = (_next_smooth(_log_int(rng, 64, 4096), even=True) for _ in range(2))
        if rng.random() < 0.4:
            n0, n1 = (1 << round(math.log2(n)) for n in (n0, n1))
        real = rng.random() < 0.5
        n1 = min(n1, MAX_POINTS // n0)
        n1 = n1 if _smooth(n1) else 1 << int(math.log2(n1))
        return dict(family="pair", precision="f32", shape="%dx%d" % (n0, n1),
                    batch=rng.randint(1, max(1, min(4, MAX_POINTS // (n0 * n1)))), real=real)
    if c < 0.85:  # volumes
        dims = [_next_smooth(_log_int(rng, 32, 192), even=True) for _ in range(3)]
        prec = rng.choice(["f32", "f32", "f64", "df64"])
        return dict(family="pair", precision=prec, shape="x".join(map(str, dims)), batch=1,
                    real=prec == "f32" and rng.random() < 0.5)
    if c < 0.95:  # long lines
        n = _length(rng, 1 << 14, 1 << 22)
        prec = rng.choice(["f32", "f32", "f64"])
        return dict(family="c2c", precision=prec, shape=str(n), batch=rng.randint(1, max(1, min(8, MAX_POINTS // n))),
                    inverse=rng.random() < 0.5, in_place=False)
    return dict(family="batch", precision="f32", count=_log_int(rng, 8, 96), mix_seed=rng.randint(0, 1 << 20))


def _shape(case):
    return [int(n) for n in case["shape"].split("x")]


def _dims(case):
    """Torch dimensions of the case's array: batch, then the axes with axis 0 last."""
    return [case["batch"]] + _shape(case)[::-1]


def _uneven(case):
    """(length, lines, first point) of every transform of an uneven batch, each
    at a 16-byte boundary of one array, and the points of that array."""
    rng, mix, at = random.Random(case["mix_seed"]), [], 0
    for _ in range(case["count"]):
        n, b = rng.choice(UNEVEN_LENGTHS), rng.randint(1, 256)
        mix.append((n, b, at))
        at += n * b + n * b % 2
    return mix, at


def _uniform(count, seed, dtype):
    """`count` values uniform in [-1, 1), made on the device from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand(count, generator=g, device="cuda", dtype=dtype).mul_(2).sub_(1)


def _input(case, seed):
    """The input array of a case in its storage format."""
    if case["family"] == "batch":
        points = _uneven(case)[1]
        return torch.view_as_complex(_uniform(2 * points, seed, torch.float32).view(-1, 2))
    dims, prec = _dims(case), case["precision"]
    points = math.prod(dims)
    if case["family"] == "r2c" or case.get("real"):
        return _uniform(points, seed, torch.float32).view(dims)
    if prec == "df64":
        v = _uniform(2 * points, seed, torch.float64)
        hi = v.float()
        return torch.stack([hi, (v - hi.double()).float()], dim=-1).view(dims + [4])
    dtype = torch.float32 if prec == "f32" else torch.float64
    return torch.view_as_complex(_uniform(2 * points, seed, dtype).view(dims + [2]))


def prepare(case, seed):
    x = _input(case, seed)
    state = {"case": case, "x": x}
    if case["family"] == "batch":
        # one input and one output array, every transform at its own place in them
        y = torch.zeros_like(x)
        state.update(y=y, batch=FftBatch([dict(n=n, batch=b, input=x[at:at + n * b], output=y[at:at + n * b])
                                          for n, b, at in _uneven(case)[0]]))
        return state
    config = FftConfig.new_nd(_shape(case)).with_batch(case["batch"]).with_precision(PRECISION[case["precision"]])
    back = config.with_direction(FftDirection.Inverse)
    if case["family"] == "c2c":
        if case["inverse"]:
            config = back
        if case["in_place"]:
            config = config.with_normalization(Normalization.Orthogonal)
        state.update(plan=FftPlan.c2c(config), y=None if case["in_place"] else torch.empty_like(x))
        return state
    if case["family"] == "pair" and not case["real"]:
        state.update(plan=FftPlan.c2c(config), inverse=FftPlan.c2c(back), y=torch.empty_like(x), z=torch.empty_like(x))
        return state
    dims = _dims(case)
    packed = torch.empty(dims[:-1] + [dims[-1] // 2 + 1], dtype=torch.complex64, device="cuda")
    state.update(plan=FftPlan.r2c(config), y=packed)
    if case["family"] == "pair":
        state.update(inverse=FftPlan.c2r(back), z=torch.empty_like(x))
    return state


def run(state):
    if "batch" in state:
        state["batch"].execute()
        return state["y"]
    if "z" in state:
        state["plan"].execute(state["x"], state["y"])
        state["inverse"].execute(state["y"], state["z"])
        return state["y"], state["z"]
    if state["y"] is None:
        state["plan"].execute_in_place(state["x"])
        return state["x"]
    state["plan"].execute(state["x"], state["y"])
    return state["y"]


def work(case):
    """Each input read once and each output written once; 5 N log2 N per
    complex transform, half of it per real one."""
    if case["family"] == "batch":
        mix = _uneven(case)[0]
        return {"bytes": sum(2 * 8 * n * b for n, b, _ in mix),
                "flops": sum(5 * n * math.log2(n) * b for n, b, _ in mix)}
    shape = _shape(case)
    n = math.prod(shape)
    real = case["family"] == "r2c" or case.get("real", False)
    if real:
        move = case["batch"] * (4 * n + 8 * (shape[0] // 2 + 1) * (n // shape[0]))
    else:
        move = case["batch"] * 2 * ELEMENT[case["precision"]] * n
    flops = (2.5 if real else 5) * n * math.log2(n) * case["batch"]
    passes = 2 if case["family"] == "pair" else 1
    return {"bytes": passes * move, "flops": passes * flops}


def exact(case, seed):
    """torch.fft in complex128 / float64 of the same inputs."""
    x = _input(case, seed)
    if case["family"] == "batch":
        y = torch.zeros(x.numel(), dtype=torch.complex128, device="cuda")
        for n, b, at in _uneven(case)[0]:
            y[at:at + n * b] = torch.fft.fft(x[at:at + n * b].to(torch.complex128).view(b, n)).view(-1)
        return y
    axes = tuple(range(1, len(_shape(case)) + 1))
    if case["family"] == "r2c" or case.get("real"):
        y = torch.fft.rfftn(x.double(), dim=axes)
        return (y, x.double()) if case["family"] == "pair" else y
    if case["precision"] == "df64":
        v = x.double()
        v = torch.complex(v[..., 0] + v[..., 1], v[..., 2] + v[..., 3])
    else:
        v = x.to(torch.complex128)
    if case["family"] == "pair":
        y, z = torch.fft.fftn(v, dim=axes), v
    elif case["inverse"]:
        y, z = torch.fft.ifftn(v, dim=axes, norm="ortho" if case["in_place"] else "backward"), None
    else:
        y, z = torch.fft.fftn(v, dim=axes, norm="ortho" if case["in_place"] else "backward"), None
    if case["precision"] == "df64":
        def words(c):
            r = torch.view_as_real(c)
            hi = r.float().double()
            return torch.stack([hi, r - hi], dim=-1).flatten(-2)
        y, z = words(y), None if z is None else words(z)
    return y if z is None else (y, z)
