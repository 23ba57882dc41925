"""Runtime-schedule register lines (mix_kernels.hpp): lengths where a tile, a
stage or a round can go wrong, against the FP64 oracle.

Bounds: f32 relative L2 <= 1e-6 (about ten stages of rounding at 6e-8 each stay
under it), f64 <= 1e-13, df64 <= 1e-11, as everywhere in this suite.
"""
import numpy as np
import pytest

import oracle
from tests.helpers import c2c_expected, empty_dev, from_dev, seeded_complex, to_dev
from wgpufft_amd import FftBatch, FftConfig, FftDirection, FftPlan, FftPrecision

pytestmark = pytest.mark.gpu

# two stages of the smallest length; odd, coprime and repeated radices; a
# stage of every compiled unroll; five stages; the longest on-chip lines
LENGTHS = [18, 22, 49, 60, 143, 169, 200, 270, 400, 540, 1000, 1080, 2187, 2401, 3125, 3993, 7203, 9216]


def run(plan, x, out_bytes):
    d = to_dev(x)
    out = empty_dev(out_bytes)
    plan.execute(d, out)
    return from_dev(out, x.dtype)


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("batch", [1, 7])
def test_contiguous_f32(torch_cuda, n, batch):
    for inverse in (False, True):
        x = seeded_complex(n + batch, n * batch)
        cfg = (FftConfig.inverse(n) if inverse else FftConfig.new(n)).with_batch(batch)
        plan = FftPlan.c2c(cfg)
        assert " nt=" in plan.describe(), plan.describe()
        y = run(plan, x, x.nbytes)
        e = oracle.rel_l2(y, c2c_expected(x, [n], batch=batch, inverse=inverse))
        assert e <= 1e-6, (n, batch, inverse, e, plan.describe())


@pytest.mark.parametrize("n,width", [(18, 5), (60, 33), (270, 17), (1000, 9), (1080, 6), (3993, 3), (7203, 2)])
def test_strided_f32(torch_cuda, n, width):
    x = seeded_complex(n, n * width * 2)
    plan = FftPlan.c2c(FftConfig.new_nd([width, n]).with_axes([1]).with_batch(2))
    y = run(plan, x, x.nbytes)
    want = np.fft.fft(x.astype(np.complex128).reshape(2, n, width), axis=1).reshape(-1)
    e = oracle.rel_l2(y, want)
    assert e <= 1e-6, (n, width, e, plan.describe())


@pytest.mark.parametrize("n", [22, 60, 540, 1000, 2401, 4608])
@pytest.mark.parametrize("prec", [FftPrecision.F64, FftPrecision.Df64])
def test_double_precision(torch_cuda, n, prec):
    batch = 5
    v = np.random.default_rng(n).uniform(-1, 1, (n * batch, 2))
    plan = FftPlan.c2c(FftConfig.new(n).with_batch(batch).with_precision(prec))
    assert " nt=" in plan.describe(), plan.describe()
    if prec == FftPrecision.F64:
        got = run(plan, v.reshape(-1), v.nbytes).reshape(-1, 2)
    else:
        hi = v.astype(np.float32)
        lo = (v - hi).astype(np.float32)
        w = run(plan, np.stack([hi, lo], -1).reshape(-1), v.nbytes).reshape(-1, 2, 2).astype(np.float64)
        got = w[..., 0] + w[..., 1]
        v = hi.astype(np.float64) + lo
    want = np.fft.fft((v[:, 0] + 1j * v[:, 1]).reshape(batch, n)).reshape(-1)
    e = oracle.rel_l2(got[:, 0] + 1j * got[:, 1], want)
    assert e <= (1e-13 if prec == FftPrecision.F64 else 1e-11), (n, e)


def test_long_axis_passes(torch_cuda):
    """Twiddle-on-store columns and transposed-store rows of a smooth split."""
    for n, inverse in ((44100, False), (30030, True)):
        x = seeded_complex(n, 2 * n)
        plan = FftPlan.c2c((FftConfig.inverse(n) if inverse else FftConfig.new(n)).with_batch(2))
        assert "post" in plan.describe(), plan.describe()
        e = oracle.rel_l2(run(plan, x, x.nbytes), c2c_expected(x, [n], batch=2, inverse=inverse))
        assert e <= 1e-6, (n, e, plan.describe())


def test_batched_tiles_equal_standalone(torch_cuda):
    """The batched kernel's 256-thread tiles of the same schedules, bit for bit."""
    import torch
    items, want = [], []
    for k, (n, b) in enumerate([(18, 3), (60, 50), (270, 11), (540, 1), (1000, 6), (1080, 2), (3993, 4)]):
        x = seeded_complex(100 + k, n * b)
        cfg = FftConfig.new(n).with_batch(b).with_direction(FftDirection(k % 2))
        want.append(run(FftPlan.c2c(cfg), x, x.nbytes))
        items.append(dict(n=n, batch=b, input=to_dev(x), output=empty_dev(x.nbytes), direction=FftDirection(k % 2)))
    FftBatch(items).execute()
    torch.cuda.synchronize()
    for it, w in zip(items, want):
        got = from_dev(it["output"], np.complex64)
        assert np.array_equal(got.view(np.uint32), w.view(np.uint32)), it["n"]


@pytest.mark.parametrize("n", [36, 60, 66, 98, 120, 286, 400, 1014, 1920, 4374, 9000])
@pytest.mark.parametrize("batch", [1, 13])
def test_half_length_real_lines(torch_cuda, n, batch):
    """Even real lines at half length; C2R drops the imaginary parts of the
    first and last bin of arbitrary packed input, as numpy's irfft does."""
    rng = np.random.default_rng(n + batch)
    x = rng.uniform(-1, 1, (batch, n)).astype(np.float32)
    r2c = FftPlan.r2c(FftConfig.new(n).with_batch(batch))
    assert "half" in r2c.describe(), r2c.describe()
    y = run(r2c, x, batch * (n // 2 + 1) * 8).view(np.complex64)
    e = oracle.rel_l2(y, np.fft.rfft(x.astype(np.float64), axis=1).reshape(-1))
    assert e <= 1e-6, (n, batch, e, r2c.describe())
    p = seeded_complex(n, batch * (n // 2 + 1))
    c2r = FftPlan.c2r(FftConfig.inverse(n).with_batch(batch))
    assert "half" in c2r.describe(), c2r.describe()
    z = run(c2r, p, batch * n * 4).view(np.float32)
    e = oracle.rel_l2(z, np.fft.irfft(p.astype(np.complex128).reshape(batch, -1), n=n, axis=1).reshape(-1))
    assert e <= 1e-6, (n, batch, e, c2r.describe())


def test_half_length_real_volume(torch_cuda):
    shape, batch = [60, 18, 35], 2
    x = np.random.default_rng(3).uniform(-1, 1, (batch, 35, 18, 60)).astype(np.float32)
    r2c, c2r = FftPlan.r2c(FftConfig.new_nd(shape).with_batch(batch)), FftPlan.c2r(FftConfig.inverse_nd(shape).with_batch(batch))
    y = run(r2c, x, batch * 35 * 18 * 31 * 8).view(np.complex64)
    assert oracle.rel_l2(y, np.fft.rfftn(x.astype(np.float64), axes=(1, 2, 3)).reshape(-1)) <= 1e-6
    z = run(c2r, y, x.nbytes).view(np.float32)
    assert oracle.rel_l2(z, x.astype(np.float64).reshape(-1)) <= 1e-6


@pytest.mark.parametrize("p,batch", [(29, 1), (29, 300), (61, 77), (73, 5), (127, 64), (257, 9), (1009, 7), (2003, 2),
                                     (4051, 1), (7561, 3)])
def test_rader_register_convolution(torch_cuda, p, batch):
    """Cyclic Rader lines on the register stages, contiguous and strided."""
    for inverse in (False, True):
        x = seeded_complex(p + batch, p * batch)
        plan = FftPlan.c2c((FftConfig.inverse(p) if inverse else FftConfig.new(p)).with_batch(batch))
        assert plan.describe().startswith("rader") and " nt=" in plan.describe(), plan.describe()
        e = oracle.rel_l2(run(plan, x, x.nbytes), c2c_expected(x, [p], batch=batch, inverse=inverse))
        assert e <= 1e-6, (p, batch, inverse, e)
    width = 3 if p > 2000 else 19
    x = seeded_complex(p, p * width)
    plan = FftPlan.c2c(FftConfig.new_nd([width, p]).with_axes([1]))
    want = np.fft.fft(x.astype(np.complex128).reshape(p, width), axis=0).reshape(-1)
    assert oracle.rel_l2(run(plan, x, x.nbytes), want) <= 1e-6, (p, plan.describe())


@pytest.mark.parametrize("n,kind", [(127, "rader"), (1019, "rader"), (3001, "rader"), (34, "bluestein"),
                                    (611, "bluestein"), (1622, "bluestein")])
def test_double_precision_convolutions(torch_cuda, n, kind):
    for prec, bound in ((FftPrecision.F64, 1e-13), (FftPrecision.Df64, 1e-11)):
        batch = 6
        v = np.random.default_rng(n).uniform(-1, 1, (n * batch, 2)).astype(np.float32).astype(np.float64)
        plan = FftPlan.c2c(FftConfig.new(n).with_batch(batch).with_precision(prec))
        assert plan.describe().startswith(kind) and " nt=" in plan.describe(), plan.describe()
        if prec == FftPrecision.F64:
            got = run(plan, v.reshape(-1), v.nbytes).reshape(-1, 2)
        else:
            w = np.stack([v, np.zeros_like(v)], -1).astype(np.float32)
            w = run(plan, w.reshape(-1), v.nbytes).reshape(-1, 2, 2).astype(np.float64)
            got = w[..., 0] + w[..., 1]
        want = np.fft.fft((v[:, 0] + 1j * v[:, 1]).reshape(batch, n)).reshape(-1)
        e = oracle.rel_l2(got[:, 0] + 1j * got[:, 1], want)
        assert e <= bound, (n, prec, e)


def test_batched_convolutions_equal_standalone(torch_cuda):
    import torch
    items, want = [], []
    for k, (n, b) in enumerate([(29, 40), (127, 9), (257, 3), (1009, 5), (2003, 2)]):
        x = seeded_complex(200 + k, n * b)
        cfg = FftConfig.new(n).with_batch(b)
        want.append(run(FftPlan.c2c(cfg), x, x.nbytes))
        items.append(dict(n=n, batch=b, input=to_dev(x), output=empty_dev(x.nbytes)))
    FftBatch(items).execute()
    torch.cuda.synchronize()
    for it, w in zip(items, want):
        got = from_dev(it["output"], np.complex64)
        assert np.array_equal(got.view(np.uint32), w.view(np.uint32)), it["n"]
