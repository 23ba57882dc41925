"""Rounding errors of single kernels against longer arithmetic, at bounds that
an extra rounding per term, per output or per bin pair exceeds.  u is the unit
roundoff; C u = 0.42 u is the rms of one rounding to nearest (uniform error,
logarithmic mantissas)."""
import numpy as np
import pytest
import torch

from wgpufft_amd import FftConfig, FftPlan, FftPrecision

pytestmark = pytest.mark.gpu

U32, U64, C = 2.0 ** -24, 2.0 ** -53, 0.42


def uniform(count, seed, dtype=torch.float32):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand(count, generator=g, device="cuda", dtype=dtype) * 2 - 1


def rel_l2(y, ref):
    return (torch.linalg.norm(y.to(ref.dtype) - ref) / torch.linalg.norm(ref)).item()


@pytest.mark.parametrize("n0,n1,volumes", [(17, 17, 256), (59, 47, 32)])
def test_small_volume_direct_sums_round_once_per_term(n0, n1, volumes):
    """A direct sum of n terms whose accumulator rounds once per term errs by C u
    sqrt(n / 2), a term by C u sqrt(2.5) (product, its difference, the factor);
    twice per term would be C u sqrt(n) (measured 1.31 and 1.36 times as much)."""
    x = torch.view_as_complex(uniform(2 * n0 * n1 * volumes, n0).view(volumes, n1, n0, 2))
    y = torch.empty_like(x)
    plan = FftPlan.c2c(FftConfig.new_nd([n0, n1]).with_batch(volumes))
    assert plan.describe().startswith("small-volume"), plan.describe()
    plan.execute(x, y)
    torch.cuda.synchronize()
    e = rel_l2(y, torch.fft.fft2(x.to(torch.complex128)))
    assert e <= 1.1 * C * U32 * np.sqrt((n0 + n1) / 2 + 5), e


@pytest.mark.parametrize("q", [1, 37, 617, 991])
def test_f64_split_twiddles_from_the_table(q):
    """The f64 split of 10^6 points: one point q < 1000 goes through the column
    pass as ones, so that the output is the pass's twiddle W^(q k1) times three
    stages of row twiddles.  One product of two table entries per output and the
    stages err by 1.7 u together; a product carried from output to output adds 3
    to 5 u over the ten of a butterfly."""
    n = 1000000
    x = torch.zeros(n, dtype=torch.complex128, device="cuda")
    x[q] = 1
    y = torch.empty_like(x)
    plan = FftPlan.c2c(FftConfig.new(n).with_precision(FftPrecision.F64))
    assert "lds N=1000" in plan.describe() and " nt=" in plan.describe(), plan.describe()
    plan.execute(x, y)
    t = (np.arange(n, dtype=np.int64) * q % n).astype(np.longdouble) / n * 2 * np.arccos(np.longdouble(-1))
    got = y.cpu().numpy()
    e = np.sqrt(np.mean((got.real - np.cos(t)) ** 2 + (got.imag + np.sin(t)) ** 2))
    assert e <= 2.4 * U64, float(e / U64)


def line_errors(kind, n, lines):
    """Relative L2 errors of a kind of real lines of n points, and of complex
    lines of half as many and as many."""
    e_c2c = []
    for m in (n // 2, n):
        cplx = torch.view_as_complex(uniform(2 * m * lines, m).view(lines, m, 2))
        y = torch.empty_like(cplx)
        FftPlan.c2c(FftConfig.new(m).with_batch(lines)).execute(cplx, y)
        e_c2c.append(rel_l2(y, torch.fft.fft(cplx.to(torch.complex128))))
    r = uniform(n * lines, n + 1).view(lines, n)
    if kind == "r2c":
        out = torch.empty(lines, n // 2 + 1, dtype=torch.complex64, device="cuda")
        plan, src, ref = FftPlan.r2c(FftConfig.new(n).with_batch(lines)), r, torch.fft.rfft(r.double())
    else:
        src = torch.fft.rfft(r.double()).to(torch.complex64).contiguous()
        out = torch.empty_like(r)
        plan, ref = FftPlan.c2r(FftConfig.inverse(n).with_batch(lines)), torch.fft.irfft(src.to(torch.complex128), n=n)
    plan.execute(src, out)
    torch.cuda.synchronize()
    return plan, rel_l2(out, ref), e_c2c


@pytest.mark.parametrize("kind", ["r2c", "c2r"])
@pytest.mark.parametrize("n", [36, 200, 400, 1000, 1920, 4374])
def test_half_length_lines_err_as_their_transform_and_one_rounding(kind, n):
    """The bin pairs of a half-length real line are joined (split) in 64 bits and
    rounded once: the line errs by its n / 2-point transform and C u.  In 32 bits
    the pairs cost 0.6 to 0.8 u, 4 to 8 % of the line's error."""
    plan, e, (e_half, _) = line_errors(kind, n, (1 << 21) // n)
    assert "half" in plan.describe(), plan.describe()
    assert e <= 1.02 * np.hypot(e_half, C * U32), e / np.hypot(e_half, C * U32)


@pytest.mark.parametrize("n", [64, 128, 256, 512])
def test_compiled_c2r_lines_err_less_than_complex_lines(n):
    """A full-length inverse of Hermitian bins spreads its error over the real
    and the imaginary part, which is dropped: 0.87 to 0.9 of a complex line's
    error, where a half-length transform has all of it (0.95 to 0.98)."""
    plan, e, (_, e_c2c) = line_errors("c2r", n, (1 << 21) // n)
    assert plan.describe().startswith("reg "), plan.describe()
    assert e <= 0.93 * e_c2c, e / e_c2c
